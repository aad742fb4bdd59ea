"""The steps of a decode layer of up to 16 rows whose norms have no launch: rows packed for the next projection, their scale behind it."""
import math

import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu


def _rows(M, H, gpu):
    x = torch.randn(M, H, device=gpu).to(torch.bfloat16)
    x[:, 5] *= 30
    return x, (1 + 0.3 * torch.randn(H, device=gpu)).to(torch.bfloat16)


def _unpack(xw, M, H):
    return xw.view(H // 32, 4, 16, 8).permute(2, 0, 1, 3).reshape(16, H)[:M]


def _normed64(x, nw):
    x = x.double()
    return x * torch.rsqrt(x.pow(2).mean(1, keepdim=True) + 1e-5) * nw.double()


# tiles of one stage a wave and of many, one and several groups of squares, more than a wave asks for at once (8,192), 16 and 32 weight rows a workgroup
@pytest.mark.parametrize("M", [1, 2, 9, 16])
@pytest.mark.parametrize("H,N", [(256, 64), (768, 1152), (2048, 4160), (4096, 6144), (4096, 14336), (8192, 192)])
@pytest.mark.parametrize("epi", [1, 2])
def test_normed_product(gpu, M, H, N, epi):
    """x w rounds to bf16 once (2^-9 of a value, independently), as a normed row does; SwiGLU's result once more."""
    torch.manual_seed(H + N + M)
    x, nw = _rows(M, H, gpu)
    w = (torch.randn((2 if epi == 2 else 1) * N, H, device=gpu) / math.sqrt(H)).to(torch.bfloat16)
    rows = ops.stream_open(x, nw)
    assert torch.equal(_unpack(rows[0], M, H), (x.float() * nw.float()).to(torch.bfloat16))
    y = ops.stream_normed(rows, M, w, 1e-5, epi)
    want = _normed64(x, nw) @ w.double().t().contiguous()
    if epi == 2:
        want = torch.nn.functional.silu(want[:, :N]) * want[:, N:]
        y = _unpack(y, M, N)
    assert y.shape == want.shape
    assert bool(((y.double() - want).norm(dim=1) <= 2 ** -8 * (3 if epi == 2 else 1) * want.norm(dim=1)).all())


@pytest.mark.parametrize("M", [1, 2, 9, 16])
@pytest.mark.parametrize("N,K", [(256, 256), (768, 2048), (4096, 4096), (4096, 14336), (8192, 512)])
@pytest.mark.parametrize("packed", [False, True])
def test_added_product(gpu, M, N, K, packed):
    """The residual as linear_add_ has it; the rows behind it are those of stream_open, with squares in another order (2^-24 each)."""
    torch.manual_seed(N + K + M)
    x = torch.randn(M, K, device=gpu).to(torch.bfloat16)
    w = (torch.randn(N, K, device=gpu) / math.sqrt(K)).to(torch.bfloat16)
    resid, nw = _rows(M, N, gpu)
    want, xs = resid.double() + x.double() @ w.double().t().contiguous(), x
    if packed:   # rows beyond the M-th hold anything
        xs = torch.full((16, K), float("nan"), device=gpu, dtype=torch.bfloat16)
        xs[:M] = x
        xs = xs.view(16, K // 32, 4, 8).permute(1, 2, 0, 3).reshape(-1).contiguous()
    other = resid.clone()
    assert ops.stream_add_(other, xs, w) is None
    rows = ops.stream_add_(resid, xs, w, nw)
    assert torch.equal(resid, other)
    slack = 2 ** -24 * math.sqrt(K) * (x.double().abs() @ w.double().abs().t().contiguous())
    assert bool(((resid.double() - want).abs() <= 2 ** -8 * want.abs() + slack + 1e-6).all())
    assert torch.equal(_unpack(rows[0], M, N), (resid.float() * nw.float()).to(torch.bfloat16))
    sq = rows[1].view(N // 64, 16, 4).double().sum((0, 2))[:M]
    assert bool(((sq - resid.double().pow(2).sum(1)).abs() <= 2 ** -20 * sq).all())


def test_refused(gpu):
    x, nw = _rows(3, 256, gpu)
    rows, w = ops.stream_open(x, nw), torch.zeros(64, 256, dtype=torch.bfloat16, device=gpu)
    for bad in (lambda: ops.stream_open(x[:, :128], nw[:128]), lambda: ops.stream_open(torch.zeros(17, 256, dtype=torch.bfloat16, device=gpu), nw),
                lambda: ops.stream_normed(rows, 17, w, 1e-5, 1), lambda: ops.stream_normed(rows, 3, w[:48], 1e-5, 1),
                lambda: ops.stream_normed(rows, 3, torch.zeros(64, 512, dtype=torch.bfloat16, device=gpu), 1e-5, 1),
                lambda: ops.stream_normed(rows, 3, w, 1e-5, 0), lambda: ops.stream_add_(x, x[:2], torch.zeros(256, 256, dtype=torch.bfloat16, device=gpu)),
                lambda: ops.stream_add_(x, x, torch.zeros(256, 256, dtype=torch.bfloat16, device=gpu), nw[:128])):
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.parametrize("M,H,Q,F,ok", [(1, 4096, 6144, 14336, False), (2, 4096, 6144, 14336, True), (16, 4096, 6144, 14336, True), (17, 4096, 6144, 14336, False),
                                        (16, 2048, 3072, 8192, True), (4, 8192, 10240, 28672, False), (4, 4096, 6144, 14368, False), (16, 3072, 5120, 8192, True)])
def test_which_layers(gpu, M, H, Q, F, ok):
    z = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device=gpu)  # noqa: E731
    assert ops.stream_layer_covers(z(M, H), z(H), z(Q, H), z(H, H), z(H), z(2 * F, H), z(H, F)) == ok


# rows of one page and of several, a row without a context, a model whose F the stream kernel leaves (no multiple of 64)
@pytest.mark.parametrize("over,ctxs,taken", [({}, [300, 64], True), ({}, [300, 1, 65, 64, 129], True), ({}, [3 * i + 1 for i in range(16)], True),
                                             ({}, [3 * i + 1 for i in range(17)], False), ({"ffn": 1056}, [7, 8], False)])
def test_a_models_step(gpu, monkeypatch, over, ctxs, taken):
    """A decode step's final rows beside the same step in launches of their own, each against 64 bits."""
    import test_decode_step_gpu as one
    from nv_genai_amd.models.config import llama_config
    from nv_genai_amd.models.llama import AttnMeta, LlamaModel

    m = LlamaModel(llama_config("llama3-8b", **{**dict(layers=3, vocab_size=512, hidden=512, heads=4, kv_heads=2, head_dim=128, ffn=1024, max_position=512), **over}), gpu)
    g = torch.Generator(gpu).manual_seed(11)
    for L in m.layers:
        for n in ("attn_norm", "mlp_norm"):
            L[n].normal_(1, 0.1, generator=g)
    m.embed.mul_(20)
    pages = [(n + 63) // 64 for n in ctxs]
    m.allocate_kv_cache(sum(pages) + 1)
    for t in (m.k_cache, m.v_cache):
        t.copy_(torch.randn(t.shape, device=gpu, generator=g).to(t.dtype))
    before, bt, slots, at = [m.k_cache.clone(), m.v_cache.clone()], torch.zeros(len(ctxs), max(pages), dtype=torch.int32, device=gpu), [], 1
    for b, n in enumerate(ctxs):
        bt[b, : pages[b]] = torch.arange(at, at + pages[b])
        at += pages[b]
        slots.append(int(bt[b, (n - 1) // 64]) * 64 + (n - 1) % 64)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)  # noqa: E731
    meta = AttnMeta(kind="decode", slots=i32(slots), cu_q=i32(list(range(len(ctxs) + 1))), ctx_lens=i32(ctxs), block_tables=bt, max_q_len=1,
                    max_ctx=max(ctxs), decode_ws=ops.DecodeWorkspace(len(ctxs), m.hq, m.hkv, max(ctxs), gpu, D=m.D))
    ids, pos = i32([7 + 3 * b for b in range(len(ctxs))]), i32([n - 1 for n in ctxs])
    want, calls = one._step64(m, ids, pos, before, bt, ctxs), []
    monkeypatch.setattr(m, "_decode_rows", lambda *a, f=m._decode_rows: calls.append(1) or f(*a))
    got = m.forward(ids, pos, meta)
    assert bool(calls) == taken
    last = torch.tensor([len(ctxs) - 1], device=gpu)
    assert torch.equal(m.forward(ids, pos, meta, last), got[-1:])
    monkeypatch.setattr(m, "_rows_decode", lambda *a: False)
    single = m.forward(ids, pos, meta)
    err = lambda y: ((y.double() - want).norm() / want.norm()).item()  # noqa: E731
    # the roundings are as many and as large: to within chance (a fifth at 512 values a row)
    assert err(got) <= 1.2 * err(single) and err(single) < 0.02, (err(got), err(single))
