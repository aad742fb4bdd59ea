"""The fused kernels of a decode step against the launches that they stand for."""
import math

import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu


def _pages(ctxs, Hkv, dev):
    pages = [(c + 63) // 64 for c in ctxs]
    nb = sum(pages) + 3
    kc = torch.randn(nb, Hkv, 64, 128, device=dev).to(torch.bfloat16)
    vc = torch.randn(nb, Hkv, 128, 64, device=dev).to(torch.bfloat16)
    perm = torch.randperm(nb).tolist()
    bt = torch.zeros(len(ctxs), max(pages), dtype=torch.int32)
    slots, k = [], 0
    for i, (c, p) in enumerate(zip(ctxs, pages)):
        for j in range(p):
            bt[i, j], k = perm[k], k + 1
        slots.append(int(bt[i, (c - 1) // 64]) * 64 + (c - 1) % 64 if c else -1)
    return kc, vc, bt.to(dev), torch.tensor(slots, dtype=torch.int32, device=dev)


@pytest.mark.parametrize("G,Hkv", [(4, 8), (1, 8), (5, 2), (16, 1)])
@pytest.mark.parametrize("ppp,window", [(None, 0), (1, 0), (3, 0), (2, 200), (None, 64)])
@pytest.mark.parametrize("slabs", [0, 1, 3])
def test_decode_step_is_rotation_and_attention(gpu, G, Hkv, ppp, window, slabs):
    """Contexts around the ends of pages and of partitions, rows without a context and rows whose key is not written. The
    cache is the same to the bit. The outputs are bf16 of the same products; only the sum over the partitions has another
    form (two fp32 sums over up to 16 parts, then one rounding): one bf16 step, 2^-8 of the value, and of the largest where
    values cancel."""
    torch.manual_seed(G * 100 + slabs)
    Hq, D, dev = Hkv * G, 128, gpu
    part = 64 * 4 * (ppp or 1)
    ctxs = [1, 0, 63, 64, 65, 700, 128, part - 1, part, part + 1, 3 * part + 1, 2500]
    kc, vc, bt, slots = _pages(ctxs, Hkv, dev)
    slots[6] = -1
    B, row = len(ctxs), (Hq + 2 * Hkv) * D
    if slabs:
        qkv = ops.PartialSum(torch.randn(slabs, B, row, device=dev))
        flat = ops.splitk_reduce(qkv.slabs)
    else:
        flat = torch.randn(B, row, device=dev).to(torch.bfloat16)
        qkv = flat.clone()
    ctx = torch.tensor(ctxs, dtype=torch.int32, device=dev)
    pos = (ctx - 1).clamp(min=0)
    cs = ops.rope_cos_sin(4096, D).to(dev)
    most, scale = max(ctxs), 1 / math.sqrt(D)
    ws = ops.DecodeWorkspace(B, Hq, Hkv, most, dev, ppp)
    k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    ops.rope_cache_(flat, pos, cs, slots, k1, v1, Hq, Hkv, D)
    want = ops.decode_attention(flat[:, : Hq * D], k1, v1, bt, ctx, Hq, Hkv, most, scale, ws=ws, window=window)
    assert ops.decode_step_covers(qkv, k2, ctx, slots, most, ws, window)
    for k in (128, 4096):   # the counters are zero again after a launch; weights to read ahead of one and of many blocks a piece
        nxt = torch.empty(16 * 37, k, dtype=torch.bfloat16, device=dev)
        got = ops.decode_step(qkv, pos, cs, slots, k2, v2, bt, ctx, Hq, Hkv, most, scale, ws, window, nxt)
        assert torch.equal(k1, k2) and torch.equal(v1, v2)
        assert not ws.done.any()
        w, g = want.float(), got.float()
        assert (g[1] == 0).all()
        assert ((g - w).abs() <= 2 ** -8 * w.abs() + 2 ** -8 * w.abs().amax(1, keepdim=True)).all()


@pytest.mark.parametrize("rows,N,K,ahead", [(1, 4096, 4096, True), (16, 4096, 4096, True), (1, 2048, 2048, True), (1, 5120, 5120, False), (1, 8192, 8192, False),
                                           (4, 6144, 4096, False), (1, 8192, 4096, False), (1, 4096, 8192, False), (17, 4096, 4096, False),
                                           (1, 4096, 4000, False)])
def test_weights_are_read_ahead_for_the_kernel_that_takes_them(gpu, rows, N, K, ahead):
    """The stream kernel with 16 weight rows a workgroup, and up to 33.5 MB."""
    assert ops.kernels().stream_gemm_reads_ahead(rows, N, K) == ahead


@pytest.mark.parametrize("rows,Hkv,one", [(64, 8, True), (65, 8, False), (16, 32, True), (17, 32, False), (256, 2, True), (512, 1, True), (513, 1, False)])
def test_many_rows_take_launches_of_their_own(gpu, rows, Hkv, one):
    """From more than two workgroups a CU on the rotation stands alone; at the line both give the same."""
    D, dev = 128, gpu
    ctxs = [1 + (37 * i) % 150 for i in range(rows)]
    kc, vc, bt, slots = _pages(ctxs, Hkv, dev)
    qkv = torch.randn(rows, 3 * Hkv * D, device=dev).to(torch.bfloat16)
    ctx, cs = torch.tensor(ctxs, dtype=torch.int32, device=dev), ops.rope_cos_sin(256, D).to(dev)
    ws = ops.DecodeWorkspace(rows, Hkv, Hkv, 192, dev)
    assert ops.decode_step_covers(qkv, kc, ctx, slots, 192, ws) == one
    if not one:
        return
    k1, v1, flat = kc.clone(), vc.clone(), qkv.clone()
    got = ops.decode_step(qkv, ctx - 1, cs, slots, kc, vc, bt, ctx, Hkv, Hkv, 192, D ** -0.5, ws).float()
    ops.rope_cache_(flat, ctx - 1, cs, slots, k1, v1, Hkv, Hkv, D)
    want = ops.decode_attention(flat[:, : Hkv * D], k1, v1, bt, ctx, Hkv, Hkv, 192, D ** -0.5, ws=ws).float()
    assert torch.equal(kc, k1) and torch.equal(vc, v1)
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2 ** -8 * want.abs().amax(1, keepdim=True)).all()   # as above


@pytest.mark.parametrize("N,K", [(4096, 4096), (6144, 4096), (16, 256), (48, 768), (1008, 2304), (14336, 4096), (512, 8192), (384, 5120),
                                 (101, 520), (33, 1032), (7, 8), (2064, 8184)])
@pytest.mark.parametrize("epi", [1, 2])
def test_norm_linear(gpu, N, K, epi, M=1):
    """Stages that do not split evenly over the waves, K below and at the kernels' ends, the GEMV for odd shapes. The norm's
    sum of squares has another order, so a normed value may fall on the next bf16 (2^-8 of it): at most 2^-8 of a row of
    products, and with SwiGLU, a product of two of them rounded to bf16, three times that."""
    torch.manual_seed(N + K)
    x = (2 * torch.randn(M, K, device=gpu)).to(torch.bfloat16)
    nw = (1 + 0.3 * torch.randn(K, device=gpu)).to(torch.bfloat16)
    w = (torch.randn((2 if epi == 2 else 1) * N, K, device=gpu) / math.sqrt(K)).to(torch.bfloat16)
    assert ops.norm_linear_covers(x, nw, w, epi == 2)
    got = ops.norm_linear(x, nw, 1e-5, w, epi).float()
    y = ops.rmsnorm(x, nw, 1e-5).double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :N]) * y[:, N:] if epi == 2 else y
    assert got.shape == want.shape
    err = (got.double() - want).norm(dim=1) / want.norm(dim=1)
    assert (err <= 2 ** -8 * (3 if epi == 2 else 1)).all()


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (2, 4096, 14336), (1, 16, 256), (7, 48, 768), (16, 4096, 4096), (8, 1024, 8192)])
def test_linear_add(gpu, M, N, K):
    """One rounding of the sum: half a bf16 step of it, and the products' fp32 sums in another order (K values, 2^-24 each)."""
    torch.manual_seed(N + K)
    x = torch.randn(M, K, device=gpu).to(torch.bfloat16)
    w = (torch.randn(N, K, device=gpu) / math.sqrt(K)).to(torch.bfloat16)
    resid = torch.randn(M, N, device=gpu).to(torch.bfloat16)
    assert ops.linear_add_covers(M, w)
    want = resid.double() + x.double() @ w.double().t()
    got = ops.linear_add_(resid, x, w)
    assert got.data_ptr() == resid.data_ptr()
    slack = 2 ** -24 * math.sqrt(K) * (x.double().abs() @ w.double().abs().t())
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + slack + 1e-6).all()


def _step64(m, ids, pos, pages, bt, ctxs):
    """Final-normed rows of one decode step in 64 bits; pages: K and V^T of every layer before it."""
    c, D = m.cfg, m.D
    d = lambda t: t.double()  # noqa: E731
    rms = lambda x, w: x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + c.eps) * d(w)  # noqa: E731
    x = d(m.embed)[ids.long()]
    cos, sin = (t[:, None] for t in d(m.cos_sin[pos.long()]).split(D // 2, -1))
    turn = lambda t: torch.cat([t[..., : D // 2] * cos - t[..., D // 2:] * sin, t[..., D // 2:] * cos + t[..., : D // 2] * sin], -1)  # noqa: E731
    for li, L in enumerate(m.layers):
        q, k, v = (t.unflatten(-1, (-1, D)) for t in (rms(x, L["attn_norm"]) @ d(L["wqkv"]).t()).split([m.hq * D, m.hkv * D, m.hkv * D], -1))
        q, k, out = turn(q), turn(k), []
        for b, n in enumerate(ctxs):
            at = bt[b, : (n + 63) // 64].long()
            K = d(pages[0][li, at].float()).transpose(1, 2).reshape(-1, m.hkv, D)[: n - 1]
            V = d(pages[1][li, at].float()).permute(0, 3, 1, 2).reshape(-1, m.hkv, D)[: n - 1]
            K, V = (torch.cat([a, t[b: b + 1]]).repeat_interleave(m.hq // m.hkv, 1) for a, t in ((K, k), (V, v)))
            out.append(torch.einsum("hk,khd->hd", torch.softmax(torch.einsum("hd,khd->hk", q[b], K) * m.scale, -1), V).flatten())
        x = x + torch.stack(out) @ d(L["wo"]).t()
        g, u = (rms(x, L["mlp_norm"]) @ d(L["wgu"]).t()).chunk(2, -1)
        x = x + (torch.nn.functional.silu(g) * u) @ d(L["wd"]).t()
    return rms(x, m.final_norm)


# one row with everything fused; pages of 256 dimensions and of fp8 behind the fused norms and residuals; a K that the GEMV takes; several rows
@pytest.mark.parametrize("over,kv,ctxs,one", [({}, "auto", [300], True), ({}, "auto", [65], True), ({"heads": 2, "kv_heads": 1, "head_dim": 256}, "auto", [300], True),
                                              ({}, "fp8", [300], True), ({"ffn": 1032}, "auto", [300], False), ({}, "auto", [300, 1, 64], False)])
def test_a_models_decode_step(gpu, monkeypatch, over, kv, ctxs, one):
    """Whether a step runs as _decode_layers, and its rows against 64 bits beside the same step in launches of their own: norms and
    sums are rounded less often, so its error is theirs to within chance (a fifth at 512 values a row)."""
    from nv_genai_amd.models.config import llama_config
    from nv_genai_amd.models.llama import AttnMeta, LlamaModel

    m = LlamaModel(llama_config("llama3-8b", **{**dict(layers=3, vocab_size=512, hidden=512, heads=4, kv_heads=2, head_dim=128, ffn=1024, max_position=512), **over}), gpu)
    g = torch.Generator(gpu).manual_seed(11)
    for L in m.layers:
        for n in ("attn_norm", "mlp_norm"):
            L[n].normal_(1, 0.1, generator=g)
    m.embed.mul_(20)   # a residual stream of the size of what is added to it
    pages = [(n + 63) // 64 for n in ctxs]
    m.allocate_kv_cache(sum(pages) + 1, kv_dtype=kv)
    for t in (m.k_cache, m.v_cache):
        t.copy_(torch.randn(t.shape, device=gpu, generator=g).to(t.dtype))
    before, bt, slots, at = [m.k_cache.clone(), m.v_cache.clone()], torch.zeros(len(ctxs), max(pages), dtype=torch.int32, device=gpu), [], 1
    for b, n in enumerate(ctxs):
        bt[b, : pages[b]] = torch.arange(at, at + pages[b])
        at += pages[b]
        slots.append(int(bt[b, (n - 1) // 64]) * 64 + (n - 1) % 64)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)  # noqa: E731
    meta = AttnMeta(kind="decode", slots=i32(slots), cu_q=i32(list(range(len(ctxs) + 1))), ctx_lens=i32(ctxs), block_tables=bt, max_q_len=1,
                    max_ctx=max(ctxs), decode_ws=ops.DecodeWorkspace(len(ctxs), m.hq, m.hkv, max(ctxs), gpu, D=m.D, kv_fp8=kv == "fp8"))
    ids, pos = i32([7 + 3 * b for b in range(len(ctxs))]), i32([n - 1 for n in ctxs])
    want, calls = _step64(m, ids, pos, before, bt, ctxs), []
    monkeypatch.setattr(m, "_decode_layers", lambda *a, f=m._decode_layers: calls.append(1) or f(*a))
    got = m.forward(ids, pos, meta)
    assert bool(calls) == one
    kept = m.k_cache.float()
    rows = m.forward(ids, pos, meta, torch.tensor([0], device=gpu))
    assert torch.equal(rows, got[:1]) and torch.equal(m.k_cache.float(), kept)
    monkeypatch.setattr(m, "_fused_decode", lambda *a: False)
    monkeypatch.setattr(ops, "decode_step_covers", lambda *a: False)
    single = m.forward(ids, pos, meta)
    err = lambda y: ((y.double() - want).norm() / want.norm()).item()  # noqa: E731
    assert err(got) <= 1.2 * err(single) and err(single) < (0.1 if kv == "fp8" else 0.02), (err(got), err(single))
