"""The training kernels and their autograd functions on the GPU: each against the same step in 64 bits, or bit for bit against
the torch operations it replaces; the models' losses and gradients against those."""
import pytest
import torch
import torch.nn.functional as F

from nv_genai_amd import ops
from nv_genai_amd.training import functional as Fn
from nv_genai_amd.training import fused

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


def _check(fn, ref, inputs, tol=6e-3):
    """fn(*inputs) and the gradients of its inputs against ref in 64 bits. bf16 results round to 2^-9 of their value, and a
    gradient sees two or three such roundings: 6e-3."""
    a = [t.detach().clone().requires_grad_(t.is_floating_point()) if torch.is_tensor(t) else t for t in inputs]
    b = [t.detach().double().requires_grad_() if torch.is_tensor(t) and t.is_floating_point() else t for t in inputs]
    x, y = fn(*a), ref(*b)
    x, y = (x if isinstance(x, tuple) else (x,)), (y if isinstance(y, tuple) else (y,))
    g = torch.Generator(device="cuda").manual_seed(7)
    dy = [torch.randn(t.shape, device="cuda", generator=g).to(t.dtype) for t in x]
    ga = torch.autograd.grad(x, [t for t in a if torch.is_tensor(t) and t.is_floating_point()], dy)
    gb = torch.autograd.grad(y, [t for t in b if torch.is_tensor(t) and t.is_floating_point()], [d.double() for d in dy])
    for p, q in zip(x, y):
        assert p.shape == q.shape and _rel(p, q) < tol, _rel(p, q)
    for i, (p, q) in enumerate(zip(ga, gb)):
        assert p.shape == q.shape and _rel(p, q) < tol, (i, _rel(p, q))


def _bf(*shape, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return (scale * torch.randn(*shape, device="cuda", generator=g)).to(BF)


def _w(n, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + n)
    return (1 + 0.3 * torch.randn(n, device="cuda", generator=g)).to(dtype)


def _bits(fn, ref, inputs, sums=(), rounded=()):
    """fn and ref, the torch operations it replaces: outputs and gradients equal to the bit, but those of the inputs in `sums`,
    which are sums over rows in another order: 1e-5, or what rounding them to bf16 makes of them (2^-8 each at most)."""
    got = []
    for f in (fn, ref):
        a = [t.detach().clone().requires_grad_() if torch.is_tensor(t) and t.is_floating_point() else t for t in inputs]
        y = f(*a)
        y = y if isinstance(y, tuple) else (y,)
        g = torch.Generator(device="cuda").manual_seed(7)
        dy = [torch.randn(t.shape, device="cuda", generator=g).to(t.dtype) for t in y]
        got.append((y, torch.autograd.grad(y, [t for t in a if torch.is_tensor(t) and t.requires_grad], dy)))
    (ya, ga), (yb, gb) = got
    for p, q in zip(ya, yb):
        assert p.dtype == q.dtype and torch.equal(p, q), (p.float() - q.float()).abs().max()
    for i, (p, q) in enumerate(zip(ga, gb)):
        assert p.dtype == q.dtype and p.shape == q.shape
        if i in sums:
            assert _rel(p, q) < (8e-3 if BF in (p.dtype, *rounded) else 1e-5), (i, _rel(p, q))
        else:
            assert torch.equal(p, q), (i, (p.float() - q.float()).abs().max(), (p != q).sum())


# one row, rows above and below the count of workgroups that leave sums, sizes at the ends of the range and off the wave's
@pytest.mark.parametrize("R,H", [(1, 8), (3, 384), (1023, 768), (1500, 1024), (5, 8192)])
@pytest.mark.parametrize("dtype", [torch.float32, BF])
def test_norms(gpu, R, H, dtype):
    eps = 1e-5
    x, o, w, b = _bf(R, H), _bf(R, H, seed=3), _w(H, dtype), _w(H, dtype, 1)
    _bits(lambda x, w: fused.rms_norm(x, w, eps), lambda x, w: Fn.rms_norm(x, w, eps), [x, w], (1,))
    _bits(lambda x, o, w: fused.add_rms_norm(x, o, w, eps), lambda x, o, w: (x + o, Fn.rms_norm(x + o, w, eps)), [x, o, w], (2,))
    _bits(lambda x, o, g, b: fused.residual_layer_norm(x, o, g, b, eps),
          lambda x, o, g, b: F.layer_norm(x.float() + o.float(), (H,), g.float(), b.float(), eps).to(BF), [x, o, w, b], (2, 3))
    rms = lambda x, w: x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w  # noqa: E731
    _check(lambda x, w: fused.rms_norm(x, w, eps, True), rms, [x, w])
    # the sum is rounded to bf16 before its norm, in both
    _check(lambda x, o, w: fused.add_rms_norm(x, o, w, eps, True),
           lambda x, o, w: (x + o, rms(x + o, w)), [x, torch.zeros_like(x), w])


def test_activations_keep_every_bit(gpu):
    """All bf16 values, infinities, NaN and subnormals with them, against a random other operand."""
    z = torch.arange(-32768, 32768, device=gpu).to(torch.int16).view(BF)
    gu = torch.stack([z, _bf(65536)], 1).reshape(-1, 2).t().reshape(1, -1)
    for fn, ref, x, n in ((fused.gelu, lambda z: F.gelu(z.float()).to(BF), z.view(8, 8192), 8192),
                          (fused.swiglu, lambda t: F.silu(t[:, :65536]) * t[:, 65536:], gu, 65536)):
        a, b = x.clone().requires_grad_(), x.clone().requires_grad_()
        dy = _bf(x.shape[0], n, seed=2)
        ya, yb = fn(a), ref(b)
        for p, q in ((ya, yb), (torch.autograd.grad(ya, a, dy)[0], torch.autograd.grad(yb, b, dy)[0])):
            assert torch.equal(p.nan_to_num(7.0), q.nan_to_num(7.0)) and torch.equal(p.isnan(), q.isnan())


@pytest.mark.parametrize("R,F_", [(1, 8), (700, 1536), (33, 2056)])
@pytest.mark.parametrize("dtype", [torch.float32, BF])
def test_activations_and_linear(gpu, R, F_, dtype):
    _bits(fused.gelu, lambda z: F.gelu(z.float()).to(BF), [_bf(R, F_)])
    _bits(fused.swiglu, lambda gu: F.silu(gu[:, :F_]) * gu[:, F_:], [_bf(R, 2 * F_)])
    _bits(fused.linear, lambda x, w, b: F.linear(x, w.to(BF), b.to(BF)),
          [_bf(R, 64), _bf(F_, 64, scale=0.1).to(dtype), _bf(F_, seed=5).to(dtype)], (2,), (BF,))


@pytest.mark.parametrize("T,P,hq,hkv,D", [(1, 1, 1, 1, 16), (130, 65, 3, 1, 64), (77, 77, 8, 2, 128)])
def test_rope(gpu, T, P, hq, hkv, D):
    a = torch.arange(P, device=gpu)[:, None] * 10000.0 ** (-torch.arange(D // 2, device=gpu) / (D // 2))
    cs = torch.cat([a.cos(), a.sin()], 1).float()
    at = torch.arange(T, device=gpu) % P
    c, s = cs[at][None, :, None, : D // 2], cs[at][None, :, None, D // 2:]

    def ref(x):
        h = x.view(1, T, hq + 2 * hkv, D)
        return torch.cat([Fn.apply_rope(h[:, :, : hq + hkv], c, s), h[:, :, hq + hkv:]], 2).reshape(T, -1)

    _bits(lambda x: fused.rope(x, cs, hq + hkv, hq + 2 * hkv, D), ref, [_bf(T, (hq + 2 * hkv) * D)])


def _causal(q, k, v, n):
    """[n, heads, D] in 64 bits; also the rows' log-sums."""
    k, v = (t.repeat_interleave(q.shape[1] // t.shape[1], 1).transpose(0, 1) for t in (k, v))
    s = q.transpose(0, 1) @ k.transpose(1, 2) * q.shape[2] ** -0.5
    s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    return (torch.softmax(s, -1) @ v).transpose(0, 1).flatten(1), torch.logsumexp(s, -1)


@pytest.mark.parametrize("lens", [[1], [64, 65], [128, 129, 31], [300, 1, 257]])
@pytest.mark.parametrize("D,hq,hkv", [(32, 3, 3), (64, 4, 1), (128, 8, 2)])
def test_attention_backward(gpu, lens, D, hq, hkv):
    T, w = sum(lens), [hq * D, hkv * D, hkv * D]
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0).tolist()), dtype=torch.int32, device="cuda")
    qkv, dout = _bf(T, sum(w)), _bf(T, hq * D, seed=4)
    x = qkv.double().requires_grad_()
    parts = [_causal(*(t[a:a + n].unflatten(1, (-1, D)) for t in x.split(w, 1)), n) for a, n in zip(cu.tolist(), lens)]
    ref = torch.cat([p[0] for p in parts])
    want = torch.autograd.grad(ref, x, dout.double())[0].split(w, 1)
    lse = torch.cat([p[1] for p in parts], 1).detach().float() * 1.4426950408889634
    d = torch.empty_like(qkv)
    ops.kernels().train_attention_backward(*d.split(w, 1), dout, *qkv.split(w, 1), ref.detach().to(BF), lse, cu, hq, hkv, D, max(lens), D ** -0.5)
    # probabilities, their gradient and the result round to bf16, 2^-9 each: 6e-3; a lone key's p (dp - delta) cancels in full
    for p, q in zip(d.split(w, 1), want):
        assert _rel(p, q) < 6e-3 or (T == 1 and (p.double() - q).abs().max() < 0.1), _rel(p, q)


@pytest.mark.parametrize("B,S,D,hq,hkv", [(1, 1, 64, 2, 2), (2, 130, 64, 4, 1), (3, 77, 128, 8, 2)])
def test_attention_matches_torch_operations(gpu, B, S, D, hq, hkv):
    a = torch.arange(B * S, device="cuda")[:, None] % S * 10000.0 ** (-torch.arange(D // 2, device="cuda") / (D // 2))
    cs = torch.cat([a.cos(), a.sin()], 1).float()
    cu = torch.arange(0, B * S + 1, S, dtype=torch.int32, device="cuda")
    x = _bf(B, S, (hq + 2 * hkv) * D).requires_grad_()
    assert fused.attention_usable(x, D, hq, hkv, D ** -0.5)
    ya = fused.attention(x, cs, cu, hq, hkv, D, D ** -0.5)
    q, k, v = fused._heads(fused.rope(x, cs, hq + hkv, hq + 2 * hkv, D), hq, hkv, D)
    yb = F.scaled_dot_product_attention(q, k, v, is_causal=True, scale=D ** -0.5, enable_gqa=hq != hkv).transpose(1, 2).reshape(ya.shape)
    dy = _bf(*ya.shape, seed=6)
    assert torch.equal(ya, yb)
    assert _rel(*(torch.autograd.grad(y, x, dy)[0] for y in (ya, yb))) < 1e-2


@pytest.mark.parametrize("R,V", [(1, 8), (3, 32768), (65, 50264)])
def test_cross_entropy(gpu, R, V):
    y = torch.randint(0, V, (R,), device="cuda")
    lg = _bf(R, V, scale=3.0)
    a, b = lg.clone().requires_grad_(), lg.double().requires_grad_()
    la, lb = fused.cross_entropy_sum(a, y, True), F.cross_entropy(b, y, reduction="sum")
    # fp32 sums of V terms: about sqrt(V) 2^-24
    assert abs(la.item() - lb.item()) <= 1e-5 * max(1.0, abs(lb.item()))
    ga, gb = torch.autograd.grad(la * 0.5, a)[0], torch.autograd.grad(lb * 0.5, b)[0]
    assert _rel(ga, gb) < 4e-3
    a, b = lg.clone().requires_grad_(), lg.clone().requires_grad_()
    la, lb = fused.cross_entropy_sum(a, y), F.cross_entropy(b.float(), y, reduction="sum")
    assert torch.equal(la, lb) and torch.equal(*(torch.autograd.grad(x * 0.3, t)[0] for x, t in ((la, a), (lb, b))))


def test_lora_linear(gpu):
    x, w, a, b = _bf(130, 256), _bf(384, 256, scale=0.05), _bf(16, 256, scale=0.05).float(), _bf(384, 16, scale=0.05).float()
    a, b = a.requires_grad_(), b.requires_grad_()
    xa, xb = x.clone().requires_grad_(), x.double().requires_grad_()
    A, B = a.detach().double().requires_grad_(), b.detach().double().requires_grad_()
    ya, yb = fused.lora_linear(xa, w, a, b, 2.0), xb @ w.double().t() + 2.0 * (xb @ A.t()) @ B.t()
    dy = _bf(130, 384, seed=9)
    h = (x @ a.detach().to(BF).t()) @ b.detach().to(BF).t()
    assert _rel(ya, yb) < 6e-3 and torch.equal(ya, x @ w.t() + h * 2.0)
    for p, q in zip(torch.autograd.grad(ya, (xa, a, b), dy), torch.autograd.grad(yb, (xb, A, B), dy.double())):
        assert p.dtype == (torch.float32 if p.shape != x.shape else BF) and _rel(p, q) < 6e-3


@pytest.mark.parametrize("name,S", [("llama-tiny", 70), ("mistral-tiny", 130), ("gemma-tiny", 40), ("mixtral-tiny", 33),
                                    ("starcoder2-tiny", 50), ("llama-small", 129)])
@pytest.mark.parametrize("how", ["params", "lora", "checkpointed"])
def test_llama_hidden_matches_torch_operations(gpu, monkeypatch, name, S, how):
    from nv_genai_amd.models.config import llama_config
    from nv_genai_amd.models.llama import LlamaModel
    from nv_genai_amd.training.lora import LoRA, LoRAConfig

    m = LlamaModel(llama_config(name), gpu, seed=3)
    ids = torch.randint(0, 1000, (2, S), device=gpu)
    lab = torch.randint(0, 1000, (2, S), device=gpu)
    lab[1, S // 2:] = -100

    def grads():
        if how == "lora":
            ad = LoRA(m, LoRAConfig(r=8, alpha=16, targets=("qkv", "o")) if not m.cfg.is_moe else LoRAConfig(r=8, alpha=16), seed=1)
            for t in ad.B.values():
                t.data.normal_(0, 0.02, generator=torch.Generator(device="cuda").manual_seed(4))
            ps, kw = list(ad.parameters()), {"linear": ad.linear}
        else:
            P = Fn.trainable_params(m, "llama")
            ps, kw = [P[k] for k in sorted(P, key=str)], {"params": P, "grad_ckpt": how == "checkpointed"}
        with torch.autocast("cuda", dtype=BF):
            loss = Fn.lm_loss(m, Fn.llama_hidden(m, ids, **kw), lab, params=kw.get("params"))
        return loss.detach(), torch.autograd.grad(loss, ps, allow_unused=True)

    la, ga = grads()
    off = lambda *a, **k: False  # noqa: E731
    for n in ("usable", "swiglu_usable", "rope_usable", "cross_entropy_usable"):
        monkeypatch.setattr(fused, n, off)
    lb, gb = grads()
    if how == "lora":
        # equal activations; the loss sums in another order, the gradients carry bf16 rounding through two to four layers
        ltol, tol = 1e-6, 3e-2
    else:
        # equal bits but for the fp32 sums of norms' weights (test_training_routes_gpu.py compares them); experts' rows are added
        # up in no fixed order
        ltol, tol = 0.0, 4e-3
    assert abs(la.item() - lb.item()) <= ltol * abs(lb.item())
    for p, q in zip(ga, gb):
        assert (p is None) == (q is None)
        if p is not None:
            assert p.dtype == q.dtype and _rel(p, q) < tol, (p.shape, _rel(p, q))


@pytest.mark.parametrize("pooling", ["cls", "mean"])
@pytest.mark.parametrize("ckpt", [False, True])
def test_encoder_embed_matches_torch_operations(gpu, monkeypatch, pooling, ckpt):
    from dataclasses import replace

    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel

    m = EncoderModel(replace(encoder_config("encoder-tiny"), pooling=pooling), gpu, seed=2)
    ids = torch.randint(0, 1000, (5, 70), device=gpu)
    lens = torch.tensor([70, 1, 33, 64, 2], device=gpu)
    mask = (torch.arange(70, device=gpu) < lens[:, None]).long()
    dy = torch.randn(5, m.cfg.hidden, device=gpu)

    def grads():
        P = Fn.trainable_params(m, "encoder")
        with torch.autocast("cuda", dtype=BF):
            y = Fn.encoder_embed(m, ids, mask, P, ckpt)
        ks = sorted(P, key=str)
        return y.detach(), dict(zip(ks, torch.autograd.grad(y, [P[k] for k in ks], dy)))

    ya, ga = grads()
    monkeypatch.setattr(fused, "usable", lambda *a: False)
    yb, gb = grads()
    assert torch.equal(ya, yb)
    for k in ga:
        # the key bias has no gradient in exact arithmetic: what either side has of it is rounding
        p, q = (t[k] if k[1] != "bqkv" else torch.cat([t[k][: m.cfg.hidden], t[k][2 * m.cfg.hidden:]]) for t in (ga, gb))
        assert _rel(p, q) < 4e-3, (k, _rel(p, q))


# one element, tails of a chunk and of eight, more tensors than a launch takes; both passes use all of them, or one leaves one out
@pytest.mark.parametrize("skip", [None, 1])
def test_half_copies_keep_every_bit(gpu, skip):
    shapes = [(1,), (7, 3), (8192,), (8193,), (3, 8190)] + [(5,)] * 70
    m = [torch.randn(s, device=gpu).mul_(3).requires_grad_() for s in shapes]
    assert fused.half_copies_usable(m)
    got, ref = fused.half_copies(m), [[t.to(BF) for t in m] for _ in range(2)]
    dy = [[torch.randn(s, device=gpu).to(BF) for s in shapes] for _ in range(2)]
    sums = []
    for use in (got, ref):
        sums.append(sum((y * d).float().sum() for u in range(2) for i, (y, d) in enumerate(zip(use[u], dy[u])) if not (u == 1 and i == skip)))
    for a, b in zip(got, ref):
        assert all(torch.equal(p, q) for p, q in zip(a, b))
    for create in (False, True):
        ga, gb = (torch.autograd.grad(s, m, retain_graph=True, create_graph=create) for s in sums)
        assert all(p.dtype == torch.float32 and torch.equal(p, q) for p, q in zip(ga, gb))


def test_half_params_keep_the_gradients(gpu):
    """A step of both passes over shared copies against each pass casting for itself."""
    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel

    m = EncoderModel(encoder_config("encoder-tiny"), gpu, seed=2)
    ids = torch.randint(0, 1000, (3, 40), device=gpu)
    got = []
    for shared in (True, False):
        P = Fn.trainable_params(m, "encoder")
        with torch.autocast("cuda", dtype=BF):
            a, b = Fn.half_params(P) if shared else (P, P)
            assert (a[(0, "wo")].dtype is BF) == shared
            y = (Fn.encoder_embed(m, ids, torch.ones_like(ids), a) * Fn.encoder_embed(m, ids[:, :9], torch.ones_like(ids[:, :9]), b)).pow(3).sum()
        y.backward()
        got.append((y.detach(), {k: v.grad for k, v in P.items()}))
    (ya, ga), (yb, gb) = got
    assert torch.equal(ya, yb)
    for k in gb:
        assert torch.equal(ga[k], gb[k]), k


def test_checkpointed_embedding_step_holds_no_copies(gpu):
    """With checkpointing a step's loss holds the layers' inputs (two short texts) and no bf16 copy of the weights (21 MB); its loss and
    gradients are those without."""
    import gc

    from nv_genai_amd.engine.embed_engine import EmbeddingEngine
    from nv_genai_amd.training.embed_finetune import embed_trainer
    from nv_genai_amd.training.sft import TrainConfig

    eng, got = EmbeddingEngine("all-minilm-l6-v2", device=gpu), []
    recs = [{"question": "one two", "pos_doc": ["three four"], "neg_doc": ["five six"]}] * 2
    for ckpt in (True, False):
        tr, P = embed_trainer(eng, recs, TrainConfig(micro_batch=2, global_batch=2, max_steps=2, log_every=0, grad_ckpt=ckpt), hard_negatives=1)
        tr.loss_fn(tr.data[0]).backward()   # libraries' workspaces are there
        for p in P.values():
            p.grad = None
        gc.collect()
        before = torch.cuda.memory_allocated()
        loss = tr.loss_fn(tr.data[0])
        assert not ckpt or torch.cuda.memory_allocated() - before < 5e6
        loss.backward()
        got.append((loss.item(), {k: p.grad for k, p in P.items()}))
    assert got[0][0] == got[1][0] and all(torch.equal(got[0][1][k], got[1][1][k]) for k in got[0][1])
