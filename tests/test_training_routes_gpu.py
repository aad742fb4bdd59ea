"""Calls that the fused training functions take or leave to the torch operations: every form that those accept gives their
results."""
import pytest
import torch

from nv_genai_amd.training import functional as Fn
from nv_genai_amd.training import fused

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


def _rows(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return torch.randn(*shape, device="cuda", generator=g).to(BF)


def _without(monkeypatch):
    """The torch operations in place of the functions."""
    for n in ("usable", "swiglu_usable", "rope_usable", "cross_entropy_usable"):
        monkeypatch.setattr(fused, n, lambda *a, **k: False)


def _llama(dev, name="llama-tiny"):
    from nv_genai_amd.models.config import llama_config
    from nv_genai_amd.models.llama import LlamaModel

    return LlamaModel(llama_config(name), dev, seed=3)


@pytest.mark.parametrize("shape", [(1, 40), (2, 1), (1, 1), (2, 40), (40,)])
def test_positions_of_any_shape(gpu, monkeypatch, shape):
    """Positions broadcast over the ids [2, 40]; a bare [40] raises, as it does without the functions."""
    m = _llama(gpu)
    ids = torch.randint(0, 1000, (2, 40), device=gpu)
    pos = torch.randint(0, 60, shape, device=gpu)

    def hidden():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF):
            return Fn.llama_hidden(m, ids, pos=pos)

    if len(shape) == 1:
        with pytest.raises(RuntimeError):
            hidden()
        return
    a = hidden()
    _without(monkeypatch)
    assert torch.equal(a, hidden())


@pytest.mark.parametrize("name", ["wo", "wd", "all"])
def test_projections_of_another_type(gpu, monkeypatch, name):
    """A caller's projections may return fp32 rows."""
    m = _llama(gpu)
    ids = torch.randint(0, 1000, (2, 40), device=gpu)

    def linear(x, li, n):
        w = m.layers[li][n]
        return x.float() @ w.float().t() if name in (n, "all") else x.to(BF) @ w.t()

    with torch.no_grad():
        a = Fn.llama_hidden(m, ids, linear=linear)
        _without(monkeypatch)
        b = Fn.llama_hidden(m, ids, linear=linear)
    assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("how", ["params", "lora", "encoder"])
def test_autocast_to_half(gpu, monkeypatch, how):
    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel
    from nv_genai_amd.training.lora import LoRA, LoRAConfig

    m = _llama(gpu) if how != "encoder" else EncoderModel(encoder_config("encoder-tiny"), gpu, seed=2)
    ids = torch.randint(0, 1000, (2, 40), device=gpu)

    def loss_and_grads():
        if how == "lora":
            ad = LoRA(m, LoRAConfig(r=8, alpha=16), seed=1)
            for t in ad.B.values():
                t.data.normal_(0, 0.02, generator=torch.Generator(device="cuda").manual_seed(4))
            ps, kw = list(ad.parameters()), {"linear": ad.linear}
        else:
            P = Fn.trainable_params(m, "llama" if how == "params" else how)
            ps, kw = [P[k] for k in sorted(P, key=str)], {"params": P}
        with torch.autocast("cuda", dtype=torch.float16):
            if how == "encoder":
                loss = Fn.encoder_embed(m, ids, torch.ones_like(ids), **kw).pow(3).sum()
            else:
                loss = Fn.lm_loss(m, Fn.llama_hidden(m, ids, **kw), ids, params=kw.get("params"))
        return loss.detach(), torch.autograd.grad(loss, ps, allow_unused=True)

    la, ga = loss_and_grads()
    _without(monkeypatch)
    lb, gb = loss_and_grads()
    assert torch.equal(la, lb)
    for p, q in zip(ga, gb):   # the same operations; torch adds the embeddings' gradient in no fixed order
        assert (p is None) == (q is None)
        assert p is None or _rel(p, q) < 1e-3, (p.shape, _rel(p, q))


def test_make_fx_records_the_operations(gpu):
    """A graph recorded from real tensors computes from its inputs."""
    from torch.fx.experimental.proxy_tensor import make_fx

    m = _llama(gpu)
    ids = torch.randint(0, 1000, (2, 40), device=gpu)

    def loss(h, w):
        with torch.autocast("cuda", dtype=BF):
            x = Fn.llama_hidden(m, ids, params={"final_norm": w}) + h
        return Fn.lm_loss(m, x, ids)

    with torch.no_grad():
        g = make_fx(loss)(_rows(2, 40, m.cfg.hidden), _rows(m.cfg.hidden))
        h, w = _rows(2, 40, m.cfg.hidden, seed=9), _rows(m.cfg.hidden, seed=9)
        assert abs(g(h, w) - loss(h, w)) < 1e-5 * abs(loss(h, w))


@pytest.mark.parametrize("dtype", [torch.float32, BF])
def test_norm_weights_at_any_address(gpu, monkeypatch, dtype):
    """Norms' weights may be views that do not begin at 16 bytes."""
    m = _llama(gpu)
    ids = torch.randint(0, 1000, (2, 40), device=gpu)
    P = {k: v.detach().to(dtype) for k, v in Fn.trainable_params(m, "llama").items()}
    for k in [k for k in P if P[k].ndim == 1]:
        P[k] = torch.empty(P[k].numel() + 1, dtype=dtype, device=gpu)[1:].copy_(P[k])
    with torch.no_grad(), torch.autocast("cuda", dtype=BF):
        a = Fn.llama_hidden(m, ids, params=P)
        _without(monkeypatch)
        assert torch.equal(a, Fn.llama_hidden(m, ids, params=P))


def _twice(monkeypatch, f, xs, tol):
    """Gradients of f and of a function of those, with the fused functions and without."""
    got = []
    for fused_too in (True, False):
        if not fused_too:
            _without(monkeypatch)
        a = [x.detach().clone().requires_grad_() for x in xs]
        g = torch.autograd.grad(f(*a), a, create_graph=True)
        s = sum((t.float() * torch.linspace(-1, 1, t.numel(), device="cuda").view(t.shape)).sum() for t in g)
        got.append(g + torch.autograd.grad(s, a, allow_unused=True))
    for i, (p, q) in enumerate(zip(*got)):
        assert (p is None) == (q is None), i
        assert p is None or (p.dtype == q.dtype and _rel(p, q) < tol), (i, p.shape, _rel(p, q))


@pytest.mark.parametrize("kind", ["llama", "encoder", "lora", "loss", "loss of adapters"])
def test_second_derivatives(gpu, monkeypatch, kind):
    """Under create_graph the gradients can be differentiated again (attention through torch's plain form, its fast ones cannot).
    Both sides compute in bf16, and the second pass carries the rounding of the first: a few times 1e-2 at most."""
    from torch.nn.attention import SDPBackend, sdpa_kernel

    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel
    from nv_genai_amd.training.lora import LoRA, LoRAConfig

    m = EncoderModel(encoder_config("encoder-tiny"), gpu, seed=2) if kind == "encoder" else _llama(gpu)
    ids = torch.randint(0, 1000, (2, 24), device=gpu)
    if kind.startswith("loss"):
        P = {"lm_head": m.lm_head.float()} if kind == "loss" else None
        _twice(monkeypatch, lambda h: Fn.lm_loss(m, h, ids, params=P), [_rows(2, 24, m.cfg.hidden)], 1e-2)
        return
    if kind == "lora":
        ad = LoRA(m, LoRAConfig(r=8, alpha=24, targets=("qkv", "o")), seed=1)
        for t in ad.B.values():
            t.data.normal_(0, 0.02, generator=torch.Generator(device="cuda").manual_seed(4))
        ks, xs = [(d, k) for d in ("A", "B") for k in sorted(ad.A)], [*(ad.A[k] for k in sorted(ad.A)), *(ad.B[k] for k in sorted(ad.A))]
    else:
        P = Fn.trainable_params(m, kind)
        ks = sorted(P, key=str)
        xs = [P[k] for k in ks]

    def f(*ps):
        with torch.autocast("cuda", dtype=BF), sdpa_kernel(SDPBackend.MATH):
            if kind == "lora":
                for (d, k), p in zip(ks, ps):
                    getattr(ad, d)[k] = p
                return Fn.lm_loss(m, Fn.llama_hidden(m, ids, linear=ad.linear), ids)
            Q = dict(zip(ks, ps))
            if kind == "llama":
                return Fn.lm_loss(m, Fn.llama_hidden(m, ids, params=Q), ids, params=Q)
            return Fn.encoder_embed(m, ids, torch.ones_like(ids), Q).pow(3).sum()

    _twice(monkeypatch, f, xs, 5e-2)


@pytest.mark.parametrize("once", [False, True])
@pytest.mark.parametrize("at,n", [(0, 8), (0, 4104), (8, 1), (4088, 8), (4096, 8), (0, 0)])
def test_logits_that_are_not_numbers(gpu, once, at, n):
    """A NaN anywhere in a row, also where a thread of the one-pass form sees nothing else, makes its loss and gradient NaN;
    -inf does not."""
    lg = _rows(2, 4104)
    lg[:, 16:24] = float("-inf")
    lg[1, at:at + n] = float("nan")
    lg.requires_grad_()
    y = torch.tensor([5, 100], device=gpu)
    loss = fused.cross_entropy_sum(lg, y, once)
    want = torch.nn.functional.cross_entropy(lg.double(), y, reduction="sum")
    assert loss.isnan() == want.isnan() == (n > 0) and (n or abs(loss - want) < 1e-4)
    g = torch.autograd.grad(loss, lg)[0]
    assert not g[0].isnan().any() and g[1].isnan().all() == (n > 0)


def test_labels_outside_the_vocabulary_raise(gpu):
    m = _llama(gpu)
    V = m.lm_head.shape[0]
    h, lab = _rows(1, 6, m.cfg.hidden), torch.tensor([[-100, 3, V - 1, -1, 0, 5]], device=gpu)
    assert torch.isfinite(Fn.lm_loss(m, h, lab))
    assert float(Fn.lm_loss(m, h, torch.full_like(lab, -100))) == 0.0
    lab[0, 4] = V
    with pytest.raises(IndexError):
        Fn.lm_loss(m, h, lab)


@pytest.mark.parametrize("how,reached", [
    ("params", {"rms_norm", "add_rms_norm", "rope", "swiglu", "cross_entropy_sum"}),
    ("checkpointed", {"rms_norm", "add_rms_norm", "rope", "swiglu", "cross_entropy_sum"}),
    ("lora", {"rms_norm", "add_rms_norm", "attention", "lora_linear", "swiglu", "cross_entropy_sum"}),
    ("encoder", {"linear", "residual_layer_norm", "gelu"})])
def test_models_reach_the_functions(gpu, monkeypatch, how, reached):
    """Comparisons of the models with and without the functions compare something: these are called, and without them none is."""
    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel
    from nv_genai_amd.training.lora import LoRA, LoRAConfig

    called = set()
    names = {"rms_norm", "add_rms_norm", "rope", "swiglu", "cross_entropy_sum", "attention", "lora_linear", "linear",
             "residual_layer_norm", "gelu"}
    for n in names:
        monkeypatch.setattr(fused, n, lambda *a, n=n, f=getattr(fused, n): called.add(n) or f(*a))
    m = EncoderModel(encoder_config("encoder-tiny"), gpu, seed=2) if how == "encoder" else _llama(gpu)
    ids = torch.randint(0, 1000, (2, 40), device=gpu)

    def run():
        with torch.autocast("cuda", dtype=BF):
            if how == "encoder":
                return Fn.encoder_embed(m, ids, torch.ones_like(ids), Fn.trainable_params(m, "encoder")).sum()
            if how == "lora":
                return Fn.lm_loss(m, Fn.llama_hidden(m, ids, linear=LoRA(m, LoRAConfig(r=8, alpha=16), seed=1).linear), ids)
            P = Fn.trainable_params(m, "llama")
            return Fn.lm_loss(m, Fn.llama_hidden(m, ids, params=P, grad_ckpt=how == "checkpointed"), ids, params=P)

    run().backward()
    assert called == reached
    called.clear()
    _without(monkeypatch)
    run().backward()
    assert not called


@pytest.mark.parametrize("how", ["llama", "checkpointed", "encoder"])
def test_all_weight_gradients_keep_their_bits(gpu, monkeypatch, how):
    """All weights trained, one step's loss and the gradients of matrices and embeddings are those of the torch operations to the
    bit; those of norms' weights and of biases are sums over the rows in another order: in fp32 1e-5 for some hundred rows, and
    biases, which round that sum to bf16, one step of it, 2^-8."""
    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel

    kind = "encoder" if how == "encoder" else "llama"
    m = EncoderModel(encoder_config("encoder-tiny"), gpu, seed=2) if kind == "encoder" else _llama(gpu, "llama-small")
    ids = torch.randint(0, 1000, (2, 129), device=gpu)
    got = []
    for fused_too in (True, False):
        if not fused_too:
            _without(monkeypatch)
        P = Fn.trainable_params(m, kind)
        with torch.autocast("cuda", dtype=BF):
            if kind == "encoder":
                loss = Fn.encoder_embed(m, ids, torch.ones_like(ids), P).pow(3).sum()
            else:
                loss = Fn.lm_loss(m, Fn.llama_hidden(m, ids, params=P, grad_ckpt=how == "checkpointed"), ids, params=P)
        ks = sorted(P, key=str)
        got.append((loss.detach(), dict(zip(ks, torch.autograd.grad(loss, [P[k] for k in ks], allow_unused=True)))))
    (la, ga), (lb, gb) = got
    assert torch.equal(la, lb)
    for k, q in gb.items():
        p, name = ga[k], k if isinstance(k, str) else k[1]
        if q is None:
            assert p is None
        elif name.startswith("b"):   # the keys' bias has no gradient but rounding
            H = m.cfg.hidden
            p, q = (torch.cat([t[:H], t[2 * H:]]) if name == "bqkv" else t for t in (p, q))
            assert _rel(p, q) < 4e-3, (k, _rel(p, q))
        elif p.ndim == 1:
            assert _rel(p, q) < 1e-5, (k, _rel(p, q))
        else:
            assert torch.equal(p, q), (k, _rel(p, q))


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="two GPUs")
def test_a_gpu_that_is_not_the_current_one(gpu):
    """Weights, rows and optimiser on the second GPU, the first the current one: as torch's operations run there."""
    from nv_genai_amd.training.optim import AdamW

    got = []
    for dev in (gpu, torch.device("cuda:1")):
        torch.manual_seed(0)
        w = {n: (0.1 * torch.randn(s)).to(dev).requires_grad_() for n, s in dict(n=(256,), i=(1024, 256), b=(1024,), o=(256, 512)).items()}
        x, y = torch.randn(48, 256).to(BF).to(dev), torch.randint(0, 256, (48,)).to(dev)
        opt = AdamW(list(w.values()), lr=0.1)
        h = fused.swiglu(fused.linear(fused.rms_norm(x, w["n"], 1e-5), w["i"], w["b"]))
        fused.cross_entropy_sum(h @ w["o"].to(BF).t(), y, True).backward()
        assert opt._covers() and torch.cuda.current_device() == 0
        opt.step(max_norm=1.0)
        got.append([t.detach().cpu() for t in w.values()])
    assert all(torch.equal(a, b) for a, b in zip(*got))


def test_many_rows_change_only_the_matrices(gpu, monkeypatch):
    """An encoder's step over 5,160 rows: its loss and its embeddings' gradients are the torch operations' to the bit, since a weight's
    gradient moves nothing behind it; the projections' are fp32 sums in another order, rounded to bf16 (2^-8 at most, here of their norm)."""
    from nv_genai_amd import ops
    from nv_genai_amd.models.config import EncoderConfig
    from nv_genai_amd.models.encoder import EncoderModel

    m = EncoderModel(EncoderConfig(name="t", vocab_size=1000, hidden=256, layers=2, heads=4, ffn=512, max_position=136), gpu, seed=3)
    ids, got, calls = torch.randint(0, 1000, (40, 129), device=gpu), [], []
    monkeypatch.setattr(ops, "weight_grad_covers", lambda *a, f=ops.weight_grad_covers: f(*a) and not calls.append(a))
    for fused_too in (True, False):
        if not fused_too:
            _without(monkeypatch)
        P = Fn.trainable_params(m, "encoder")
        with torch.autocast("cuda", dtype=BF):
            loss = Fn.encoder_embed(m, ids, torch.ones_like(ids), P).pow(3).sum()
        loss.backward()
        got.append((loss.detach(), {k: p.grad for k, p in P.items()}))
    (la, ga), (lb, gb) = got
    assert len(calls) == 8 and torch.equal(la, lb)   # four projections a layer
    for k in ga:
        if not isinstance(k, tuple) and "emb_ln" not in k:
            assert torch.equal(ga[k], gb[k]), k
        elif ga[k].dim() == 2:
            assert ((ga[k] - gb[k]).norm() <= 2 ** -8 * gb[k].norm()), k
