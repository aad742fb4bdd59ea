"""Encoder forwards that the native call takes or leaves to the steps in Python."""
import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu


def _model(dev):
    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel

    return EncoderModel(encoder_config("encoder-tiny"), dev, seed=2)


def _tokens(dev, n):
    """n tokens in sequences of up to 60."""
    g = torch.Generator().manual_seed(n)
    ids = torch.randint(0, 1000, (n,), generator=g, dtype=torch.int32)
    cu = torch.tensor([*range(0, n, 60), n], dtype=torch.int32)
    return ids.to(dev), (torch.arange(n) % 60).int().to(dev), cu.to(dev), 60


def _close(a, b):
    """Two forms that round to bf16 at different places, some 2^-9 of a value each, through a few layers."""
    assert a.shape == b.shape and ((a - b).norm() / b.norm()).item() < 2e-2


def _native(m, t):
    """What the model's forward asks first: the hidden rows, or None for weights that the native call leaves."""
    return ops.encoder_forward(t[0], t[1], None, t[2], t[3], m.word, m.pos, m.type, m.emb_ln, m.layers, m.cfg.heads, m.cfg.eps, m.scale, covered_only=True)


def _odd(t):
    return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)


def _apart(t):
    return torch.stack([t, t], -1)[..., 0]


@pytest.mark.parametrize("n", [30, 1200])
@pytest.mark.parametrize("what,how", [(w, _odd) for w in ("word", "pos", "type", "emb_ln", "wqkv", "bqkv", "bi", "ln1_g", "wo2")]
                         + [(w, _apart) for w in ("word", "pos", "type", "wqkv")])
def test_weights_of_any_layout(gpu, n, what, how):
    """Views that do not begin at 16 bytes, and tables and projections whose elements lie apart."""
    m, t = _model(gpu), _tokens(gpu, n)
    want = m.forward(*t)
    assert torch.equal(m._pool(_native(m, t), t[2]), want)
    if what in m.layers[0]:
        m.layers[0][what] = how(m.layers[0][what])
    else:
        setattr(m, what, tuple(how(w) for w in m.emb_ln) if what == "emb_ln" else how(getattr(m, what)))
    assert not ops.encoder_covers(m.word, m.layers, m.cfg.heads, (m.pos, m.type, *m.emb_ln)) and _native(m, t) is None
    _close(m.forward(*t), want)


@pytest.mark.parametrize("name,size", [("wi", (192, 64)), ("bi", (64,))])
def test_weights_of_other_shapes_are_not_covered(gpu, name, size):
    m = _model(gpu)
    tables = (m.pos, m.type, *m.emb_ln)
    assert ops.encoder_covers(m.word, m.layers, m.cfg.heads, tables)
    m.layers[1][name] = torch.zeros(size, dtype=torch.bfloat16, device=gpu)
    assert not ops.encoder_covers(m.word, m.layers, m.cfg.heads, tables) and _native(m, _tokens(gpu, 30)) is None
    with pytest.raises(RuntimeError):   # asked for by name it raises
        ops.encoder_forward(*_tokens(gpu, 30)[:2], None, *_tokens(gpu, 30)[2:], m.word, m.pos, m.type, m.emb_ln, m.layers, m.cfg.heads, m.cfg.eps, m.scale)
    with pytest.raises(RuntimeError):
        m.forward(*_tokens(gpu, 30))


def test_one_type_for_all_tokens(gpu):
    m, t = _model(gpu), _tokens(gpu, 30)
    one = torch.ones(1, device=gpu, dtype=torch.int32)
    _close(m.forward(*t, one), m.forward(*t, one.expand(30).contiguous()))


def test_other_threads_run_during_the_launches(gpu):
    """The native call gives up the interpreter lock: with switching by time off, a waiting thread can only run while it does."""
    import sys
    import threading

    m, (ids, pos, cu, longest) = _model(gpu), _tokens(gpu, 30)
    w = [L[n] for L in m.layers for n in ops.ENCODER_LAYER] * 40   # as long as a large model's
    go, ran = threading.Event(), []
    t = threading.Thread(target=lambda: (go.wait(), ran.append(1)))
    t.start()
    was = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        f = ops.kernels().encoder_forward
        go.set()
        for _ in range(20):
            f(ids, pos, None, cu, longest, m.word, m.pos, m.type, m.emb_ln[0], m.emb_ln[1], w, m.cfg.heads, m.cfg.eps, m.scale)
        seen = bool(ran)
    finally:
        sys.setswitchinterval(was)
    t.join()
    assert seen
