"""Two encoder passes a layer in turn against one after the other: the same operations on the same inputs, so the same bits, of the
results and of the gradients, in which each weight has two terms and their order is free."""
import pytest
import torch

from nv_genai_amd.training import functional as Fn


def _check(dev, grad_ckpt, rows):
    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel

    m = EncoderModel(encoder_config("encoder-tiny"), dev, seed=2)
    g = torch.Generator().manual_seed(4)

    def batch(B, S):
        lens = torch.randint(1, S + 1, (B, 1), generator=g)
        return torch.randint(0, 1000, (B, S), generator=g).to(dev), (torch.arange(S) < lens).long().to(dev)

    many, few = batch(4 * rows, 50), batch(rows, 9)
    got = []
    for paired in (True, False):
        P = Fn.trainable_params(m, "encoder")
        with torch.autocast(torch.device(dev).type, dtype=torch.bfloat16):
            one, two = (P, P) if grad_ckpt else Fn.half_params(P)
            if paired:
                p, q = Fn.encoder_embed_pair(m, (*many, two), (*few, one), grad_ckpt)
            else:
                q = Fn.encoder_embed(m, *few, one, grad_ckpt)
                p = Fn.encoder_embed(m, *many, two, grad_ckpt)
        (q @ p.t()).logsumexp(-1).sum().backward()
        got.append((p, q, {k: v.grad for k, v in P.items()}))
    (pa, qa, ga), (pb, qb, gb) = got
    assert torch.equal(pa, pb) and torch.equal(qa, qb)
    for k in gb:
        assert torch.equal(ga[k], gb[k]), k


@pytest.mark.parametrize("grad_ckpt", [False, True])
@pytest.mark.parametrize("rows", [1, 3])
def test_passes_in_turn_keep_the_bits(grad_ckpt, rows):
    _check("cpu", grad_ckpt, rows)


@pytest.mark.gpu
@pytest.mark.parametrize("grad_ckpt", [False, True])
@pytest.mark.parametrize("rows", [1, 3])
def test_passes_in_turn_keep_the_bits_gpu(gpu, grad_ckpt, rows):
    _check(gpu, grad_ckpt, rows)
