"""Tokens outside an encoder's tables are refused where they come in."""
import pytest
import torch

from nv_genai_amd.engine.embed_engine import EmbeddingEngine


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_tokens_outside_the_tables_raise(device):
    eng = EmbeddingEngine("encoder-tiny", device=device)
    n, longest = eng.cfg.vocab_size, eng.cfg.max_position
    for seqs, types in (([[5, n]], None), ([[7], [-1, 3]], None), ([[9] * (longest + 1)], None), ([[5, 6]], [[0, eng.cfg.type_vocab]])):
        with pytest.raises(IndexError):
            eng.embed_ids(seqs, types)
    out = eng.embed_ids([[0, n - 1], [9] * longest], [[0, eng.cfg.type_vocab - 1], [0] * longest])
    assert torch.isfinite(out).all()
