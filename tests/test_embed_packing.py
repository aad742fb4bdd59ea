"""An encoder's packed batch, written by native code, against the lists that it stands for."""
import numpy as np
import pytest
import torch

from nv_genai_amd._native import rt
from nv_genai_amd.engine.embed_engine import EmbeddingEngine

SEQS = [[5, 9, 2], [7], [], [3, 3, 3, 3, 3], [1, 8]]


@pytest.mark.parametrize("form", [list, tuple, np.array, lambda s: np.array(s, dtype=np.int64), torch.tensor, lambda s: [float(t) for t in s]])
@pytest.mark.parametrize("types", [None, [[0] * len(s) for s in SEQS], [[1] * len(s) for s in SEQS]])
@pytest.mark.parametrize("batch", [[0], [2], [0, 1], [1, 4, 0, 3], [4, 3, 2, 1, 0]])
def test_packed_batch(form, types, batch):
    eng = EmbeddingEngine("encoder-tiny", device="cpu")
    seqs = [form(s) if len(s) or form is list else s for s in SEQS]
    tok = sum(len(SEQS[b]) for b in batch)
    ids, pos, cu, tt, rows, longest = eng._packed(seqs, batch, tok, types)
    assert ids.tolist() == [t for b in batch for t in SEQS[b]] and pos.tolist() == [p for b in batch for p in range(len(SEQS[b]))]
    assert cu.tolist() == np.cumsum([0] + [len(SEQS[b]) for b in batch]).tolist() and rows.tolist() == batch
    assert longest == max(len(SEQS[b]) for b in batch)
    assert tt is None if types is None else tt.tolist() == [t for b in batch for t in types[b]]
    assert all(t.dtype == torch.int32 for t in (ids, pos, cu)) and rows.dtype == torch.int64


def test_refused_batches():
    eng = EmbeddingEngine("encoder-tiny", device="cpu")
    with pytest.raises(RuntimeError):
        eng.embed_ids([[1, 1 << 40]])
    with pytest.raises(ValueError):
        eng.embed_ids([["a"]])
    buf = np.zeros(16, dtype=np.int32)
    ok = (SEQS, [0], None, buf, 4, 8, 12, 16, 3)
    assert rt.pack_tokens(*ok) == (3, 2, 9, 2 ** 31 - 1, -2 ** 31) and buf.tolist() == [0, 0, 0, 0, 0, 3, 0, 0, 5, 9, 2, 0, 0, 1, 2, 0]
    for at, bad in ((1, [9]), (4, 15), (4, -1), (5, 14), (6, 1 << 62), (8, 2), (8, 9), (3, buf[::2]), (3, buf.astype(np.int64)), (2, [[0]]), (2, [])):
        args = list(ok)
        args[at] = bad
        with pytest.raises(ValueError):
            rt.pack_tokens(*args)
