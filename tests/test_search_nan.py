"""Vectors that are no numbers are found by no search, however many results it asks for."""
import pytest
import torch

from nv_genai_amd import ops
from nv_genai_amd.index.flat import FlatIndex
from nv_genai_amd.ops import reference


def _index(dev, metric, dim=96):
    g = torch.Generator().manual_seed(4)
    X = torch.randn(700, dim, generator=g)
    bad = torch.arange(0, 700, 7)
    X[bad] = float("nan")
    X[bad[::2]] *= -1   # NaN of either sign
    idx = FlatIndex(dim, metric, dev)
    idx.add(X)
    return idx, set(bad.tolist()), torch.randn(5, dim, generator=g)


def _check(idx, bad, q, k):
    v, i = idx.search(q.to(idx.X.device), k)
    live = 700 - len(bad)
    assert v.shape == (5, k) and bool(torch.isfinite(v[:, :live]).all()) and bool((v[:, live:] == float("-inf")).all())
    for row in i[:, :live].tolist():
        assert len(set(row)) == min(k, live) and not bad & set(row) and -1 not in row
    assert bool((i[:, live:] == -1).all())


@pytest.mark.parametrize("metric", ["ip", "cosine", "l2"])
@pytest.mark.parametrize("k", [4, 100, 640])
def test_flat(metric, k):
    _check(*_index("cpu", metric), k)


# dimensions of the native search, and those of a score matrix
@pytest.mark.gpu
@pytest.mark.parametrize("dim", [128, 96])
@pytest.mark.parametrize("metric", ["ip", "cosine", "l2"])
@pytest.mark.parametrize("k", [4, 25, 200])
def test_flat_gpu(gpu, dim, metric, k):
    _check(*_index(gpu, metric, dim), k)


def test_lists():
    g = torch.Generator().manual_seed(5)
    X = torch.randn(300, 32, generator=g)
    X[::3] = float("nan")
    q = torch.randn(2, 32, generator=g)
    beg, end = torch.tensor([0, 100, 150]), torch.tensor([100, 150, 300])
    v, i = reference.ivf_search_topk(q, X, None, 1.0, torch.tensor([[0, 2], [1, 2]]), beg, end, 80)
    assert bool(torch.isfinite(v).all()) and bool((i % 3 != 0).all()) and bool((v.diff() <= 0).all())
    assert torch.equal(v, ops.ivf_search_topk(q, X, None, 1.0, torch.tensor([[0, 2], [1, 2]]), beg, end, 150, 80)[0])
