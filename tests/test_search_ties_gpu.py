"""Equal scores: of vectors that score the same the ones that come first in the index are returned, in that order, on every call."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N, D = 40_000, 256


def _vectors(nq, copies):
    """N vectors, `copies` of them the same, and queries that score highest with those."""
    g = torch.Generator(device="cuda").manual_seed(nq + copies)
    X = torch.randn(N, D, device="cuda", generator=g)
    same = torch.randperm(N, device="cuda", generator=g)[:copies]
    X[same] = X[same[0]].clone()
    return X, same, X[same[:1]].expand(nq, D).contiguous()


# register lists of 4 to 16 and 8, scores with their selection; 9,000 copies are more than the selection ranks at once
@pytest.mark.parametrize("nq,k", [(1, 1), (1, 4), (5, 16), (20, 25), (40, 8), (40, 25), (100, 4), (3, 200)])
@pytest.mark.parametrize("copies", [300, 9000])
def test_flat(gpu, nq, k, copies):
    from nv_genai_amd.index.flat import FlatIndex

    X, same, q = _vectors(nq, copies)
    idx = FlatIndex(D, "ip", "cuda", capacity=N)
    idx.add(X, torch.arange(N))
    want = same.sort().values[:k]
    for _ in range(3):
        assert (idx.search(q, k)[1] == want).all()


@pytest.mark.parametrize("nq,k", [(1, 4), (5, 32), (40, 8), (40, 32)])
@pytest.mark.parametrize("copies", [300, 9000])
def test_lists(gpu, nq, k, copies):
    from nv_genai_amd.index.ivf import IVFFlatIndex

    X, same, q = _vectors(nq, copies)
    idx = IVFFlatIndex(D, 16, 8, "ip", "cuda")
    idx.train(X[:8000], iters=2, seed=1)
    idx.add(X, torch.arange(N))
    idx.search(q, k)   # brings the rows in list order
    want = idx.ids[torch.isin(idx.ids, same).nonzero().squeeze(1)[:k]]
    for _ in range(3):
        assert (idx.search(q, k)[1] == want).all()
