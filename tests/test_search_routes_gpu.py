"""Searches of many queries: which kernels take them, and that both give the same."""
import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu


def _spy(monkeypatch, name):
    calls, f = [], getattr(ops, name)
    monkeypatch.setattr(ops, name, lambda *a: calls.append(1) or f(*a))
    return calls


def _same(a, b):
    """Scores to the order of their fp32 sums, and for cosine to one element of a query that the norm's last bit rounds to the
    other bf16 neighbour: 2^-8 of a product of two elements of unit vectors, which stay below 0.16 at 1,024 dimensions. Ids
    but for neighbours whose scores that turns round."""
    assert torch.allclose(a[0], b[0], rtol=1e-5, atol=1e-4) and (a[1] == b[1]).float().mean() > 0.999


@pytest.mark.parametrize("nq,rows,k,here", [(4096, 10_728, 4, True), (4096, 10_730, 4, False), (4096, 10_730, 9, True),
                                            (4096, 10_730, 8, False), (4033, 10_730, 1, False), (4032, 10_730, 1, True)])
@pytest.mark.parametrize("metric", ["cosine", "l2"])
def test_flat_of_many_queries(gpu, monkeypatch, nq, rows, k, here, metric):
    from nv_genai_amd.index.flat import FlatIndex

    g = torch.Generator(device="cuda").manual_seed(rows + k)
    idx = FlatIndex(1024, metric, "cuda", capacity=rows)
    idx.add(torch.randn(rows, 1024, device=gpu, generator=g), torch.arange(rows) + 7)
    idx.remove([9, 11])
    q = torch.randn(nq, 1024, device=gpu, generator=g)
    calls = _spy(monkeypatch, "flat_search")
    a = idx.search(q, k)
    assert bool(calls) == here
    monkeypatch.setattr(ops, "search_many", lambda *a: here)   # the other route
    _same(idx.search(q, k), a)


def test_flat_of_many_short_vectors_or_few_queries(gpu):
    assert not ops.search_many(10_000, 10 ** 7, 128, 4) and not ops.search_many(64, 10 ** 8, 1024, 4)


# points that were timed, the faster one by more than a twentieth each
@pytest.mark.parametrize("D,rows,nq,k,topk", [(256, 300_000, 256, 4, True), (256, 100_000, 128, 4, False), (384, 300_000, 512, 4, True), (384, 100_000, 256, 4, False),
                                              (512, 1_000_000, 256, 4, True), (512, 300_000, 128, 4, False), (640, 1_000_000, 512, 4, True),
                                              (640, 1_000_000, 128, 4, False), (768, 1_000_000, 1024, 4, True), (768, 1_000_000, 128, 4, False),
                                              (768, 300_000, 192, 4, False), (896, 300_000, 256, 4, False), (896, 1_000_000, 128, 4, False),
                                              (384, 300_000, 256, 8, True), (640, 300_000, 256, 8, True), (768, 300_000, 192, 8, False),
                                              (896, 100_000, 512, 8, False), (512, 100_000, 256, 9, False), (1024, 1_000_000, 512, 4, False)])
def test_flat_line_agrees_with_the_measurements(gpu, D, rows, nq, k, topk):
    assert ops.search_many(nq, rows, D, k) == topk


@pytest.mark.parametrize("nq,nprobe,k,here", [(1024, 2, 4, False), (1024, 2, 9, True), (700, 2, 4, True)])
def test_lists_of_many_queries(gpu, monkeypatch, nq, nprobe, k, here):
    """Two lists of 100,000 x 1,024 rows, both probed."""
    from nv_genai_amd.index.ivf import IVFFlatIndex

    g = torch.Generator(device="cuda").manual_seed(nq + k)
    X = torch.randn(200_000, 1024, device=gpu, generator=g)
    idx = IVFFlatIndex(1024, 2, nprobe, "l2", "cuda")
    idx.train(X[:2000], iters=1, seed=1)
    idx.add(X, torch.arange(200_000) + 7)
    q = torch.randn(nq, 1024, device=gpu, generator=g)
    calls = _spy(monkeypatch, "ivf_search")
    a = idx.search(q, k)
    assert bool(calls) == here
    if k <= 8:   # the other route; above, it goes query by query
        monkeypatch.setattr(ops, "search_many_lists", lambda *a: here)
        _same(idx.search(q, k), a)


def test_lists_that_stay(gpu):
    """Short lists, short vectors, few probes."""
    for rows, D, nlist, nprobe in ((300_000, 1024, 64, 64), (1_000_000, 512, 64, 64), (1_000_000, 1024, 64, 4)):
        assert not ops.search_many_lists(4096, rows, D, 4, nlist, nprobe)
    assert ops.search_many_lists(4096, 1_000_000, 1024, 4, 64, 8) and ops.search_many_lists(256, 1_000_000, 1024, 8, 64, 64)
