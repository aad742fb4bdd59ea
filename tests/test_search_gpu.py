"""Fused vector-search kernels on the GPU against fp32 PyTorch references: the MFMA score +
per-block register top-k (flat search, K13) and the batched IVF list scan over (list,
query-chunk) work items (K14)."""
import pytest
import torch

from nv_genai_amd import ops
from nv_genai_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _data(N, D, nq, seed, dev):
    g = torch.Generator(device="cpu").manual_seed(seed)
    X = torch.nn.functional.normalize(torch.randn(N, D, generator=g), dim=1).to(dev, torch.bfloat16)
    Q = torch.nn.functional.normalize(torch.randn(nq, D, generator=g), dim=1).to(dev, torch.bfloat16)
    return X, Q


def _check_topk(v, r, X, Q, bias, scale, k):
    """Returned scores are the exact scores of the returned rows, sorted, and no row outside
    the result scores above the k-th (ties aside)."""
    S = ref.score(Q, X, bias, scale)                       # fp32 reference [nq, N]
    rv, _ = torch.topk(S, k, dim=1)
    assert v.shape == (Q.shape[0], k) and r.shape == (Q.shape[0], k)
    fin = torch.isfinite(rv)
    assert torch.equal(torch.isfinite(v), fin)
    assert torch.allclose(v[fin], rv[fin], atol=2e-3, rtol=1e-3)
    assert bool((r[~fin] == -1).all()) and bool((r[fin] >= 0).all())
    got = torch.gather(S, 1, r.clamp_min(0))
    assert torch.allclose(got[fin], v[fin], atol=2e-3, rtol=1e-3)
    assert bool((v[:, :-1] >= v[:, 1:]).all())
    for row in r.tolist():                                  # distinct rows
        live = [x for x in row if x >= 0]
        assert len(set(live)) == len(live)


@pytest.mark.parametrize("N,D,nq,k", [(1000, 128, 1, 4), (100_003, 1024, 1, 4), (100_003, 1024, 8, 8),
                                      (50_000, 384, 33, 16), (70_001, 1024, 64, 4), (70_001, 1024, 100, 8),
                                      (3, 128, 5, 4), (20_000, 1024, 17, 1),
                                      # LDS-DMA form: 256- and 512-dim chunks, partial last tile
                                      (30_011, 768, 16, 16), (20_000, 2048, 3, 4), (5_000, 256, 2, 4),
                                      (777, 1024, 16, 8)])
def test_search_topk_matches_reference(gpu, N, D, nq, k):
    X, Q = _data(N, D, nq, N + nq, gpu)
    bias = torch.zeros(N, device=gpu)
    bias[::7] = float("-inf")                                # tombstones
    v, r = ops.search_topk(Q, X, bias, 1.0, k)
    _check_topk(v, r, X, Q, bias, 1.0, min(k, N))


def test_search_topk_l2_bias_and_no_bias(gpu):
    X, Q = _data(30_000, 256, 12, 5, gpu)
    bias = -ops.row_sqnorm(X)
    v, r = ops.search_topk(Q, X, bias, 2.0, 8)
    _check_topk(v, r, X, Q, bias, 2.0, 8)
    v, r = ops.search_topk(Q, X, None, 1.0, 8)
    _check_topk(v, r, X, Q, None, 1.0, 8)


def test_search_topk_large_k_falls_back(gpu):
    X, Q = _data(10_000, 128, 4, 9, gpu)
    v, r = ops.search_topk(Q, X, None, 1.0, 50)                # beyond the register lists
    _check_topk(v, r, X, Q, None, 1.0, 50)


@pytest.mark.parametrize("nq,nprobe,k", [(1, 16, 4), (8, 16, 8), (64, 16, 4), (70, 5, 8), (20, 16, 16)])
def test_ivf_scan_matches_reference(gpu, nq, nprobe, k):
    N, D, nlist = 60_000, 256, 64
    X, Q = _data(N, D, nq, 11 + nq, gpu)
    # list-sorted slab with uneven lists, some empty
    sizes = torch.randint(0, 2 * N // nlist, (nlist,), generator=torch.Generator().manual_seed(1))
    sizes[3] = 0
    sizes[10] = 0
    off = torch.cat([torch.zeros(1, dtype=torch.int64), sizes.cumsum(0)])
    Xs = X[: int(off[-1])].contiguous()
    beg, end = off[:-1].to(gpu), off[1:].to(gpu)
    bias = torch.zeros(Xs.shape[0], device=gpu)
    bias[::5] = float("-inf")
    g = torch.Generator().manual_seed(nq)
    probes = torch.stack([torch.randperm(nlist, generator=g)[:nprobe] for _ in range(nq)]).to(gpu)
    probes[0, 0] = 3                                            # an empty list is probed
    v, r = ops.ivf_search_topk(Q, Xs, bias, 1.0, probes, beg, end, int(sizes.max()), k)
    rv, rr = ref.ivf_search_topk(Q, Xs, bias, 1.0, probes, beg, end, k)
    fin = torch.isfinite(rv)
    assert torch.equal(torch.isfinite(v), fin)
    assert torch.allclose(v[fin], rv[fin], atol=2e-3, rtol=1e-3)
    S = ref.score(Q, Xs, bias, 1.0)
    assert torch.allclose(torch.gather(S, 1, r.clamp_min(0))[fin], v[fin], atol=2e-3, rtol=1e-3)
    assert bool((r[~fin] == -1).all())


def test_ivf_scan_splits_past_item_limit(gpu):
    """nlist 4,096 with 1,100 queries is 4,096 x 18 = 73,728 (list, query-chunk) items, past
    the scan launch's 65,535: the queries run in two sub-batches and still match the reference."""
    N, D, nlist, nq, nprobe, k = 40_000, 128, 4096, 1100, 4, 4
    X, Q = _data(N, D, nq, 23, gpu)
    sizes = torch.randint(0, 2 * N // nlist, (nlist,), generator=torch.Generator().manual_seed(2))
    off = torch.cat([torch.zeros(1, dtype=torch.int64), sizes.cumsum(0)])
    Xs = X[: int(off[-1])].contiguous()
    beg, end = off[:-1].to(gpu), off[1:].to(gpu)
    g = torch.Generator().manual_seed(5)
    probes = torch.stack([torch.randperm(nlist, generator=g)[:nprobe] for _ in range(nq)]).to(gpu)
    assert nlist * -(-nq // 64) > ops.IVF_MAX_ITEMS
    v, r = ops.ivf_search_topk(Q, Xs, None, 1.0, probes, beg, end, int(sizes.max()), k)
    rv, rr = ref.ivf_search_topk(Q, Xs, None, 1.0, probes, beg, end, k)
    fin = torch.isfinite(rv)
    assert v.shape == (nq, k) and torch.equal(torch.isfinite(v), fin)
    assert torch.allclose(v[fin], rv[fin], atol=2e-3, rtol=1e-3)


def test_ivf_index_recall_vs_flat_nlist64_nprobe16(gpu):
    """The reference's GPU_IVF_FLAT setting (nlist 64, nprobe 16) on clustered data: batched
    IVF search finds >= 95% of the flat index's top-10 (RetrievalAugmentedGeneration/common/
    utils.py:198-203)."""
    from nv_genai_amd.index.flat import FlatIndex
    from nv_genai_amd.index.ivf import IVFFlatIndex

    g = torch.Generator().manual_seed(7)
    centers = torch.randn(200, 512, generator=g)
    X = centers[torch.randint(0, 200, (200_000,), generator=g)] + 0.4 * torch.randn(200_000, 512, generator=g)
    Q = X[torch.randint(0, 200_000, (48,), generator=g)] + 0.1 * torch.randn(48, 512, generator=g)
    ids = torch.arange(200_000) * 3 + 1
    flat = FlatIndex(512, "cosine", gpu, capacity=200_000)
    flat.add(X, ids)
    ivf = IVFFlatIndex(512, nlist=64, nprobe=16, metric="cosine", device=gpu)
    ivf.train(X[:50_000])
    ivf.add(X, ids)
    assert len(ivf) == 200_000
    fv, fi = flat.search(Q, 10)
    iv, ii = ivf.search(Q, 10)
    recall = sum(len(set(a) & set(b)) for a, b in zip(ii.tolist(), fi.tolist())) / fi.numel()
    assert recall >= 0.95, recall
    assert ivf.remove(ii[:, 0].tolist()) == len(set(ii[:, 0].tolist()))
    assert len(ivf) == 200_000 - len(set(ii[:, 0].tolist()))
    _, ii2 = ivf.search(Q, 10)
    assert not set(ii[:, 0].tolist()) & set(ii2.reshape(-1).tolist())


def _check_found(v, i, S, k):
    """Scores sorted and those of the returned ids (row = id); none outside the result is larger. Sums of at most 1,024
    products of bf16 values in fp32: 1,024 * 2^-24 of the summed magnitudes, which are at most 4 here."""
    S = S.double()
    rv = torch.topk(S, k, dim=1).values
    fin = torch.isfinite(rv)
    assert torch.equal(torch.isfinite(v), fin) and torch.equal(i >= 0, fin)
    assert bool((v[fin].double() - rv[fin]).abs().max() <= 2.5e-4) if fin.any() else True
    assert bool((torch.gather(S, 1, i.clamp_min(0))[fin] - v[fin].double()).abs().max() <= 2.5e-4) if fin.any() else True
    for row in i.tolist():
        live = [x for x in row if x >= 0]
        assert len(set(live)) == len(live)


# one tile and less, tile and run edges, each unit width (512, 384, 256, 128 dims), each query group count, lists and
# scores (k above 16, or above 8 with more than 32 queries), several query groups
@pytest.mark.parametrize("N,D,nq,k,metric", [(1, 128, 1, 1, "ip"), (127, 1024, 3, 25, "cosine"), (129, 384, 16, 4, "l2"),
                                             (33_000, 1024, 17, 16, "cosine"), (32_769, 768, 33, 8, "l2"), (40_001, 768, 64, 9, "ip"),
                                             (20_003, 512, 31, 17, "cosine"), (9_001, 640, 65, 4, "cosine"), (8_193, 896, 5, 256, "l2"),
                                             (70_000, 1024, 48, 25, "l2"), (50_001, 384, 100, 16, "cosine")])
def test_flat_search_against_fp64(gpu, N, D, nq, k, metric):
    from nv_genai_amd.index.flat import FlatIndex

    g = torch.Generator().manual_seed(N + D + nq)
    idx = FlatIndex(D, metric, gpu, capacity=N)
    x = torch.randn(N, D, generator=g) / D ** 0.5
    idx.add(x)
    if N > 200:
        idx.remove(list(range(0, N, 9)))
    q = torch.randn(nq, D, generator=g).to(gpu) / D ** 0.5
    assert ops.search_covers(idx.X, k)
    v, i = idx.search(q, k)
    k = min(k, N)
    assert v.shape == i.shape == (nq, k)
    qb = idx._prep(q).to(torch.bfloat16).double()
    S = qb @ idx.X[:N].double().t()
    if metric == "l2":
        S = 2 * S - idx.X[:N].double().pow(2).sum(1) - q.double().pow(2).sum(1, keepdim=True)
    _check_found(v, i, S.masked_fill(idx.bias[:N] == float("-inf"), float("-inf")), k)


# rows around the ends of units, tiles and one tile a workgroup; groups of queries that are full, have one query, or fill a second item;
# register lists of each length, and scores
@pytest.mark.parametrize("D", [384, 768, 1024])
@pytest.mark.parametrize("N,nq,k", [(1, 17, 1), (16, 33, 4), (33, 64, 8), (8191, 49, 9), (8193, 32, 16), (24_577, 48, 17), (100_001, 17, 4),
                                    (100_001, 65, 25), (70_000, 129, 8), (300, 64, 256)])
def test_flat_search_of_many_against_fp64(gpu, D, N, nq, k):
    test_flat_search_against_fp64(gpu, N, D, nq, k, ("ip", "cosine", "l2")[N % 3])


# the other dimensions, with the ring's length of each: the last rows of a workgroup's units, one workgroup's only tile
@pytest.mark.parametrize("D", [128, 256, 512, 640, 896])
@pytest.mark.parametrize("N,nq,k", [(1, 17, 1), (33, 64, 8), (8193, 32, 16), (24_577, 48, 17), (100_001, 33, 4), (100_001, 65, 25), (70_000, 129, 8)])
def test_flat_search_of_many_of_other_dimensions_against_fp64(gpu, D, N, nq, k):
    test_flat_search_against_fp64(gpu, N, D, nq, k, ("ip", "cosine", "l2")[N % 3])


def test_flat_search_takes_what_it_was_measured_for(gpu):
    """17 to 32, 33 to 48 and 49 to 64 queries of each dimension with the queries in registers, but where the other kernel is faster."""
    took = {D: [ng for ng in (1, 2, 3, 4, 5) if ops.kernels().scan_wide_covers(D, ng)] for D in (64, *range(128, 1153, 128))}
    assert took == {64: [], 128: [], 256: [2, 4], 640: [3, 4], 1152: [], **{D: [2, 3, 4] for D in (384, 512, 768, 896, 1024)}}


def test_flat_search_equal_scores_and_strided_queries(gpu):
    """More equal scores than the selection sorts at once (one vector many times), with lists and with scores; queries
    that are every second row of a wider matrix."""
    from nv_genai_amd.index.flat import FlatIndex

    idx = FlatIndex(256, "ip", gpu, capacity=20_000)
    one = torch.randn(1, 256) / 16
    x = one.repeat(20_000, 1)
    x[5] = 0
    idx.add(x)
    big = torch.randn(12, 300, device=gpu) / 16
    q = big[::2, 7:263]
    S = q.to(torch.bfloat16).double() @ idx.X[: idx.n].double().t()
    for k in (4, 40, 256):
        v, i = idx.search(q, k)
        _check_found(v, i, S, k)
    idx.remove(list(range(19_998)))                     # fewer live rows than asked for
    v, i = idx.search(q, 16)
    assert bool((i[:, 2:] == -1).all()) and bool(torch.isinf(v[:, 2:]).all()) and bool((i[:, :2] >= 0).all())


# queries per list of each group count, register lists of each length, more than 64 probing queries of one list
@pytest.mark.parametrize("D,nq,nprobe,k,metric", [(1024, 1, 16, 4, "cosine"), (256, 1, 1, 32, "l2"), (384, 16, 16, 25, "cosine"),
                                                  (768, 33, 7, 8, "ip"), (128, 150, 50, 4, "l2"), (256, 70, 50, 32, "cosine")])
def test_ivf_search_against_fp64(gpu, D, nq, nprobe, k, metric):
    from nv_genai_amd.index.ivf import IVFFlatIndex

    N, nlist = 21_011, 50
    g = torch.Generator().manual_seed(D + nq)
    idx = IVFFlatIndex(D, nlist, nprobe, metric, gpu)
    c = torch.randn(5, D, generator=g)
    x = (torch.randn(N, D, generator=g) + c[torch.randint(0, 5, (N,), generator=g)]) / (2 * D) ** 0.5   # uneven lists
    idx.train(x[:4000].to(gpu))
    idx.add(x.to(gpu), torch.arange(N))
    idx.remove(list(range(0, N, 11)))
    q = (x[:nq] + 0.02 * torch.randn(nq, D, generator=g)).to(gpu)
    v, i = idx.search(q, k)
    qb = idx._prep(q).to(torch.bfloat16)
    probes = torch.topk(qb.double() @ idx.centroids.to(torch.bfloat16).double().t(), nprobe, dim=1).indices
    lists = torch.repeat_interleave(torch.arange(nlist), idx.offsets[1:] - idx.offsets[:-1]).to(gpu)
    S = qb.double() @ idx.X.double().t()
    if metric == "l2":
        S = 2 * S - idx.X.double().pow(2).sum(1) - q.double().pow(2).sum(1, keepdim=True)
    seen = (lists[None, :, None] == probes[:, None, :]).any(-1) if nq <= 40 else torch.stack([torch.isin(lists, p) for p in probes])
    S = S.masked_fill(~seen | (idx.bias == float("-inf"))[None], float("-inf"))
    by_id = torch.full((nq, N), float("-inf"), dtype=torch.float64, device=gpu)
    by_id[:, idx.ids] = S
    _check_found(v, i, by_id, k)
