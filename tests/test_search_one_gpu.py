"""List search of one query in one launch (ivf_one_kernel) beside the launches of several: the same query twice takes those. Sums, their order
and the order of results are the same, so are the bits."""
import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu
METRIC = {"ip": 0, "cosine": 1, "l2": 2}


def _both(q, X, bias, ids, cent, beg, end, metric, nprobe, k):
    one = ops.ivf_search(q, X, bias, ids, cent, beg, end, metric, nprobe, k)
    two = ops.ivf_search(q.expand(2, -1), X, bias, ids, cent, beg, end, metric, nprobe, k)
    assert torch.equal(one[1][0], two[1][0]) and torch.equal(one[0][0], two[0][0])
    return one


# lists of any sizes, empty ones too, and in any order of rows; runs that end with a list, in its last tile and behind several short ones
@pytest.mark.parametrize("D,rows,nlist,nprobe,k,metric", [
    (1024, 1, 1, 1, 1, "cosine"), (384, 31, 3, 3, 4, "l2"), (768, 33, 64, 64, 5, "ip"), (512, 5000, 64, 16, 8, "cosine"),
    (1024, 33_000, 128, 7, 9, "l2"), (384, 40_001, 256, 31, 25, "cosine"), (768, 70_003, 170, 170, 32, "ip"), (512, 100_000, 37, 1, 4, "l2")])
def test_same_as_of_several(gpu, D, rows, nlist, nprobe, k, metric):
    assert ops.kernels().ivf_one_covers(1, nlist, D, k) and not ops.kernels().ivf_one_covers(2, nlist, D, k)
    g = torch.Generator().manual_seed(D + rows)
    X = (torch.randn(rows, D, generator=g) / D ** 0.5).to(torch.bfloat16)
    X[rows // 2:] = torch.where(torch.rand(rows - rows // 2, 1, generator=g) < 0.1, X[:1], X[rows // 2:])   # equal scores
    bias = -X.float().pow(2).sum(1) if metric == "l2" else torch.zeros(rows)
    bias[torch.rand(rows, generator=g) < 0.1] = float("-inf")   # removed
    ids = torch.randperm(rows, generator=g)
    cut = torch.randint(0, rows + 1, (nlist - 1,), generator=g).sort().values
    off = torch.cat([torch.tensor([0]), cut, torch.tensor([rows])])
    order = torch.randperm(nlist, generator=g)
    cent = torch.randn(nlist, D, generator=g)
    q = torch.randn(3, 2 * D, generator=g)[1:2, D:] / D ** 0.5   # a row of a wider matrix
    X, bias, ids, cent, q, beg, end = (t.to(gpu) for t in (X, bias, ids, cent, q, off[:-1][order], off[1:][order]))
    v, i = _both(q, X, bias, ids, cent, beg, end, metric, nprobe, min(k, rows))
    qf = q.float()
    qb = (qf / qf.norm() if metric == "cosine" else qf).to(torch.bfloat16).double()
    probes = torch.topk(qb @ cent.to(torch.bfloat16).double().t(), nprobe).indices[0].tolist()
    at = torch.cat([torch.arange(int(beg[p]), int(end[p]), device=gpu) for p in probes])
    at = at[torch.isfinite(bias[at])]
    s = X[at].double() @ qb[0]
    if metric == "l2":
        s = 2 * s - X[at].double().pow(2).sum(1) - q.double().pow(2).sum()
    n = min(k, at.numel(), rows)
    assert bool((i[0, n:] == -1).all()) and bool((v[0, n:] == float("-inf")).all())
    # at most 1,024 products of bf16 in fp32: 1,024 x 2^-24 of the summed magnitudes, at most 4 here
    assert n == 0 or bool((v[0, :n].double() - torch.topk(s, n).values).abs().max() <= 2.5e-4)


def test_which_calls_it_takes(gpu):
    took = [(D, n) for D in range(128, 1025, 128) for n in (1, 128, 129, 256, 257) if ops.kernels().ivf_one_covers(1, n, D, 32)]
    assert took == [(D, n) for D in (384, 512, 768, 1024) for n in (1, 128, 129, 256) if n * D <= 131072]
    assert not ops.kernels().ivf_one_covers(1, 64, 1024, 33)
