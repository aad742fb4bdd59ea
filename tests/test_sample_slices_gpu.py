"""Sampling by slices of a row beside the passes over whole rows, which a batch too large for slices takes: the tokens are the same, the
log-probabilities up to the order of their sums."""
import pytest
import torch

from nv_genai_amd import ops
from nv_genai_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
# temperature, top_k, top_p
HOW = [(0.0, 0, 1.0), (0.2, 0, 0.7), (0.2, 40, 0.95), (1.0, 0, 0.9), (1.0, 1, 1.0), (1.0, 0, 1.0), (0.7, 50, 1.0), (0.05, 3, 0.5), (0.2, 0, 0.9999999)]


def _rows(V, g):
    """Logits as a trained model has them, flat ones, a slice that lists too many, equal largest values, and rows with and of -inf."""
    x = 2.5 * torch.randn(9, V, device="cuda", generator=g)
    x[0, V // 3] += 12
    x[1] *= 0.01
    x[2, :2048] = x[2].max() - 0.1 * torch.rand(min(2048, V), device="cuda", generator=g)[: x[2, :2048].numel()]
    x[3, [5, 2047, 2048, V - 1]] = x[3].max() + 1
    x[4, V // 2:] = float("-inf")
    x[5] = float("-inf")
    x[6] = float("-inf")
    x[6, V - 1] = 3.0
    x[7, 100:] = x[7, :1].clone()
    x[8, 7] = float("nan")
    return x


@pytest.mark.parametrize("V", [22_529, 24_576, 24_580, 30_721, 32_768, 47_104, 47_105, 50_257, 120_836, 128_256, 262_144])
@pytest.mark.parametrize("temp,k,p", HOW)
def test_same_tokens(gpu, V, temp, k, p):
    n = -(-V // 2048)
    g = torch.Generator(device="cuda").manual_seed(V)
    x = _rows(V, g)
    B = 4096 // n + 1   # one row too many
    assert B > len(x)
    full = torch.cat([x, x[:1].expand(B - len(x), V)]) if B * V < 1 << 27 else None
    if full is None:
        pytest.skip("a batch of several GiB")

    def run(lg, seed, first=0):
        b = lg.shape[0]
        arg = (torch.full((b,), temp, device=gpu), torch.full((b,), k, dtype=torch.int32, device=gpu), torch.full((b,), p, device=gpu))
        at = first + torch.arange(b, device=gpu)
        return ops.sample(lg, *arg, seed + at, at)

    for seed in (0, 1000):
        # 4 rows at a time: more are not sliced below 24 slices
        ta, la = (torch.cat(t) for t in zip(*(run(x[i:i + 4].clone(), seed, i) for i in range(0, len(x), 4))))
        tb, lb = run(full.clone(), seed)
        tb, lb = tb[: len(x)], lb[: len(x)]
        assert torch.equal(ta, tb)
        # sums of up to 262,144 terms in fp32, in two orders: about sqrt(V) 2^-24 of them
        assert torch.allclose(la, lb, rtol=1e-5, atol=1e-5, equal_nan=True)


def test_a_penalty_changes_the_row_first(gpu):
    V = 32_000
    g = torch.Generator(device="cuda").manual_seed(1)
    x = 2.5 * torch.randn(3, V, device="cuda", generator=g)
    hist = x.topk(3, 1).indices.int()
    pen = torch.tensor([1.0, 5.0, 1.3], device=gpu)
    arg = (torch.zeros(3, device=gpu), torch.zeros(3, dtype=torch.int32, device=gpu), torch.ones(3, device=gpu), torch.arange(3, device=gpu),
           torch.arange(3, device=gpu))
    want = x.clone()
    for r in range(3):
        v = want[r, hist[r].long()]
        want[r, hist[r].long()] = torch.where(v > 0, v / pen[r], v * pen[r])
    tok, lp = ops.sample(x.clone(), *arg, pen, hist)
    assert torch.equal(tok.long(), want.argmax(1))
    assert torch.allclose(lp, torch.log_softmax(want.double(), 1).max(1).values.float(), atol=1e-5)


def test_the_same_draw_again(gpu):
    """top-k and top-p together: the target of top-p comes of a sum of what top-k keeps, so that must add up in one order. Rows whose
    target lies at the boundary between two values, give or take an ulp, draw again what they drew."""
    V, K, B = 128_256, 1000, 64
    g = torch.Generator().manual_seed(5)
    near = torch.randperm(V, generator=g)[:K + 200]
    x = torch.full((V,), -30.0)
    x[near] = -6 * torch.rand(K + 200, generator=g)
    w = x[near].double().sort(descending=True).values[:K].exp()
    at = torch.randint(50, K - 200, (B,), generator=g)
    p = (w.cumsum(0) / w.sum())[at].float() + (torch.arange(B) % 9 - 4) * 2.0 ** -25
    x = x.expand(B, V).contiguous().to(gpu)
    arg = (torch.ones(B, device=gpu), torch.full((B,), K, dtype=torch.int32, device=gpu), p.to(gpu))
    row = torch.arange(B, device=gpu)
    for s in range(300):
        first = ops.sample(x, *arg, 1000 * s + row, row)[0]
        for _ in range(6):
            assert torch.equal(ops.sample(x, *arg, 1000 * s + row, row)[0], first)


def test_many_equal_largest_values(gpu):
    """A slice of more largest values than it can list, where the largest value less the lists' distance of 16 rounds to itself. The two
    seeds' noise is 16.6 for one of these values, which rounds up there, and so decides."""
    V, temp = 32_000, torch.tensor(1e-6)
    M = 400.0 * (1.0 / temp)
    assert M - 16.0 == M and M + 16.6 > M
    x = torch.randn(V)
    x[4096:4296] = 400.0
    x = x.expand(2, V).contiguous()
    arg = (temp.expand(2).contiguous(), torch.zeros(2, dtype=torch.int32), torch.full((2,), 0.9), torch.tensor([33_800, 77_349]), torch.zeros(2, dtype=torch.long))
    assert ref.sample(x, *arg)[0].tolist() == [4165, 4167]
    assert ops.sample(x.to(gpu), *(a.to(gpu) for a in arg))[0].tolist() == [4165, 4167]


@pytest.mark.parametrize("V", [1000, 128_256])
@pytest.mark.parametrize("temp,k,p", [(0.0, 0, 1.0), (1.0, 0, 1.0), (0.2, 40, 0.9)])
def test_rows_without_a_value(gpu, V, temp, k, p):
    """A row of NaN or of -inf gives the first token: there is none that it could draw."""
    x = torch.full((3, V), float("nan"), device=gpu)
    x[1] = float("-inf")
    x[2] = torch.arange(V, device=gpu) / V
    arg = (torch.full((3,), temp, device=gpu), torch.full((3,), k, dtype=torch.int32, device=gpu), torch.full((3,), p, device=gpu))
    tok, _ = ops.sample(x, *arg, torch.arange(3, device=gpu), torch.arange(3, device=gpu))
    assert tok[:2].tolist() == [0, 0] and 0 <= int(tok[2]) < V
