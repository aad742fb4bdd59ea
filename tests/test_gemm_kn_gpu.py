"""The 256 x 256 tiles: a projection's input gradient, x [M, K] . w [K, N] (gemm_kn.hip), and an
encoder's GELU(x . w [N, K]^T + bias) (gemm_nt.hip), against 64 bits."""
import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# rows around a tile and its quarters, K slices of one count and of several, stages that end anywhere in the ring's round, rows
# apart from one another
@pytest.mark.parametrize("M,N,K,apart", [(1, 256, 256, 0), (17, 256, 288, 8), (255, 512, 320, 0), (256, 256, 352, 0), (257, 256, 2080, 40),
                                         (513, 768, 4096, 0), (1024, 4096, 6144, 0), (130, 4096, 14336, 0), (300, 16640, 1056, 0),
                                         (4097, 4096, 512, 0)])
def test_gemm_kn(gpu, M, N, K, apart):
    """The fp32 sum's error grows with the root of the terms (2^-24 of their magnitudes each), then one rounding to bf16."""
    g = torch.Generator(gpu).manual_seed(M + K)
    x = torch.randn(M, K + apart, device=gpu, generator=g).to(BF)[:, :K]
    w = torch.randn(K, N, device=gpu, generator=g).to(BF)
    got = ops.kernels().gemm_kn(x, w, False)
    want, mag = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -24 * K ** 0.5 * mag).all()
    assert torch.equal(got, ops.kernels().gemm_kn(x, w, False))


# last stages of each kind: whole, one row, all but one; slices of each count; columns of a wider matrix
@pytest.mark.parametrize("K,M,N,apart", [(256, 256, 256, 0), (257, 256, 512, 8), (287, 512, 256, 0), (1000, 768, 1024, 0), (10_240, 1024, 4096, 0),
                                         (8_743, 3072, 1024, 0), (4_096, 4096, 4096, 64), (300, 16384, 1024, 0)])
def test_gemm_kn_of_transposed_rows(gpu, K, M, N, apart):
    """The bound of test_gemm_kn; infinities in rows that the last stage has twice come once."""
    g = torch.Generator(gpu).manual_seed(M + K)
    x = torch.randn(K, M + apart, device=gpu, generator=g).to(BF)[:, :M]
    w = torch.randn(K, N, device=gpu, generator=g).to(BF)
    got = ops.kernels().gemm_kn(x, w, True)
    want, mag = x.double().t() @ w.double(), x.double().abs().t() @ w.double().abs()
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -24 * K ** 0.5 * mag).all()
    x[K - 30, 3], w[K - 30] = float("inf"), w[K - 30].abs() + 1
    got = ops.kernels().gemm_kn(x, w, True)
    assert (got[3] == float("inf")).all() and got.isfinite().sum() == got.numel() - N


@pytest.mark.parametrize("shape,N", [((2, 40), 16384), ((700,), 16384), ((3, 0), 16384), ((100,), 4096), ((100,), 4128)])
def test_frozen_linear(gpu, shape, N):
    """Outputs are the product's to the bit; the gradient has other sums than the library's (both fp32, one rounding each: 2^-8), and
    can be differentiated again."""
    from nv_genai_amd.training import fused

    w = torch.randn(N, 512, device=gpu).to(BF)
    x = torch.randn(*shape, 512, device=gpu).to(BF).requires_grad_()
    ok = fused.frozen_linear_usable(x, w)
    assert ok == (x.numel() > 0)
    if not ok:
        return
    y = fused.frozen_linear(x, w)
    assert torch.equal(y, x @ w.t())
    dy = torch.randn_like(y).requires_grad_()
    got, = torch.autograd.grad(y, x, dy, create_graph=True)
    assert torch.equal(got, dy @ w)
    once, = torch.autograd.grad(fused.frozen_linear(x, w), x, dy)
    want = dy.double() @ w.double()
    assert ((once.double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -24 * N ** 0.5 * (dy.double().abs() @ w.double().abs())).all()
    assert torch.autograd.grad(got.float().pow(2).sum(), dy)[0].isfinite().all()
    for v, u in ((x.detach(), w), (x, w.clone().requires_grad_()), (x, w.float()), (x.float(), w), (x, w.t().contiguous().t())):
        assert not fused.frozen_linear_usable(v, u)


# one tile, tiles of rows that are not full, blocks of eight of them and one more, more tiles than CUs (a workgroup's second and third),
# stages that end anywhere in the ring's round
@pytest.mark.parametrize("M,N,K,apart", [(1, 256, 256, 0), (256, 768, 288, 8), (257, 256, 320, 0), (2100, 512, 352, 0), (2305, 1024, 1024, 0),
                                         (4200, 4096, 1024, 24), (9000, 3072, 768, 0), (3000, 1024, 4096, 0)])
def test_gemm_nt_gelu(gpu, M, N, K, apart):
    """The fp32 sum's error grows with the root of the terms (2^-24 of their magnitudes each); GELU's slope is at most 1.13, and its form
    here is within 1e-7 of the exact one; then one rounding to bf16."""
    g = torch.Generator(gpu).manual_seed(M + K)
    x = torch.randn(M, K + apart, device=gpu, generator=g).to(BF)[:, :K]
    w = torch.randn(N, K, device=gpu, generator=g).mul_(2 / K ** 0.5).to(BF)
    b = torch.randn(N, device=gpu, generator=g).to(BF)
    sums, mag = x.double() @ w.double().t() + b.double(), x.double().abs() @ w.double().abs().t() + b.double().abs()
    want = torch.nn.functional.gelu(sums)
    got = ops.kernels().gemm_nt_gelu(x, w, b)
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 1.13 * 2 ** -24 * K ** 0.5 * mag + 1e-7 * sums.abs()).all()


def test_gemm_nt_gelu_at_the_ends(gpu):
    """Sums of every size, infinities and NaN: K values of which one counts. Down to -7.5 a small result has its digits (relative 1.3e-4
    before its rounding to bf16, where 1 + erf has none); below, GELU is at most 2.4e-13, and its form, which lacks the logarithm's last
    change there, less than twice that."""
    v = torch.cat([torch.linspace(-12, 12, 4001), torch.tensor([0.0, -0.0, 1e-30, -1e-30, 3e38, -3e38, float("inf"), float("-inf"), float("nan")])])
    x = torch.zeros(v.numel(), 256, device=gpu, dtype=BF)
    x[:, 0] = v.to(gpu)
    w = torch.zeros(256, 256, device=gpu, dtype=BF)
    w[:, 0] = 1
    got = ops.kernels().gemm_nt_gelu(x, w, torch.zeros(256, device=gpu, dtype=BF))
    a = x[:, 0].double()
    want = torch.where(a == 0, a, a * 0.5 * torch.erfc(-a * 0.5 ** 0.5))   # torch's own loses the digits of a small 1 + erf
    fin = want.isfinite()
    assert torch.equal(got.isnan(), want.isnan()[:, None].expand_as(got)) and (got[want == float("inf")] == float("inf")).all()
    rel = 2 ** -8 + torch.where(a < -7.5, 1.0, 1.4e-4)   # half a bf16 step, and GELU's own
    assert ((got[fin].double() - want[fin, None]).abs() <= (rel * want.abs())[fin, None] + 2.0 ** -133).all()


@pytest.mark.parametrize("T", [4999, 5000, 6003])
def test_weight_gradients(gpu, T):
    """fused.linear's weight gradient on both sides of the line, of rows that lie apart in memory: the library's to one bf16 step."""
    from nv_genai_amd.training import fused

    x = torch.randn(T, 264, device=gpu).to(BF)[:, :256]
    w = torch.randn(512, 256, device=gpu).requires_grad_()
    b = torch.zeros(512, device=gpu, requires_grad=True)
    assert ops.weight_grad_covers(T, 512, 256) == (T >= 5000)
    dy = torch.randn(T, 512, device=gpu).to(BF)
    got, = torch.autograd.grad(fused.linear(x, w, b), w, dy)
    want, mag = dy.double().t() @ x.double(), dy.double().abs().t() @ x.double().abs()
    assert got.dtype == torch.float32 and ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -24 * T ** 0.5 * mag).all()


@pytest.mark.parametrize("N,K,here", [(2048, 4096, True), (6144, 1536, False), (7680, 1280, False), (5120, 2048, True), (4096, 4096, True), (4096, 4352, False),
                                      (6144, 3072, False), (5120, 4608, True), (8192, 4096, True), (256, 256, True), (256, 128, False), (300, 256, False)])
def test_weight_gradients_by_their_tiles(gpu, N, K, here):
    """128 tiles, 144, 150, 160, 256, 272, 288, 360, 512, 1: the counts that leave CUs idle are the library's."""
    assert ops.weight_grad_covers(8192, N, K) == here
