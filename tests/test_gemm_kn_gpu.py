"""Gradient of a projection's inputs, x [M, K] . w [K, N] (gemm_kn.hip), against 64 bits."""
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
    got = ops.kernels().gemm_kn(x, w)
    want, mag = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -24 * K ** 0.5 * mag).all()
    assert torch.equal(got, ops.kernels().gemm_kn(x, w))


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
