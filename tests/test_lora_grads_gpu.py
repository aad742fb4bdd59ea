"""A low-rank adapter's gradients (lora.hip) against 64-bit products, with each value's bound from the roundings on its way."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# edges of the 32 rows of a step, the 64 of a workgroup and the slices (from 2,048 rows); of the 64 columns of a sum, the 512 of dx and
# the 256 of a chunk; of the 16, 32 and 64 columns that r is laid out in
@pytest.mark.parametrize("T,K,N,r", [(1, 8, 8, 8), (31, 72, 520, 16), (33, 512, 256, 24), (64, 520, 64, 32), (65, 64, 264, 40),
                                     (257, 1032, 776, 64), (1025, 136, 4096, 8), (2048, 256, 128, 32), (2100, 72, 1544, 56)])
@pytest.mark.parametrize("wants", ["all", "no dx", "a", "b", "dx"])
def test_lora_grads(gpu, T, K, N, r, wants):
    from nv_genai_amd import ops

    g = torch.Generator("cuda").manual_seed(T + r)
    rn = lambda *s: torch.randn(*s, device=gpu, generator=g).to(BF)  # noqa: E731
    dy, x, h, a, b, dxw = rn(T, N), rn(T, K), rn(T, r), rn(r, K), rn(N, r), rn(T, K)
    scale = 0.7
    want_a, want_b = wants in ("all", "no dx", "a"), wants in ("all", "no dx", "b")
    dx = dxw.clone() if wants in ("all", "dx") else None
    da, db = ops.kernels().lora_grads(dy, x, h, a, b, dx, scale, want_a, want_b)
    assert (da is not None) == want_a and (db is not None) == want_b
    D = lambda t: t.double()  # noqa: E731
    e = 2.0 ** -23   # of one fp32 operation, twice over: the matrix units' own roundings
    near = lambda got, ref, bound: bool(((D(got) - ref).abs() <= bound).all())  # noqa: E731
    if want_b:
        ref, size = scale * D(dy).t() @ D(h), scale * D(dy).abs().t() @ D(h).abs()
        assert db.dtype is torch.float32 and near(db, ref, (T + 4) * e * size)
    dh = scale * D(dy) @ D(b)
    off = 2.0 ** -8 * dh.abs() + (N + 4) * e * scale * D(dy).abs() @ D(b).abs()   # dh as bf16 (half an ulp: 2^-9), of a sum in fp32
    if want_a:
        assert da.dtype is torch.float32 and near(da, dh.t() @ D(x), off.t() @ D(x).abs() + (T + 4) * e * dh.abs().t() @ D(x).abs())
    if dx is not None:
        add = D(dxw) + dh @ D(a)
        bound = off @ D(a).abs() + (r + 4) * e * (dh.abs() @ D(a).abs() + D(dxw).abs())
        assert near(dx, add, bound + 2.0 ** -8 * (add.abs() + bound))


def test_batched_gradients_take_single_operations(gpu):
    """A backward under vmap, which no kernel of ours sees the rows of."""
    from nv_genai_amd.training import fused

    g = torch.Generator("cuda").manual_seed(1)
    rn = lambda *s: (0.1 * torch.randn(*s, device=gpu, generator=g)).to(BF)  # noqa: E731
    x, w, a, b = rn(6, 64).requires_grad_(), rn(40, 64), rn(8, 64).float().requires_grad_(), rn(40, 8).float().requires_grad_()
    y, dy = fused.lora_linear(x, w, a, b, 2.0), rn(3, 6, 40)
    many = torch.autograd.grad(y, (x, a, b), dy, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for p, q in zip(many, torch.autograd.grad(y, (x, a, b), dy[i], retain_graph=True)):
            assert torch.allclose(p[i].float(), q.float(), rtol=2.0 ** -6, atol=2.0 ** -6 * q.float().abs().max().item())


@pytest.mark.parametrize("T,N,K,r", [(2, 16, 24, 0), (1 << 24, 8, 8, 8)])
def test_sizes_that_it_leaves_to_single_operations(gpu, T, N, K, r):
    """No rank at all, and more rows than its kernels count."""
    from nv_genai_amd import ops
    from nv_genai_amd.training import fused

    assert not ops.lora_grads_covers(T, N, K, r)
    rn = lambda *s: torch.randn(*s, device=gpu, dtype=BF)  # noqa: E731
    x, w, a, b = rn(T, K).requires_grad_(), rn(N, K), rn(r, K).float().requires_grad_(), rn(N, r).float().requires_grad_()
    y = fused.lora_linear(x, w, a, b, 0.5)
    y.backward(torch.ones_like(y))
    assert a.grad.shape == a.shape and b.grad.shape == b.shape
    want = w.double().sum(0) + 0.5 * (b.detach().to(BF).double().sum(0) @ a.detach().to(BF).double())
    # every row's is the same: sums of N and r terms, rounded to bf16 once or twice of magnitudes up to their own sums
    size = w.double().abs().sum(0) + 0.5 * (b.detach().double().abs().sum(0) @ a.detach().double().abs())
    assert ((x.grad[::max(1, T // 100)].double() - want).abs() <= 2.0 ** -6 * size).all()
