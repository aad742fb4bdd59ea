"""The fused kernels of a decode step against the launches that they stand for."""
import math

import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu


def _pages(ctxs, Hkv, dev):
    pages = [(c + 63) // 64 for c in ctxs]
    nb = sum(pages) + 3
    kc = torch.randn(nb, Hkv, 64, 128, device=dev).to(torch.bfloat16)
    vc = torch.randn(nb, Hkv, 128, 64, device=dev).to(torch.bfloat16)
    perm = torch.randperm(nb).tolist()
    bt = torch.zeros(len(ctxs), max(pages), dtype=torch.int32)
    slots, k = [], 0
    for i, (c, p) in enumerate(zip(ctxs, pages)):
        for j in range(p):
            bt[i, j], k = perm[k], k + 1
        slots.append(int(bt[i, (c - 1) // 64]) * 64 + (c - 1) % 64 if c else -1)
    return kc, vc, bt.to(dev), torch.tensor(slots, dtype=torch.int32, device=dev)


@pytest.mark.parametrize("G,Hkv", [(4, 8), (1, 8), (5, 2), (16, 1)])
@pytest.mark.parametrize("ppp,window", [(None, 0), (1, 0), (3, 0), (2, 200), (None, 64)])
@pytest.mark.parametrize("slabs", [0, 1, 3])
def test_decode_step_is_rotation_and_attention(gpu, G, Hkv, ppp, window, slabs):
    """Contexts around the ends of pages and of partitions, rows without a context and rows whose key is not written. The
    cache is the same to the bit. The outputs are bf16 of the same products; only the sum over the partitions has another
    form (two fp32 sums over up to 16 parts, then one rounding): one bf16 step, 2^-8 of the value, and of the largest where
    values cancel."""
    torch.manual_seed(G * 100 + slabs)
    Hq, D, dev = Hkv * G, 128, gpu
    part = 64 * 4 * (ppp or 1)
    ctxs = [1, 0, 63, 64, 65, 700, 128, part - 1, part, part + 1, 3 * part + 1, 2500]
    kc, vc, bt, slots = _pages(ctxs, Hkv, dev)
    slots[6] = -1
    B, row = len(ctxs), (Hq + 2 * Hkv) * D
    if slabs:
        qkv = ops.PartialSum(torch.randn(slabs, B, row, device=dev))
        flat = ops.splitk_reduce(qkv.slabs)
    else:
        flat = torch.randn(B, row, device=dev).to(torch.bfloat16)
        qkv = flat.clone()
    ctx = torch.tensor(ctxs, dtype=torch.int32, device=dev)
    pos = (ctx - 1).clamp(min=0)
    cs = ops.rope_cos_sin(4096, D).to(dev)
    most, scale = max(ctxs), 1 / math.sqrt(D)
    ws = ops.DecodeWorkspace(B, Hq, Hkv, most, dev, ppp)
    k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    ops.rope_cache_(flat, pos, cs, slots, k1, v1, Hq, Hkv, D)
    want = ops.decode_attention(flat[:, : Hq * D], k1, v1, bt, ctx, Hq, Hkv, most, scale, ws=ws, window=window)
    assert ops.decode_step_covers(qkv, k2, ctx, slots, most, ws, window)
    for k in (128, 4096):   # the counters are zero again after a launch; weights to read ahead of one and of many blocks a piece
        nxt = torch.empty(16 * 37, k, dtype=torch.bfloat16, device=dev)
        got = ops.decode_step(qkv, pos, cs, slots, k2, v2, bt, ctx, Hq, Hkv, most, scale, ws, window, nxt)
        assert torch.equal(k1, k2) and torch.equal(v1, v2)
        assert not ws.done.any()
        w, g = want.float(), got.float()
        assert (g[1] == 0).all()
        assert ((g - w).abs() <= 2 ** -8 * w.abs() + 2 ** -8 * w.abs().amax(1, keepdim=True)).all()


@pytest.mark.parametrize("rows,N,K,ahead", [(1, 4096, 4096, True), (16, 4096, 4096, True), (1, 2048, 2048, True), (1, 5120, 5120, False), (1, 8192, 8192, False),
                                           (4, 6144, 4096, False), (1, 8192, 4096, False), (1, 4096, 8192, False), (17, 4096, 4096, False),
                                           (1, 4096, 4000, False)])
def test_weights_are_read_ahead_for_the_kernel_that_takes_them(gpu, rows, N, K, ahead):
    """The stream kernel with 16 weight rows a workgroup, and up to 33.5 MB."""
    assert ops.kernels().stream_gemm_reads_ahead(rows, N, K) == ahead


@pytest.mark.parametrize("rows,Hkv,one", [(64, 8, True), (65, 8, False), (16, 32, True), (17, 32, False), (256, 2, True), (512, 1, True), (513, 1, False)])
def test_many_rows_take_launches_of_their_own(gpu, rows, Hkv, one):
    """From more than two workgroups a CU on the rotation stands alone; at the line both give the same."""
    D, dev = 128, gpu
    ctxs = [1 + (37 * i) % 150 for i in range(rows)]
    kc, vc, bt, slots = _pages(ctxs, Hkv, dev)
    qkv = torch.randn(rows, 3 * Hkv * D, device=dev).to(torch.bfloat16)
    ctx, cs = torch.tensor(ctxs, dtype=torch.int32, device=dev), ops.rope_cos_sin(256, D).to(dev)
    ws = ops.DecodeWorkspace(rows, Hkv, Hkv, 192, dev)
    assert ops.decode_step_covers(qkv, kc, ctx, slots, 192, ws) == one
    if not one:
        return
    k1, v1, flat = kc.clone(), vc.clone(), qkv.clone()
    got = ops.decode_step(qkv, ctx - 1, cs, slots, kc, vc, bt, ctx, Hkv, Hkv, 192, D ** -0.5, ws).float()
    ops.rope_cache_(flat, ctx - 1, cs, slots, k1, v1, Hkv, Hkv, D)
    want = ops.decode_attention(flat[:, : Hkv * D], k1, v1, bt, ctx, Hkv, Hkv, 192, D ** -0.5, ws=ws).float()
    assert torch.equal(kc, k1) and torch.equal(vc, v1)
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2 ** -8 * want.abs().amax(1, keepdim=True)).all()   # as above


@pytest.mark.parametrize("N,K", [(4096, 4096), (6144, 4096), (16, 256), (48, 768), (1008, 2304), (14336, 4096), (512, 8192), (384, 5120),
                                 (101, 520), (33, 1032), (7, 8), (2064, 8184)])
@pytest.mark.parametrize("epi", [1, 2])
def test_norm_linear(gpu, N, K, epi, M=1):
    """Stages that do not split evenly over the waves, K below and at the kernels' ends, the GEMV for odd shapes. The norm's
    sum of squares has another order, so a normed value may fall on the next bf16 (2^-8 of it): at most 2^-8 of a row of
    products, and with SwiGLU, a product of two of them rounded to bf16, three times that."""
    torch.manual_seed(N + K)
    x = (2 * torch.randn(M, K, device=gpu)).to(torch.bfloat16)
    nw = (1 + 0.3 * torch.randn(K, device=gpu)).to(torch.bfloat16)
    w = (torch.randn((2 if epi == 2 else 1) * N, K, device=gpu) / math.sqrt(K)).to(torch.bfloat16)
    assert ops.norm_linear_covers(x, nw, w, epi == 2)
    got = ops.norm_linear(x, nw, 1e-5, w, epi).float()
    y = ops.rmsnorm(x, nw, 1e-5).double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :N]) * y[:, N:] if epi == 2 else y
    assert got.shape == want.shape
    err = (got.double() - want).norm(dim=1) / want.norm(dim=1)
    assert (err <= 2 ** -8 * (3 if epi == 2 else 1)).all()


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (2, 4096, 14336), (1, 16, 256), (7, 48, 768), (16, 4096, 4096), (8, 1024, 8192)])
def test_linear_add(gpu, M, N, K):
    """One rounding of the sum: half a bf16 step of it, and the products' fp32 sums in another order (K values, 2^-24 each)."""
    torch.manual_seed(N + K)
    x = torch.randn(M, K, device=gpu).to(torch.bfloat16)
    w = (torch.randn(N, K, device=gpu) / math.sqrt(K)).to(torch.bfloat16)
    resid = torch.randn(M, N, device=gpu).to(torch.bfloat16)
    assert ops.linear_add_covers(M, w)
    want = resid.double() + x.double() @ w.double().t()
    got = ops.linear_add_(resid, x, w)
    assert got.data_ptr() == resid.data_ptr()
    slack = 2 ** -24 * math.sqrt(K) * (x.double().abs() @ w.double().abs().t())
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + slack + 1e-6).all()
