"""Where the weight-stream kernel takes a projection of few rows."""
import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("M,N,K,swiglu,here", [
    (1, 4096, 4096, False, True), (1, 4112, 3072, False, False), (1, 7168, 4096, False, True), (1, 7184, 4096, False, False), (1, 8176, 1024, False, False),
    (1, 8192, 1024, False, True), (1, 8208, 1024, False, False), (1, 2816, 1024, True, False), (1, 4096, 2048, True, True),
    (2, 6144, 4096, False, True), (2, 5504, 4096, True, False), (2, 5504, 2048, True, True), (3, 5504, 4096, True, True),
    (2, 6144, 4096, True, True), (2, 4096, 4096, True, True), (16, 14336, 4096, True, True), (17, 4096, 4096, False, False),
    (8, 4096, 8192, False, True), (9, 4096, 8192, False, False), (8, 4112, 8192, False, False)])
def test_rule(gpu, M, N, K, swiglu, here):
    assert ops.kernels().stream_gemm_covers(M, N, K, swiglu) == here


def _odd(t):
    return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("M", [5, 16])
def test_rows_at_any_address(gpu, M):
    """Rows that do not begin at 16 bytes take the library's product, as from 17 rows on; weights that do not are refused."""
    from nv_genai_amd.models.config import llama_config
    from nv_genai_amd.models.llama import LlamaModel

    m = LlamaModel(llama_config("llama-tiny"), gpu, seed=1)
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = torch.randn(M, 512, device=gpu, generator=g).to(BF), (0.05 * torch.randn(272, 512, device=gpu, generator=g)).to(BF)
    assert ops.stream_covers(x, w)
    want = x.double() @ w.double().t()
    for y in (m._lin(_odd(x), {"wo": w}, "wo"), m._lin(_odd(x), {"wo": w}, "wo", partial_ok=True)):
        assert ((y.double() - want).norm() / want.norm()).item() < 4e-3   # fp32 sums, one rounding to bf16
    with pytest.raises(ValueError):
        m._lin(x, {"wo": _odd(w)}, "wo")
