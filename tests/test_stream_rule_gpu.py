"""Where the weight-stream kernel takes a projection of few rows."""
import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("M,N,K,swiglu,here", [
    (1, 4096, 4096, False, True), (1, 4112, 4096, False, False), (1, 6144, 4096, False, False), (1, 8176, 1024, False, False),
    (1, 8192, 1024, False, True), (1, 8208, 1024, False, False), (1, 2816, 1024, True, False), (1, 4096, 2048, True, True),
    (2, 6144, 4096, False, True), (2, 5504, 4096, True, False), (2, 5504, 2048, True, True), (3, 5504, 4096, True, True),
    (2, 6144, 4096, True, True), (2, 4096, 4096, True, True), (16, 14336, 4096, True, True), (17, 4096, 4096, False, False),
    (8, 4096, 8192, False, True), (9, 4096, 8192, False, False), (8, 4112, 8192, False, False)])
def test_rule(gpu, M, N, K, swiglu, here):
    assert ops.kernels().stream_gemm_covers(M, N, K, swiglu) == here
