"""The narrow tile of split columns (csrc/kernels/rows_gemm.hip): the wide tile's sums bit for bit."""
import pytest
import torch

from penroz.ops import _ext, gemm


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(32, 4096), (64, 2048), (64, 1026), (17, 2057), (250, 512), (241, 509)])
@pytest.mark.parametrize("K", [8, 264, 1016, 2048, 6144])
def test_same_bits_as_the_wide_tile(M, N, K):
    wide = 8192 * 32 // (32 * -(-M // 32))  # columns that one round of narrow tiles does not hold
    assert _ext.kernels().rows_gemm_tile(M, N, K) == _ext.kernels().rows_gemm_tile(M, wide, K) == 1
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(wide, K, generator=g, device="cuda").bfloat16()
    want = gemm.rows_linear(x, w, fp32=True)
    got = gemm.rows_linear(x, w[:N], fp32=True)
    assert torch.equal(got, want[:, :N])
    assert torch.linalg.norm(got.double() - x.double() @ w[:N].double().t()) <= 2.0 ** -24 * (K / 32 + 32) ** 0.5 * torch.linalg.norm(got.double())
