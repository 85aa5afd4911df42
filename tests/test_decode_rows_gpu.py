"""Decode products of a few rows (csrc/kernels/decode_linear.hip): the LayerNorm products at the edges of
their tiles and shares, against fp32 torch."""
import pytest
import torch
import torch.nn.functional as F

from penroz.ops import _ext

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _near(got, ref, spread):
    """One bf16 rounding of the result (2^-8) and operands whose fp32 value lies so near a tie that the two sides round it apart:
    ``spread`` is the root of the sum of the products' squares, of which such a step moves single ones by 2^-8."""
    err = (got.float() - ref).abs()
    bound = 2.0 ** -8 * (ref.abs() + spread) + 1e-5
    assert torch.all(err <= bound), float((err / bound).max())


def _ln_case(M, K, N, offset=0.5):
    torch.manual_seed(M * 131 + K + N)
    rin = torch.randn(M, K, device=DEV) * 2 + offset
    gamma, beta = torch.randn(K, device=DEV), torch.randn(K, device=DEV)
    w = (torch.randn(N, K, device=DEV) / K ** 0.5).to(torch.bfloat16)
    b = torch.randn(N, device=DEV).to(torch.bfloat16)
    return rin, gamma, beta, w, b


def _ln_ref(s, gamma, beta, w, b):
    y = F.layer_norm(s.double(), s.shape[1:], gamma.double(), beta.double(), 1e-5).to(torch.bfloat16).float()
    ref = y @ w.float().t() + b.float()
    return ref, (y.square() @ w.float().square().t()).sqrt()


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("K,N", [(32, 16), (96, 48), (256, 80), (288, 4112), (512, 1040), (544, 64), (768, 2304), (800, 3088),
                                 (1024, 4096)])
def test_ln_product(M, K, N):
    rin, gamma, beta, w, b = _ln_case(M, K, N)
    before = rin.clone()
    big = torch.full((M + 1, N + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    _ext.kernels().decode_ln_gemm(rin, gamma, beta, 1e-5, w, b, big[:M, :N], 0)
    _near(big[:M, :N], *_ln_ref(rin, gamma, beta, w, b))
    assert torch.equal(rin, before) and (big[M] == 7).all() and (big[:, N:] == 7).all()


@pytest.mark.parametrize("M", [1, 4, 16])
def test_ln_product_rows_far_from_zero(M):
    """A row whose mean is a thousand times its spread: the squares are taken about the mean, not of the values."""
    K, N = 768, 64
    rin, gamma, beta, w, b = _ln_case(M, K, N, offset=2000.0)
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    _ext.kernels().decode_ln_gemm(rin, gamma, beta, 1e-5, w, b, out, 0)
    ref, spread = _ln_ref(rin, gamma, beta, w, b)
    # an fp32 mean of 2000 is off by up to 2^-13, a 16000th of the spread of 2, in every value alike: below one bf16 rounding
    _near(out, ref, 2 * spread)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K", [32, 288, 768, 1024])
def test_ln_product_of_embeddings(M, K):
    N = 48
    _, gamma, beta, w, b = _ln_case(M, K, N)
    wte, wpe = (torch.randn(9, K, device=DEV).to(torch.bfloat16) for _ in range(2))
    idx, pos = torch.tensor([8, 0, 3, 11][:M], device=DEV), torch.tensor([12], device=DEV)  # (past the ends: the last row)
    rows, out = torch.empty(M, K, device=DEV), torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    _ext.kernels().decode_gemv(None, None, None, None, rows, gamma, beta, 1e-5, w, b, out, 0, emb_idx=idx, emb_wte=wte,
                               emb_wpe=wpe, emb_pos=pos)
    s = wte[idx.clamp(max=8)].float() + wpe[8].float()
    assert torch.equal(rows, s)
    _near(out, *_ln_ref(s, gamma, beta, w, b))
