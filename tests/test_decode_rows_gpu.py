"""Decode products of a few rows (csrc/kernels/decode_linear.hip): the LayerNorm products, the GEMV whose waves share a row,
the paired rows, at the edges of their tiles, shares and lengths, against fp32 torch."""
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


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K", [8, 512, 520, 1024, 1032, 1536, 1544, 3072, 3080, 4608, 4616, 7168, 7176, 8192])
@pytest.mark.parametrize("N", [1, 33])
def test_gemv_rows(M, K, N):
    """Every length class of the GEMV, exact and one chunk over; a last workgroup with one row of its two."""
    torch.manual_seed(M + K + N)
    x = torch.randn(M, K + 8, device=DEV).to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K, device=DEV) / K ** 0.5).to(torch.bfloat16)
    b = torch.randn(N, device=DEV).to(torch.bfloat16)
    big = torch.full((M + 1, N + 3), 7.0, device=DEV, dtype=torch.bfloat16)
    _ext.kernels().decode_gemv(x, None, None, None, None, None, None, 0.0, w, b, big[:M, :N], 0)
    ref = x.float() @ w.float().t() + b.float()
    _near(big[:M, :N], ref, 0 * ref)
    assert (big[M] == 7).all() and (big[:, N:] == 7).all()


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("K", [32, 768, 3072, 4640, 8192, 8224])
def test_gemv_adds_to_the_residual(M, K):
    """decode_gemm_acc around the GEMV's limits (4 rows, 8192 columns): fp32 sums of exact products, so within K roundings."""
    torch.manual_seed(M + K)
    N = 48
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) / K ** 0.5).to(torch.bfloat16)
    b = torch.randn(N, device=DEV).to(torch.bfloat16)
    old = torch.randn(M, N, device=DEV)
    got = old.clone()
    _ext.kernels().decode_gemm_acc(x, w, b, got)
    ref = old.double() + x.double() @ w.double().t() + b.double()
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + old.double().abs() + b.double().abs())
    assert torch.all((got.double() - ref).abs() <= bound)


@pytest.mark.parametrize("M", [1, 3, 4])
@pytest.mark.parametrize("K,I", [(8, 1), (256, 5), (768, 4), (1032, 17), (1792, 3)])
@pytest.mark.parametrize("ppw", [0, 2, 4])
def test_gemv_pairs_of_few_rows(M, K, I, ppw):
    """Pairs that end inside a wave and inside a workgroup, columns that end inside a chunk group; infinities stay in their row."""
    torch.manual_seed(M + K + I)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    gu = (torch.randn(2 * I, K, device=DEV) / K ** 0.5).to(torch.bfloat16)
    gu[0, K - 1] = float("inf")
    big = torch.full((M + 1, I + 3), 7.0, device=DEV, dtype=torch.bfloat16)
    _ext.kernels().decode_gemv_pair(x, gu, big[:M, :I], 1, 2, pairs_per_wave=ppw)
    y = (x.float() @ gu.float().t()).to(torch.bfloat16).float()
    ref = F.silu(y[:, :I]) * y[:, I:]
    got = big[:M, :I].float()
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(got), fin)
    # gate and up, rounded from sums of another order, may be a bf16 step apart each; the result is rounded once more
    assert torch.all((got - ref)[fin].abs() <= 2.0 ** -8 * 4 * (ref.abs() + y[:, :I].abs() + y[:, I:].abs())[fin] + 1e-5)
    assert (big[M] == 7).all() and (big[:, I:] == 7).all()


def _step_ref(x, a, w1, w2, mode, eps1, eps2):
    """rms_residual's step in fp32 with its bf16 rounding points, from 64-bit sums."""
    b16 = lambda t: t.to(torch.bfloat16).float()
    rms = lambda t, eps: b16(t * torch.rsqrt(t.double().square().mean(-1, keepdim=True) + eps).float())
    x = x.float()
    if mode == 0:
        v = b16(rms(b16(x + a.float()), eps1) * w1.float())
    elif mode == 1:
        v = b16(x + b16(rms(a.float(), eps1) * w1.float()))
    else:
        v = b16(x + a.float()) if mode == 2 else x
    return v, b16(rms(v, eps2) * w2.float())


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K", [8, 264, 768, 1032, 1152, 1792])
@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("gated", [True, False])
def test_norm_pair(M, K, mode, gated):
    """The step between two sublayers in front of a pair product: its residual row by row, its product against the product of
    the reference's rows; pairs that end inside a wave and a workgroup."""
    torch.manual_seed(M + K + mode)
    k = _ext.kernels()
    x, a = (torch.randn(M, K, device=DEV).to(torch.bfloat16) for _ in range(2))
    w1, w2 = ((1 + 0.1 * torch.randn(K, device=DEV)).to(torch.bfloat16) for _ in range(2))
    D, N = 16, 2 * 37 if gated else 5 * 16
    w = (torch.randn(N, K, device=DEV) / K ** 0.5).to(torch.bfloat16)
    big = torch.full((M + 1, N + 3), 7.0, device=DEV, dtype=torch.bfloat16)
    out = big[:M, :N // 2 if gated else N]
    h = torch.empty(M, K, device=DEV, dtype=torch.bfloat16)
    ang = torch.rand(D // 2, device=DEV) * 6
    cs, sn = ang.cos(), ang.sin()
    if mode == 3:
        table, idx = torch.randn(9, K, device=DEV).to(torch.bfloat16), torch.tensor([8, 0, 3, 5][:M], device=DEV)
        x = (table[idx] * 3.5)
        k.decode_norm_pair(None, None, None, w2, 3, 0.0, 1e-6, h, w, out, 1 if gated else 2, 2, D, 4, cs, sn, idx, table, 3.5)
    else:
        k.decode_norm_pair(x, a, w1, w2, mode, 1e-6, 1e-5, h, w, out, 1 if gated else 2, 2, D, 4, cs, sn)
    v, y = _step_ref(x, a, w1, w2, mode, 1e-6, 1e-6 if mode == 3 else 1e-5)
    # a value near a tie may be rounded apart at each of the step's four roundings
    assert torch.all((h.float() - v).abs() <= 4 * 2.0 ** -8 * (v.abs() + x.float().abs()) + 1e-6)
    z = (y @ w.float().t())
    slack = 2.0 ** -8 * (z.abs() + 4 * (y.square() @ w.float().square().t()).sqrt())
    if gated:
        I = N // 2
        ref = F.silu(z[:, :I]) * z[:, I:]
        # |silu'| <= 1.1
        bound = slack[:, :I] * 1.1 * z[:, I:].abs() + F.silu(z[:, :I]).abs() * slack[:, I:] + slack[:, :I] * slack[:, I:]
        bound = bound + 2.0 ** -8 * ref.abs() + 1e-5
    else:
        zz, s2 = z.view(M, 5, D), slack.view(M, 5, D)
        lo, hi = zz[..., :D // 2], zz[..., D // 2:]
        rot = torch.cat([lo * cs - hi * sn, hi * cs + lo * sn], -1)
        ref = torch.cat([rot[:, :4], zz[:, 4:]], 1).view(M, N)
        both = s2[..., :D // 2] + s2[..., D // 2:]
        bound = torch.cat([both, both], -1).view(M, N) + 2.0 ** -8 * ref.abs() + 1e-5
    assert torch.all((out.float() - ref).abs() <= bound), float(((out.float() - ref).abs() / bound).max())
    assert (big[M] == 7).all() and (big[:, out.shape[1]:] == 7).all()


@pytest.mark.parametrize("T,n,pos", [(1, 128, 0), (1, 4, 8191), (5, 33, 1000)])
def test_rope_table_at_a_device_position(T, n, pos):
    from penroz.ops import rope
    inv = 1.0 / (1e6 ** (torch.arange(n, device=DEV, dtype=torch.float32) / n))
    got = rope.rope_table(inv, 0, T, DEV, offset_dev=torch.tensor([pos], device=DEV))
    for g, r in zip(got, rope.rope_table(inv, pos, T, DEV)):
        assert g.shape == r.shape and torch.all((g - r).abs() <= 2.0 ** -22)
