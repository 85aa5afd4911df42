"""Linear layers of short steps (csrc/kernels/rows_gemm.hip) against float64."""
import pytest
import torch

from penroz.ops import _ext, gemm


@pytest.mark.skipif(not _ext.available("penroz_serve"), reason="HIP extension not built")
@pytest.mark.parametrize("M,N,K,tile", [(1, 8, 8, 6), (64, 768, 768, 6), (65, 832, 768, 1), (256, 1024, 1024, 1), (257, 1024, 1024, 2),
                                        (64, 8192, 2048, 2), (256, 3072, 768, 3), (64, 12288, 2048, 3), (65, 12288, 2048, 0),
                                        (512, 3072, 768, 4), (1024, 3072, 768, 5), (64, 32768, 2048, 5), (4096, 3072, 768, 0),
                                        (64, 768, 772, 0), (0, 768, 768, 0), (64, 1 << 21, 768, 0)])
def test_rows_gemm_rule(M, N, K, tile):
    assert _ext.kernels().rows_gemm_tile(M, N, K) == tile
    in_order = _ext.kernels().rows_gemm_tile(M, N, K, True)
    assert in_order == (1 if tile in (2, 6) else tile)


@pytest.mark.skipif(not _ext.available("penroz_serve"), reason="HIP extension not built")
@pytest.mark.parametrize("M,N,K,tile", [(5, 32768, 2048, 0), (8, 32768, 2048, 0), (9, 32768, 2048, 5), (5, 50304, 768, 5)])
def test_wide_outputs_of_few_rows(M, N, K, tile):
    """Up to 8 rows of more than 1024 columns stay with skinny_gemm."""
    assert _ext.kernels().rows_gemm_tile(M, N, K) == tile


# every tile: less than one, its edges, ragged rows and columns; K of less than a stage, whole stages, ragged ones
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,tile", [(1, 8, 6), (31, 33, 6), (33, 250, 6), (64, 1022, 6), (70, 1001, 1),
                                      (256, 1024, 1), (300, 1026, 2), (17, 9001, 2),
                                      (200, 3001, 3), (64, 12288, 3), (500, 3001, 4), (700, 3100, 5), (64, 40000, 5)])
@pytest.mark.parametrize("K", [8, 56, 64, 72, 256, 264, 760, 1024])
def test_rows_gemm(M, N, tile, K):
    assert _ext.kernels().rows_gemm_tile(M, N, K) == tile
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K]  # strided rows
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    bias = torch.randn(N, generator=g, device="cuda").bfloat16()
    want = x.double() @ w.double().t()
    full = gemm.rows_linear(x, w, fp32=True)
    # fp32 sums of K products: in blocks of 32 in the MFMA, K / 32 of them
    assert full.dtype == torch.float32
    assert torch.linalg.norm(full.double() - want) <= 2.0 ** -24 * (K / 32 + 32) ** 0.5 * torch.linalg.norm(want)
    act = gemm.rows_linear(x, w, bias, gelu=True)
    lin = gemm.rows_linear(x, w, bias).double()
    gelu = torch.nn.functional.gelu(lin)  # one rounding to bf16, and erff's cancellation at negative values
    assert ((act.double() - gelu).abs() <= 2.0 ** -8 * gelu.abs() + 2.0 ** -22 * lin.abs()).all()
    for b, in_order in ((None, True), (None, False), (bias, True), (bias, False)):
        ref = want if b is None else want + b.double()
        got = gemm.rows_linear(x, w, b, in_order=in_order)
        if got is None:
            assert in_order and tile == 2
            got = gemm.rows_linear(x, w, b)
        assert got.dtype == torch.bfloat16
        # half a step of bf16 at each value, and the sums' own error where they cancel
        assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -18 * K ** 0.5).all()
    buf = torch.full((M, N + 8), 7.0, device="cuda", dtype=torch.bfloat16)  # rows of a wider buffer
    assert gemm.rows_linear(x, w, bias, buf[:, :N]) is not None
    assert torch.equal(buf[:, :N], got) and (buf[:, N:] == 7.0).all()
    if K % 32 == 0 and N % 16 == 0:  # added to an fp32 residual
        w = w.contiguous()
        resid = torch.randn(M, N, generator=g, device="cuda")
        ref = resid.double() + want + bias.double()
        _ext.kernels().decode_gemm_acc(x, w, bias, resid)
        assert torch.linalg.norm(resid.double() - ref) <= 2.0 ** -24 * (K / 32 + 32) ** 0.5 * torch.linalg.norm(ref)


@pytest.mark.gpu
def test_rows_gemm_leaves_other_forms():
    """What the kernel does not read goes to the library with the result it always had."""
    x, w = (torch.randn(64, 256, device="cuda").bfloat16() for _ in range(2))
    forms = [(x[:, 1:249], w[:, 1:249]), (x.t().contiguous().t(), w), (x, w.t().contiguous().t()), (x[:, :100], w[:, :100])]
    for a, b in forms:
        assert gemm.rows_linear(a, b) is None
        assert torch.equal(gemm.linear(a, b), torch.mm(a, b.t()))
    off = torch.randn(64 * 256 + 1, device="cuda").bfloat16()[1:].view(64, 256)
    assert gemm.rows_linear(off, w) is None
    assert gemm.rows_linear(x, w, torch.zeros(64, device="cuda")) is None  # an fp32 bias
    assert gemm.rows_linear(x.float(), w.float()) is None
    with pytest.raises(RuntimeError):
        gemm.linear(x, w[:, :248])
    wp = w.clone().requires_grad_()
    gemm.linear(x, wp).sum().backward()
    assert wp.grad is not None


@pytest.mark.gpu
def test_rows_gemm_propagates_what_is_not_finite():
    x = torch.ones(40, 96, device="cuda").bfloat16()
    w = torch.ones(72, 96, device="cuda").bfloat16()
    x[3, 95], w[5, 0], x[7, 1] = float("inf"), float("nan"), -float("inf")
    got, ref = gemm.rows_linear(x, w), torch.mm(x.float(), w.float().t())
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(got[3, :5], ref[3, :5].bfloat16())
    assert torch.equal(got[7, :5], ref[7, :5].bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["residual off 16 bytes", "no columns", "rows far apart"])
def test_residual_products_of_every_form(form):
    g = torch.Generator(device="cuda").manual_seed(1)
    M, N, K = 5, 768, 96
    x, w = torch.randn(M, K, generator=g, device="cuda").bfloat16(), torch.randn(N, K, generator=g, device="cuda").bfloat16()
    bias, resid = torch.randn(N, generator=g, device="cuda").bfloat16(), torch.randn(M, N, generator=g, device="cuda")
    if form == "residual off 16 bytes":
        flat = torch.zeros(M * N + 3, device="cuda")
        resid = flat[3:].view(M, N).copy_(resid)
    elif form == "no columns":
        x, w = x[:, :0], w[:, :0].contiguous()
    else:  # a row stride beyond 32 bits
        M, resid = 2, resid[:2].contiguous()
        far = torch.empty((1 << 31) + K, dtype=torch.bfloat16, device="cuda").as_strided((2, K), (1 << 31, 1))
        x = far.copy_(x[:2])
    ref = resid.double() + x.double() @ w.double().t() + bias.double()
    _ext.kernels().decode_gemm_acc(x, w, bias, resid)
    assert torch.linalg.norm(resid.double() - ref) <= 2.0 ** -24 * 6 * torch.linalg.norm(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 256, 640, 768, 832, 1024])
def test_sums_in_order_are_the_librarys_bits(K):
    """What training steps rest on: from 32 rows on, of up to 1024 columns (GPT-2's and Gemma's outputs, ragged rows)."""
    g = torch.Generator(device="cuda").manual_seed(K)
    taken = 0
    for N in (256, 768, 1024, 1152, 2304, 3072):
        w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
        bias = torch.randn(N, generator=g, device="cuda").bfloat16()
        for M in (gemm.TRAIN_ROWS_MIN, 33, 64, 100, 255, 256, 257, 513, 1000, 1100, 2048):
            x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
            for b, want in ((None, torch.mm(x, w.t())), (bias, torch.addmm(bias, x, w.t()))):
                got = gemm.rows_linear(x, w, b, in_order=True)
                if got is not None:
                    taken += 1
                    assert torch.equal(got, want), (M, N, b is not None)
    assert taken >= 100


@pytest.mark.gpu
def test_training_products_of_few_rows_are_the_librarys():
    for M in (1, 5, 16, 31):
        x, w = torch.randn(M, 768, device="cuda").bfloat16(), torch.randn(768, 768, device="cuda").bfloat16()
        assert torch.equal(gemm.train_linear(x, w), torch.mm(x, w.t()))


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["x", "w", "bias"])
def test_operands_that_need_gradients_go_to_the_library(which):
    t = {"x": torch.randn(64, 256, device="cuda").bfloat16(), "w": torch.randn(128, 256, device="cuda").bfloat16(),
         "bias": torch.randn(128, device="cuda").bfloat16()}
    t[which].requires_grad_()
    gemm.linear(**t).sum().backward()
    assert t[which].grad is not None and t[which].grad.any()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(33, 250), (256, 1024), (700, 3100)])
def test_gelu_is_the_erf_form(M, N):
    """Of values of order 1 to 4, where the forms differ."""
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = torch.randn(M, 256, generator=g, device="cuda").bfloat16(), torch.randn(N, 256, generator=g, device="cuda") / 8
    lin = gemm.rows_linear(x, w.bfloat16()).double()
    act = gemm.rows_linear(x, w.bfloat16(), gelu=True).double()
    erf, tanh = (torch.nn.functional.gelu(lin, approximate=form) for form in ("none", "tanh"))
    bound = 2.0 ** -8 * erf.abs() + 2.0 ** -22 * lin.abs()
    assert ((act - erf).abs() <= bound).all()
    assert ((tanh - erf).abs() > bound).float().mean() > 0.05  # the other form would not pass


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(9, 32768, 1032), (16, 30001, 1280), (13, 32768, 2048), (16, 17000, 1992), (16, 8192, 1032),
                                   (64, 50304, 192), (64, 9001, 1024), (33, 9000, 1024)])
def test_large_weights_of_few_rows(M, N, K):
    """Outputs of up to 16 rows in tiles of 16 x 64, and large weights in other tiles: ragged rows, columns and stages."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    bias = torch.randn(N, generator=g, device="cuda").bfloat16()
    want = x.double() @ w.double().t()
    full = gemm.rows_linear(x, w, fp32=True)
    # fp32 sums of K products: in blocks of 32 in the MFMA, K / 32 of them
    assert torch.linalg.norm(full.double() - want) <= 2.0 ** -24 * (K / 32 + 32) ** 0.5 * torch.linalg.norm(want)
    got, ref = gemm.rows_linear(x, w, bias), want + bias.double()
    # half a step of bf16 at each value, and the sums' own error where they cancel
    assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -18 * K ** 0.5).all()
