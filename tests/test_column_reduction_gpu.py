"""Column sums of many rows (csrc/kernels/reduce.h) on the main stream and beside a second one."""
import pytest
import torch

from penroz.ops import _ext


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 15, 16, 33, 272, 1025, 4133])
@pytest.mark.parametrize("cols", [8, 40, 520, 3072])
def test_column_reduction(rows, cols):
    K = _ext.kernels()
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g, device="cuda").bfloat16()
    start = torch.randn(cols, generator=g, device="cuda")
    want = start.double() + x.double().sum(0)
    main = start.clone()
    K.colsum(x, main)
    # fp32 sums of `rows` values of order 1, in blocks: no longer a chain than rows
    assert ((main.double() - want).abs() <= 2.0 ** -24 * (rows + 8) * (x.double().abs().sum(0) + start.double().abs())).all()
    side, beside = torch.cuda.Stream(), start.clone()
    torch.cuda.synchronize()
    K.set_deferred_reduce_stream(side.cuda_stream, 0)
    try:
        K.colsum(x, beside)
    finally:
        K.set_deferred_reduce_stream(0, 0)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(main, beside)


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [40, 3072])
def test_column_reduction_of_many_rows(cols):
    """1024 partial rows and more: one launch on either stream, of 32 slices or of 8 at a time, the same bits."""
    test_column_reduction(16500, cols)
