"""RMS norms of rows in registers (csrc/kernels/rmsnorm.hip) at the edges of their widths, against float64."""
import pytest
import torch

from penroz.ops import _ext

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("C", [8, 504, 512, 520, 1152, 2056, 3080, 4104, 6144, 6152])
@pytest.mark.parametrize("N", [1, 5])
def test_rmsnorm_rows_in_registers(dt, C, N):
    torch.manual_seed(C + N)
    x, w = torch.randn(N, C, device=DEV).to(dt), (1 + 0.1 * torch.randn(C, device=DEV)).to(dt)
    y, rstd = _ext.kernels().rmsnorm_fwd(x, w, 1e-6)
    ref = torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-6)
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -22}[dt]
    assert torch.all((rstd.double()[:, None] - ref).abs() <= 2.0 ** -20 * ref)
    # the normalised value and its product with the weight are rounded once each
    want = x.double() * ref * w.double()
    assert torch.all((y.double() - want).abs() <= 2 * u * want.abs() + 1e-7)
