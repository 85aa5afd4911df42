"""Expert rows read several at a time (csrc/kernels/packed_rows.hip): counts around the groups of 4 and 8."""
import pytest
import torch

from penroz.ops import _ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top", [1, 4, 5, 8, 9, 17])
@pytest.mark.parametrize("C", [7, 100, 2048, 4100])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shared", [False, True])
def test_weighted_rows(top, C, dt, shared):
    g = torch.Generator(device="cuda").manual_seed(top * C)
    N, eps = 3, 1e-5
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y, pw, nw = r(N, C), r(N * top, C).to(dt), r(N, top + shared), r(C)
    ys = r(N, C).to(dt) if shared else None
    y[0, 0], y[N * top - 1, 1] = float("inf"), float("nan")
    out, h = torch.empty_like(x), torch.empty(N, C, device="cuda", dtype=dt)
    _ext.kernels().residual_norm(None, None, None, x, out, y, None, None, None, 1.0, 0.0, pw, ys, nw, eps, None, False, h)
    rows, w = y.double().view(N, top, C), pw.double()
    want = x.double() + (rows * w[:, :top, None]).sum(1) + (w[:, top:] * ys.double() if shared else 0)
    mass = x.abs() + (rows * w[:, :top, None]).abs().sum(1) + (w[:, top:] * ys.double() if shared else torch.zeros(1, device="cuda")).abs()
    ok = want.isfinite()
    assert (~ok).sum() == 2 and torch.equal(out.double()[~ok].isnan(), want[~ok].isnan())
    assert ((out.double() - want).abs()[ok] <= 2.0 ** -24 * (top + 3) * mass[ok]).all()  # top + 2 fp32 steps
    full = ok.all(1)
    ref = want[full] * torch.rsqrt(want[full].square().mean(1, keepdim=True) + eps) * nw.double()
    tol = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -22 * (top + 3)
    assert ((h.double()[full] - ref).abs() <= tol * ref.abs() + 2.0 ** -22 * (top + 3) * mass[full] * nw.double().abs()).all()
