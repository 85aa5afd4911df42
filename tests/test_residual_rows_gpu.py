"""Expert rows read several at a time (csrc/kernels/packed_rows.hip): counts around the groups of 4 and 8."""
import pytest
import torch

from penroz.ops import _ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top", [1, 2, 3, 4, 5, 8, 9, 17])
@pytest.mark.parametrize("C", [7, 100, 2048, 2052, 4096, 4100])
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


@pytest.mark.parametrize("top", [0, 1, 4, 5, 9])  # 0: one plain row
@pytest.mark.parametrize("taps", [0, 1, 2, 4, 5, 16])
@pytest.mark.parametrize("C,dt", [(96, torch.bfloat16), (2048, torch.bfloat16), (4096, torch.float32), (2056, torch.bfloat16)])
def test_rows_with_a_convolution(top, taps, C, dt):
    g = torch.Generator(device="cuda").manual_seed(top * C + taps)
    N, groups, eps = 4, 2, 1e-5
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y, nw = r(N, C), r(N * max(top, 1), C).to(dt), r(C)
    pw = r(N, top) if top else None
    pos = torch.tensor([0, 1, 3, 40], device="cuda", dtype=torch.int32)
    slot = torch.tensor([2, 0, 5, 1], device="cuda", dtype=torch.int32)
    cw = r(taps, C) if taps else None
    state = r(6, taps - 1, C) if taps else None
    if taps > 1:
        state[2] = float("nan")  # a slot taken again: nothing before position 0 is read
    before = None if state is None else state.clone()
    out, h = torch.empty_like(x), torch.empty(N, C, device="cuda", dtype=dt)
    _ext.kernels().row_norm_add(None, None, x, out, y, pw, nw, groups, eps, cw, state, slot, pos, False, h)
    v = y.double().view(N, -1, C)
    v = (v * pw.double()[..., None]).sum(1) if top else v[:, 0]
    v = v.view(N, groups, -1)
    want = x.double() + (v * torch.rsqrt(v.square().mean(2, keepdim=True) + eps)).view(N, C) * nw.double()
    scale = want.abs().amax(1, keepdim=True)
    assert ((out.double() - want).abs() <= 2.0 ** -20 * (top + 4) * scale).all()
    conv = want.clone()
    if taps:
        conv = conv + cw[-1].double() * want
        for n in range(N):
            for k in range(taps - 1):
                if int(pos[n]) - (taps - 1) + k >= 0:
                    conv[n] += cw[k].double() * before[slot[n], k].double()
            if taps > 1:
                assert torch.equal(state[slot[n], :-1].nan_to_num(7.0), before[slot[n], 1:].nan_to_num(7.0))
                assert torch.equal(state[slot[n], -1], out[n])
    lim = (2.0 ** -8 if dt == torch.bfloat16 else 0.0) * conv.abs() + 2.0 ** -19 * (top + taps + 4) * conv.abs().amax(1, keepdim=True)
    assert ((h.double() - conv).abs() <= lim).all()
