"""The router's rounds of experts per wave and its choice in registers (csrc/kernels/experts.hip), against float64."""
import pytest
import torch

from penroz.ops import packed as P

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("E,top", [(1, 1), (16, 16), (17, 3), (33, 4), (48, 48), (63, 6), (64, 6), (64, 64), (79, 5), (80, 6), (129, 7)])
@pytest.mark.parametrize("C,gate", [(8, False), (520, True), (2048, True), (2056, False), (4104, True), (1023, False)])
def test_router_rounds(dt, E, top, C, gate):
    torch.manual_seed(E + C)
    h = torch.randn(3, C, device=DEV).to(dt)
    wr = (torch.randn(E + gate, C, device=DEV) * C ** -0.5).to(dt)
    corr = 0.1 * torch.randn(E, device=DEV)
    ids, wts = P.route(h, wr, top, sigmoid=True, correction=corr, scale=1.5, gate=gate)
    s = torch.sigmoid(h.double() @ wr.double().t())
    key = s[:, :E] + corr.double()
    # fp32 sums of C terms: C roundings of the largest partial sum
    tol = C * 2.0 ** -24 * float((h.double().abs() @ wr.double().abs().t()).max()) + 2.0 ** -21
    assert all(len(set(r)) == top for r in ids.tolist())
    got = key.gather(1, ids.long())
    assert torch.all((got - key.topk(top, dim=1).values).abs() <= 2 * tol), "choice"
    assert torch.all((wts[:, :top].double() - 1.5 * s.gather(1, ids.long())).abs() <= 2 * tol)
    if gate:
        assert torch.all((wts[:, top].double() - s[:, E]).abs() <= tol)


def test_router_ties_go_to_the_lower_index():
    h = torch.ones(2, 64, device=DEV, dtype=torch.bfloat16)
    wr = torch.zeros(64, 64, device=DEV, dtype=torch.bfloat16)
    wr[40:44] = 0.125
    ids, wts = P.route(h, wr, 6)
    assert ids.tolist() == [[40, 41, 42, 43, 0, 1]] * 2 and torch.equal(wts[:, 4], wts[:, 5])
