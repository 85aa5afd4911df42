"""Experts of few pairs (csrc/kernels/experts.hip): weights by whole lines, each width's kernel and the one for any width, against
float64."""
import pytest
import torch

from penroz.ops import packed as P

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _chosen(N, E, top, spread):
    """ids [N, top]: ``spread`` experts share all pairs, each row's are distinct."""
    if top == 1:
        return torch.randint(0, spread, (N, 1))
    return torch.stack([torch.randperm(spread)[:top] for _ in range(N)])


# pairs per expert: 8, 9, 16, 17 and many; pairs fewer than experts (and several of one), as many, more; blocks of 16 and 32 rows
@pytest.mark.parametrize("N,E,top,spread", [(1, 1, 1, 1), (8, 1, 1, 1), (9, 4, 1, 1), (16, 1, 1, 1), (17, 2, 1, 1), (100, 3, 2, 2),
                                            (1, 64, 6, 64), (5, 64, 3, 4), (16, 48, 3, 48), (60, 16, 4, 16), (260, 20, 3, 20),
                                            (512, 64, 2, 64)])
# widths: every kernel of 256 columns per step, and widths in between, off 64 columns, and above
@pytest.mark.parametrize("kind,C,F", [(P.UNGATED, 256, 512), (1, 512, 256), (1, 768, 1024), (P.UNGATED, 1024, 768), (1, 1536, 32),
                                      (P.UNGATED, 2048, 1536), (0, 2304, 96), (P.UNGATED, 32, 2048), (1, 160, 1280), (0, 2080, 64),
                                      (0, 1664, 448)])
def test_expert_rows(N, E, top, spread, kind, C, F):
    torch.manual_seed(N + 31 * E + C)
    ids = _chosen(N, E, top, spread)
    h = torch.randn(N, C).bfloat16().to(DEV)
    g, u = ((torch.randn(E, F, C) * C ** -0.5).bfloat16().to(DEV) for _ in range(2))
    d = (torch.randn(E, C, F) * F ** -0.5).bfloat16().to(DEV)
    gated = kind != P.UNGATED
    w = P.pack_experts(g if gated else None, u, d)
    y = P.experts(h, ids.int().to(DEV), w, kind, 0.7).view(N, top, C).double()
    for e in range(spread):
        r, k = (ids == e).nonzero(as_tuple=True)
        if not r.numel():
            continue
        x = h[r.to(DEV)].double()
        a = P.expert_activation(x @ g[e].double().t() if gated else None, x @ u[e].double().t(), kind, 0.7)
        want = a @ d[e].double().t()
        # the hidden row is rounded to bf16 (2^-9), and the result (2^-9); fp32 sums of C and F terms are far below
        tol = 2.0 ** -8 * (a.abs() @ d[e].double().abs().t()) + 2.0 ** -8 * want.abs() + 1e-6
        assert torch.all((y[r.to(DEV), k.to(DEV)] - want).abs() <= tol), (e, r.numel())


@pytest.mark.parametrize("N,E,top", [(1, 8, 2), (3, 8, 3), (8, 2, 2), (9, 40, 4), (16, 3, 3), (16, 64, 6), (17, 8, 2)])
@pytest.mark.parametrize("C,F,S", [(256, 256, 512), (512, 1024, 2048), (1024, 768, 1536), (2048, 512, 1024), (1536, 256, 512),
                                   (512, 256, 768), (256, 1536, 3072), (288, 256, 512)])
def test_shared_expert_beside(N, E, top, C, F, S):
    """The shared expert in the experts' launches, and where it keeps its own (17 rows, other widths)."""
    torch.manual_seed(N + C + F)
    ids = _chosen(N, E, top, E).int().to(DEV)
    h = torch.randn(N, C).bfloat16().to(DEV)
    u, d = ((torch.randn(E, *s) * s[1] ** -0.5).bfloat16().to(DEV) for s in ((F, C), (C, F)))
    su, sd = ((torch.randn(*s) * s[1] ** -0.5).bfloat16().to(DEV) for s in ((S, C), (C, S)))
    w = P.pack_experts(None, u, d)
    both = P.kernels().experts_rows_shared(h, ids, w["gu"], w["down"], 0.0, su, sd)
    assert (both is not None) == (N <= 16 and S == 2 * F and F <= 1024 and C % 256 == 0)
    y, out = P.experts_beside_shared(h, ids, w, P.UNGATED, 0.0, {"up": su, "down": sd})
    if both is not None:
        assert torch.equal(y, both[0]) and torch.equal(out, both[1])
    assert torch.equal(y, P.experts(h, ids, w, P.UNGATED, 0.0))
    pre = h.double() @ su.double().t()
    a = torch.nn.functional.gelu(pre)
    # the hidden row is rounded to bf16 before (|gelu'| < 1.2) and after the activation, and the result: 2^-9 each
    tol = 2.0 ** -9 * (1.2 * pre.abs() + a.abs()) @ sd.double().abs().t() + 2.0 ** -8 * (a @ sd.double().t()).abs() + 1e-5
    assert torch.all((out.double() - a @ sd.double().t()).abs() <= tol)


@pytest.mark.parametrize("N,C,F,S", [(16, 512, 256, 768), (4, 512, 256, 256), (17, 512, 256, 512), (2, 288, 96, 192)])
def test_refused_shared_expert_allocates_nothing(N, C, F, S):
    """Where the shared expert keeps its own launches, a step allocates what those do."""
    ids = _chosen(N, 8, 2, 8).int().to(DEV)
    r = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    h, w, shared = r(N, C), {"gu": r(8, F, C), "down": r(8, C, F)}, {"up": r(S, C), "down": r(C, S)}
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]

    def both():
        return P.experts_beside_shared(h, ids, w, P.UNGATED, 0.0, shared)

    def alone():
        return P.experts(h, ids, w, P.UNGATED, 0.0), P.gelu_mlp(h, **shared)

    used = []
    for f in (both, alone, both, alone):
        n = count()
        out = f()
        used.append(count() - n)
        del out
    assert used[2] == used[3]
