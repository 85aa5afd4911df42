"""Which kernel a step's experts take (ops/packed.py: few_pairs), and both against float64 on either side of the line."""
import pytest
import torch

from penroz.ops import packed as P

DEV = "cuda"


def _w(E, C, F, gated=True):
    t = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device="meta")
    return {"gu": t(E, 2 * F if gated else F, C), "down": t(E, C, F)}


@pytest.mark.parametrize("w,P_,few", [
    (_w(64, 2048, 1024), 1024, True), (_w(64, 2048, 1024), 1025, False),  # the pair list
    (_w(8, 2048, 1024), 255, True), (_w(8, 2048, 1024), 256, False),      # 32 pairs per expert of large ones
    (_w(4, 2048, 1024), 128, False), (_w(4, 2048, 1024, gated=False), 128, True),  # 48 and 32 MB
    (_w(4, 64, 64), 383, True), (_w(4, 64, 64), 384, False),              # 96 of any
    (_w(2, 4096, 4096), 255, True), (_w(1, 64, 64), 256, False),          # of two or one, 256 in all
    (_w(1, 32768, 32768), 1024, True),                                    # past the tiles' 32-bit offsets
    (_w(8, 2048, 1024), 0, True),
])
def test_rule(w, P_, few):
    assert P.few_pairs(P_, w) == few


@pytest.mark.gpu
@pytest.mark.parametrize("kind,E,C,F,N,top", [(1, 8, 2048, 800, 127, 2), (1, 8, 2048, 800, 128, 2), (P.UNGATED, 3, 96, 160, 95, 3),
                                              (P.UNGATED, 3, 96, 160, 96, 3), (0, 1, 32, 32, 255, 1), (0, 1, 32, 32, 256, 1), (1, 5, 544, 64, 200, 5)])
def test_either_side(kind, E, C, F, N, top):
    g = torch.Generator().manual_seed(E + N)
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(N)])
    r = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).bfloat16().to(DEV)
    h, wg, u, d = r(N, C), r(E, F, C, scale=C ** -0.5), r(E, F, C, scale=C ** -0.5), r(E, C, F, scale=F ** -0.5)
    gated = kind != P.UNGATED
    y = P.experts(h, ids.int().to(DEV), P.pack_experts(wg if gated else None, u, d), kind, 0.7).view(N, top, C).double()
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        x = h[t.to(DEV)].double()
        a = P.expert_activation(x @ wg[e].double().t() if gated else None, x @ u[e].double().t(), kind, 0.7)
        want = a @ d[e].double().t()
        # the hidden row is rounded to bf16 (2^-9), and the result (2^-9); fp32 sums of C and F terms are far below
        tol = 2.0 ** -8 * (a.abs() @ d[e].double().abs().t()) + 2.0 ** -8 * want.abs() + 1e-6
        assert torch.all((y[t.to(DEV), k.to(DEV)] - want).abs() <= tol), e


@pytest.mark.gpu
@torch.inference_mode()  # (as decoders capture; torch's generator state of a process is of the first capture's mode)
def test_tiles_in_a_captured_step():
    """What was a captured step of the few-pairs kernel is one of the sort and the tiles: every replay on new rows and choices."""
    E, C, F, N, top = 8, 2048, 800, 128, 2
    g = torch.Generator(device=DEV).manual_seed(5)
    r = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).bfloat16()
    w = {"gu": r(E, F, C, scale=C ** -0.5), "down": r(E, C, F, scale=F ** -0.5)}
    assert not P.few_pairs(N * top, w)
    choose = lambda: torch.rand(N, E, generator=g, device=DEV).topk(top, dim=1).indices.int()
    h, ids = r(N, C), choose()
    P.experts(h, ids, w, P.UNGATED, 0.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = P.experts(h, ids, w, P.UNGATED, 0.0)
    for _ in range(4):
        h.copy_(r(N, C))
        ids.copy_(choose())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, P.experts(h, ids, w, P.UNGATED, 0.0))


class _Kernels:
    """Notes the elements of each call's input and hidden rows, and counts its pairs."""

    def __init__(self):
        self.calls, self.rows = [], 0

    def experts_rows(self, h, ids, gu, down, kind, limit, act, y, past):
        self.calls.append((h.numel(), act.numel()))
        assert ids.shape[0] == h.shape[0] and act.shape[0] == y.shape[0] == ids.numel() and past
        self.rows += y.shape[0]


@pytest.mark.parametrize("N,top,C,F,calls", [(16, 6, 2048, 1024, 1), (100, 2, 32, (1 << 24) - 32, 2), (64, 1, 32, 1 << 25, 2),
                                             (127, 1, 1 << 24, 32, 1), (128, 1, 1 << 24, 32, 2), (3, 2, 32, (1 << 30) - 32, 3)])
def test_few_pairs_within_32_bit_offsets(monkeypatch, N, top, C, F, calls):
    """One call where the input rows lie within them, more of fewer tokens where not."""
    K = _Kernels()
    monkeypatch.setattr(P, "kernels", lambda: K)
    monkeypatch.setattr(P, "use_kernels", lambda h: True)
    t = lambda *s, dtype=torch.bfloat16: torch.empty(*s, dtype=dtype, device="meta")
    w = {"gu": t(8, F, C), "down": t(8, C, F)}
    assert P.few_pairs(N * top, w)
    P.experts(t(N, C), t(N, top, dtype=torch.int32), w, P.UNGATED, 0.0, True)
    assert K.rows == N * top and len(K.calls) == calls and max(max(c) for c in K.calls) < 1 << 31


@pytest.mark.gpu
@pytest.mark.parametrize("C,F", [(32, (1 << 24) + (1 << 15)), ((1 << 24) + (1 << 15), 32)])
def test_rows_past_32_bit_offsets(C, F):
    """Input or hidden rows of 4 GiB and more: the last pairs, of another expert than the first, have the bits that they have alone."""
    N = 128
    ids = (torch.arange(N, device=DEV) >= N // 2).int().view(N, 1)
    g = torch.Generator(device=DEV).manual_seed(C)
    r = lambda *s, scale: torch.empty(*s, dtype=torch.bfloat16, device=DEV).normal_(0, scale, generator=g)
    h, w = r(N, C, scale=1.0), {"gu": r(2, F, C, scale=C ** -0.5), "down": r(2, C, F, scale=F ** -0.5)}
    assert P.few_pairs(N, w)
    y = P.experts(h, ids, w, P.UNGATED, 0.0)
    last = P.experts(h[-4:], ids[-4:], w, P.UNGATED, 0.0)
    assert torch.equal(y[-4:], last) and last.float().std() > 0.1 and not torch.equal(y[:4], last)
