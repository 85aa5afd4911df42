"""Weights read past the caches: what a decode step's weights are together decides (ops/gemm.py: past_caches), not the kernel's
layout, and the sums are the same bits either way."""
import pytest
import torch

import bench
import zozenex_util as Z
from penroz.models import graph_decode as gd
from penroz.models import zozenex
from penroz.models.mapper import Mapper
from penroz.models.model import NeuralNetworkModel
from penroz.models.packed import PackedProgram
from penroz.ops import _ext, gemm
from penroz.ops import packed as P

DEV = "cuda"
MB = 1 << 20


def _w(sizes):
    return [torch.empty(m * MB, dtype=torch.uint8, device="meta") for m in sizes]


@pytest.mark.parametrize("weights,experts,want", [
    ([], [], (gemm.KEEP, False)),
    ([1] * 20 + [64], [], (gemm.KEEP, False)),                    # fits whole
    ([192], [], (gemm.KEEP, False)),
    ([193], [], (193 * MB, True)),
    ([3] * 40 + [77], [], (77 * MB, True)),                       # the layers do
    ([77] + [4] * 40, [], (4 * MB, True)),
    ([2] * 26 + [4] * 12 + [32] * 26 + [604], [], (32 * MB, True)),
    ([4] * 20, [50] * 8, (gemm.KEEP, True)),                      # beside experts that pass
    ([4] * 20 + [64], [50] * 8, (64 * MB, True)),
    ([4] * 10, [25] * 4, (gemm.KEEP, False)),                     # a small mixture
])
def test_rule(weights, experts, want):
    assert gemm.past_caches(_w(weights), _w(experts)) == want


def test_programs_ask_for_their_own_weights(monkeypatch):
    cfg = Z.config()
    sd = Z.weights(cfg)
    m = NeuralNetworkModel("t", Mapper(zozenex.layers_from_config(cfg, sd), {"adamw": {"lr": 1e-3}})).to(torch.bfloat16)

    def thresholds():
        p = PackedProgram.build(m)
        subs = [s for _, s, _ in p.steps]
        subs += [q for s in subs if hasattr(s, "left") for q in (s.left, s.right)]
        return p, {(s.past, s.experts_past) for s in subs}

    p, seen = thresholds()
    assert seen == {(p.past, False)} == {(gemm.KEEP, False)}  # some kilobytes
    monkeypatch.setattr(gemm, "CACHE_BYTES", 0)
    monkeypatch.setattr(gemm, "HELD_BYTES", p.head.nbytes)
    p, seen = thresholds()
    assert p.past < gemm.KEEP and seen == {(p.past, True)}
    gpt = NeuralNetworkModel("g", Mapper(bench.gpt2_layers(V=256, C=128, L=2, H=2, P=16), {"sgd": {"lr": 0.1}})).to(torch.bfloat16)
    monkeypatch.setattr(gemm, "HELD_BYTES", 2 * 128 * (2 * 128 + 256 + 2 * 384))  # projections, head and QKV
    prog = gd.GPTDecodeProgram.build(gpt)
    assert prog.past == prog.spec.blocks[0].fc.weight.nbytes


gpu = pytest.mark.gpu


def _randn(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


@gpu
@pytest.mark.parametrize("M,N,K,rpw", [(1, 16384, 256, 0), (3, 16391, 520, 0), (4, 20000, 1152, 0), (2, 16400, 3000, 0), (1, 16385, 8192, 0),
                                       (1, 50, 4616, 0), (4, 333, 6912, 0), (3, 64, 8192, 0), (2, 999, 768, 8)])
def test_gemv(M, N, K, rpw):
    """The vocabulary's waves and long rows; their ends."""
    x, w, b = _randn(M, K, seed=1), _randn(N, K, seed=2), _randn(N, seed=3)
    out = torch.full((2, M, N), 7.0, device=DEV, dtype=torch.bfloat16)
    for past in (False, True):
        _ext.kernels().decode_gemv(x, None, None, None, None, None, None, 0.0, w, b, out[int(past)], 0, rpw, past=past)
    assert torch.equal(out[0], out[1])
    want = x.double() @ w.double().t() + b.double()
    assert ((out[1].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -18 * K ** 0.5).all()


@gpu
@pytest.mark.parametrize("M,I,K", [(1, 512, 256), (2, 1000, 520), (3, 6912, 1152), (4, 24, 1792)])
def test_gated_gemv(M, I, K):
    x, w = _randn(M, K, seed=4), _randn(2 * I, K, seed=5, scale=K ** -0.5)
    a, b = (P.gated_linear(x, w, 0, past=past) for past in (gemm.KEEP, 0))
    assert torch.equal(a, b) and a.isfinite().all()


@gpu
@pytest.mark.parametrize("M,N,K,tile", [(16, 4096, 2048, 6), (16, 4090, 2304, 6), (32, 4608, 2048, 1), (33, 3000, 4096, 1), (64, 8192, 2048, 2),
                                        (17, 8200, 1032, 2), (64, 12288, 2048, 3), (48, 9001, 1024, 3), (64, 16400, 1024, 4),
                                        (16, 32768, 1024, 4), (64, 50304, 768, 5), (12, 50304, 192, 5), (16, 32768, 2048, 5)])
def test_rows_gemm(M, N, K, tile):
    """Every tile with weights of 16 MB and more (and, of the same tile, of less)."""
    assert _ext.kernels().rows_gemm_tile(M, N, K) == tile
    x, w = _randn(M, K, seed=6), _randn(N, K, seed=7)
    a, b = (gemm.rows_linear(x, w, past=past) for past in (False, True))
    assert torch.equal(a, b)
    want = x.double() @ w.double().t()
    assert ((b.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -18 * K ** 0.5).all()


@gpu
@pytest.mark.parametrize("kind,C,F", [(P.UNGATED, 256, 512), (1, 768, 1024), (1, 2048, 1536), (0, 160, 576), (1, 1664, 416)])
@pytest.mark.parametrize("N,E,top", [(1, 16, 2), (9, 2, 1), (40, 3, 2)])
def test_experts(N, E, top, kind, C, F):
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(i))[:top] for i in range(N)]).int().to(DEV)
    w = {"gu": _randn(E, F if kind == P.UNGATED else 2 * F, C, seed=8, scale=C ** -0.5), "down": _randn(E, C, F, seed=9, scale=F ** -0.5)}
    h = _randn(N, C, seed=10)
    assert P.few_pairs(N * top, w)
    a, b = (P.experts(h, ids, w, kind, 0.7, past) for past in (False, True))
    assert torch.equal(a, b) and a.isfinite().all()


@gpu
@pytest.mark.parametrize("N", [3, 16])
def test_shared_expert(N):
    C, F, E = 512, 256, 8
    ids = torch.randint(0, E, (N, 2), generator=torch.Generator().manual_seed(1)).int().to(DEV)
    w = {"gu": _randn(E, F, C, seed=11, scale=C ** -0.5), "down": _randn(E, C, F, seed=12, scale=F ** -0.5)}
    shared = {"up": _randn(2 * F, C, seed=13, scale=C ** -0.5), "down": _randn(C, 2 * F, seed=14, scale=(2 * F) ** -0.5)}
    h = _randn(N, C, seed=15)
    (a, sa), (b, sb) = (P.experts_beside_shared(h, ids, w, P.UNGATED, 0.0, shared, experts_past=past) for past in (False, True))
    assert torch.equal(a, b) and torch.equal(sa, sb)
