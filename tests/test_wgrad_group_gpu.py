"""Weight gradients of several linears in one launch (csrc/kernels/gemm_wgrad.hip: wgrad_group_kernel) against float64."""
import pytest
import torch

from penroz.ops import _ext, gemm

GPT2 = [(768, 3072), (3072, 768), (768, 768), (2304, 768)]


@pytest.mark.skipif(not _ext.available(), reason="HIP extension not built")
@pytest.mark.parametrize("shapes,K,tile", [(GPT2, 1, 128), (GPT2, 3885, 128), (GPT2, 16384, 256), (GPT2, 65536, 0),
                                           ([(50304, 768)], 256, 128), ([(50304, 768)], 4096, 0), ([(768, 768)], 0, 0),
                                           ([(0, 768)], 64, 0), ([(768, 768)] * 9, 64, 128)])
def test_wgrad_group_rule(shapes, K, tile):
    assert _ext.kernels().wgrad_group_tile([m for m, _ in shapes], [n for _, n in shapes], K, 256) == tile
    beside = 0 if shapes[0][0] == 50304 else tile  # several rounds of workgroups: not beside another stream
    assert _ext.kernels().wgrad_group_tile([m for m, _ in shapes], [n for _, n in shapes], K, 256, True) == beside


@pytest.mark.skipif(not _ext.available(), reason="HIP extension not built")
@pytest.mark.parametrize("shape", [*GPT2, (1152, 6912), (1536, 1152), (64, 64)])
@pytest.mark.parametrize("K", [64, 1024, 4096])
def test_a_product_by_itself_beside_a_second_stream_is_the_split_kernels(shape, K):
    assert _ext.kernels().wgrad_group_tile([shape[0]], [shape[1]], K, 256, True) == 0


def _products(shapes, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for m, n in shapes:
        rows = torch.randn(K, (m + 7) // 8 * 8, generator=g, device="cuda").bfloat16()  # m % 8 != 0: padded rows
        out.append((rows[:, :m], torch.randn(K, n, generator=g, device="cuda").bfloat16(),
                    torch.randn(m, n, generator=g, device="cuda")))
    return out


def _check(shapes, K, accumulate, products):
    want = [dy.double().t() @ x.double() + (g.double() if a else 0.0) for (dy, x, g), a in zip(products, accumulate)]
    gemm.wgrad_group(*zip(*products), accumulate)
    for (dy, x, g), w in zip(products, want):
        # fp32 sums: of 32 products in the MFMA, of 8 of those, of K / 256 of these
        bound = 2.0 ** -24 * (K / 256 + 8 + 32) ** 0.5
        assert torch.linalg.norm(g.double() - w) <= bound * torch.linalg.norm(w)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [1, 31, 32, 33, 95, 129, 257, 1000, 2049])
@pytest.mark.parametrize("shapes", [[(128, 128)], [(8, 8)], [(77, 136)], [(129, 264), (8, 1000), (300, 8), (256, 128)],
                                    [(40, 24)] * 8, [(768, 768), (1003, 72)]])
def test_wgrad_group(shapes, K):
    for accumulate in ([False] * len(shapes), [i % 2 == 0 for i in range(len(shapes))]):
        _check(shapes, K, accumulate, _products(shapes, K))


@pytest.mark.gpu
@pytest.mark.parametrize("shapes,K", [(GPT2, 16384), ([(777, 3080), (3072, 776), (768, 768), (2304, 768)], 16385)])
def test_wgrad_group_wide_tiles(shapes, K):
    assert _ext.kernels().wgrad_group_tile([m for m, _ in shapes], [n for _, n in shapes], K, 256) == 256
    _check(shapes, K, [True, False, True, False], _products(shapes, K))


@pytest.mark.gpu
def test_wgrad_group_of_other_forms():
    """More than 8 products, several K, no rows at all, operands off 16 bytes: as one after the other."""
    _check(*(lambda s: (s, 64, [True] * 9, _products(s, 64)))([(64, 64)] * 9))
    a, b = _products([(64, 128)], 40)[0], _products([(128, 64)], 72)[0]
    _check(None, 72, [False, True], [a, b])
    dy, x, g = _products([(64, 64)], 0)[0]
    gemm.wgrad_group([dy], [x], [g], [False])
    assert not g.any()
    dy, x, g = _products([(64, 64)], 32)[0]
    flat = torch.zeros(64 * 64 + 1, device="cuda")
    off = flat[1:].view(64, 64)
    off.copy_(g)
    _check(None, 32, [True], [(dy, x, off)])


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [(0, 128), (64, 192)])  # the same gradient, half of it
def test_gradients_that_share_memory_are_written_in_order(rows):
    g = torch.Generator(device="cuda").manual_seed(0)
    dys = [torch.randn(96, 128, generator=g, device="cuda").bfloat16() for _ in range(2)]
    xs = [torch.randn(96, 64, generator=g, device="cuda").bfloat16() for _ in range(2)]
    buf = torch.randn(192, 64, generator=g, device="cuda")
    assert _ext.kernels().wgrad_group_tile([128, 128], [64, 64], 96, 256) == 128  # apart they go in one launch
    want = buf.double()
    want[:128] = dys[0].double().t() @ xs[0].double()
    want[rows[0]:rows[1]] += dys[1].double().t() @ xs[1].double()
    gemm.wgrad_group(dys, xs, [buf[:128], buf[rows[0]:rows[1]]], [False, True])
    assert torch.linalg.norm(buf.double() - want) <= 2.0 ** -24 * 8 * torch.linalg.norm(want)
