"""Decode attention of short contexts (csrc/kernels/decode_attn.hip: decode_small_kernel) where its work is split: heads of a group
over workgroups, keys over waves and blocks of 16, many items; the new key and value from this step's rows, NaN behind the length."""
import pytest
import torch

from penroz.ops import _ext

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _reference(q, k, v, scale):
    """float64: q [B, H, D], k, v [B, Hkv, S, D]; products element by element (no library product)."""
    G = q.shape[1] // k.shape[1]
    k, v = k.double().repeat_interleave(G, 1), v.double().repeat_interleave(G, 1)
    w = ((q.double()[:, :, None] * k).sum(-1) * scale).softmax(-1)
    return (w[..., None] * v).sum(2)


@pytest.mark.parametrize("D,G,B,Hkv", [
    (64, 1, 5, 13), (64, 4, 1, 2), (64, 4, 7, 5), (64, 16, 3, 1), (128, 1, 9, 1), (128, 2, 40, 2), (128, 8, 2, 3), (128, 16, 17, 1),
    (256, 1, 3, 1), (256, 4, 3, 1), (256, 4, 9, 1), (256, 4, 33, 1), (256, 8, 2, 1), (256, 16, 1, 1), (256, 1, 257, 1), (512, 1, 1, 1),
    (512, 2, 33, 1), (512, 4, 2, 1), (512, 8, 5, 1)])
@pytest.mark.parametrize("S", [1, 16, 17, 63, 129, 1000])
def test_decode_small(D, G, B, Hkv, S):
    torch.manual_seed(D + G + B + S)
    cap, H = 1024, G * Hkv
    kc, vc = (torch.full((B, Hkv, cap, D), float("nan"), device=DEV, dtype=torch.bfloat16) for _ in range(2))
    kc[:, :, :S - 1] = torch.randn(B, Hkv, S - 1, D, device=DEV).to(torch.bfloat16)
    vc[:, :, :S - 1] = torch.randn(B, Hkv, S - 1, D, device=DEV).to(torch.bfloat16)
    qkv = torch.randn(B, 1, (H + 2 * Hkv) * D, device=DEV).to(torch.bfloat16)
    q = qkv[:, :, :H * D].view(B, 1, H, D)
    k, v = (qkv[:, :, (H + i * Hkv) * D:(H + (i + 1) * Hkv) * D].view(B, 1, Hkv, D) for i in (0, 1))
    K, scale = _ext.kernels(), D ** -0.5
    assert K.decode_small_applies(B, 1, H, Hkv, D, cap) == (B * Hkv <= 256 or D != 256)
    full = [t.clone() for t in (kc, vc)]
    for t, new in zip(full, (k, v)):
        t[:, :, S - 1] = new[:, 0]
    length = torch.tensor([S], device=DEV)
    out = K.decode_attn(q, kc, vc, None, None, cap, cap - 1, scale, length, k, v)
    ref = _reference(q[:, 0], full[0][:, :, :S], full[1][:, :, :S], scale).view(B, 1, H * D)
    # scores and weights in fp32: one bf16 rounding of the result (2^-9) and fp32 sums of up to 1024 terms
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -14
    assert torch.all((out.double() - ref).abs() <= bound), float(((out.double() - ref).abs() / bound).max())
    for t, f in zip((kc, vc), full):
        assert torch.equal(t.view(torch.int16), f.view(torch.int16)), "cache"


@pytest.mark.parametrize("D,G,rope", [(128, 8, False), (128, 2, True), (256, 4, False), (256, 4, True), (512, 2, False)])
@pytest.mark.parametrize("S", [1, 40, 200])
def test_cache_off_16_bytes(D, G, rope, S):
    """A cache that is a view at an odd offset: read without LDS-DMA, by another kernel or straight, the same answer."""
    torch.manual_seed(D + G + S)
    B, Hkv, cap = 2, 1, 256
    H = G * Hkv

    def cache():
        return torch.randn(B * Hkv * cap * D + 1, device=DEV).to(torch.bfloat16)[1:].view(B, Hkv, cap, D)

    kc, vc = cache(), cache()
    qkv = torch.randn(B, 1, (H + 2 * Hkv) * D, device=DEV).to(torch.bfloat16)
    q = qkv[:, :, :H * D].view(B, 1, H, D)
    k, v = (qkv[:, :, (H + i * Hkv) * D:(H + (i + 1) * Hkv) * D].view(B, 1, Hkv, D) for i in (0, 1))
    ang = torch.rand(D // 2, device=DEV) * 6
    cos, sin = ang.cos(), ang.sin()

    def turn(x):  # rotate-half in fp32, rounded to bf16 as the kernel keeps it
        if not rope:
            return x
        a, b = x.float().split(D // 2, -1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1).to(torch.bfloat16)

    full = [t.clone() for t in (kc, vc)]
    full[0][:, :, S - 1], full[1][:, :, S - 1] = turn(k)[:, 0], v[:, 0]
    ref = _reference(turn(q)[:, 0], full[0][:, :, :S], full[1][:, :, :S], D ** -0.5).view(B, 1, H * D)
    out = _ext.kernels().decode_attn(q, kc, vc, None, None, cap, cap - 1, D ** -0.5, torch.tensor([S], device=DEV), k, v, None,
                                     *((cos, sin) if rope else (None, None)))
    # as above; a fused multiply-add in the rotation may round a query or the new key to its other neighbour: 2^-9 of each of D
    # products of a score, whose spread is 1
    bound = 2.0 ** -8 * ref.abs() + (2.0 ** -5 if rope else 2.0 ** -14)
    assert torch.all((out.double() - ref).abs() <= bound), float(((out.double() - ref).abs() / bound).max())
    assert torch.equal(vc, full[1]) and torch.equal(kc[:, :, :S - 1], full[0][:, :, :S - 1]) and torch.equal(kc[:, :, S:], full[0][:, :, S:])
    assert torch.all((kc[:, :, S - 1].float() - full[0][:, :, S - 1].float()).abs() <= 2.0 ** -7 * full[0][:, :, S - 1].float().abs() + 2.0 ** -14)
