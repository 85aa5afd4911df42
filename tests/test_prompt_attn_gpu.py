"""Attention of several query rows per sequence over a bf16 cache (csrc/kernels/prompt_attn.hip, and decode_kernel where the
rows are few) against float64."""
import math

import pytest
import torch

from penroz.ops import _ext

pytestmark = pytest.mark.gpu


def exact(q, k, v, off):
    B, T, H, D = q.shape
    k, v = (t.double().repeat_interleave(H // t.shape[1], 1) for t in (k[:, :, :off + T], v[:, :, :off + T]))
    s = torch.matmul(q.double().transpose(1, 2), k.transpose(2, 3).contiguous()) / math.sqrt(D)
    dead = torch.ones(T, off + T, dtype=torch.bool, device=q.device).triu(off + 1)
    p = s.masked_fill(dead, float("-inf")).softmax(-1)
    return torch.matmul(p, v).transpose(1, 2).reshape(B, T, H * D)


def make(B, T, H, Hkv, D, off, cap, seed=0):
    B = max(B, -(-1024 // T)) if D > 128 and T > 1 else B  # from where wide heads take the kernel
    g = torch.Generator(device="cuda").manual_seed(seed)
    qkv = torch.randn(B, T, (H + 2) * D, generator=g, device="cuda").bfloat16()
    q = qkv[..., :H * D].unflatten(-1, (H, D))  # a view into wider rows, as the fused projection gives it
    k, v = (torch.randn(B, Hkv, cap, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    k[:, :, off + T:], v[:, :, off + T:] = float("nan"), float("nan")  # slots that nothing may read into a result
    return q, k, v


def attend(q, k, v, off):
    T, D = q.shape[1], q.shape[3]
    return _ext.kernels().decode_attn(q, k, v, None, None, off + T, off, 1 / math.sqrt(D), None, None, None, None, None,
                                      None)


@pytest.mark.parametrize("D", [64, 128, 256, 512])
@pytest.mark.parametrize("B,T,H,Hkv,off", [
    (1, 2, 4, 4, 0), (3, 16, 4, 2, 5), (2, 17, 3, 1, 0), (1, 63, 2, 2, 1), (2, 64, 2, 2, 0), (2, 65, 4, 1, 64),
    (9, 33, 4, 4, 31), (1, 5, 4, 1, 1043), (1, 130, 16, 1, 300), (1, 1, 2, 1, 40)])
def test_prompt_attention(D, B, T, H, Hkv, off):
    q, k, v = make(B, T, H, Hkv, D, off, off + T + 7)
    ref = exact(q, k, v, off)
    out = attend(q, k, v, off).double()
    # the result's own rounding to bf16 is at most 2^-8 of it; the weights' 16 bits and exponentials are 2^-16 of the
    # largest value that they weigh
    bound = 2 ** -7.9 * ref.abs() + 2 ** -16 * v[:, :, :off + T].abs().max().double()
    assert ((out - ref).abs() <= bound).all()


@pytest.mark.parametrize("D", [64, 128, 256, 512])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_value_that_is_not_finite_stays_with_the_rows_that_see_it(D, bad):
    q, k, v = make(2, 70, 4, 2, D, 3, 80)
    ref = exact(q, k, v, 3)
    v[1, 1, 40, 7] = bad
    out = attend(q, k, v, 3).double().view(-1, 70, 4, D)
    ref = ref.view(-1, 70, 4, D)
    hit = torch.zeros_like(ref, dtype=torch.bool)
    hit[1, 37:, 2:, 7] = True  # position 3 + tq >= 40, the heads of KV head 1
    assert ((out - ref).abs()[~hit] <= 0.02).all()
    assert (torch.isnan(out[hit]) if bad != bad else out[hit] == bad).all()


@pytest.mark.parametrize("score", [float("inf"), float("nan")])
def test_scores_without_a_softmax_give_zero(score):
    q, k, v = make(1, 40, 2, 2, 64, 0, 40)
    q = q.contiguous()
    q[0, 20, 1] = 1.0
    k[0, 1, 5] = score  # (the row's score is then inf or NaN; the general kernel gives 0 for such a row)
    out = attend(q, k, v, 0).view(1, 40, 2, 64)
    ref = torch.cat([attend(q[:, i:i + 1].contiguous(), k, v, i) for i in range(40)], 1).view(1, 40, 2, 64)
    assert torch.equal(out == 0, ref == 0)
    assert (out[0, 20, 1] == 0).all()


def test_rows_off_sixteen_bytes_and_repeat():
    q, k, v = make(2, 20, 2, 2, 64, 4, 30)
    wide = torch.zeros(2, 20, 2 * 64 + 3, device="cuda", dtype=torch.bfloat16)
    wide[..., 1:129] = q.reshape(2, 20, 128)
    a = attend(wide[..., 1:129].unflatten(-1, (2, 64)), k, v, 4)
    assert torch.equal(a, attend(q, k, v, 4)) and torch.equal(a, attend(q, k, v, 4))


@pytest.mark.parametrize("D", [64, 128, 256, 512])
def test_weights_keep_all_of_fp32(D):
    """Values of the last three keys that cancel the others' sum, to bf16 each: what is left of it is the weights' own error."""
    B, T, H, Hkv = (512 if D > 128 else 24), 2, 4, 1
    g = torch.Generator(device="cuda").manual_seed(D)
    q = torch.randn(B, T, H, D, generator=g, device="cuda").bfloat16()
    q[:] = q[:, :, :1].clone()  # the heads of the group weigh alike, so that one value cancels for all of them
    k, v = (torch.randn(B, Hkv, 6, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    k[:, :, 3:], v[:, :, 3:] = 0, 0
    p = torch.matmul(q[:, 1, :1].double().unsqueeze(1), k.double().transpose(2, 3).contiguous()).div(math.sqrt(D)).softmax(-1)
    for c in (3, 4, 5):
        v[:, :, c] = (-torch.matmul(p, v.double())[:, :, 0] / p[:, :, 0, c:c + 1]).bfloat16()
    ref, size = torch.matmul(p, v.double())[:, 0], torch.matmul(p, v.double().abs())[:, 0]
    out = attend(q, k, v, 4).view(B, T, H, D)[:, 1].double()
    # fp32 exponentials and sums of six values: a few steps of 2^-24 each; weights of 16 bits are off by up to 2^-18
    assert ((out - ref).abs() <= 2.0 ** -20 * size + 2.0 ** -8 * ref.abs()).all()


# D, B, Tq, H, Hkv, keys -> the kernel of many rows (True) or a workgroup per row
@pytest.mark.parametrize("sizes,many", [
    ((64, 1, 64, 12, 12, 64), True), ((64, 1, 16, 12, 12, 416), False), ((64, 1, 16, 12, 12, 1016), True),
    ((64, 64, 4, 12, 12, 40), True), ((64, 16, 4, 8, 8, 100), False), ((64, 1, 2, 8, 2, 2), True),
    ((128, 1, 2, 8, 8, 402), False), ((128, 1, 2, 8, 8, 1002), True), ((128, 16, 4, 8, 8, 404), True),
    ((256, 1, 2, 8, 8, 240), False), ((256, 1, 2, 8, 8, 241), True), ((256, 3, 200, 4, 1, 200), True),
    ((256, 1, 9, 4, 1, 9), True), ((512, 1, 2, 8, 8, 202), False), ((512, 1, 2, 8, 8, 402), True),
    ((512, 1, 2, 8, 2, 20), False), ((512, 1, 2, 8, 2, 32), True), ((512, 8, 100, 8, 8, 100), True),
    ((32, 8, 100, 8, 8, 100), False), ((64, 8, 1, 8, 8, 100), False)])
def test_rule_of_rows_and_keys(sizes, many):
    D, B, Tq, H, Hkv, keys = sizes
    assert _ext.kernels().prompt_attn_applies(B, Tq, H, Hkv, D, keys) == many


def test_keys_of_a_part_as_asked_for():
    splits = _ext.kernels().prompt_attn_splits
    assert splits(12, 64, 1000, 64) == 5 and splits(12, 64, 1000, 64, 64) == 16 and splits(12, 64, 1000, 64, 4096) == 1
    assert splits(600, 64, 1000, 64, 64) == 1 and splits(256, 64, 1000, 64, 64) == 2


@pytest.mark.parametrize("D", [64, 128, 256, 512])
@pytest.mark.parametrize("B,T,H,Hkv,off", [(260, 2, 2, 2, 0), (65, 16, 2, 2, 5), (33, 17, 3, 1, 0), (9, 63, 1, 1, 1),
                                           (130, 3, 2, 2, 130), (20, 33, 4, 4, 31)])
def test_prompt_attention_of_many_sequences(D, B, T, H, Hkv, off):
    assert _ext.kernels().prompt_attn_applies(B, T, H, Hkv, D, off + T)
    q, k, v = make(B, T, H, Hkv, D, off, off + T + 3)
    ref = exact(q, k, v, off)
    bound = 2 ** -7.9 * ref.abs() + 2 ** -16 * v[:, :, :off + T].abs().max().double()
    assert ((attend(q, k, v, off).double() - ref).abs() <= bound).all()
