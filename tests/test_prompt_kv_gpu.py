"""A prompt's rotation and cache append in one kernel against the separate passes: the same bits in the caches and in q."""
import pytest
import torch

from penroz.models import layers as L
from penroz.models.kv_cache import KVCache, TurboQuantKVCache
from penroz.ops.attention import DECODE_HEAD_DIMS

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _both(B, T, H, Hkv, D, theta, inv_dtype, before=0):
    torch.manual_seed(B * T + D)
    att = L.CausalSelfAttention(H, num_kv_heads=Hkv, rope_theta=theta, head_dim=D).to("cuda")
    if theta is not None:
        att.inv_freq = att.inv_freq.to(inv_dtype)
    rows = [torch.randn(B, n, (H + 2 * Hkv) * D, device="cuda").to(BF) for n in (before, T) if n]
    outs = []
    for fast in (True, False):
        cache = KVCache(1, capacity=before + T // 2 + 1)  # grows on the way
        att.set_kv_cache(cache, 0)
        with torch.inference_mode() if fast else torch.no_grad():
            y = [att(x) for x in rows]
        outs.append((y, cache, cache.get(0)))
    return outs


@pytest.mark.parametrize("B,T,H,Hkv,D,theta,inv", [
    (1, 1, 1, 1, 16, 1e4, torch.float32), (3, 200, 4, 1, 256, 1e6, torch.float32), (2, 7, 5, 5, 48, 1e4, BF),
    (3, 5, 8, 2, 80, 1e4, torch.float32), (1, 33, 64, 16, 256, 1e6, BF), (1, 9, 12, 12, 64, None, None),
    (5, 64, 12, 12, 64, None, None), (2, 3, 4, 2, 128, None, None)])
@pytest.mark.parametrize("before", [0, 11])
def test_prompt_append(B, T, H, Hkv, D, theta, inv, before):
    (y, fast, kv), (want, slow, ref) = _both(B, T, H, Hkv, D, theta, inv, before)
    assert fast.seq_len(0) == slow.seq_len(0) == before + T
    assert fast.metrics.memory_bytes == slow.metrics.memory_bytes and fast.metrics.num_appends == slow.metrics.num_appends
    for g, w in zip(kv, ref):
        assert torch.equal(g, w)
    if D in DECODE_HEAD_DIMS:  # other widths' attention is a library product, whose order of sums may follow q's strides
        for g, w in zip(y, want):
            assert torch.equal(g, w)


def test_what_keeps_the_separate_passes(monkeypatch):
    from penroz.models import kv_cache as kvc

    def refuse():
        raise AssertionError("the fused kernel was asked for")

    monkeypatch.setattr(kvc, "kernels", refuse)

    class Own(KVCache):
        def attend(self, layer_idx, q, k, v):
            return super().attend(layer_idx, q, k, v)

    x = torch.randn(2, 4, 3 * 64, device="cuda")
    for cache, dtype, mode in ((Own(1), BF, torch.inference_mode), (TurboQuantKVCache(1), BF, torch.inference_mode),
                               (KVCache(1), torch.float32, torch.inference_mode), (KVCache(1), BF, torch.no_grad)):
        att = L.CausalSelfAttention(1)
        att.set_kv_cache(cache, 0)
        with mode():
            assert att(x.to(dtype)).shape == (2, 4, 64)
        assert cache.seq_len(0) == 4
