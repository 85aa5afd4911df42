"""Preallocated KV cache for incremental decoding, plus the int8 "TurboQuant" variant.

API parity with the reference (``kv_cache.py:14-206``): ``KVCacheMetrics``, ``KVCache.append /
get / clear / seq_len / log_metrics``, ``TurboQuantKVCache`` (per-token absmax/127 int8 with
fp32 scales), ``create_kv_cache`` keyed on ``TURBO_QUANT_KV_CACHE=1``.

MI355X-first differences:
  * storage is preallocated ``[B, Hkv, capacity, D]`` per layer and written in place (the
    reference re-``torch.cat``s the whole cache every token — O(S) copies per step);
    capacity doubles only if a sequence outgrows it;
  * only the KV heads are stored (no GQA expansion before caching);
  * ``attend`` runs the decode-attention HIP kernel directly on the cache — for the int8
    cache the dequantisation is fused into the kernel, so the full cache is never
    materialised in fp32 (the reference dequantises the *whole* cache every step and returns
    fp32, which also breaks bf16 models);
  * ``seq_len(layer_idx)`` is per layer, so each layer's RoPE offset is its own.
"""
from __future__ import annotations

import logging
import os
import time
from dataclasses import dataclass

import numpy as np
import torch
from torch import Tensor

from penroz.ops._ext import kernels, plain_call
from penroz.ops import attention as attn_ops
from penroz.ops import packed as packed_ops
from penroz.ops import sampling as samp_ops

log = logging.getLogger(__name__)

TURBO_QUANT_ENABLED = os.environ.get("TURBO_QUANT_KV_CACHE", "0") == "1"
DEFAULT_CAPACITY = 256


@dataclass
class KVCacheMetrics:
    num_appends: int = 0
    total_entries: int = 0
    memory_bytes: int = 0
    compressed_memory_bytes: int = 0
    compression_ratio: float = 1.0
    last_append_latency_ms: float = 0.0


class KVCache:
    """Per-layer preallocated key/value storage."""

    def __init__(self, num_layers: int = 0, capacity: int | None = None):
        self.num_layers = num_layers
        self._capacity_hint = capacity
        self._k: list[Tensor | None] = [None] * num_layers
        self._v: list[Tensor | None] = [None] * num_layers
        self._len: list[int] = [0] * num_layers
        self._metrics = KVCacheMetrics()

    # ------------------------------------------------------------------ bookkeeping
    @property
    def metrics(self) -> KVCacheMetrics:
        return self._metrics

    def reserve(self, capacity: int):
        """Capacity to allocate on first use (e.g. the generation block size)."""
        self._capacity_hint = capacity

    def seq_len(self, layer_idx: int = 0) -> int:
        return self._len[layer_idx]

    def clear(self):
        """Forget every cached token (storage is kept for reuse)."""
        self._len = [0] * self.num_layers
        self._metrics = KVCacheMetrics()

    def _record(self, t0: float, new_tokens: int, raw_bytes: int, stored_bytes: int):
        m = self._metrics
        m.num_appends += 1
        m.total_entries += new_tokens
        m.memory_bytes += raw_bytes
        m.compressed_memory_bytes += stored_bytes
        m.compression_ratio = (m.memory_bytes / m.compressed_memory_bytes
                               if m.compressed_memory_bytes > 0 else 1.0)
        m.last_append_latency_ms = (time.monotonic() - t0) * 1000

    def log_metrics(self):
        m = self._metrics
        log.info(f"KVCache metrics: entries={m.total_entries}, memory={m.memory_bytes / 1024:.1f}KB, "
                 f"compression_ratio={m.compression_ratio:.2f}, last_append={m.last_append_latency_ms:.3f}ms")

    # ------------------------------------------------------------------ storage
    def _alloc(self, like: Tensor, B: int, Hkv: int, cap: int, D: int, dtype=None):
        return torch.empty(B, Hkv, cap, D, dtype=dtype or like.dtype, device=like.device)

    def _ensure(self, layer_idx: int, like: Tensor, B: int, Hkv: int, D: int, new_tokens: int):
        """Make room for ``new_tokens`` more (a shape / device change resets the layer first)."""
        k = self._k[layer_idx]
        if k is not None and (k.shape[0] != B or k.shape[1] != Hkv or k.shape[3] != D
                              or k.device != like.device):
            k = None
            self._len[layer_idx] = 0
        needed = self._len[layer_idx] + new_tokens
        if k is None:
            cap = max(needed, self._capacity_hint or DEFAULT_CAPACITY)
            self._k[layer_idx] = self._alloc(like, B, Hkv, cap, D)
            self._v[layer_idx] = self._alloc(like, B, Hkv, cap, D)
        elif k.shape[2] < needed:
            cap = max(needed, 2 * k.shape[2])
            n = self._len[layer_idx]
            for store in (self._k, self._v):
                new = self._alloc(store[layer_idx], B, Hkv, cap, D)
                new[:, :, :n] = store[layer_idx][:, :, :n]
                store[layer_idx] = new

    def _write(self, layer_idx: int, k_bthd: Tensor, v_bthd: Tensor) -> int:
        """Store k/v given as [B, T, Hkv, D]; returns the new length."""
        B, T, Hkv, D = k_bthd.shape
        self._ensure(layer_idx, k_bthd, B, Hkv, D, T)
        pos = self._len[layer_idx]
        samp_ops.kv_store_into(k_bthd, self._k[layer_idx], pos)
        samp_ops.kv_store_into(v_bthd, self._v[layer_idx], pos)
        self._len[layer_idx] = pos + T
        return pos + T

    # ------------------------------------------------------------------ reference API
    def append(self, layer_idx: int, key: Tensor, value: Tensor) -> tuple[Tensor, Tensor]:
        """Append ``key``/``value`` of shape (B, Hkv, S_new, D); return the full (B, Hkv, S, D) views."""
        t0 = time.monotonic()
        raw = key.nelement() * key.element_size() + value.nelement() * value.element_size()
        n = self._write(layer_idx, key.transpose(1, 2), value.transpose(1, 2))
        self._record(t0, key.shape[2], raw, raw)
        return self._k[layer_idx][:, :, :n], self._v[layer_idx][:, :, :n]

    def get(self, layer_idx: int) -> tuple[Tensor | None, Tensor | None]:
        n = self._len[layer_idx]
        if n == 0:
            return None, None
        return self._k[layer_idx][:, :, :n], self._v[layer_idx][:, :, :n]

    # ------------------------------------------------------------------ decode attention
    def attend(self, layer_idx: int, q: Tensor, k: Tensor, v: Tensor) -> Tensor:
        """Append k/v ([B, T, Hkv, D]) then attend q ([B, T, H, D]) over the cache -> [B, T, H*D]."""
        t0 = time.monotonic()
        raw = k.nelement() * k.element_size() + v.nelement() * v.element_size()
        n = self._write(layer_idx, k, v)
        self._record(t0, k.shape[1], raw, raw)
        return attn_ops.decode_attention(q, self._k[layer_idx], self._v[layer_idx], n)

    def attend_qkv(self, layer_idx: int, qkv: Tensor, H: int, Hkv: int, D: int, inv_freq: Tensor | None,
                   offset: int) -> Tensor | None:
        """``attend`` of the fused projection [B, T, (H + 2 Hkv) * D] at position ``offset``, rotated on the way
        (``inv_freq``): one kernel in place of table, rotation and two copies. None, and nothing stored, where that kernel
        does not apply."""
        cls = type(self)
        if not (cls.attend in _STORES_AS_GIVEN and cls._write is KVCache._write and qkv.dtype == torch.bfloat16 and plain_call(qkv)):
            return None
        t0 = time.monotonic()
        B, T, _ = qkv.shape
        self._ensure(layer_idx, qkv, B, Hkv, D, T)
        kc, vc, pos = self._k[layer_idx], self._v[layer_idx], self._len[layer_idx]
        if pos != offset or kc.dtype != qkv.dtype:
            return None
        q = kernels().prompt_kv(qkv, inv_freq, kc, vc, pos, H, Hkv)
        if q is None:
            return None
        self._len[layer_idx] = pos + T
        raw = 2 * B * T * Hkv * D * qkv.element_size()
        self._record(t0, T, raw, raw)
        return attn_ops.decode_attention(q, kc, vc, pos + T)


# the ``attend`` methods that ``attend_qkv`` may stand in for (a subclass's own is always called)
_STORES_AS_GIVEN = {KVCache.attend}


class TurboQuantKVCache(KVCache):
    """int8 KV cache with per-token fp32 scales (``kv_cache.py:101-195``)."""

    def __init__(self, num_layers: int = 0, capacity: int | None = None):
        super().__init__(num_layers, capacity)
        self._sk: list[Tensor | None] = [None] * num_layers
        self._sv: list[Tensor | None] = [None] * num_layers
        self._dtype: list[torch.dtype | None] = [None] * num_layers

    # per-token quantisation helpers kept with the reference's names for parity tests
    @staticmethod
    def _quantize(tensor: Tensor) -> tuple[Tensor, Tensor]:
        return samp_ops.reference_quantize(tensor)

    @staticmethod
    def _dequantize(quantized: Tensor, scale: Tensor) -> Tensor:
        return quantized.float() * scale

    def _ensure(self, layer_idx: int, like: Tensor, B: int, Hkv: int, D: int, new_tokens: int):
        """Make room for ``new_tokens`` more (a shape / device change resets the layer first)."""
        k = self._k[layer_idx]
        if k is not None and (k.shape[0] != B or k.shape[1] != Hkv or k.shape[3] != D
                              or k.device != like.device):
            k = None
            self._len[layer_idx] = 0
        needed = self._len[layer_idx] + new_tokens
        if k is None:
            cap = max(needed, self._capacity_hint or DEFAULT_CAPACITY)
            self._k[layer_idx] = self._alloc(like, B, Hkv, cap, D, torch.int8)
            self._v[layer_idx] = self._alloc(like, B, Hkv, cap, D, torch.int8)
            self._sk[layer_idx] = torch.ones(B, Hkv, cap, dtype=torch.float32, device=like.device)
            self._sv[layer_idx] = torch.ones(B, Hkv, cap, dtype=torch.float32, device=like.device)
        elif k.shape[2] < needed:
            cap = max(needed, 2 * k.shape[2])
            n = self._len[layer_idx]
            for store in (self._k, self._v):
                new = self._alloc(store[layer_idx], B, Hkv, cap, D, torch.int8)
                new[:, :, :n] = store[layer_idx][:, :, :n]
                store[layer_idx] = new
            for store in (self._sk, self._sv):
                new = torch.ones(B, Hkv, cap, dtype=torch.float32, device=like.device)
                new[:, :, :n] = store[layer_idx][:, :, :n]
                store[layer_idx] = new

    def _write(self, layer_idx: int, k_bthd: Tensor, v_bthd: Tensor) -> int:
        B, T, Hkv, D = k_bthd.shape
        self._ensure(layer_idx, k_bthd, B, Hkv, D, T)
        pos = self._len[layer_idx]
        samp_ops.kv_quantize_into(k_bthd, self._k[layer_idx], self._sk[layer_idx], pos)
        samp_ops.kv_quantize_into(v_bthd, self._v[layer_idx], self._sv[layer_idx], pos)
        self._dtype[layer_idx] = k_bthd.dtype
        self._len[layer_idx] = pos + T
        return pos + T

    def _stored_bytes(self, k: Tensor) -> int:
        n_tok = k.nelement() // k.shape[-1]
        return 2 * (k.nelement() * 1 + n_tok * 4)

    def append(self, layer_idx: int, key: Tensor, value: Tensor) -> tuple[Tensor, Tensor]:
        """Quantise and append (B, Hkv, S_new, D); return the dequantised full cache in key's dtype."""
        t0 = time.monotonic()
        raw = key.nelement() * key.element_size() + value.nelement() * value.element_size()
        n = self._write(layer_idx, key.transpose(1, 2), value.transpose(1, 2))
        self._record(t0, key.shape[2], raw, self._stored_bytes(key))
        k = self._dequantize(self._k[layer_idx][:, :, :n], self._sk[layer_idx][:, :, :n, None])
        v = self._dequantize(self._v[layer_idx][:, :, :n], self._sv[layer_idx][:, :, :n, None])
        return k.to(key.dtype), v.to(value.dtype)

    def get(self, layer_idx: int) -> tuple[Tensor | None, Tensor | None]:
        n = self._len[layer_idx]
        if n == 0:
            return None, None
        dt = self._dtype[layer_idx] or torch.float32
        return (self._dequantize(self._k[layer_idx][:, :, :n], self._sk[layer_idx][:, :, :n, None]).to(dt),
                self._dequantize(self._v[layer_idx][:, :, :n], self._sv[layer_idx][:, :, :n, None]).to(dt))

    def get_quantized(self, layer_idx: int):
        n = self._len[layer_idx]
        return self._k[layer_idx], self._v[layer_idx], self._sk[layer_idx], self._sv[layer_idx], n

    def attend(self, layer_idx: int, q: Tensor, k: Tensor, v: Tensor) -> Tensor:
        t0 = time.monotonic()
        raw = k.nelement() * k.element_size() + v.nelement() * v.element_size()
        n = self._write(layer_idx, k, v)
        self._record(t0, k.shape[1], raw, self._stored_bytes(k))
        return attn_ops.decode_attention(q, self._k[layer_idx], self._v[layer_idx], n,
                                         self._sk[layer_idx], self._sv[layer_idx])


class SequenceState:
    """State manager of the packed step: slots of per-sequence state, taken and given back while other
    sequences go on.

    Per slot: the latent cache rows of every latent-attention layer that has its own (``latent_widths``),
    ``[slots, capacity, width]`` in the model's dtype; the last ``taps - 1`` inputs of every causal convolution
    (``convs``), fp32 ``[slots, taps - 1, channels]``; key / value rows per head and the means of their blocks of
    ``pool`` tokens for every window layer (``windows``: heads, row width, pool), ``[slots, heads, capacity (or
    blocks), width]`` in the model's dtype; the matrix state of every linear-attention layer (``linear``: its
    shape), fp32 ``[slots, *shape]``. A slot needs no clearing when it is taken again: a sequence's reads never
    reach behind its own position 0, and its first token starts a matrix state from zero. Slots and capacity
    double when they run out; ``limit`` bounds the tokens of a sequence (learned positions)."""

    def __init__(self, latent_widths: list[int], convs: list[tuple[int, int]], rotations, dtype: torch.dtype, device,
                 slots: int = 1, capacity: int | None = None, *, windows=(), linear=(), limit: int | None = None):
        self.dtype, self.device = dtype, torch.device(device)
        self.num_layers = len(latent_widths) + len(windows) + len(linear)
        self.limit = limit
        self.capacity = max(1, capacity or DEFAULT_CAPACITY)
        if limit is not None:
            self.capacity = min(self.capacity, limit)
        self.slots = max(1, slots)
        n, cap = self.slots, self.capacity
        self.latent = [torch.zeros(n, cap, w, dtype=dtype, device=self.device) for w in latent_widths]
        self.conv = [torch.zeros(n, taps - 1, C, dtype=torch.float32, device=self.device) for C, taps in convs]
        self._pools = [pool for _, _, pool in windows]
        self.window = [torch.zeros(n, heads, cap, w, dtype=dtype, device=self.device) for heads, w, _ in windows]
        self.pooled = [torch.zeros(n, heads, -(-cap // pool), w, dtype=dtype, device=self.device)
                       for heads, w, pool in windows]
        self.linear = [torch.zeros(n, *shape, dtype=torch.float32, device=self.device) for shape in linear]
        self._rotations = sorted(set(rotations))
        self.tables: dict = {}
        self._build_tables()
        self._len: dict[int, int] = {}
        self._free = list(range(self.slots - 1, -1, -1))
        self._metrics = KVCacheMetrics()

    def _build_tables(self):
        for base, dims in self._rotations:
            self.tables[(base, dims)] = packed_ops.rotation_table(base, dims, self.capacity, self.device)

    _STORES = ("latent", "conv", "window", "pooled", "linear")

    def moving(self) -> list[Tensor]:
        """The stores a step replaces (running it twice would move them twice); the others are written per
        position."""
        return self.conv + self.linear

    # ------------------------------------------------------------------ slots
    def acquire(self) -> int:
        if not self._free:
            n = self.slots
            self.slots = 2 * n
            for store in self._STORES:
                setattr(self, store, [self._grown(t, 0, self.slots) for t in getattr(self, store)])
            self._free = list(range(self.slots - 1, n - 1, -1))
        slot = self._free.pop()
        self._len[slot] = 0
        return slot

    def release(self, slot: int):
        del self._len[slot]
        self._free.append(slot)

    @staticmethod
    def _grown(t: Tensor, dim: int, n: int) -> Tensor:
        shape = list(t.shape)
        shape[dim] = n
        new = t.new_zeros(shape)
        new.narrow(dim, 0, t.shape[dim]).copy_(t)
        return new

    def reserve(self, capacity: int):
        """Room for ``capacity`` tokens per sequence."""
        if self.limit is not None and capacity > self.limit:
            raise ValueError(f"a sequence of {capacity} tokens exceeds the model's {self.limit} positions")
        if capacity > self.capacity:
            self.capacity = max(capacity, 2 * self.capacity)
            if self.limit is not None:
                self.capacity = min(self.capacity, self.limit)
            self.latent = [self._grown(t, 1, self.capacity) for t in self.latent]
            self.window = [self._grown(t, 2, self.capacity) for t in self.window]
            self.pooled = [self._grown(t, 2, -(-self.capacity // p)) for t, p in zip(self.pooled, self._pools)]
            self._build_tables()

    def length(self, slot: int) -> int:
        return self._len[slot]

    def seq_len(self, layer_idx: int = 0) -> int:
        return max(self._len.values(), default=0)

    @property
    def metrics(self) -> KVCacheMetrics:
        return self._metrics

    def clear(self):
        """Forget every sequence (storage is kept for reuse)."""
        for slot in list(self._len):
            self.release(slot)
        self._metrics = KVCacheMetrics()

    def log_metrics(self):
        held = sum(self._len.values())
        size = sum(t.nelement() * t.element_size() for store in self._STORES for t in getattr(self, store))
        log.info(f"Sequence state: tokens={held}, sequences={len(self._len)}, memory={size / 1024:.1f}KB")

    # ------------------------------------------------------------------ steps
    def advance(self, slots: list[int], count: int):
        """Account for ``count`` tokens per slot that a captured step has already written."""
        for s in slots:
            self._len[s] += count

    def begin(self, entries: list[tuple[int, int]]) -> packed_ops.PackedBatch:
        """Descriptor of a step that brings ``count`` new tokens to each ``(slot, count)``; advances the
        slots' lengths."""
        if any(n < 1 for _, n in entries) or len({s for s, _ in entries}) != len(entries):
            raise ValueError("a step brings at least one token to each of distinct slots")
        self.reserve(max(self._len[s] + n for s, n in entries))
        seq = np.array([s for s, _ in entries], dtype=np.int32)
        count = np.array([n for _, n in entries], dtype=np.int32)
        start = np.array([self._len[s] for s, _ in entries], dtype=np.int32)
        cu = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
        first = np.repeat(cu[:-1], count)
        slot = np.repeat(seq, count)
        pos = np.arange(cu[-1], dtype=np.int32) - first + np.repeat(start, count)
        for s, n in entries:
            self._len[s] += n
        lens, counts = (start + count).tolist(), count.tolist()
        flat = torch.from_numpy(np.concatenate([slot, pos, first, cu, seq]))
        if self.device.type == "cuda":
            flat = flat.pin_memory().to(self.device, non_blocking=True)
        parts = flat.split([len(slot), len(pos), len(first), len(cu), len(seq)])
        m = self._metrics
        m.num_appends += 1
        m.total_entries += sum(counts)
        # (slices of one upload start at any 4-byte offset: the kernels read them as scalars)
        return packed_ops.PackedBatch(*parts, single=all(n == 1 for n in counts),
                                      fresh=all(l == n for l, n in zip(lens, counts)), counts=counts, lens=lens,
                                      max_len=max(lens))


def create_kv_cache(num_layers: int, capacity: int | None = None) -> KVCache:
    """``TurboQuantKVCache`` when ``TURBO_QUANT_KV_CACHE=1`` (module constant), else ``KVCache``."""
    if TURBO_QUANT_ENABLED:
        log.info("TurboQuant KV cache enabled (TURBO_QUANT_KV_CACHE=1)")
        return TurboQuantKVCache(num_layers, capacity)
    return KVCache(num_layers, capacity)
