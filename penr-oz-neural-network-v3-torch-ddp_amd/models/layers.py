"""Layer library for the JSON layer vocabulary.

Behavioural parity with the reference's custom modules (``neural_net_layers.py:7-225``):
``CausalSelfAttention``, ``PositionEmbedding``, ``Summation``, ``ResidualConnection``,
``SoftmaxOnLast``, ``RMSNorm``, ``GatedMLP``, ``ScaledEmbedding``, ``TransformerBlock``.
Parameter names and module nesting are identical, so state_dict keys match the reference's
checkpoints (``mappers.py:326-353``).

What differs (MI355X-first):
  * attention goes through ``penroz.ops.attention`` — the hand-written CDNA4 flash-attention
    kernels on GPU (fused QKV read, head merge in the epilogue, GQA by index math, no expand);
    torch SDPA math on CPU only;
  * the KV cache is preallocated and written in place, stores the *KV* heads (the reference
    expands GQA before caching, ``neural_net_layers.py:76-88``) and each layer reads its own
    cache length for the RoPE offset (reference bug: layer 0's length for every layer, ``:72``);
  * RMSNorm / RoPE / gated-MLP activation / LayerNorm / GELU use HIP kernels on GPU.
"""
from __future__ import annotations

import torch
from torch import Tensor
import torch.nn as nn

from penroz.models.kv_cache import KVCache
from penroz.ops import attention as attn_ops
from penroz.ops.gemm import apply
from penroz.ops import norms as norm_ops
from penroz.ops import activations as act_ops
from penroz.ops import packed as packed_ops
from penroz.ops import rope as rope_ops
from penroz.ops import linear_attn as linear_ops
from penroz.ops import window as window_ops


class CausalSelfAttention(nn.Module):
    """Causal self-attention over a fused QKV input ``[B, T, (H + 2*Hkv) * D]``.

    Mirrors ``neural_net_layers.py:7-95``: optional RoPE (``rope_theta``), grouped-query
    attention (``num_kv_heads``), attention dropout while training, optional KV cache.
    """

    def __init__(self, num_heads: int, dropout: float = 0.0,
                 num_kv_heads: int = None, rope_theta: float = None,
                 head_dim: int = None):
        super().__init__()
        self.num_heads = num_heads
        self.num_kv_heads = num_kv_heads if num_kv_heads is not None else num_heads
        if self.num_heads % self.num_kv_heads != 0:
            raise ValueError(f"num_heads {num_heads} not divisible by num_kv_heads {self.num_kv_heads}")
        self.dropout = dropout
        self.rope_theta = rope_theta
        self.head_dim = head_dim
        self._kv_cache = None
        self._layer_idx = 0
        if rope_theta is not None and head_dim is not None:
            inv_freq = 1.0 / (rope_theta ** (torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim))
            self.register_buffer("inv_freq", inv_freq, persistent=False)

    def set_kv_cache(self, kv_cache, layer_idx: int):
        """Attach (or detach with ``None``) a KV cache slot for incremental decoding."""
        self._kv_cache = kv_cache
        self._layer_idx = layer_idx

    def _inv_freq(self, head_dim: int, device) -> Tensor:
        if hasattr(self, "inv_freq"):
            return self.inv_freq.to(device)
        return 1.0 / (self.rope_theta ** (torch.arange(0, head_dim, 2, device=device,
                                                       dtype=torch.float32) / head_dim))

    def forward(self, query_key_value: Tensor) -> Tensor:
        batch_size, block_size, total_dim = query_key_value.size()
        head_dim = total_dim // (self.num_heads + 2 * self.num_kv_heads)
        q_dim = self.num_heads * head_dim
        kv_dim = self.num_kv_heads * head_dim

        cache = self._kv_cache
        offset = cache.seq_len(self._layer_idx) if cache is not None else 0

        inv_freq = None if self.rope_theta is None else self._inv_freq(head_dim, query_key_value.device)
        if isinstance(cache, KVCache) and not getattr(cache, "graph_mode", False):
            out = cache.attend_qkv(self._layer_idx, query_key_value, self.num_heads, self.num_kv_heads, head_dim, inv_freq, offset)
            if out is not None:
                return out

        if inv_freq is not None:
            # graph-replayed decode: positions come from the cache's device counter (one table per
            # (theta, head_dim) and step, shared by the layers)
            table = (cache.rope_table((self.rope_theta, head_dim), inv_freq, block_size)
                     if getattr(cache, "graph_mode", False) else None)
            qkv = rope_ops.apply_rope_qkv(query_key_value, self.num_heads, self.num_kv_heads, head_dim,
                                          inv_freq, offset, table=table)
        else:
            qkv = query_key_value

        if cache is None:
            dropout = self.dropout if self.training else 0.0
            return attn_ops.causal_attention_qkv(qkv, self.num_heads, self.num_kv_heads, head_dim,
                                                 dropout_p=dropout)

        # Incremental path: append this step's K/V (KV heads only) in place, attend over the cache.
        q, k, v = qkv.split([q_dim, kv_dim, kv_dim], dim=2)
        k = k.view(batch_size, block_size, self.num_kv_heads, head_dim)
        v = v.view(batch_size, block_size, self.num_kv_heads, head_dim)
        q = q.reshape(batch_size, block_size, self.num_heads, head_dim)
        return cache.attend(self._layer_idx, q, k, v)


class PositionEmbedding(nn.Embedding):
    """Learned absolute positions ``arange(offset, offset + T)`` (``neural_net_layers.py:98-118``)."""

    def __init__(self, *args, **kwargs):
        super().__init__(*args, **kwargs)
        self._position_offset = 0
        self.position_offset_tensor: Tensor | None = None  # device int64 [1] (graph-replayed decode)

    @property
    def position_offset(self) -> int:
        return self._position_offset

    @position_offset.setter
    def position_offset(self, value: int):
        self._position_offset = value

    def forward(self, input_data: Tensor) -> Tensor:
        _, num_positions = input_data.shape
        if self.position_offset_tensor is not None:  # offset read on the device (caller bounds it)
            positions = self.position_offset_tensor + torch.arange(num_positions, dtype=torch.long,
                                                                   device=input_data.device)
            return super().forward(positions)
        if self._position_offset + num_positions > self.num_embeddings:
            raise ValueError(f"positions {self._position_offset}..{self._position_offset + num_positions} "
                             f"exceed the position table ({self.num_embeddings})")
        positions = torch.arange(self._position_offset, self._position_offset + num_positions,
                                 dtype=torch.long, device=input_data.device)
        return super().forward(positions)


class Summation(nn.Sequential):
    """Sum of every child applied to the same input (token + position embedding)."""

    def forward(self, input_data: Tensor) -> Tensor:
        forwarded = self[0](input_data)
        for layer in self[1:]:
            forwarded = forwarded + layer(input_data)
        return forwarded


class ResidualConnection(nn.Sequential):
    """``x = x + child(x)`` for each child in order."""

    def forward(self, forwarded: Tensor) -> Tensor:
        for layer in self:
            if torch.jit.is_scripting():
                forwarded = forwarded + layer(forwarded)
            else:
                forwarded = forwarded + apply(layer, forwarded)
        return forwarded


class SoftmaxOnLast(nn.Softmax):
    """Softmax over the last position's logits ``logits[:, -1, :]``."""

    def forward(self, logits: Tensor) -> Tensor:
        return super().forward(logits[:, -1, :])


class LayerNorm(nn.LayerNorm):
    """``nn.LayerNorm`` whose GPU path is the HIP LayerNorm kernel (fp32 statistics).

    Same parameters/keys as ``nn.LayerNorm``; the ``layernorm`` algo compiles to this class.
    """

    def forward(self, x: Tensor) -> Tensor:
        if len(self.normalized_shape) == 1 and self.elementwise_affine:
            w, b = self.weight, self.bias
            if w.dtype != torch.float32 and b is not None and not torch.is_grad_enabled():
                w, b = self._fp32_affine()  # inference on bf16 weights: no per-call casts
            return norm_ops.layer_norm(x, w, b, self.eps)
        return super().forward(x)

    def _fp32_affine(self):
        """fp32 copies of (weight, bias) — the kernel's parameter dtype — cached until the
        parameters change (storage or in-place version)."""
        key = (self.weight.data_ptr(), self.weight._version, self.bias.data_ptr(), self.bias._version)
        c = self.__dict__.get("_fp32_cache")
        if c is None or c[0] != key:
            c = (key, self.weight.detach().float(), self.bias.detach().float())
            self.__dict__["_fp32_cache"] = c
        return c[1], c[2]


class GELU(nn.GELU):
    """``nn.GELU`` (erf or tanh) whose GPU path is the vectorised HIP GELU kernel."""

    def forward(self, x: Tensor) -> Tensor:
        return act_ops.gelu(x, self.approximate)


class RMSNorm(nn.Module):
    """Root-mean-square norm computed in fp32 (``neural_net_layers.py:144-155``)."""

    def __init__(self, normalized_shape: int, eps: float = 1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(normalized_shape))
        self.eps = eps

    def forward(self, x: Tensor) -> Tensor:
        return norm_ops.rms_norm(x, self.weight, self.eps)


class GatedMLP(nn.Module):
    """``down(act(gate(x)) * up(x))`` with silu / gelu_tanh / gelu (``neural_net_layers.py:158-174``)."""

    def __init__(self, in_features: int, intermediate_size: int,
                 bias: bool = False, activation: str = "gelu_pytorch_tanh"):
        super().__init__()
        self.gate_proj = nn.Linear(in_features, intermediate_size, bias=bias)
        self.up_proj = nn.Linear(in_features, intermediate_size, bias=bias)
        self.down_proj = nn.Linear(intermediate_size, in_features, bias=bias)
        if activation in ("silu", "swish"):
            self.act_kind = "silu"
            self.act = nn.SiLU()
        elif activation == "gelu_pytorch_tanh":
            self.act_kind = "gelu_tanh"
            self.act = nn.GELU(approximate="tanh")
        else:
            self.act_kind = "gelu"
            self.act = nn.GELU()

    def forward(self, x: Tensor) -> Tensor:
        return apply(self.down_proj, act_ops.gated_act(apply(self.gate_proj, x), apply(self.up_proj, x), self.act_kind))


class ScaledEmbedding(nn.Embedding):
    """Embedding whose output is multiplied by a fixed ``scale`` (Gemma: sqrt(hidden))."""

    def __init__(self, num_embeddings: int, embedding_dim: int, scale: float = 1.0, **kwargs):
        super().__init__(num_embeddings, embedding_dim, **kwargs)
        self.scale = scale

    def forward(self, input_data: Tensor) -> Tensor:
        return super().forward(input_data) * self.scale


class TransformerBlock(nn.Module):
    """Decoder block with optional post-norms (``neural_net_layers.py:188-225``).

    ``post_norm_on_residual=True`` (Gemma 3+): ``h = post_norm(x + attn(x))``;
    ``False`` (Gemma 2): ``h = x + post_norm(attn(x))``. Without an ``mlp_block`` the block ends at ``h``.
    """

    def __init__(self, attn_block: nn.Module, mlp_block: nn.Module = None,
                 post_attn_norm: nn.Module = None, post_mlp_norm: nn.Module = None,
                 post_norm_on_residual: bool = True):
        super().__init__()
        self.attn_block = attn_block
        self.mlp_block = mlp_block
        self.post_attn_norm = post_attn_norm
        self.post_mlp_norm = post_mlp_norm
        self.post_norm_on_residual = post_norm_on_residual

    def forward(self, x: Tensor) -> Tensor:
        if torch.jit.is_scripting():
            attn_out = self.attn_block(x)
        else:
            attn_out = apply(self.attn_block, x)
        if self.post_attn_norm is not None and not self.post_norm_on_residual:
            attn_out = self.post_attn_norm(attn_out)
        h = x + attn_out
        if self.post_attn_norm is not None and self.post_norm_on_residual:
            h = self.post_attn_norm(h)
        if self.mlp_block is None:
            return h
        if torch.jit.is_scripting():
            mlp_out = self.mlp_block(h)
        else:
            mlp_out = apply(self.mlp_block, h)
        if self.post_mlp_norm is not None and not self.post_norm_on_residual:
            mlp_out = self.post_mlp_norm(mlp_out)
        out = h + mlp_out
        if self.post_mlp_norm is not None and self.post_norm_on_residual:
            out = self.post_mlp_norm(out)
        return out


# --------------------------------------------------------------------------- packed-step layers
# Layers of the designs that the packed program runs (models/packed.py): state per sequence beyond
# keys and values, an fp32 residual stream. Their forward runs whole fresh sequences [B, T, C] through
# the same ops (ops/packed.py), without gradients.
def _no_grad_only(module: nn.Module, x: Tensor):
    if torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in module.parameters())):
        raise NotImplementedError(f"{type(module).__name__} has no backward: run it under torch.no_grad()")


def fresh_batch(B: int, T: int, device) -> packed_ops.PackedBatch:
    """B sequences of T tokens, each from its first one, in slots 0..B-1."""
    i32 = dict(dtype=torch.int32, device=device)
    rows = torch.arange(B * T, **i32)
    seq = rows // T
    return packed_ops.PackedBatch(slot=seq, pos=rows - seq * T, first=seq * T, cu=torch.arange(B + 1, **i32) * T,
                                  seq_slot=torch.arange(B, **i32), single=False, fresh=True, counts=[T] * B,
                                  lens=[T] * B, max_len=T)


class GroupedRMSNorm(nn.Module):
    """RMS norm over ``groups`` equal consecutive parts of the vector, each by its own root mean
    square, times one weight; fp32 output (an fp32 residual stream adds it)."""

    def __init__(self, normalized_shape: int, groups: int = 1, eps: float = 1e-6):
        super().__init__()
        if normalized_shape % groups:
            raise ValueError(f"{normalized_shape} values do not split into {groups} groups")
        self.weight = nn.Parameter(torch.ones(normalized_shape))
        self.groups, self.eps = groups, eps

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        x2 = x.reshape(-1, x.shape[-1]).float().contiguous()
        return packed_ops.row_norm(x2, self.weight.float(), self.groups, self.eps, torch.float32).view(x.shape)


class CausalConv(nn.Module):
    """``x + conv(x)``: a causal convolution over time on each channel (weight [channels, taps], the last
    tap at the token itself), fp32 in and in the state, output in the weight's dtype."""

    def __init__(self, channels: int, taps: int):
        super().__init__()
        if not 1 <= taps <= 16:
            raise ValueError(f"causal convolution of {taps} taps (1 to 16)")
        self.weight = nn.Parameter(torch.randn(channels, taps) / taps)
        self.taps = taps

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        B, T, C = x.shape
        state = torch.zeros(B, self.taps - 1, C, dtype=torch.float32, device=x.device)
        x2 = x.reshape(B * T, C).float().contiguous()
        _, h = packed_ops.residual_conv(fresh_batch(B, T, x.device), self.weight.dtype, x=x2,
                                        conv=(self.weight.float().t().contiguous(), state))
        return h.view(B, T, C)


class LatentAttention(nn.Module):
    """Causal attention over compressed keys and values: per token one normed latent of ``kv_rank`` values
    and one rotated key part of ``rot_dim`` values shared by all heads, from which every head forms its
    unrotated key (``uk``) and value (``uv``). Queries are laid out per head [dim | rot_dim]; rotate-half
    rotary positions on the rotated parts. ``kv_from``: index (among the model's latent-attention layers)
    of an earlier layer whose latents this one attends over instead of its own."""

    def __init__(self, in_features: int, num_heads: int, dim: int, rot_dim: int, v_dim: int, kv_rank: int,
                 scale: float, rope_theta: float, eps: float = 1e-6, kv_from: int = None, out_features: int = None):
        super().__init__()
        self.sizes = packed_ops.LatentSizes(num_heads, dim, rot_dim, v_dim, kv_rank, float(scale), float(rope_theta),
                                            float(eps))
        if rot_dim % 2 or rot_dim < 2:
            raise ValueError(f"rot_dim {rot_dim} must be even and positive")
        self.kv_from = kv_from
        self.q = nn.Linear(in_features, num_heads * (dim + rot_dim), bias=False)
        if kv_from is None:
            self.dkv = nn.Linear(in_features, kv_rank + rot_dim, bias=False)
            self.dkv_norm = nn.Parameter(torch.ones(kv_rank))
        self.uk = nn.Linear(kv_rank, num_heads * dim, bias=False)
        self.uv = nn.Linear(kv_rank, num_heads * v_dim, bias=False)
        self.o = nn.Linear(num_heads * v_dim, out_features or in_features, bias=False)
        self._source = ()
        self._cache = None

    def bind(self, layers: list["LatentAttention"]):
        """Resolve ``kv_from`` (kept in a tuple: not a submodule)."""
        if self.kv_from is None:
            return
        own = next(i for i, m in enumerate(layers) if m is self)
        src = layers[self.kv_from] if 0 <= self.kv_from < own else None
        if (src is None or src.kv_from is not None or src.sizes.rank != self.sizes.rank
                or src.sizes.rot != self.sizes.rot or src.sizes.base != self.sizes.base):
            raise ValueError(f"latent layer {own}: kv_from {self.kv_from} is no earlier layer with its own latents of "
                             "the same rank and rotation")
        self._source = (src,)

    def packed(self) -> dict:
        s = self.sizes
        return packed_ops.pack_latent(s, self.q.weight, None if self.kv_from is not None else self.dkv.weight,
                                      self.uk.weight, self.uv.weight, self.o.weight)

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        s = self.sizes
        B, T, C = x.shape
        w = self.packed()
        b = fresh_batch(B, T, x.device)
        if self.kv_from is None:
            self._cache = torch.zeros(B, T, s.cache_width, dtype=x.dtype, device=x.device)
        cache = self._cache if self.kv_from is None else self._source[0]._cache
        z = packed_ops.linear(x.reshape(B * T, C).contiguous(), w["z"])
        tab = packed_ops.rotation_table(s.base, s.rot, T, x.device)
        o = packed_ops.latent_attention(s, w, z, cache, self.dkv_norm.float() if self.kv_from is None else None, tab, b)
        return packed_ops.linear(o, w["o"]).view(B, T, -1)


def _rows(x: Tensor, dtype: torch.dtype) -> Tensor:
    """[B, T, C] -> contiguous [B·T, C] in ``dtype``."""
    return x.reshape(-1, x.shape[-1]).to(dtype).contiguous()


class WindowAttention(nn.Module):
    """Attention over a sliding window of ``window`` tokens and, before it, the means of blocks of ``pool`` tokens;
    sigmoid weights (not normalised) of softcapped scores plus a bias per head (``pb``); grouped key / value
    heads; rotate-half rotary positions on the first ``rot_dim`` dimensions of queries and keys, and on the
    values, whose sum is turned back by the query's position."""

    def __init__(self, in_features: int, num_heads: int, num_kv_heads: int, dim: int, v_dim: int, rot_dim: int,
                 rope_theta: float, scale: float, softcap: float, window: int, pool: int, out_features: int = None):
        super().__init__()
        self.sizes = window_ops.WindowSizes(num_heads, num_kv_heads, dim, v_dim, rot_dim, float(rope_theta),
                                            float(scale), float(softcap), window, pool)
        self.sizes.check()
        self.q = nn.Linear(in_features, num_heads * dim, bias=False)
        self.k = nn.Linear(in_features, num_kv_heads * dim, bias=False)
        self.v = nn.Linear(in_features, num_kv_heads * v_dim, bias=False)
        self.pb = nn.Parameter(torch.zeros(num_heads))
        self.o = nn.Linear(num_heads * v_dim, out_features or in_features, bias=False)

    def packed(self) -> dict:
        return window_ops.pack_window(self.sizes, self.q.weight, self.k.weight, self.v.weight, self.o.weight)

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        s, (B, T, _), dt = self.sizes, x.shape, self.q.weight.dtype
        w, b = self.packed(), fresh_batch(B, T, x.device)
        kv = torch.zeros(B, s.kv_heads, T, s.row, dtype=dt, device=x.device)
        pooled = torch.zeros(B, s.kv_heads, -(-T // s.pool), s.row, dtype=dt, device=x.device)
        tables = {r: packed_ops.rotation_table(*r, T, x.device) for r in s.rotations}
        o = window_ops.window_attention(s, packed_ops.linear(_rows(x, dt), w["z"]), kv, pooled, self.pb.float(), tables, b)
        return packed_ops.linear(o, w["o"]).view(B, T, -1)


class _LinearAttention(nn.Module):
    """Linear attention with a decayed matrix state (``ops/linear_attn.py``), gated and normed per head."""

    def __init__(self, sizes: linear_ops.LinearSizes, in_features: int, out_features: int | None):
        super().__init__()
        sizes.check()
        self.sizes = sizes
        H = sizes.heads
        self.q = nn.Linear(in_features, H * sizes.dim, bias=False)
        self.k = nn.Linear(in_features, H * sizes.dim, bias=False)
        self.v = nn.Linear(in_features, H * sizes.vdim, bias=False)
        self.g = nn.Linear(in_features, H * sizes.vdim, bias=False)
        self.o = nn.Linear(H * sizes.vdim, out_features or in_features, bias=False)

    def packed(self) -> dict:
        raise NotImplementedError

    def _pack(self, **extra) -> dict:
        return linear_ops.pack_linear(self.sizes, self.q.weight, self.k.weight, self.v.weight, self.g.weight,
                                      self.o.weight, **extra)

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        B, T, _ = x.shape
        w = self.packed()
        state = torch.zeros(B, *self.sizes.state, dtype=torch.float32, device=x.device)
        z = packed_ops.linear(_rows(x, self.q.weight.dtype), w["z"])
        o = linear_ops.linear_attention(self.sizes, w, z, state, fresh_batch(B, T, x.device))
        return packed_ops.linear(o, w["o"]).view(B, T, -1)


class Retention(_LinearAttention):
    """Linear attention with a fixed ``decay`` per head (keys scaled by dim^-1/2, outputs normed per head without
    a weight, gated by silu)."""

    def __init__(self, in_features: int, num_heads: int, dim: int, v_dim: int, decay: list, eps: float = 1e-6,
                 out_features: int = None):
        super().__init__(linear_ops.LinearSizes(num_heads, dim, v_dim, dim ** -0.5, float(eps)), in_features,
                         out_features)
        if len(decay) != num_heads or not all(0.0 <= d <= 1.0 for d in decay):
            raise ValueError(f"{num_heads} heads need a decay in [0, 1] each, not {decay}")
        self.decay = [float(d) for d in decay]

    def packed(self) -> dict:
        return self._pack(decay=torch.tensor(self.decay, dtype=torch.float32, device=self.q.weight.device))


class GatedLinearAttention(_LinearAttention):
    """Linear attention whose decay per token, head and key channel is sigmoid(a2 a1 h + bias)^(1/tau) (queries
    scaled by dim^-1/2, outputs normed per head with a weight shared by the heads, gated by silu)."""

    def __init__(self, in_features: int, num_heads: int, dim: int, v_dim: int, decay_rank: int, tau: float,
                 eps: float = 1e-6, out_features: int = None):
        super().__init__(linear_ops.LinearSizes(num_heads, dim, v_dim, dim ** -0.5, float(eps), decay_rank, float(tau)),
                         in_features, out_features)
        if decay_rank < 1:
            raise ValueError(f"decay_rank {decay_rank} must be positive")
        self.a1 = nn.Linear(in_features, decay_rank, bias=False)
        self.a2 = nn.Linear(decay_rank, num_heads * dim)
        self.norm = nn.Parameter(torch.ones(v_dim))

    def packed(self) -> dict:
        return self._pack(a1=self.a1.weight, a2=self.a2.weight, bias=self.a2.bias, norm=self.norm)


class ParallelMixers(nn.Module):
    """Two mixers that read the same input, side by side: half the sum of their outputs, each RMS-normed with
    its own weight (fp32 out: an fp32 residual stream adds it)."""

    def __init__(self, features: int, left: nn.Module, right: nn.Module, eps: float = 1e-6):
        super().__init__()
        self.left, self.right = left, right
        self.left_out = nn.Parameter(torch.ones(features))
        self.right_out = nn.Parameter(torch.ones(features))
        self.eps = eps

    def forward(self, x: Tensor) -> Tensor:
        y, y2 = self.left(x), self.right(x)
        d = packed_ops.Delta(y.flatten(0, 1), y2.flatten(0, 1), self.left_out.float(), self.right_out.float(), 0.5, self.eps)
        return d.value().view(y.shape)


class GeluMLP(nn.Module):
    """down(gelu(up(x))), erf form, no biases."""

    def __init__(self, in_features: int, intermediate_size: int):
        super().__init__()
        self.up = nn.Linear(in_features, intermediate_size, bias=False)
        self.down = nn.Linear(intermediate_size, in_features, bias=False)

    def packed(self) -> dict:
        to = (self.up.weight.shape[0] + 7) // 8 * 8  # zero rows up to the kernels' vector width
        return {"up": packed_ops._pad(self.up.weight, 0, to).contiguous(),
                "down": packed_ops._pad(self.down.weight, 1, to).contiguous()}

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        w = self.packed()
        return packed_ops.gelu_mlp(_rows(x, w["up"].dtype), w["up"], w["down"]).view(x.shape)


class MixtureOfExperts(nn.Module):
    """Routed feed-forward: ``num_experts`` experts without biases, ``top_k`` per token by the ``scoring`` of an
    fp32 router — "softmax" over all experts, or a "sigmoid" each, chosen by score plus ``correction`` — and
    weighted by those scores times ``scale`` (``renormalize``: by their share among the chosen).
    ``activation``: gated "silu", or "clamped_swiglu" — g = min(gate, limit), u = clamp(up, ±limit),
    g · sigmoid(1.702 g) · (u + 1) — or ungated "gelu" (erf form). ``shared_size``: a shared expert of that
    width (ungated gelu) runs for every token, times sigmoid of its own gate row."""

    def __init__(self, in_features: int, intermediate_size: int, num_experts: int, top_k: int,
                 activation: str = "silu", limit: float = 0.0, renormalize: bool = False, scoring: str = "softmax",
                 scale: float = 1.0, correction: bool = False, shared_size: int = None):
        super().__init__()
        if activation not in packed_ops.EXPERT_KINDS:
            raise ValueError(f"unknown expert activation {activation!r}")
        if not 1 <= top_k <= num_experts:
            raise ValueError(f"top_k {top_k} of {num_experts} experts")
        if scoring not in ("softmax", "sigmoid") or (correction and scoring != "sigmoid"):
            raise ValueError(f"router scoring {scoring!r} (a correction goes with sigmoid scores)")
        self.top_k, self.limit, self.renormalize = top_k, float(limit), renormalize
        self.kind = packed_ops.EXPERT_KINDS[activation]
        self.scoring, self.scale = scoring, float(scale)
        self.router = nn.Linear(in_features, num_experts, bias=False)
        if self.kind != packed_ops.UNGATED:
            self.gate = nn.Parameter(torch.randn(num_experts, intermediate_size, in_features) * in_features ** -0.5)
        self.up = nn.Parameter(torch.randn(num_experts, intermediate_size, in_features) * in_features ** -0.5)
        self.down = nn.Parameter(torch.randn(num_experts, in_features, intermediate_size) * intermediate_size ** -0.5)
        if correction:
            self.correction = nn.Parameter(torch.zeros(num_experts))
        self.shared = None
        if shared_size is not None:
            self.shared = GeluMLP(in_features, shared_size)
            self.shared_gate = nn.Linear(in_features, 1, bias=False)

    def packed(self) -> dict:
        return packed_ops.pack_experts(None if self.kind == packed_ops.UNGATED else self.gate, self.up, self.down)

    def routing(self) -> tuple[Tensor, dict]:
        """(router rows, the shared expert's gate row last; keyword arguments) of ``ops.packed.route``."""
        wr, c = self.router.weight, getattr(self, "correction", None)
        if self.shared is not None:
            wr = torch.cat([wr, self.shared_gate.weight])
        return wr.contiguous(), dict(top=self.top_k, renorm=self.renormalize, sigmoid=self.scoring == "sigmoid",
                                     correction=None if c is None else c.float().contiguous(), scale=self.scale,
                                     gate=self.shared is not None)

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        h = _rows(x, self.up.dtype)
        wr, rule = self.routing()
        ids, wts = packed_ops.route(h, wr, **rule)
        y = packed_ops.experts(h, ids, self.packed(), self.kind, self.limit)
        shared = None if self.shared is None else self.shared(h)
        return packed_ops.Delta(y, pair_w=wts, shared=shared).value().view(x.shape)


class OutputLinear(nn.Linear):
    """Output projection without a bias: fp32 logits of rows rounded to the weight's dtype."""

    def __init__(self, in_features: int, out_features: int):
        super().__init__(in_features, out_features, bias=False)

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        return packed_ops.logits(_rows(x, self.weight.dtype), self.weight).float().view(*x.shape[:-1], -1)


class TiedLinear(nn.Module):
    """Output projection with the weight of an embedding layer (``source``: its index in the layer list),
    times ``scale``."""

    def __init__(self, source: int = 0, scale: float = 1.0):
        super().__init__()
        self.source, self.scale = source, float(scale)
        self._table = ()

    def bind(self, layers):
        self._table = (layers[self.source],)

    @property
    def weight_source(self) -> nn.Embedding:
        return self._table[0]

    def forward(self, x: Tensor) -> Tensor:
        _no_grad_only(self, x)
        w = self._table[0].weight
        h = (x.float() * self.scale).to(w.dtype).reshape(-1, x.shape[-1]).contiguous()
        return packed_ops.logits(h, w).float().view(*x.shape[:-1], -1)


def bind_layers(layers: nn.ModuleList):
    """Resolve the references between layers of one model (tied weights, shared latents)."""
    latent = [m for m in layers.modules() if isinstance(m, LatentAttention)]
    for m in latent:
        m.bind(latent)
    for m in layers:
        if isinstance(m, TiedLinear):
            m.bind(layers)
