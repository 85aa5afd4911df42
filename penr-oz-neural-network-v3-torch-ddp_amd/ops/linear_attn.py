"""Linear attention with a decayed matrix state (retention, gated linear attention) on the packed step's rows
(``ops/packed.py``).

Per head: S_t = diag(alpha_t) S_(t-1) + k_t v_tᵀ, o_t = scale · S_tᵀ q_t; alpha is a constant per head, or per
token and key channel sigmoid(z)^(1/tau), z = W (low-rank input) + b. The output is o over its root mean square
(times a weight over the value size when there is one), times silu of the gate columns. The state is fp32.
GPU: ``csrc/kernels/linear_attn.hip`` (token by token), ``linear_mfma.hip`` (prompts in chunks). CPU: torch.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
from torch import Tensor

from penroz.ops import gemm as gemm_ops, packed as P
from penroz.ops._ext import kernels, use_kernels
from penroz.ops.window import head_columns, head_rows

MAX_DIM = 256  # widest key or value of a head, and the decay's low rank


@dataclass(frozen=True)
class LinearSizes:
    """One layer: heads, key and value size per head, scale of the output, eps of the output norm; for decays
    from the input their low rank and tau. The padded sizes (multiples of 8, zero weight rows) are the
    kernels' layout."""
    heads: int
    dim: int
    vdim: int
    scale: float
    eps: float
    rank: int = 0
    tau: float = 1.0

    def check(self):
        if max(self.dim, self.vdim, self.rank) > MAX_DIM or min(self.dim, self.vdim) < 1:
            raise ValueError(f"head sizes {self.dim} / {self.vdim}, decay rank {self.rank} (at most {MAX_DIM})")
        if self.rank and self.tau <= 0:
            raise ValueError(f"tau {self.tau} must be positive")

    @property
    def d8(self):
        return (self.dim + 7) // 8 * 8

    @property
    def v8(self):
        return (self.vdim + 7) // 8 * 8

    @property
    def r8(self):
        return (self.rank + 7) // 8 * 8

    @property
    def width(self):  # projection columns
        return 2 * self.heads * (self.d8 + self.v8) + self.r8

    @property
    def state(self):
        return (self.heads, self.d8, self.v8)

    @property
    def kernel_sizes(self):
        return [self.heads, self.d8, self.v8, self.vdim, self.r8]


def pack_linear(s: LinearSizes, q: Tensor, k: Tensor, v: Tensor, g: Tensor, o: Tensor, *, decay: Tensor | None = None,
                a1: Tensor | None = None, a2: Tensor | None = None, bias: Tensor | None = None,
                norm: Tensor | None = None) -> dict:
    """``z`` = the stacked projection [q; k; v; g; a1], ``o``, the decays (fp32 ``decay`` per head, or the second
    low-rank projection ``a2`` [heads · d8, r8] with fp32 ``bias``) and the fp32 output ``norm``, padded."""
    H = s.heads
    z = [head_rows(q, H, s.d8), head_rows(k, H, s.d8), head_rows(v, H, s.v8), head_rows(g, H, s.v8)]
    w = {"o": head_columns(o, H, s.v8), "decay": None if decay is None else decay.float().contiguous(), "a2": None,
         "bias": None, "norm": None if norm is None else P._pad(norm.float(), 0, s.v8).contiguous()}
    if a1 is not None:
        z.append(P._pad(a1, 0, s.r8))
        w["a2"] = P._pad(head_rows(a2, H, s.d8), 1, s.r8).contiguous()
        w["bias"] = P._pad(bias.float().view(H, s.dim), 1, s.d8).reshape(-1).contiguous()
    w["z"] = torch.cat(z)
    return w


# portions up to this many tokens are stepped token by token, longer ones run in chunks
STEP_MAX_PORTION = 16
CHUNK = 64
# workgroups (span of a sequence × head) aimed at when sequences are cut into spans: two per CU, one where the key's
# width leaves registers and LDS for no second (8 × 1024 tokens, 16 heads of 128: 102 µs at 256, 112 at 512; 8 heads of
# 64: 42 and 35)
CHUNK_WORKGROUPS = 512


def span(s: LinearSizes, counts: list) -> int:
    """Tokens per span: sequences in one piece unless that leaves the GPU empty."""
    chunks = sum(-(-n // CHUNK) for n in counts)
    longest = -(-max(counts) // CHUNK)
    target = CHUNK_WORKGROUPS // (2 if s.d8 > 64 else 1)
    return CHUNK * min(longest, max(1, -(-chunks * s.heads // target)))


def linear_attention(s: LinearSizes, w: dict, z: Tensor, state: Tensor, b: P.PackedBatch) -> Tensor:
    """The layer's output rows [N, heads · v8] (normed and gated) of the projection rows z [N, width]; ``state``
    [slots, heads, d8, v8] moves on."""
    N = z.shape[0]
    if use_kernels(z):
        out = torch.empty(N, s.heads * s.v8, dtype=z.dtype, device=z.device)
        args = (z, s.kernel_sizes, s.scale, s.eps, s.tau, w["decay"], w["a2"], w["bias"], state, w["norm"], b.cu,
                b.seq_slot, b.pos)
        K = kernels()
        if (z.dtype == torch.bfloat16 and not b.single and max(b.counts) > STEP_MAX_PORTION
                and K.linear_chunk_ok(s.d8, s.v8)):
            length = span(s, b.counts)
            spans, cs = b.spans(length)
            zdec = ws = wdec = None
            if s.rank:  # bf16 operands: the products are exact, their sums fp32
                zdec = gemm_ops.linear_fp32(z[:, s.width - s.r8:s.width], w["a2"])
            if spans.shape[0] > len(b.counts):
                ws = torch.empty(spans.shape[0], *s.state, dtype=torch.float32, device=z.device)
                wdec = torch.empty(spans.shape[0], s.heads, s.d8, dtype=torch.float32, device=z.device)
            K.linear_chunk(*args, zdec, spans, cs, length, ws, wdec, out)
        elif b.single:
            K.linear_decode(*args, out)
        else:
            K.linear_step(*args, out)
        return out
    H = s.heads
    parts = z.float().split([H * s.d8, H * s.d8, H * s.v8, H * s.v8, s.r8], dim=1)
    q, k, v, g = (t.reshape(N, H, -1) for t in parts[:4])
    if w["decay"] is not None:
        alpha = w["decay"].view(1, H, 1).expand(N, H, s.d8)
    else:
        alpha = torch.exp(torch.nn.functional.logsigmoid(parts[4] @ w["a2"].float().t() + w["bias"]) / s.tau)
        alpha = alpha.view(N, H, s.d8)
    o = torch.empty(N, H, s.v8)
    cu = b.cu.tolist()
    for i, slot in enumerate(b.seq_slot.tolist()):
        S = torch.zeros_like(state[slot]) if int(b.pos[cu[i]]) == 0 else state[slot].clone()
        for t in range(cu[i], cu[i + 1]):
            S = alpha[t].unsqueeze(-1) * S + k[t].unsqueeze(-1) * v[t].unsqueeze(1)
            o[t] = (q[t].unsqueeze(1) @ S).squeeze(1) * s.scale
        state[slot] = S
    o = o * torch.rsqrt(o.square().sum(-1, keepdim=True) / s.vdim + s.eps)
    if w["norm"] is not None:
        o = o * w["norm"]
    return (o * torch.nn.functional.silu(g)).reshape(N, -1).to(z.dtype)
