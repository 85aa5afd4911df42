"""Ops of the packed decoder step: the new tokens of several sequences laid end to end, no padding.

A :class:`PackedBatch` (made by the state manager, ``models/kv_cache.py: SequenceState``) describes the
rows; the residual stream is fp32 ``[N, C]``, sublayer inputs and outputs have the model's dtype.
GPU: ``csrc/kernels/packed_rows.hip``, ``latent_attn.hip``, ``latent_mfma.hip``, ``experts.hip``.
Window and linear attention: ``ops/window.py``, ``ops/linear_attn.py``.
CPU: the torch forms below (also what the GPU parity tests may compare single kernels with).
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
from torch import Tensor

from penroz.ops._ext import kernels, use_kernels
from penroz.ops import gemm as gemm_ops


def upload(values, dtype: torch.dtype, device: torch.device) -> Tensor:
    """Host values as a tensor on ``device``. By way of pinned memory, whose copy is one more piece of the stream's work: a copy from
    pageable memory waits for all that the stream has been given, and the GPU then idles until the next kernels arrive (64 sequences
    of Golepel stepped token by token, 0.15 of 1.25 ms a step)."""
    t = torch.tensor(values, dtype=dtype)
    if device.type != "cuda" or t.numel() == 0:
        return t.to(device)
    if torch.cuda.is_current_stream_capturing():  # each replay would copy what the pinned block holds by then
        raise RuntimeError("a captured graph cannot bring values from the host: make them tensors before the capture")
    return t.pin_memory().to(device, non_blocking=True)


@dataclass
class PackedBatch:
    """Rows of one step. Per row (int32 [N]): ``slot`` of its sequence, ``pos`` in it, ``first`` row of the
    sequence in this step. Per sequence (int32): ``cu`` [S + 1] row offsets, ``seq_slot`` [S]. Host side:
    ``single`` — one new token per sequence (a decode step); ``fresh`` — every sequence starts at position
    0; ``lens`` / ``counts`` — tokens held after the step and new tokens, per sequence (empty in a captured
    step, where positions live on the device only); ``max_len`` bounds them."""
    slot: Tensor
    pos: Tensor
    first: Tensor
    cu: Tensor
    seq_slot: Tensor
    single: bool
    fresh: bool
    counts: list
    lens: list
    max_len: int
    advance: bool = False  # the step's first kernel increments pos (captured decode step)
    _kv: dict | None = None
    _blocks: Tensor | None = None
    _spans: dict | None = None

    @property
    def rows(self) -> int:
        return self.slot.numel()

    def key_rows(self) -> tuple[Tensor, int]:
        """(int32 [S + 1] offsets of every sequence's keys laid end to end, their total)."""
        if self._kv is None:
            off = [0]
            for n in self.lens:
                off.append(off[-1] + n)
            self._kv = {"cu": upload(off, torch.int32, self.slot.device), "n": off[-1]}
        return self._kv["cu"], self._kv["n"]

    def query_blocks(self, size: int = 128) -> Tensor:
        """int32 [blocks, 2]: (sequence, first query) of every block of ``size`` queries, the ones with the
        most keys first."""
        if self._blocks is None:
            blk = [(l - n + min(q + size, n), s, q) for s, (n, l) in enumerate(zip(self.counts, self.lens))
                   for q in range(0, n, size)]
            blk.sort(key=lambda b: -b[0])
            self._blocks = upload([b[1:] for b in blk], torch.int32, self.slot.device)
        return self._blocks

    def spans(self, size: int) -> tuple[Tensor, Tensor]:
        """(int32 [spans, 2]: (sequence, first new token) of every piece of ``size`` new tokens, in order; int32
        [S + 1] offsets of the sequences' pieces)."""
        if self._spans is None:
            self._spans = {}
        if size not in self._spans:
            rows = [(s, q) for s, n in enumerate(self.counts) for q in range(0, n, size)]
            off = [0]
            for n in self.counts:
                off.append(off[-1] - (-n // size))
            self._spans[size] = tuple(upload(t, torch.int32, self.slot.device) for t in (rows, off))
        return self._spans[size]


# --------------------------------------------------------------------------- rotation table
def rotation_table(base: float, dims: int, positions: int, device) -> Tensor:
    """fp32 [positions, dims]: cos then sin of position · base^(-2i/dims), angles formed in float64."""
    f = torch.pow(torch.tensor(float(base), dtype=torch.float64),
                  -torch.arange(0, dims, 2, dtype=torch.float64) / dims)
    a = torch.arange(positions, dtype=torch.float64)[:, None] * f
    return torch.cat([a.cos(), a.sin()], dim=1).float().to(device)


def _rotate(x: Tensor, tab: Tensor) -> Tensor:
    """Rotate-half of fp32 x [..., rot] with table rows [..., rot] (broadcast)."""
    h = x.shape[-1] // 2
    u, v, c, s = x[..., :h], x[..., h:], tab[..., :h], tab[..., h:]
    return torch.cat([u * c - v * s, v * c + u * s], dim=-1)


# --------------------------------------------------------------------------- norms
def grouped_rms(x: Tensor, groups: int, eps: float) -> Tensor:
    """fp32: each of ``groups`` equal parts of the last dimension over its own root mean square."""
    p = x.float().unflatten(-1, (groups, -1))
    return (p * torch.rsqrt(p.square().mean(-1, keepdim=True) + eps)).flatten(-2)


def row_norm(x: Tensor, w: Tensor, groups: int, eps: float, dtype: torch.dtype, rows: Tensor | None = None) -> Tensor:
    """Grouped RMS norm of (selected) fp32 rows [N, C], times fp32 w, in ``dtype``."""
    if use_kernels(x):
        out = torch.empty(x.shape[0] if rows is None else rows.numel(), x.shape[1], dtype=dtype, device=x.device)
        kernels().row_norm(x, rows, w, groups, eps, out)
        return out
    x = x if rows is None else x[rows.long()]
    return (grouped_rms(x, groups, eps) * w).to(dtype)


# --------------------------------------------------------------------------- residual + convolution
def _conv_torch(x: Tensor, cw: Tensor, state: Tensor, b: PackedBatch) -> Tensor:
    """x + causal convolution, sequence by sequence; updates ``state`` rows of the batch."""
    taps = cw.shape[0]
    out = x.clone()
    cu, slots = b.cu.tolist(), b.seq_slot.tolist()
    for s, slot in enumerate(slots):
        r0, r1 = cu[s], cu[s + 1]
        p0 = int(b.pos[r0])
        old = state[slot].clone()
        if p0 < taps - 1:
            old[:taps - 1 - p0] = 0
        seq = torch.cat([old, x[r0:r1]])
        for j in range(taps):
            out[r0:r1] += cw[j] * seq[j:j + r1 - r0]
        state[slot] = seq[seq.shape[0] - (taps - 1):]
    return out


def _norm_conv_fits(x: Tensor, y: Tensor, w: Tensor, groups: int, cw: Tensor, state: Tensor, dtype: torch.dtype) -> bool:
    """Whether the residual add, its norm and the convolution of a prompt run as one pass: a norm group is what one
    wave holds, its registers keep the rows of up to 4 taps (8192 rows of 2048: 56 us as two passes, 38 as one), and y
    and the output are of one type."""
    return (y.dtype == dtype and x.shape[1] in (256 * groups, 512 * groups) and cw.shape[0] <= 4
            and all(t.data_ptr() % 16 == 0 for t in (x, y, w, cw, state)))


def residual_conv(b: PackedBatch, dtype: torch.dtype, *, x: Tensor | None = None, embed: tuple[Tensor, Tensor] | None = None,
                  y: Tensor | None = None, pair_w: Tensor | None = None, norm: tuple[Tensor, int, float] | None = None,
                  conv: tuple[Tensor, Tensor] | None = None) -> tuple[Tensor, Tensor | None]:
    """The step between two sublayers: x (fp32, or the embedding rows of ``embed`` = (ids, table)) +=
    norm(y), then, with ``conv`` = (fp32 taps [taps, C], state), the next sublayer's input x + conv(x) in
    ``dtype``. ``norm`` = (fp32 w, groups, eps). ``pair_w`` [N, top]: y holds ``top`` expert rows per token,
    summed with these weights. The GPU updates x in place, or leaves it and returns another buffer
    (``_norm_conv_fits``). Returns (x, h or None)."""
    ref = x if x is not None else embed[1]
    if use_kernels(ref):
        K = kernels()
        N, C = b.rows, ref.shape[1]
        tok, table = (embed[0], embed[1]) if embed is not None else (None, None)
        xo = x if x is not None else torch.empty(N, C, dtype=torch.float32, device=ref.device)
        cw, st = conv if conv is not None else (None, None)
        w, g, eps = norm if norm is not None else (None, 1, 0.0)
        h = torch.empty(N, C, dtype=dtype, device=ref.device) if conv is not None else None
        if conv is None or b.single:
            adv = b.advance and embed is not None
            K.row_norm_add(tok, table, x, xo, y, pair_w, w, g, eps, cw, st, b.slot, b.pos, adv, h)
        elif embed is None and y is not None and pair_w is None and _norm_conv_fits(x, y, w, g, cw, st, dtype):
            xo = torch.empty_like(x)
            K.norm_conv_rows(x, xo, y, w, g, eps, cw, st, b.slot, b.pos, b.first, b.cu, b.seq_slot, h)
        else:
            if embed is not None or y is not None:
                K.row_norm_add(tok, table, x, xo, y, pair_w, w, g, eps, None, None, None, None, False, None)
            K.conv_rows(xo, cw, st, b.slot, b.pos, b.first, b.cu, b.seq_slot, h)
        return xo, h
    if embed is not None:
        x = embed[1][embed[0].reshape(-1)].float()
    if y is not None:
        yf = y.float()
        if pair_w is not None:
            yf = (yf.view(pair_w.shape[0], pair_w.shape[1], -1) * pair_w.unsqueeze(-1)).sum(1)
        x = x + grouped_rms(yf, norm[1], norm[2]) * norm[0]
    return x, (_conv_torch(x, *conv, b).to(dtype) if conv is not None else None)


# --------------------------------------------------------------------------- residual + pre-norm
@dataclass
class Delta:
    """What a sublayer adds to the residual stream: ``y`` [N, C], or ``coef`` · (y + y2), each RMS-normed over C
    with its fp32 weight ``w`` / ``w2`` where it has one; or, with ``pair_w`` [N, top], the weighted sum of y's
    ``top`` expert rows per token, plus ``shared`` [N, C] times the last column of pair_w [N, top + 1]."""
    y: Tensor
    y2: Tensor | None = None
    w: Tensor | None = None
    w2: Tensor | None = None
    coef: float = 1.0
    eps: float = 0.0
    pair_w: Tensor | None = None
    shared: Tensor | None = None

    def value(self) -> Tensor:
        """fp32 [N, C] (torch form)."""
        y = self.y.float()
        if self.pair_w is not None:
            top = self.pair_w.shape[1] - (self.shared is not None)
            y = (y.view(self.pair_w.shape[0], top, -1) * self.pair_w[:, :top, None]).sum(1)
            return y if self.shared is None else y + self.shared.float() * self.pair_w[:, top:]
        parts = [(y, self.w)] + ([(self.y2.float(), self.w2)] if self.y2 is not None else [])
        return self.coef * sum(p if w is None else grouped_rms(p, 1, self.eps) * w for p, w in parts)


def residual_norm(b: PackedBatch, dtype: torch.dtype, *, x: Tensor | None = None,
                  embed: tuple[Tensor, Tensor, Tensor | None] | None = None, delta: Delta | None = None,
                  norm: tuple[Tensor, float] | None = None) -> tuple[Tensor, Tensor | None]:
    """The step between two sublayers of pre-norm blocks: x (fp32, or the rows of ``embed`` = (ids, token table,
    position table or None)) += delta, then, with ``norm`` = (fp32 w, eps), the next sublayer's input
    rms_norm(x) · w in ``dtype``. x is updated in place on the GPU. Returns (x, h or None)."""
    ref = x if x is not None else embed[1]
    if use_kernels(ref):
        N, C = b.rows, ref.shape[1]
        tok, table, ptable = embed if embed is not None else (None, None, None)
        xo = x if x is not None else torch.empty(N, C, dtype=torch.float32, device=ref.device)
        h = torch.empty(N, C, dtype=dtype, device=ref.device) if norm is not None else None
        w, eps = norm if norm is not None else (None, 0.0)
        d = delta if delta is not None else Delta(None)
        kernels().residual_norm(tok, table, ptable, x, xo, d.y, d.w, d.y2, d.w2, d.coef, d.eps, d.pair_w, d.shared, w,
                                eps, b.pos, b.advance and embed is not None, h)
        return xo, h
    if embed is not None:
        x = embed[1][embed[0].reshape(-1)].float()
        if embed[2] is not None:
            x = x + embed[2][b.pos.long()].float()
    if delta is not None:
        x = x + delta.value()
    return x, ((grouped_rms(x, 1, norm[1]) * norm[0]).to(dtype) if norm is not None else None)


# --------------------------------------------------------------------------- projections
def _gemv_ok(x: Tensor, w: Tensor, max_k: int) -> bool:
    """1-4 bf16 rows on the decode GEMV (csrc/kernels/decode_linear.hip)."""
    K = x.shape[1]
    return (x.dtype == torch.bfloat16 and 1 <= x.shape[0] <= 4 and K % 8 == 0 and K <= max_k
            and w.data_ptr() % 16 == 0 and x.data_ptr() % 16 == 0 and x.is_contiguous())


def linear(x: Tensor, w: Tensor, past: int = gemm_ops.KEEP) -> Tensor:
    """x [M, K] · wᵀ in x's dtype (decode-shaped kernels at few rows, the library GEMM otherwise). ``past``, here and below:
    weights from this size on are read past the caches (``gemm.past_caches``)."""
    if x.is_cuda and x.dtype == torch.bfloat16:
        if _gemv_ok(x, w, 8192):
            out = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
            kernels().decode_gemv(x, None, None, None, None, None, None, 0.0, w, None, out, 0, past=w.nbytes >= past)
            return out
        from penroz.models.graph_decode import _linear
        return _linear(x, w, w.nbytes >= past)
    return torch.mm(x, w.t())


def logits(h: Tensor, table: Tensor, past: int = gemm_ops.KEEP) -> Tensor:
    """fp32 (bf16 at decode-shaped row counts) logits of normed rows over the embedding table."""
    if h.is_cuda and h.dtype == torch.bfloat16:
        if h.shape[0] <= 4 and _gemv_ok(h, table, 8192):
            return linear(h, table, past)
        if h.shape[0] <= 16 and gemm_ops.skinny_ok(h, table):
            y = gemm_ops.rows_linear(h, table, past=table.nbytes >= past)
            return gemm_ops.skinny_linear(h, table, None) if y is None else y
        return gemm_ops.linear_fp32(h, table, past=table.nbytes >= past)
    return torch.mm(h, table.t()).float()


def gated_linear(x: Tensor, gu: Tensor, kind: int, limit: float = 0.0, past: int = gemm_ops.KEEP) -> Tensor:
    """act(x·Wgᵀ, x·Wuᵀ) of the packed [gate; up] weight; kind 0 silu, 1 clamped (``expert_activation``)."""
    if x.is_cuda:
        from penroz.models.graph_decode import DECODE_EPILOGUES, SKINNY_MAX_ROWS
        if kind == 0 and DECODE_EPILOGUES and _gemv_ok(x, gu, 1792):
            out = torch.empty(x.shape[0], gu.shape[0] // 2, dtype=x.dtype, device=x.device)
            kernels().decode_gemv_pair(x, gu, out, 1, 2, past=gu.nbytes >= past)
            return out
        if (kind == 0 and DECODE_EPILOGUES and x.shape[0] <= SKINNY_MAX_ROWS and gemm_ops.skinny_ok(x, gu)):
            return gemm_ops.skinny_gated(x, gu, 2)
        z = linear(x, gu, past)
        out = torch.empty(x.shape[0], gu.shape[0] // 2, dtype=x.dtype, device=x.device)
        kernels().gated_rows(z, kind, float(limit), out)
        return out
    g, u = torch.mm(x, gu.t()).chunk(2, dim=1)
    return expert_activation(g.float(), u.float(), kind, limit).to(x.dtype)


def gelu_mlp(x: Tensor, up: Tensor, down: Tensor, past: int = gemm_ops.KEEP) -> Tensor:
    """gelu(x · upᵀ) · downᵀ (erf form, no biases)."""
    if x.is_cuda:
        if _gemv_ok(x, up, 8192):
            u = torch.empty(x.shape[0], up.shape[0], dtype=x.dtype, device=x.device)
            kernels().decode_gemv(x, None, None, None, None, None, None, 0.0, up, None, u, 1, past=up.nbytes >= past)
        else:
            u = gemm_ops.rows_linear(x, up, gelu=True, past=up.nbytes >= past)
            if u is None:
                u = linear(x, up, past)
                kernels().gelu_rows(u)
    else:
        u = torch.nn.functional.gelu(torch.mm(x, up.t()).float()).to(x.dtype)
    return linear(u, down, past)


def expert_activation(g: Tensor | None, u: Tensor, kind: int, limit: float) -> Tensor:
    if kind == UNGATED:
        return torch.nn.functional.gelu(u)
    if kind == 1:
        g = g.clamp(max=limit)
        return g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1.0)
    return g * torch.sigmoid(g) * u


# --------------------------------------------------------------------------- latent attention
@dataclass
class LatentSizes:
    """One latent-attention layer: heads and, per head, unrotated / rotated query-key and value sizes;
    the latent's rank. The padded sizes (multiples of 8, zero weight rows) are the kernels' layout."""
    heads: int
    dim: int
    rot: int
    vdim: int
    rank: int
    scale: float
    base: float
    eps: float

    @staticmethod
    def pad8(n: int) -> int:
        return (n + 7) // 8 * 8

    @property
    def d8(self):
        return self.pad8(self.dim)

    @property
    def r8(self):
        return self.pad8(self.rot)

    @property
    def v8(self):
        return self.pad8(self.vdim)

    @property
    def R8(self):
        return self.pad8(self.rank)

    @property
    def cache_width(self):
        return self.R8 + self.r8

    @property
    def q_width(self):
        return self.heads * (self.d8 + self.r8)


def _pad(w: Tensor, dim: int, to: int) -> Tensor:
    if w.shape[dim] == to:
        return w
    shape = list(w.shape)
    shape[dim] = to - w.shape[dim]
    return torch.cat([w, w.new_zeros(shape)], dim=dim)


def pack_latent(s: LatentSizes, q: Tensor, dkv: Tensor | None, uk: Tensor, uv: Tensor, o: Tensor) -> dict:
    """The layer's weights in the kernels' layout: ``z`` [q rows; latent rows], ``uk`` [H, d8, R8],
    ``uka`` (the absorbing kernel's form), ``uv`` [H, v8, R8], ``ukv`` = both up-projections stacked for the
    expanded form, ``o`` [C, H·v8]."""
    C = q.shape[1]
    qp = q.view(s.heads, s.dim + s.rot, C)
    z = torch.cat([_pad(qp[:, :s.dim], 1, s.d8), _pad(qp[:, s.dim:], 1, s.r8)], dim=1).reshape(-1, C)
    if dkv is not None:
        z = torch.cat([z, _pad(dkv[:s.rank], 0, s.R8), _pad(dkv[s.rank:], 0, s.r8)])
    ukp = _pad(_pad(uk.view(s.heads, s.dim, s.rank), 1, s.d8), 2, s.R8).contiguous()
    uvp = _pad(_pad(uv.view(s.heads, s.vdim, s.rank), 1, s.v8), 2, s.R8).contiguous()
    op = _pad(o.view(-1, s.heads, s.vdim), 2, s.v8).reshape(o.shape[0], -1)
    # the absorbing kernel reads uk by its reduction: bf16 (MFMA) wants it contiguous per latent column
    uka = ukp.transpose(1, 2).contiguous() if q.dtype == torch.bfloat16 else ukp
    return {"z": z.contiguous(), "uk": ukp, "uka": uka, "uv": uvp, "o": op.contiguous(),
            "ukv": torch.cat([ukp.reshape(-1, s.R8), uvp.reshape(-1, s.R8)]).contiguous()}


def _latent_rows_torch(s: LatentSizes, zl: Tensor, nw: Tensor, tab: Tensor, dtype) -> Tensor:
    """Cache rows [n, R8 + r8] of latent projection rows zl (fp32 math)."""
    c = grouped_rms(zl[:, :s.rank], 1, s.eps) * nw
    k = _rotate(zl[:, s.R8:s.R8 + s.rot].float(), tab)
    return torch.cat([_pad(c, 1, s.R8), _pad(k, 1, s.r8)], dim=1).to(dtype)


def latent_attention(s: LatentSizes, w: dict, z: Tensor, cache: Tensor, nw: Tensor | None, tab: Tensor,
                     b: PackedBatch) -> Tensor:
    """Attention of the packed projection rows z (``w["z"]`` output) over the sequences' latent caches,
    after writing this step's own latent rows when the layer has them (``nw``: their norm weight; None:
    ``cache`` belongs to an earlier layer, which wrote it). Returns [N, H·v8]."""
    N, dt = z.shape[0], z.dtype
    if use_kernels(z):
        return _latent_attention_gpu(s, w, z, cache, nw, tab, b)
    pos, slot = b.pos.long(), b.slot.long()
    if nw is not None:
        cache[slot, pos] = _latent_rows_torch(s, z[:, s.q_width:], nw, tab[pos], dt)
    q = z[:, :s.q_width].view(N, s.heads, s.d8 + s.r8).float()
    qr = _rotate(q[..., s.d8:s.d8 + s.rot], tab[pos].unsqueeze(1))
    qa = torch.cat([torch.einsum("nhd,hdr->nhr", q[..., :s.d8], w["uk"].float()), _pad(qr, 2, s.r8)], dim=2)
    out = torch.empty(N, s.heads, s.v8)
    for i in range(N):
        keys = cache[slot[i], :int(pos[i]) + 1].float()
        p = torch.softmax(qa[i] @ keys.t() * s.scale, dim=-1)
        out[i] = torch.einsum("hr,hvr->hv", p @ keys[:, :s.R8], w["uv"].float())
    return out.reshape(N, -1).to(dt)


# bf16 steps whose longest new portion is at most this many tokens run every row through the decode
# kernel (queries in latent space, no keys are formed); longer portions expand keys and values once
DECODE_MAX_PORTION = 4
# workgroups aimed at when a row's keys are split: one per CU, two where the latent is narrow (decode +
# value up-projection, R = 512, H = 16: 16 rows × 1024 keys 16.0 µs at 16 ranges, 23.4 at 32; 64 × 4096
# 72.5 µs at 4, 78.8 at 8. R = 256, H = 8: 64 × 4096 43.7 µs at 4, 33.8 at 8)
DECODE_WORKGROUPS = 256
MAX_KEY_RANGES = 64


def key_ranges(rows: int, heads: int, max_len: int, rank: int = 512) -> int:
    """Key ranges per row of the decode kernel: fill the GPU, at least 64 keys each."""
    target = DECODE_WORKGROUPS * (2 if rank <= 256 else 1)
    want = -(-target // (rows * -(-heads // 32)))
    return max(1, min(want, -(-max_len // 64), MAX_KEY_RANGES))


def _latent_attention_gpu(s, w, z, cache, nw, tab, b):
    K = kernels()
    N, dev = z.shape[0], z.device
    out = torch.empty(N, s.heads * s.v8, dtype=z.dtype, device=dev)
    bf = z.dtype == torch.bfloat16
    dims = (s.heads, s.d8, s.r8, s.rot, s.rank)
    if bf and not b.single and max(b.counts) > DECODE_MAX_PORTION and K.latent_flash_ok(s.d8 + s.r8, s.v8):
        # expanded form: this step's latents (and the sequences' earlier ones) to keys and values per head
        fresh = b.fresh and nw is not None
        kcu, M = (b.cu, N) if b.fresh else b.key_rows()
        c = torch.empty(M, s.R8, dtype=z.dtype, device=dev)
        kr = torch.empty(M, s.r8, dtype=z.dtype, device=dev)
        K.latent_store(z, *dims, s.R8, nw, s.eps, tab, cache if nw is not None else None, b.slot, b.pos,
                       c if fresh else None, kr if fresh else None, True)
        if not fresh:
            K.latent_gather(cache, kcu, b.seq_slot, s.R8, s.r8, c, kr)
        K.latent_flash(z, gemm_ops.linear(c, w["ukv"]), kr, b.query_blocks(), b.cu, kcu, s.heads, s.d8, s.r8, s.v8,
                       s.scale, out)
        return out
    qa = torch.empty(N, s.heads, s.cache_width, dtype=z.dtype, device=dev)
    K.latent_absorb(z, *dims, w["uka"], tab, b.slot, b.pos, qa, nw, s.eps, cache if nw is not None else None)
    if bf and K.latent_decode_ok(s.R8, s.r8):
        P = key_ranges(N, s.heads, b.max_len, s.R8)
        ol = torch.empty(P, N, s.heads, s.R8, dtype=torch.float32, device=dev)
        ml = torch.empty(P, N, s.heads, 2, dtype=torch.float32, device=dev)
        K.latent_decode(qa, cache, b.slot, b.pos, s.R8, s.scale, ol, ml)
    else:
        ol, ml = torch.empty(1, N, s.heads, s.R8, dtype=torch.float32, device=dev), None
        K.latent_attn_row(qa, cache, b.slot, b.pos, s.R8, s.scale, ol)
    K.latent_uv(ol, ml, w["uv"], out)
    return out


# --------------------------------------------------------------------------- experts
EXPERT_ROWS_MAX_PAIRS = 1024  # the few-pairs kernel's pair list (csrc/kernels/experts.hip kMaxPairs)
EXPERT_KINDS = {"silu": 0, "clamped_swiglu": 1, "gelu": 2}
UNGATED = 2  # expert(x) = down · gelu(up · x): no gate


def pack_experts(gate: Tensor | None, up: Tensor, down: Tensor) -> dict:
    """gate / up [E, F, C], down [E, C, F] -> the kernels' layout: F padded to a multiple of 32, blocks of
    32 gate rows followed by the matching 32 up rows (the up rows alone without a gate)."""
    E, F, C = up.shape
    Fp = (F + 31) // 32 * 32
    if gate is None:
        return {"gu": _pad(up, 1, Fp).contiguous(), "down": _pad(down, 2, Fp).contiguous()}
    g, u = (_pad(t, 1, Fp).view(E, Fp // 32, 1, 32, C) for t in (gate, up))
    return {"gu": torch.cat([g, u], dim=2).reshape(E, 2 * Fp, C).contiguous(), "down": _pad(down, 2, Fp).contiguous()}


def route(h: Tensor, wr: Tensor, top: int, renorm: bool = False, *, sigmoid: bool = False,
          correction: Tensor | None = None, scale: float = 1.0, gate: bool = False) -> tuple[Tensor, Tensor]:
    """Choice by the scores of fp32 logits h·wrᵀ — softmax over all experts, or ``sigmoid`` each, then chosen by
    score + ``correction`` (fp32 [E]) — as int32 ids and fp32 weights (scores · ``scale``) [N, top], largest
    first. ``gate``: wr's last row is a shared expert's gate, whose sigmoid is one more weight column."""
    N = h.shape[0]
    if use_kernels(h):
        ids = torch.empty(N, top, dtype=torch.int32, device=h.device)
        wts = torch.empty(N, top + gate, dtype=torch.float32, device=h.device)
        rule = (sigmoid, correction, scale, renorm)
        if N <= 64:
            kernels().router_topk(None, h, wr, *rule, ids, wts)
        else:
            z = gemm_ops.linear_fp32(h, wr) if h.dtype == torch.bfloat16 else torch.mm(h, wr.t())
            kernels().router_topk(z, None, None, *rule, ids, wts)
        return ids, wts
    z = h.float() @ wr.float().t()
    z, g = (z[:, :-1], z[:, -1:]) if gate else (z, None)
    s = torch.sigmoid(z) if sigmoid else torch.softmax(z, dim=-1)
    ids = (s if correction is None else s + correction).topk(top, dim=-1).indices
    wts = s.gather(1, ids) * scale
    if renorm:
        wts = wts / wts.sum(-1, keepdim=True)
    return ids.int(), (wts if g is None else torch.cat([wts, torch.sigmoid(g)], dim=1))


def experts_beside_shared(h: Tensor, ids: Tensor, w: dict, kind: int, limit: float, shared: dict, past: int = gemm_ops.KEEP,
                          experts_past: bool = False) -> tuple[Tensor, Tensor]:
    """:func:`experts` and :func:`gelu_mlp` of a shared expert on the same rows, in the same launches where there are kernels for that
    (``experts_rows_shared`` in csrc/kernels/experts.hip)."""
    if kind == UNGATED and h.shape[0] <= 16 and h.dtype == torch.bfloat16 and use_kernels(h):
        both = kernels().experts_rows_shared(h, ids, w["gu"], w["down"], float(limit), shared["up"], shared["down"], experts_past)
        if both is not None:
            return both
    return experts(h, ids, w, kind, limit, experts_past), gelu_mlp(h, **shared, past=past)


def few_pairs(P: int, w: dict) -> bool:
    """Whether ``P`` (token, choice) pairs of bf16 experts are the few-pairs kernel's: it reads an expert's weights again for every 16 of
    its pairs, where the tiles of ``experts_grouped`` read them once behind a sort (13 to 20 us). Both products, gated, us, few pairs /
    tiles at 32 and 96 pairs per expert: 8 experts, C 2048, F 1024 54 / 38 and 129 / 53; 4 of them (48 MB) 36 / 34 and 81 / 50; 8, C 1024,
    F 768 (36 MB) 29 / 26 and 63 / 36; 8, C 512, F 512 (12 MB) 15 / 17 and 29 / 22; 2, C 2048, F 1024 24 / 33 and 47 / 49, but 59 / 50 at 128."""
    E, F, C = w["gu"].shape[0], w["down"].shape[2], w["down"].shape[1]
    large = E >= 4 and w["gu"].nbytes + w["down"].nbytes >= 36 << 20
    many = P >= max(96 * E, 256) or (large and P >= 32 * E)
    return P <= EXPERT_ROWS_MAX_PAIRS and not (many and 2 * F * C < 1 << 31)  # (the tiles' byte offsets have 32 bits)


def experts(h: Tensor, ids: Tensor, w: dict, kind: int, limit: float, past: bool = False) -> Tensor:
    """Outputs of the chosen experts, one row per (token, choice): [N·top, C]. ``past``: few pairs read the weights past the caches
    (``gemm.past_caches``)."""
    P, C, F = ids.numel(), h.shape[1], w["down"].shape[2]
    if use_kernels(h):
        act = torch.empty(P, F, dtype=h.dtype, device=h.device)
        y = torch.empty(P, C, dtype=h.dtype, device=h.device)
        K, a = kernels(), (h, ids, w["gu"], w["down"], kind, float(limit), act, y)
        if h.dtype != torch.bfloat16 or C % 32:
            K.experts_plain(*a)
        else:
            i32 = dict(dtype=torch.int32, device=h.device)
            top, E, few = ids.shape[1], w["gu"].shape[0], few_pairs(P, w)
            # the kernels' 32-bit byte offsets bound the rows of one call
            rows = max(1, (1 << 31) // max(C, top * F, 1) - 1)
            for r in range(0, h.shape[0], rows):
                n = min(rows, h.shape[0] - r)
                if n < h.shape[0]:
                    p = slice(r * top, (r + n) * top)
                    a = (h[r:r + n], ids[r:r + n], *a[2:6], act[p], y[p])
                if few:
                    K.experts_rows(*a, past)
                else:
                    K.experts_grouped(*a, torch.empty(n * top, **i32), torch.empty(1 + 3 * (n * top // 128 + E), **i32))
        return y
    y = torch.empty(P, C, dtype=h.dtype)
    flat, top = ids.reshape(-1).long(), ids.shape[1]
    for e in flat.unique().tolist():
        sel = (flat == e).nonzero().squeeze(1)
        gu = (h[sel // top] @ w["gu"][e].t()).float()
        if kind == UNGATED:
            a = expert_activation(None, gu, kind, limit).to(h.dtype)
        else:
            gu = gu.view(len(sel), -1, 2, 32)
            a = expert_activation(gu[:, :, 0], gu[:, :, 1], kind, limit).reshape(len(sel), F).to(h.dtype)
        y[sel] = a @ w["down"][e].t()
    return y
