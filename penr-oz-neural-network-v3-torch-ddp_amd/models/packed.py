"""The packed step: prefill, continued portions and batched decode of layer lists whose sequences carry
more state than keys and values (latent attention, causal convolutions, windows with pooled blocks, matrix
states), as one explicit kernel sequence over :class:`penroz.models.kv_cache.SequenceState`.

``PackedProgram`` is compiled from the model's own modules (patterns below) and serves every kind of step:
sequences of unequal length are laid end to end, so a batch computes no padding, and a sequence's result
does not depend on the others. ``GraphDecoder`` (``models/graph_decode.py``) captures its decode step;
``PackedSession`` is the step function by sequence name that generation and ``bin/trace_run`` use.

Patterns: embedding (or the sum of token and position embeddings), transformer blocks, grouped norm, output
projection (tied or its own), softmax on the last position. A block's two parts are [entry, sublayer]:
  * post-norm blocks — entry: causal convolution; a grouped norm on each sublayer's output;
  * pre-norm blocks — entry: RMS norm; no post-norms.
Sublayers: latent attention, retention, gated linear attention, window attention, two of them side by side;
gated MLP, mixture of experts. The feed-forward part may be absent.

Between two sublayers runs one op (``residual_conv`` / ``residual_norm``): the fp32 residual takes the last
sublayer's output (:class:`penroz.ops.packed.Delta`) and the next sublayer's input leaves in the model's dtype;
in a decode step that is one kernel, the convolution states included.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
from torch import Tensor, nn

from penroz.models import layers as L
from penroz.models.kv_cache import SequenceState
from penroz.ops import gemm as gemm_ops
from penroz.ops import linear_attn as linear_ops
from penroz.ops import packed as ops
from penroz.ops import window as window_ops


# --------------------------------------------------------------------------- sublayers
class _Sublayer:
    """``weights``, ``experts``: what a decode step multiplies its rows with; ``past``, ``experts_past``: what of it is read past
    the caches (``gemm.past_caches``, of the whole program's)."""
    past, experts, experts_past = gemm_ops.KEEP, (), False

    @property
    def weights(self) -> list[Tensor]:
        return [t for t in self.w.values() if t is not None and t.dim() > 1]


class _LatentMixer(_Sublayer):
    def __init__(self, m: L.LatentAttention, cache_index: int):
        self.s, self.w = m.sizes, m.packed()
        self.nw = m.dkv_norm.float() if m.kv_from is None else None
        self.cache_index = cache_index
        self.rotation = (m.sizes.base, m.sizes.rot)

    @property
    def weights(self) -> list[Tensor]:
        return [self.w[k] for k in ("z", "uka", "uv", "o")]

    def run(self, h: Tensor, b: ops.PackedBatch, st: SequenceState) -> ops.Delta:
        z = ops.linear(h, self.w["z"], self.past)
        o = ops.latent_attention(self.s, self.w, z, st.latent[self.cache_index], self.nw, st.tables[self.rotation], b)
        return ops.Delta(ops.linear(o, self.w["o"], self.past))


class _WindowMixer(_Sublayer):
    def __init__(self, m: L.WindowAttention, index: int):
        self.s, self.w, self.index = m.sizes, m.packed(), index
        self.pb = m.pb.float().contiguous()

    def attend(self, z: Tensor, b: ops.PackedBatch, st: SequenceState) -> Tensor:
        o = window_ops.window_attention(self.s, z, st.window[self.index], st.pooled[self.index], self.pb, st.tables, b)
        return ops.linear(o, self.w["o"], self.past)

    def run(self, h, b, st) -> ops.Delta:
        return ops.Delta(self.attend(ops.linear(h, self.w["z"], self.past), b, st))


class _LinearMixer(_Sublayer):
    def __init__(self, m, index: int):
        self.s, self.w, self.index = m.sizes, m.packed(), index

    def attend(self, z: Tensor, b: ops.PackedBatch, st: SequenceState) -> Tensor:
        return ops.linear(linear_ops.linear_attention(self.s, self.w, z, st.linear[self.index], b), self.w["o"],
                          self.past)

    def run(self, h, b, st) -> ops.Delta:
        return ops.Delta(self.attend(ops.linear(h, self.w["z"], self.past), b, st))


class _ParallelMixer(_Sublayer):
    """Two mixers on one stacked projection of the same input."""

    def __init__(self, m: L.ParallelMixers, left, right):
        self.left, self.right, self.eps = left, right, m.eps
        self.z = torch.cat([left.w["z"], right.w["z"]]).contiguous()
        self.lw, self.rw = m.left_out.float().contiguous(), m.right_out.float().contiguous()

    @property
    def weights(self) -> list[Tensor]:
        return [self.z] + [t for m in (self.left, self.right) for t in m.weights if t is not m.w["z"]]

    def run(self, h, b, st) -> ops.Delta:
        z, n = ops.linear(h, self.z, self.past), self.left.s.width
        return ops.Delta(self.left.attend(z[:, :n], b, st), self.right.attend(z[:, n:], b, st), self.lw, self.rw, 0.5,
                         self.eps)


class _DenseFF(_Sublayer):
    def __init__(self, m: L.GatedMLP):
        F, C = m.gate_proj.weight.shape
        Fp = (F + 7) // 8 * 8  # zero rows up to the kernels' vector width
        self.gu = torch.cat([ops._pad(m.gate_proj.weight, 0, Fp), ops._pad(m.up_proj.weight, 0, Fp)]).contiguous()
        self.down = ops._pad(m.down_proj.weight, 1, Fp).contiguous()

    @property
    def weights(self) -> list[Tensor]:
        return [self.gu, self.down]

    def run(self, h: Tensor, b, st) -> ops.Delta:
        return ops.Delta(ops.linear(ops.gated_linear(h, self.gu, 0, past=self.past), self.down, self.past))


class _Experts(_Sublayer):
    def __init__(self, m: L.MixtureOfExperts):
        self.w, self.kind, self.limit = m.packed(), m.kind, m.limit
        self.router, self.rule = m.routing()
        self.shared = None if m.shared is None else m.shared.packed()
        self.experts = (self.w["gu"], self.w["down"])

    @property
    def weights(self) -> list[Tensor]:
        return [self.router] + ([] if self.shared is None else list(self.shared.values()))

    def run(self, h: Tensor, b, st) -> ops.Delta:
        ids, wts = ops.route(h, self.router, **self.rule)
        if self.shared is None:
            return ops.Delta(ops.experts(h, ids, self.w, self.kind, self.limit, self.experts_past), pair_w=wts)
        y, shared = ops.experts_beside_shared(h, ids, self.w, self.kind, self.limit, self.shared, self.past, self.experts_past)
        return ops.Delta(y, pair_w=wts, shared=shared)


# --------------------------------------------------------------------------- entries
class _ConvEntry:
    """x += norm(last output); h = x + conv(x)."""

    def __init__(self, m: L.CausalConv, index: int):
        self.taps, self.index = m.weight.float().t().contiguous(), index

    def run(self, p: "PackedProgram", b, st, x, embed, delta, norm):
        y, pw = (delta.y, delta.pair_w) if delta is not None else (None, None)
        return ops.residual_conv(b, p.dtype, x=x, embed=embed, y=y, pair_w=pw, norm=norm,
                                 conv=(self.taps, st.conv[self.index]))


class _NormEntry:
    """x += last output; h = rms_norm(x)."""

    def __init__(self, m: L.GroupedRMSNorm):
        self.norm = (m.weight.float().contiguous(), m.eps)

    def run(self, p: "PackedProgram", b, st, x, embed, delta, norm):
        return ops.residual_norm(b, p.dtype, x=x, embed=None if embed is None else (*embed, p.positions), delta=delta,
                                 norm=self.norm)


# --------------------------------------------------------------------------- patterns
@dataclass
class _Plan:
    tokens: nn.Embedding
    positions: nn.Embedding | None
    parts: list            # (entry module, sublayer module, post-norm module or None)
    norm: L.GroupedRMSNorm
    head: Tensor           # output projection [vocab, C]
    head_scale: float


_SINGLE_MIXERS = (L.Retention, L.GatedLinearAttention, L.WindowAttention)


def _is_mixer(m) -> bool:
    if isinstance(m, L.ParallelMixers):
        return isinstance(m.left, _SINGLE_MIXERS) and isinstance(m.right, _SINGLE_MIXERS)
    return isinstance(m, _SINGLE_MIXERS)


def _is_ff(m) -> bool:
    return isinstance(m, L.MixtureOfExperts) or (isinstance(m, L.GatedMLP) and m.act_kind == "silu"
                                                 and m.gate_proj.bias is None)


def _pair(block) -> tuple | None:
    """(entry, sublayer) of a block part."""
    m = list(block) if isinstance(block, nn.Sequential) else []
    return tuple(m) if len(m) == 2 else None


def _post_norm_parts(blk: L.TransformerBlock):
    out = [(_pair(blk.attn_block), blk.post_attn_norm)]
    if blk.mlp_block is not None:
        out.append((_pair(blk.mlp_block), blk.post_mlp_norm))
    for i, (pair, norm) in enumerate(out):
        if pair is None or not isinstance(pair[0], L.CausalConv) or not isinstance(norm, L.GroupedRMSNorm):
            return None
        if not (isinstance(pair[1], L.LatentAttention) if i == 0 else _is_ff(pair[1]) and
                getattr(pair[1], "shared", None) is None):
            return None
    return None if blk.post_norm_on_residual else [(*pair, norm) for pair, norm in out]


def _pre_norm_parts(blk: L.TransformerBlock):
    out = [_pair(blk.attn_block)] + ([_pair(blk.mlp_block)] if blk.mlp_block is not None else [])
    if blk.post_attn_norm is not None or blk.post_mlp_norm is not None:
        return None
    for i, pair in enumerate(out):
        if (pair is None or not isinstance(pair[0], L.GroupedRMSNorm) or pair[0].groups != 1
                or not (_is_mixer if i == 0 else _is_ff)(pair[1])):
            return None
    return [(*pair, None) for pair in out]


class PackedProgram:
    @staticmethod
    def match(model) -> _Plan | None:
        """The model's plan when it has one of the patterns, else None."""
        mods = list(model.layers)
        if mods and isinstance(mods[-1], L.SoftmaxOnLast):
            mods = mods[:-1]
        if len(mods) < 4 or not isinstance(mods[-2], L.GroupedRMSNorm):
            return None
        emb, positions = mods[0], None
        if isinstance(emb, L.Summation) and len(emb) == 2 and type(emb[1]) is L.PositionEmbedding:
            emb, positions = emb[0], emb[1]
        if type(emb) is not nn.Embedding:
            return None
        head = mods[-1]
        if isinstance(head, L.TiedLinear) and head.weight_source is emb:
            weight, scale = emb.weight, head.scale
        elif isinstance(head, L.OutputLinear):
            weight, scale = head.weight, 1.0
        else:
            return None
        if not all(isinstance(blk, L.TransformerBlock) for blk in mods[1:-2]):
            return None
        for style in (_post_norm_parts, _pre_norm_parts):
            parts = [style(blk) for blk in mods[1:-2]]
            if all(p is not None for p in parts) and not (positions is not None and style is _post_norm_parts):
                return _Plan(emb, positions, [p for blk in parts for p in blk], mods[-2], weight, scale)
        return None

    @staticmethod
    @torch.no_grad()
    def build(model) -> "PackedProgram | None":
        plan = PackedProgram.match(model)
        if plan is None:
            return None
        dtypes = {p.dtype for p in model.parameters()}
        if dtypes not in ({torch.bfloat16}, {torch.float32}):
            raise ValueError(f"the packed step runs bfloat16 or float32 parameters, not {sorted(map(str, dtypes))}")
        return PackedProgram(plan)

    def __init__(self, plan: _Plan):
        self.table, self.head = plan.tokens.weight, plan.head
        self.positions = None if plan.positions is None else plan.positions.weight
        self.limit = None if self.positions is None else self.positions.shape[0]  # tokens per sequence
        self.dtype, self.device = self.table.dtype, self.table.device
        self.latent_widths, self.convs, self.windows, self.linear, self.rotations = [], [], [], [], []
        self._caches: dict = {}
        self.steps = []  # (entry, sublayer, post-norm or None)
        for entry, sub, norm in plan.parts:
            if isinstance(entry, L.CausalConv):
                e = _ConvEntry(entry, len(self.convs))
                self.convs.append((entry.weight.shape[0], entry.taps))
            else:
                e = _NormEntry(entry)
            post = None if norm is None else (norm.weight.float().contiguous(), norm.groups, norm.eps)
            self.steps.append((e, self._sublayer(sub), post))
        # the output scale rides on the final norm's weight
        self.norm_f = (plan.norm.weight.float() * plan.head_scale, plan.norm.groups, plan.norm.eps)
        subs = [sub for _, sub, _ in self.steps]
        self.past, experts_past = gemm_ops.past_caches([w for s in subs for w in s.weights] + [self.head],
                                                       [w for s in subs for w in s.experts])
        for s in subs + [m for s in subs if isinstance(s, _ParallelMixer) for m in (s.left, s.right)]:
            s.past = self.past
            s.experts_past = experts_past

    def _sublayer(self, m: nn.Module):
        if isinstance(m, L.MixtureOfExperts):
            return _Experts(m)
        if isinstance(m, L.GatedMLP):
            return _DenseFF(m)
        if isinstance(m, L.ParallelMixers):
            return _ParallelMixer(m, self._sublayer(m.left), self._sublayer(m.right))
        if isinstance(m, L.WindowAttention):
            s = m.sizes
            self.windows.append((s.kv_heads, s.row, s.pool))
            self.rotations += s.rotations
            return _WindowMixer(m, len(self.windows) - 1)
        if isinstance(m, (L.Retention, L.GatedLinearAttention)):
            self.linear.append(m.sizes.state)
            return _LinearMixer(m, len(self.linear) - 1)
        if m.kv_from is None:
            self._caches[id(m)] = len(self.latent_widths)
            self.latent_widths.append(m.sizes.cache_width)
        mixer = _LatentMixer(m, self._caches[id(m if m.kv_from is None else m._source[0])])
        self.rotations.append(mixer.rotation)
        return mixer

    def new_state(self, slots: int, capacity: int) -> SequenceState:
        return SequenceState(self.latent_widths, self.convs, self.rotations, self.dtype, self.device, slots, capacity,
                             windows=self.windows, linear=self.linear, limit=self.limit)

    @torch.inference_mode()
    def forward(self, tokens: Tensor, b: ops.PackedBatch, st: SequenceState, want: Tensor | None = None,
                trace: list | None = None) -> Tensor | None:
        """Run the step's tokens (int64 [N], the descriptor's rows) and return the logits of the rows
        ``want`` (int32; None: all). ``trace`` receives the residual stream after every sublayer."""
        with torch.autocast(self.device.type, enabled=False):  # the program picks its own precisions
            return self._forward(tokens, b, st, want, trace)

    def _forward(self, tokens, b, st, want, trace):
        x = delta = norm = None
        embed = (tokens.reshape(-1), self.table)
        for entry, sub, post in self.steps:
            x, h = entry.run(self, b, st, x, embed, delta, norm)
            if trace is not None and embed is None:
                trace.append(x.clone())
            embed = None
            delta, norm = sub.run(h, b, st), post
        if norm is not None:
            x, _ = ops.residual_conv(b, self.dtype, x=x, y=delta.y, pair_w=delta.pair_w, norm=norm)
        else:
            x, _ = ops.residual_norm(b, self.dtype, x=x, delta=delta)
        if trace is not None:
            trace.append(x.clone())
        if want is not None and want.numel() == 0:
            return None
        w, groups, eps = self.norm_f
        return ops.logits(ops.row_norm(x, w, groups, eps, self.dtype, rows=want), self.head, self.past)


class PackedSession:
    """Steps of named sequences through a model's packed program: ``step([(name, tokens, want), ...])`` runs
    the new tokens of each from the state earlier steps left and returns the logits at the wanted places
    (fp32 [wanted, vocab]); a new name opens a sequence, ``end`` gives its slot back."""

    def __init__(self, model, slots: int = 1, capacity: int | None = None):
        self.program = model.packed_program()
        if self.program is None:
            raise ValueError("the model's layer list has no packed step")
        self.state = self.program.new_state(slots, capacity)
        self._slot: dict = {}

    def step(self, entries) -> Tensor | None:
        vocab = self.program.table.shape[0]
        toks, want, plan = [], [], []
        for name, tokens, places in entries:
            if not tokens or min(tokens) < 0 or max(tokens) >= vocab:
                raise ValueError(f"sequence {name!r}: token ids must be in [0, {vocab}), at least one")
            if any(not 0 <= p < len(tokens) for p in places):
                raise ValueError(f"sequence {name!r}: wanted places outside its {len(tokens)} tokens")
        for name, tokens, places in entries:
            if name not in self._slot:
                self._slot[name] = self.state.acquire()
            want += [len(toks) + p for p in places]
            toks += tokens
            plan.append((self._slot[name], len(tokens)))
        b = self.state.begin(plan)
        dev = self.program.device
        out = self.program.forward(ops.upload(toks, torch.long, dev), b, self.state, ops.upload(want, torch.int32, dev))
        return None if out is None else out.float()

    def slots(self, names) -> list[int]:
        return [self._slot[n] for n in names]

    def reset(self):
        """End every sequence."""
        for name in list(self._slot):
            self.end(name)

    def length(self, name) -> int:
        return self.state.length(self._slot[name])

    def end(self, name):
        self.state.release(self._slot.pop(name))
