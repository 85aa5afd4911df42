"""GEMM entry points.

* ``wgrad(dy, x, grad)`` — ``grad += dyᵀ·x`` for weight gradients (bf16 operands, fp32
  accumulate into the flat gradient buffer). GPU: the hand-written MFMA split-K kernel in
  ``csrc/kernels/gemm_wgrad.hip`` (256×256 tile, LDS-DMA staging, transposed LDS reads,
  wave-quantisation-aware split-K, deterministic slab reduction fused with the accumulate).
  Measured at GPT-2 124M shapes (K = 65 536 tokens, profiles/kernel_bench_r1_wgrad_ring16.log): 800–1100 TF
  vs hipBLASLt's 270–950 TF on the same calls; a layer's gradients together: ``wgrad_group``.
* ``train_linear`` — the forward / dgrad GEMMs of training steps: hipBLASLt through ``torch.addmm``/``torch.mm``
  (≈0.9–1.4 PF at the headline shapes), in short steps ``csrc/kernels/rows_gemm.hip`` where its bits are the same.
* ``rows_linear`` / ``linear`` / ``linear_fp32`` — linear layers of short steps (decode, prompts): ``rows_gemm.hip`` by the
  rule of its sizes, else the library.
"""
from __future__ import annotations

import functools
import os

import torch
from torch import Tensor

from penroz.ops import _ext
from penroz.ops._ext import use_kernels, kernels

# "auto"/"1": the native kernel (faster than hipBLASLt on every measured GPT-2 shape);
# "0": hipBLASLt (A/B switch for benchmarking).
NATIVE_WGRAD = os.environ.get("PENROZ_NATIVE_WGRAD", "auto")
# pipeline variant of the 256-tile kernel (csrc/kernels/gemm_wgrad.hip): 8 (fragment prefetch), 6,
# 4 — A/B knob. Unset: 8 for long token dimensions (GPT-2 B=64: K = 65 536), 6 for K <= 16 384,
# where the prefetch's extra prologue does not pay (Gemma-3 1B B=8, K = 8192: 67.05 / 67.11 ->
# 66.62 / 66.66 ms; GPT-2: 8 beats 6, 61.28 / 61.35 vs 61.49 / 61.43 ms; profiles/knobs_ab_r4.log)
_WGRAD_VARIANT_ENV = os.environ.get("PENROZ_WGRAD_VARIANT")
WGRAD_VARIANT = int(_WGRAD_VARIANT_ENV) if _WGRAD_VARIANT_ENV else 0  # 0: by K
WGRAD_SHORT_K = 16384


def _wgrad_variant(k: int) -> int:
    if WGRAD_VARIANT:
        return WGRAD_VARIANT
    return 6 if k <= WGRAD_SHORT_K else 8


def _native_ok(m: int, n: int, lda: int | None = None) -> bool:
    """m need not be a multiple of 8 when dy's rows are padded to it (lda >= round_up(m, 8))."""
    return NATIVE_WGRAD != "0" and n % 8 == 0 and (m % 8 == 0 or (lda is not None and lda >= (m + 7) // 8 * 8))


def reference_wgrad(dy: Tensor, x: Tensor, grad: Tensor, accumulate: bool = True) -> None:
    if accumulate:
        grad.add_(dy.float().t() @ x.float())
    else:
        grad.copy_(dy.float().t() @ x.float())


def _native_wgrad(dy: Tensor, x: Tensor) -> bool:
    return (use_kernels(dy) and _native_ok(dy.shape[1], x.shape[1], dy.stride(0)) and dy.dtype == torch.bfloat16
            and x.dtype == torch.bfloat16 and dy.stride(0) % 8 == 0 and x.stride(0) % 8 == 0)


def wgrad(dy: Tensor, x: Tensor, grad: Tensor, accumulate: bool = True) -> None:
    """grad += dyᵀ·x, or grad = dyᵀ·x with accumulate=False (the first weight-gradient write of a
    step whose zero_grad skipped this range)."""
    if _native_wgrad(dy, x):
        if WGRAD_VARIANT:
            kernels().wgrad_gemm(dy, x, grad, 256, WGRAD_VARIANT, accumulate)
        else:
            kernels().wgrad_group([dy], [x], [grad], [accumulate], _wgrad_variant(dy.shape[0]))
    elif dy.is_cuda:
        prod = torch.mm(dy.t(), x, out_dtype=torch.float32)
        grad.add_(prod) if accumulate else grad.copy_(prod)
    else:
        reference_wgrad(dy, x, grad, accumulate)


def wgrad_group(dys, xs, grads, accumulate, shared: bool = False) -> None:
    """:func:`wgrad` for each of several products over the same tokens, in one launch where that is faster (the rule,
    ``plan_wgrad_group`` in ``csrc/kernels/host_plan.h``, knows their sizes; ``shared``: another stream works beside)."""
    if not WGRAD_VARIANT and all(_native_wgrad(dy, x) for dy, x in zip(dys, xs)):
        kernels().wgrad_group(list(dys), list(xs), list(grads), list(accumulate), _wgrad_variant(dys[0].shape[0]), shared)
        return
    for args in zip(dys, xs, grads, accumulate):
        wgrad(*args)


@functools.lru_cache(maxsize=256)
def _wgrad_tile(shapes: tuple, tokens: int, cus: int, shared: bool) -> int:
    return kernels().wgrad_group_tile([m for m, _ in shapes], [n for _, n in shapes], tokens, cus, shared)


def wgrad_together(shapes: tuple, tokens: int, device: torch.device, shared: bool = False) -> bool:
    """Whether :func:`wgrad_group` takes products [m, n] of these ``shapes`` over ``tokens`` in one launch."""
    if WGRAD_VARIANT or NATIVE_WGRAD == "0":
        return False
    return _wgrad_tile(shapes, tokens, torch.cuda.get_device_properties(device).multi_processor_count, shared) != 0


# ---- weights that a decode step reads past the caches ----------------------------------------
# Of the 256 MB in front of the memory keys, values, states and activations have a part. A model of up to CACHE_BYTES is left to them;
# of a larger one they are to hold the smaller weights, up to HELD_BYTES. ms with nothing past them / this rule / all of the larger ones:
# 32 tokens of GPT-2 124M (247 MB), 1 and 64 rows 8.44 / 8.31 / 8.38 and 15.4 / 14.8 / 14.7, with 5 layers (148 MB), 1 row 4.12 / 4.12 /
# 4.14; Gemma-3 1B, 3 rows 33.3 / 31.7 / 32.0; two layers of its width and a vocabulary of 32768 (150 MB), 1 row 3.08 / 3.08 / 3.14. Room for
# 192 MB instead of 128 beside experts that pass: Zozenex small, 48 tokens, 16 rows 26.2 -> 26.7, 64 rows 32.2 -> 32.9.
CACHE_BYTES, HELD_BYTES = 192 << 20, 128 << 20
KEEP = 1 << 62  # a size that no weight has


def past_caches(weights, experts=()) -> tuple[int, bool]:
    """What of the weights that a decode step multiplies its rows with should pass the caches (loads that keep nothing): the size
    in bytes from which on ``weights`` do, and whether ``experts`` (of which each step reads others) do."""
    sizes = sorted(w.nbytes for w in weights)
    if sum(sizes) + sum(w.nbytes for w in experts) <= CACHE_BYTES:
        return KEEP, False
    held = 0
    for size in dict.fromkeys(sizes):
        held += size * sizes.count(size)
        if held > HELD_BYTES:
            return size, True
    return KEEP, True


# ---- linear layers of short steps (csrc/kernels/rows_gemm.hip) ------------------------------
ROWS_GEMM = os.environ.get("PENROZ_ROWS_GEMM", "1") != "0"  # "0": the library (A/B)


def rows_linear(x: Tensor, w: Tensor, bias: Tensor | None = None, out: Tensor | None = None,
                fp32: bool = False, in_order: bool = False, gelu: bool = False, past: bool = False) -> Tensor | None:
    """x [M, K] · wᵀ (+ bias), bf16 (``fp32``: the sums themselves; ``in_order``: each sum in one chain over k; ``gelu``: the
    erf gelu of the bf16 result; ``past``: :func:`past_caches`), by the kernel of short steps; None for what its rule
    (``rows_gemm_plan`` in ``csrc/kernels/host_plan.h``) leaves to the library."""
    if not (ROWS_GEMM and x.is_cuda and x.dtype == torch.bfloat16 and use_kernels(x)):
        return None
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, w, bias)):
        return None
    return kernels().rows_gemm(x, w, bias, out, fp32, in_order, gelu, past)


def linear(x: Tensor, w: Tensor, bias: Tensor | None = None, out: Tensor | None = None) -> Tensor:
    """x [M, K] · wᵀ (+ bias): :func:`rows_linear` or the library."""
    y = rows_linear(x, w, bias, out)
    if y is not None:
        return y
    return torch.mm(x, w.t(), out=out) if bias is None else torch.addmm(bias, x, w.t(), out=out)


# Training steps take the kernel where its results are the library's bit for bit (tests/test_rows_gemm_gpu.py): up to this many
# columns the library does not split the sums (of 2304 and 3072 it splits those of some row counts and not of others), from this
# many rows on (32 to 3000 measured, of 64 to 1024 columns; of 1 to 24 rows its other kernels round one value in 1e4 otherwise).
# A rounding that falls otherwise is as good, but AdamW's first steps carry it through every weight.
TRAIN_ROWS_MAX_K, TRAIN_ROWS_MIN = 1024, 32


def train_linear(x: Tensor, w: Tensor, bias: Tensor | None = None, out: Tensor | None = None) -> Tensor:
    """x [M, K] · wᵀ (+ bias) of a training step's forward or data gradient."""
    y = None
    if x.shape[1] <= TRAIN_ROWS_MAX_K and x.shape[0] >= TRAIN_ROWS_MIN:
        y = rows_linear(x, w, bias, out, in_order=True)
    if y is not None:
        return y
    return torch.mm(x, w.t(), out=out) if bias is None else torch.addmm(bias, x, w.t(), out=out)


def _rows_sized(M: int, N: int, K: int) -> bool:
    """``rows_gemm_plan`` (``csrc/kernels/host_plan.h``) may have a tile for these sizes: what it certainly leaves to the library
    is not asked for, at 5 µs of the host a layer."""
    n = M * N
    return n <= 1 << 19 or (n <= 1 << 22 and K <= 1024) or (K <= 2048 and (n <= 1 << 20 or (M <= 64 and n <= 1 << 22)))


def _bare(mod: torch.nn.Module) -> bool:
    """A call of ``mod`` is its class's forward and nothing else: no hooks, no forward of its own (but for ``decode_gemms``'s)."""
    f = mod.__dict__.get("forward")
    return ((f is None or getattr(f, "of_decode_gemms", False)) and mod._compiled_call_impl is None
            and not (mod._forward_hooks or mod._forward_pre_hooks or mod._backward_hooks or mod._backward_pre_hooks))


def apply(mod: torch.nn.Module, x: Tensor) -> Tensor:
    """``mod(x)``, where the ``nn.Linear`` layers of prompts (inference mode, bf16 on the GPU; ``mod`` itself or in the
    ``nn.Sequential`` that it is) take :func:`rows_linear` where its rule does. The model and its containers call their
    children so, and the layers stay ``nn.Linear`` for whatever traces, compiles or replaces them. A short prompt's pass is
    bound by the host, and the library's call costs it 19 µs against 4: GPT-2's pass over one prompt of 64 tokens
    2.60 -> 1.71 ms, of 512 2.64 -> 1.79, Gemma 3 1B's over 3 of 200 7.6 -> 7.0."""
    kind = type(mod)
    if ((kind is torch.nn.Sequential or kind is torch.nn.Linear) and _ext.plain_call(x)
            and not torch.nn.modules.module._has_any_global_hook()):
        return _apply(mod, x, x.get_device())
    return mod(x)


def _apply(mod: torch.nn.Module, x: Tensor, device: int) -> Tensor:
    """:func:`apply` where its call is plain: a child leaves the modes as it found them, so they are asked for once."""
    kind = type(mod)
    if kind is torch.nn.Linear:
        if (type(x) is Tensor and x.dtype == torch.bfloat16 and x.get_device() == device and x.dim() >= 2 and x.numel() > 0
                and _bare(mod)):
            w, b, K = mod.weight, mod.bias, x.shape[-1]
            if (type(w) is torch.nn.Parameter and (b is None or type(b) is torch.nn.Parameter)
                    and _rows_sized(x.numel() // K, w.shape[0], K)):
                y = rows_linear(x.reshape(-1, K), w, b)
                if y is not None:
                    return y.view(*x.shape[:-1], w.shape[0])
    elif kind is torch.nn.Sequential and _bare(mod):
        for m in mod:
            x = _apply(m, x, device)
        return x
    return mod(x)


def linear_fp32(x: Tensor, w: Tensor, past: bool = False) -> Tensor:
    """x [M, K] · wᵀ of bf16 operands in fp32."""
    y = rows_linear(x, w, fp32=True, past=past)
    return torch.mm(x, w.t(), out_dtype=torch.float32) if y is None else y


# ---- library GEMM solution choice (hipBLASLt / rocBLAS through torch) -----------------------
# The forward / dgrad GEMMs of steps beyond rows_gemm's sizes are library calls; which hipBLASLt (or rocBLAS) solution runs
# each shape is measured, not left to the heuristic: bench/tune_gemms.sh runs PyTorch TunableOp's
# solution search over every GEMM the executor issues at the GPT-2 headline shapes (and the HF
# import layout) and ops/tuned/tunableop_gfx950.csv ships the winners (validated against the
# PyTorch / HIP / hipBLASLt / rocBLAS versions and the gfx950 arch at load; a mismatch is refused
# by torch and the heuristic picks stay). Loaded read-only (no tuning at run time; shapes not in
# the file keep the default solution). PENROZ_TUNED_GEMMS=0 disables.
TUNED_GEMM_FILE = os.environ.get("PENROZ_TUNED_GEMM_FILE") or os.path.join(
    os.path.dirname(os.path.abspath(__file__)), "tuned", "tunableop_gfx950.csv")
_tuned_state: dict = {}


def load_tuned_gemms() -> bool:
    """Enable TunableOp in read-only mode with the shipped results (once per process)."""
    if "loaded" in _tuned_state:
        return _tuned_state["loaded"]
    ok = False
    if (os.environ.get("PENROZ_TUNED_GEMMS", "1") != "0" and os.environ.get("PYTORCH_TUNABLEOP_TUNING") != "1"
            and torch.cuda.is_available() and os.path.exists(TUNED_GEMM_FILE)):
        import torch.cuda.tunable as tunable
        tunable.enable(True)
        tunable.tuning_enable(False)
        tunable.record_untuned_enable(False)
        ok = bool(tunable.read_file(TUNED_GEMM_FILE))
        if not ok:
            tunable.enable(False)
    _tuned_state["loaded"] = ok
    return ok


def set_tuned_gemms(on: bool) -> bool:
    """Switch the loaded table's solutions on or off at run time (off: hipBLASLt's own heuristic
    for every shape). Returns whether the table is now in use."""
    if not _tuned_state.get("loaded"):
        return False
    import torch.cuda.tunable as tunable
    tunable.enable(bool(on))
    _tuned_state["active"] = bool(on)
    return bool(on)


def guard_tuned_gemms(run_steps, steps: int = 3, rounds: int = 2, margin: float = 1.0, agree=None) -> dict:
    """The shipped table must never cost time (it once drifted to 1 ms/step SLOWER than
    hipBLASLt's heuristic and nothing noticed). Times ``run_steps(steps)`` (returns seconds) with the
    table off and on, ``rounds`` interleaved times each, keeps the table only if its best time is
    <= ``margin`` × the heuristic's best, and leaves that choice switched on. ``agree`` (optional)
    maps a local time to the group's (MAX over ranks) so every rank decides the same.
    {} when no table is loaded."""
    if not _tuned_state.get("loaded"):
        return {}
    best = {False: float("inf"), True: float("inf")}
    for _ in range(rounds):
        for on in (False, True):
            set_tuned_gemms(on)
            dt = run_steps(steps)
            if agree is not None:
                dt = agree(dt)
            best[on] = min(best[on], dt / steps)
    keep = best[True] <= margin * best[False]
    set_tuned_gemms(keep)
    return {"table": os.path.basename(TUNED_GEMM_FILE), "with_table_ms": round(best[True] * 1e3, 3),
            "heuristic_ms": round(best[False] * 1e3, 3), "table_kept": keep}


# ---- linear + GELU / GELU backward (library GEMM + the HIP GELU kernels) -------------------
# Two native fused designs were built and measured against this pair: an 8-phase
# persistent MFMA GEMM with a bias/GELU epilogue and a 4-wave deferred-epilogue GEMM whose
# stores (and GELU' / bias-column work) stream inside the next tile. Both lost on every GPT-2
# shape and on the headline step (profiles/gemm_epi_r4.log, profiles/native_gemm_r4.md), so the
# forward / dgrad GEMMs are plain ones (train_linear) and the GELU work stays in elementwise.hip.
def linear_gelu(x: Tensor, w: Tensor, bias: Tensor, pre: Tensor, act: Tensor, approximate: str = "none"):
    """pre = x·wᵀ + bias (:func:`train_linear`), act = GELU(pre) (bf16; ``approximate`` "none" = erf,
    "tanh" = gelu_new; the HIP GELU kernel)."""
    train_linear(x, w, bias, pre)
    if use_kernels(pre):
        from penroz.ops import activations as act_ops
        act_ops.gelu_fwd(pre, approximate, out=act)
    else:
        act.copy_(torch.nn.functional.gelu(pre.float(), approximate=approximate))
    return pre, act


def dgrad_gelu(dy: Tensor, wt: Tensor, pre: Tensor, out: Tensor, dbias: Tensor | None, approximate: str = "none"):
    """Data gradient into a GELU's input: out = bf16(dy·wtᵀ) (:func:`train_linear`; ``wt`` = the
    transposed weight copy, [in, out] row-major), then out *= GELU'(pre) and dbias (fp32) += the
    column sums of out in one HIP kernel. The GPT executor's fc2 data gradient + GELU backward +
    fc bias gradient."""
    train_linear(dy, wt, None, out)
    from penroz.ops import activations as act_ops
    act_ops.gelu_bwd(out, pre, approximate, dbias, out=out)
    return out


# ---- decode-shaped GEMMs (csrc/kernels/skinny_gemm.hip) --------------------------------------
# out[M<=64, N] = x·Wᵀ (+ bias), bf16: one 16-column MFMA slice per workgroup over all rows,
# K split across the 4 waves (and across workgroups, with an in-launch slab reduction, when the
# output is narrow). Used for the graph-captured decode step (models/graph_decode.py), where a
# library GEMM tile at M = 64 leaves most CUs idle (~10 µs for a 3.5 MB weight read).
SKINNY_GEMM = os.environ.get("PENROZ_SKINNY_GEMM", "1") != "0"
_skinny_ws: dict = {}


def skinny_workspace(device: torch.device) -> tuple[Tensor, Tensor]:
    """Per-device split-K workspace and arrival counters (zeroed once, outside any graph
    capture; every launch leaves the counters zero again)."""
    key = (device.type, device.index if device.index is not None else torch.cuda.current_device())
    buf = _skinny_ws.get(key)
    if buf is None:
        dev = torch.device(*key)
        buf = (torch.empty(1 << 19, device=dev, dtype=torch.float32), torch.zeros(1 << 12, device=dev, dtype=torch.int32))
        _skinny_ws[key] = buf
    return buf


def skinny_ok(x: Tensor, w: Tensor) -> bool:
    if not (SKINNY_GEMM and x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16):
        return False
    K = x.shape[-1]
    rows = x.numel() // K if K else 0
    return (0 < rows <= 64 and K % 32 == 0 and w.is_contiguous() and w.shape[1] == K and w.data_ptr() % 16 == 0
            and use_kernels(x))


def skinny_linear(x: Tensor, w: Tensor, bias: Tensor | None) -> Tensor:
    """nn.Linear forward for ≤ 64 rows of bf16 activations (any leading shape)."""
    K, N = x.shape[-1], w.shape[0]
    x2 = x.reshape(-1, K)
    if x2.stride(1) != 1 or x2.stride(0) % 8 or x2.data_ptr() % 16:
        x2 = x2.contiguous()
    out = torch.empty(x2.shape[0], N, device=x.device, dtype=x.dtype)
    ws, cnt = skinny_workspace(x.device)
    kernels().skinny_gemm(x2, w, bias if bias is None or bias.dtype == torch.bfloat16 else bias.to(torch.bfloat16),
                          out, ws, cnt)
    return out.view(*x.shape[:-1], N)


def skinny_gated(x: Tensor, gu: Tensor, kind: int) -> Tensor:
    """Gated-MLP decode projection in one launch: act(x·gu[:I]ᵀ) ⊙ (x·gu[I:]ᵀ) for ≤ 64 rows,
    ``gu`` the packed [gate; up] weight [2I, K]; kind 0 gelu, 1 gelu_tanh, 2 silu. Bit-identical to
    ``skinny_linear`` + the packed gated-activation kernel (csrc/kernels/skinny_gemm.hip)."""
    out = torch.empty(x.shape[0], gu.shape[0] // 2, device=x.device, dtype=x.dtype)
    kernels().skinny_gated(x, gu, out, kind)
    return out


def skinny_qkv_rope_ok(x: Tensor, w: Tensor, D: int) -> bool:
    """The fused QKV + RoPE decode kernel applies: skinny shapes, whole heads of D % 32 == 0, and
    its split-K slabs fit the shared workspace."""
    if not (skinny_ok(x, w) and D % 32 == 0 and w.shape[0] % D == 0):
        return False
    return qkv_rope_plan_fits(x.numel() // x.shape[-1], w.shape[0], x.shape[-1])


def qkv_rope_plan_fits(rows: int, n: int, k: int) -> bool:
    """The kernel's own split-K plan (csrc/kernels/skinny_gemm.hip skinny_qkv_rope_plan: the rule
    its launcher applies) fits the shared workspace and counters of ``skinny_workspace``."""
    _, ws_floats, counters = kernels().skinny_qkv_rope_plan(rows, n, k)
    return ws_floats <= (1 << 19) and counters <= (1 << 12)


def skinny_qkv_rope(x: Tensor, w: Tensor, cos: Tensor, sin: Tensor, D: int, nrot: int) -> Tensor:
    """Decode QKV projection with RoPE (one position's cos / sin [D/2]) applied to the first
    ``nrot`` heads in the GEMM epilogue (csrc/kernels/skinny_gemm.hip); ≤ 64 rows."""
    out = torch.empty(x.shape[0], w.shape[0], device=x.device, dtype=x.dtype)
    ws, cnt = skinny_workspace(x.device)
    kernels().skinny_qkv_rope(x, w, cos, sin, D, nrot, out, ws, cnt)
    return out


class decode_gemms:
    """Context: the ``nn.Linear`` modules of ``model`` run decode-shaped inputs that :func:`apply` leaves to them through the
    skinny kernel (others keep ``F.linear``). Entered by the graph decoder around the captured step of a
    model without a decode program. Only that model's own Linear instances are re-routed (an
    instance-level ``forward``, removed on exit): other models, and other threads serving them,
    are untouched; the serving lock keeps concurrent requests off the same model."""

    def __init__(self, model: torch.nn.Module, max_rows: int = 64):
        self.model = model
        self.max_rows = max_rows
        self._patched: list[torch.nn.Linear] = []

    def __enter__(self):
        if not (SKINNY_GEMM and self.max_rows > 0):
            return self
        max_rows = self.max_rows
        for mod in self.model.modules():
            if type(mod) is not torch.nn.Linear or "forward" in mod.__dict__:
                continue

            def forward(x, mod=mod):
                if (x.numel() <= max_rows * x.shape[-1] and skinny_ok(x, mod.weight)
                        and (mod.bias is None or mod.bias.is_contiguous())):
                    return skinny_linear(x, mod.weight, mod.bias)
                return torch.nn.functional.linear(x, mod.weight, mod.bias)

            forward.of_decode_gemms = True
            mod.forward = forward
            self._patched.append(mod)
        return self

    def __exit__(self, *exc):
        for mod in self._patched:
            mod.__dict__.pop("forward", None)
        self._patched.clear()
        return False
