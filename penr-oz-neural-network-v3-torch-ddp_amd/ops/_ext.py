"""Loader for the in-tree HIP extensions ``penroz_kernels`` and ``penroz_serve`` (built for gfx950 by
``setup.py``).

GPU tensors MUST go through the extension: if a CUDA (= HIP) tensor reaches an op and the
extension is not importable, :func:`kernels` raises instead of silently falling back to eager
PyTorch.  CPU tensors use the pure-torch reference implementations that the GPU parity tests
compare against.
"""
from __future__ import annotations

import importlib
import os
import sys

import torch

_REPO_ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
# PENROZ_EXT_DIR: load the extension from another in-tree build (same-box A/B benchmarking)
_BUILD_DIR = os.environ.get("PENROZ_EXT_DIR") or os.path.join(_REPO_ROOT, "build_ext")

# penroz_serve: decode-shaped GEMMs and the packed decoder step; penroz_kernels: everything else
MODULES = ("penroz_serve", "penroz_kernels")
_mods: dict = {}
_errs: dict = {}


def _load(name: str = "penroz_kernels"):
    if name in _mods or name in _errs:
        return _mods.get(name)
    if _BUILD_DIR not in sys.path:
        sys.path.insert(0, _BUILD_DIR)
    try:
        # torch must be imported first so libc10_hip / libamdhip64 are already mapped
        _mods[name] = importlib.import_module(name)
    except Exception as e:  # pragma: no cover - exercised on boxes without a build
        _errs[name] = e
    return _mods.get(name)


class _Kernels:
    """Attribute access into the kernel modules, each loaded when first asked for."""

    def __getattr__(self, fn: str):
        for name in MODULES:
            mod = _load(name)
            if mod is not None and hasattr(mod, fn):
                f = getattr(mod, fn)
                setattr(self, fn, f)  # the next access skips the lookup
                return f
        if _errs:
            raise RuntimeError(
                f"HIP kernel {fn!r}: extension not built/importable ({_errs!r}); run "
                "`python setup.py build_ext` (gfx950) before using GPU tensors")
        raise AttributeError(fn)


_KERNELS = _Kernels()


def available(module: str | None = None) -> bool:
    """The given kernel module (all of them without one) can be loaded."""
    return all(_load(n) is not None for n in ([module] if module else MODULES))


def kernels():
    """The compiled kernels (a function whose module is missing raises loudly)."""
    return _KERNELS


def on_gpu(*tensors) -> bool:
    return any(isinstance(t, torch.Tensor) and t.is_cuda for t in tensors)


# Set by the ``reference`` engine only (stock-PyTorch baseline for speedup claims).
FORCE_TORCH = False


def use_kernels(*tensors) -> bool:
    """True when the HIP path must be taken (any operand on the GPU)."""
    if FORCE_TORCH:
        return False
    if on_gpu(*tensors):
        return True  # kernels() raises if the extension is missing
    return False


def plain_mode() -> bool:
    """Nothing but values is asked of ops: inference mode (no backward, no tangents), no trace, transform, mode or autocast
    that has to see the operators themselves."""
    return (not torch.compiler.is_compiling()  # first: a compiler's trace cannot ask for the others
            and torch.is_inference_mode_enabled() and not torch.is_autocast_enabled("cuda")
            and torch._C._get_tracing_state() is None and torch._C._functorch.peek_interpreter_stack() is None
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0 and not FORCE_TORCH)


def plain_call(x) -> bool:
    """:func:`plain_mode`, and ``x`` is a GPU tensor of no subclass that holds something, on the current device (the kernels
    start there, whatever device their operands are on)."""
    return (plain_mode() and type(x) is torch.Tensor and x.is_cuda and x.numel() > 0
            and x.get_device() == torch._C._cuda_getDevice())
