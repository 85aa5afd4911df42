"""Linear layers of prompts: inference mode on bf16 takes the kernel of short steps, every other call the library."""
import pytest
import torch
import torch.nn.functional as F

from penroz.ops import _ext
from penroz.ops import gemm as gemm_ops
from penroz.ops.gemm import apply

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _layer(K, N, bias, dtype=BF):
    torch.manual_seed(K + N)
    lin = torch.nn.Linear(K, N, bias=bias).to("cuda", dtype)
    return lin


@pytest.fixture
def taken(monkeypatch):
    calls, inner = [], gemm_ops.rows_linear

    def spy(*a, **k):
        y = inner(*a, **k)
        calls.append(y is not None)
        return y

    monkeypatch.setattr(gemm_ops, "rows_linear", spy)
    return calls


@pytest.mark.parametrize("shape,N,bias", [((1, 1, 8), 1, True), ((1, 7, 768), 2304, True), ((3, 200, 1152), 1536, False),
                                          ((64, 776), 130, True), ((2, 3, 5, 64), 96, False), ((1, 512, 768), 50304, False)])
def test_prompt_products(shape, N, bias, taken):
    lin = _layer(shape[-1], N, bias)
    wide = torch.randn(*shape[:-1], 2 * shape[-1], device="cuda", dtype=BF)
    x = wide[..., :shape[-1]]  # rows of a wider buffer
    with torch.inference_mode():
        y = apply(lin, x)
        t = apply(lin, x.movedim(0, -2))  # leading axes that reshape has to copy
    want = F.linear(x.double(), lin.weight.double(), lin.bias.double() if bias else None)
    mass = F.linear(x.double().abs(), lin.weight.double().abs(), lin.bias.double().abs() if bias else None)
    # one bf16 rounding of the result and K fp32 additions
    bound = want.abs() * 2.0 ** -8 + mass * shape[-1] * 2.0 ** -24 + 1e-30
    assert y.shape == (*shape[:-1], N) and y.dtype == BF
    assert ((y.double() - want).abs() <= bound).all()
    assert ((t.double() - want.movedim(0, -2)).abs() <= bound.movedim(0, -2)).all()
    assert True not in taken if N == 50304 else len(taken) == 2 and taken[0]


def test_other_calls_keep_the_library(taken):
    lin = _layer(64, 96, True)
    x = torch.randn(4, 64, device="cuda", dtype=BF)
    apply(lin, x.requires_grad_()).sum().backward()
    assert x.grad is not None and lin.weight.grad is not None
    with torch.no_grad():
        apply(lin, x)
    with torch.inference_mode():
        lin(x)  # the layer by itself
        torch.func.vmap(lambda t: apply(lin, t))(x.detach()[None])
        apply(lin, x[0])
        apply(lin, x[:0])
        apply(lin.float(), x.float())
        lin.to(BF)
        with torch.autocast("cuda", dtype=torch.float16):
            assert apply(lin, x).dtype == torch.float16
    assert taken == []


def test_hooks_are_called(taken):
    """A layer, or a sequence of layers, that does more than its class's forward is called as a module."""
    seen = []
    for hook in ("register_forward_hook", "register_forward_pre_hook"):
        model = torch.nn.Sequential(_layer(64, 96, True))
        x = torch.randn(4, 64, device="cuda", dtype=BF)
        with torch.inference_mode():
            for mod in (model[0], model):
                handle = getattr(mod, hook)(lambda *a: seen.append(a[0]))
                apply(model, x)
                handle.remove()
                assert seen.pop() is mod and not seen
            assert taken == []
            apply(model, x)
            assert taken == [True]
        taken.clear()
    model[0].forward = lambda t: seen.append(t)
    with torch.inference_mode():
        assert apply(model, x) is None and len(seen) == 1 and taken == []


@pytest.mark.parametrize("rows", [1, 5, 64])
def test_a_captured_step_takes_the_same_kernel(rows, taken):
    model = torch.nn.Sequential(_layer(128, 384, True), _layer(384, 128, False))
    x = torch.randn(rows, 1, 128, device="cuda", dtype=BF)
    with torch.inference_mode():
        want = apply(model, x)
        with gemm_ops.decode_gemms(model):
            got = apply(model, x)
    assert torch.equal(got, want) and taken == [True] * 4


def test_an_input_on_another_device_is_the_librarys(monkeypatch):
    """The kernels start on the current device; the library goes to its operands' own."""
    x = torch.randn(4, 64, device="cuda", dtype=BF)
    with torch.inference_mode():
        assert _ext.plain_call(x)
        monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: x.get_device() + 1)
        assert not _ext.plain_call(x)
