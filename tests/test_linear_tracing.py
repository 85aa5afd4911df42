"""The vocabulary's linear layers are torch's own to whatever traces, compiles, scripts or replaces them."""
import pytest
import torch
import torch.nn as nn

from penroz.models import layers as L
from penroz.models.mapper import Mapper
from penroz.models.model import NeuralNetworkModel

MODES = {"grad": torch.enable_grad, "no_grad": torch.no_grad, "inference": torch.inference_mode}


def _linear(a, b):
    return {"linear": {"in_features": a, "out_features": b}}


def _sequence():
    return nn.Sequential(*[Mapper._to_layer(d) for d in (_linear(8, 16), {"relu": {}}, _linear(16, 8))])


def _block():
    return L.TransformerBlock(_sequence(), nn.Sequential(nn.Linear(8, 8)))


def _model():
    return NeuralNetworkModel("linears", Mapper([_linear(8, 16), {"relu": {}}, _linear(16, 8)], {"sgd": {"lr": 0.1}}))


def _build(make, dtype=torch.bfloat16):
    torch.manual_seed(3)
    model = make()
    model.to(dtype=dtype)
    return model.eval(), torch.randn(4, 8, dtype=dtype)


def _out(y):
    return y[0][-1] if isinstance(y, tuple) else y


def _residual():
    return L.ResidualConnection(_sequence(), nn.Linear(8, 8))


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("make", [_sequence, _residual, _block])
def test_symbolic_trace_and_script(make, mode):
    model, x = _build(make)
    with MODES[mode]():
        want = model(x)
        graph = torch.fx.symbolic_trace(model)
        assert torch.equal(graph(x), want)
        assert sum(type(graph.get_submodule(n.target)) is nn.Linear for n in graph.graph.nodes if n.op == "call_module") >= 2
        if mode != "inference":  # torch keeps a script's plan of a run with gradients, which is refused there
            assert torch.equal(torch.jit.script(model)(x), want)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("make", [_sequence, _residual, _block, lambda: L.GatedMLP(8, 16), _model])
def test_compile_in_one_graph(make, mode):
    model, x = _build(make)
    torch._dynamo.reset()
    with MODES[mode]():
        assert torch.equal(_out(torch.compile(model, fullgraph=True, backend="eager")(x)), _out(model(x)))
    torch._dynamo.reset()


@pytest.mark.parametrize("make", [_sequence, _residual, _block, lambda: L.GatedMLP(8, 16), _model])
def test_dynamic_quantization_finds_the_layers(make):
    model, _ = _build(make, torch.float32)
    linears = sum(type(m) is nn.Linear for m in model.modules())
    quantized = torch.ao.quantization.quantize_dynamic(model, {nn.Linear})
    assert linears >= 2 and not any(type(m) is nn.Linear for m in quantized.modules())
