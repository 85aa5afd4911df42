"""Decode steps of models whose small parameters are views off the alignment that the widest kernels ask for."""
import pytest
import torch

from penroz.models import graph_decode as gd
from test_graph_decode_gpu import _gemma_model, _model

pytestmark = pytest.mark.gpu


def _shift(p):
    """The same values, one element off their buffer's start."""
    buf = torch.empty(p.numel() + 1, device=p.device, dtype=p.dtype)
    view = buf[1:].view(p.shape)
    view.copy_(p.data)
    p.data = view


def _step(m, rows):
    dec = gd.GraphDecoder(m, rows, 32, 0.0, None)
    assert dec.program is not None
    idx = torch.randint(0, 256, (rows, 7), device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    with torch.inference_mode():
        dec.attach()
        try:
            m(idx[:, :6], skip_softmax=True)
            dec._set_state(idx[:, 6:], 6)
            dec.cache.graph_mode = True
            dec.cache.begin_step()
            return dec.program.forward(idx[:, 6:], dec.cache).float()
        finally:
            dec.cache.graph_mode = False
            dec.detach()


@pytest.mark.parametrize("what", ["in_norm", "pre_mlp", "post_attn", "post_mlp", "embedding"])
@pytest.mark.parametrize("rows", [1, 4])
def test_gemma_norms_and_table(rows, what):
    m = _gemma_model(64)
    want = _step(m, rows)
    prog = gd.GemmaDecodeProgram.build(m)
    for mod in [prog.emb] if what == "embedding" else [b[what] for b in prog.blocks]:
        _shift(mod.weight)
    got = _step(m, rows)
    # the same products behind the same norms, whose row sums run in another order in the kernel by itself: roundings of
    # the bf16 residual stream, as test_gemma_program_step_matches_module_step's bound has them
    assert (got - want).norm() / want.norm() < 2e-2


@pytest.mark.parametrize("rows,what", [(r, w) for r in (1, 4, 5, 8) for w in ("qkv", "fc", "proj", "fc2")] +
                         [(r, w) for r in (5, 8) for w in ("proj.weight", "fc2.weight")])
def test_gpt_biases_and_weights(rows, what):
    m = _model(torch.bfloat16)
    blocks = gd.GPTDecodeProgram.build(m).spec.blocks
    for b in blocks:  # (they are zero at first)
        for lin in (b.qkv, b.proj, b.fc, b.fc2):
            torch.nn.init.normal_(lin.bias, std=0.1)
    want = _step(m, rows)
    for b in blocks:
        lin = getattr(b, what.split(".")[0])
        if what.endswith("weight"):
            _shift(lin.weight)
        elif what in ("qkv", "fc"):
            _shift(lin.bias)
        else:  # every second element of a longer one
            view = torch.zeros(2 * lin.bias.numel(), device="cuda", dtype=torch.bfloat16)[::2]
            view.copy_(lin.bias.data)
            lin.bias.data = view
    got = _step(m, rows)
    # bf16 operands in sums of another order: test_decode_program_step_matches_module_step's bound
    assert (got - want).norm() / want.norm() < 2e-2
