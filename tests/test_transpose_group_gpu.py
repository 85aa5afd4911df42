"""Transposed copies of several matrices in one launch (csrc/kernels/elementwise.hip): every bit, in any mix and number."""
import pytest
import torch

from penroz.ops import _ext


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[], [(64, 64)], [(64, 192), (0, 64), (320, 64), (64, 64)], [(64, 128)] * 64, [(128, 64)] * 131])
def test_transpose_group(shapes):
    ins = [torch.randn(r, c, device="cuda").bfloat16() for r, c in shapes]
    outs = [torch.zeros(c, r, device="cuda", dtype=torch.bfloat16) for r, c in shapes]
    _ext.kernels().transpose_bf16_group(ins, outs)
    for a, b in zip(ins, outs):
        assert torch.equal(a.t(), b)
