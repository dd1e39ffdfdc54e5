"""The rule that hands fp32 prompts to the tile projections (fused_ops), on the
CPU: what it refuses goes to the framework's linear, which answers or raises
as it does by itself."""
import pytest
import torch

from serving import fused_ops


def operands(m=300, n=96, k=128):
    return torch.randn(m, k), torch.randn(n, k)


def test_plain_operands_fit():
    x, w = operands()
    assert fused_ops._tiles_fit(x, w, None)
    assert fused_ops._tiles_fit(x, w, torch.randn(96))


@pytest.mark.parametrize("shape", [(1,), (), (95,), (97,), (300, 96), (1, 96), (0,)])
def test_other_biases_do_not_fit(shape):
    # one value per weight row is all the kernel reads
    x, w = operands()
    assert not fused_ops._tiles_fit(x, w, torch.randn(shape))
