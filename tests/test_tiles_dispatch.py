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


def test_rotary_tables():
    """A prompt's projection refuses tables of different length, as rope()
    does; the few-row kernels rotate at the positions both tables hold."""
    cos, sin = torch.randn(50, 16), torch.randn(40, 16)
    with pytest.raises(ValueError, match="equal shape"):
        fused_ops._rope_tables(cos, sin, 32, "rope", True)
    assert fused_ops._rope_tables(cos, sin, 32, "rope", False)[2] == 40
    assert fused_ops._rope_tables(cos, cos, 32, "rope", True)[2] == 50
    with pytest.raises(ValueError, match="fp32"):
        fused_ops._rope_tables(cos.double(), sin, 32, "rope", False)
