"""The rule that hands fp32 prompts to the tile projections (fused_ops), on the
CPU: what it refuses goes to the framework's linear, which answers or raises
as it does by itself."""
import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.flop_counter import FlopCounterMode

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


def test_forms_only_the_framework_takes():
    x, w = operands()
    assert not fused_ops._tiles_fit(x, w[0], None)                    # a vector
    assert not fused_ops._tiles_fit(x, w[:0], None)                   # no features
    assert not fused_ops._tiles_fit(x[:, :0], w[:, :0], None)         # empty sums
    assert not fused_ops._tiles_fit(x, w.to_sparse(), None)
    assert not fused_ops._tiles_fit(x, w[:, :96], None)               # an error there
    assert not fused_ops._tiles_fit(torch._neg_view(x), w, None)
    assert not fused_ops._tiles_fit(x, torch._neg_view(w), None)
    assert not fused_ops._tiles_resid_fit(torch._neg_view(torch.zeros(300, 96)), x, 96)
    assert not fused_ops._tiles_fit(x.double(), w.double(), None)
    assert not fused_ops._tiles_fit(x[:256], w, None)


@pytest.mark.parametrize("rows,n,k,plain,fused", [
    (257, 96, 32, True, True), (5000, 512, 128, True, True), (300, 513, 128, False, True),
    (300, 128, 160, False, True), (257, 64, 384, False, True),
    (512, 512, 512, False, False), (513, 512, 512, False, True), (257, 1024, 416, False, True),
    (1024, 16384, 544, False, False), (2240, 1024, 1024, False, False),
    (2305, 1024, 1024, False, True), (8192, 96, 1024, False, False),
    (2305, 1024, 1056, False, False)])
def test_sizes_the_tiles_are_faster_at(rows, n, k, plain, fused):
    """Both sides of each line of the size rule."""
    x, w = torch.empty(rows, k), torch.empty(n, k)
    assert fused_ops._tiles_fit(x, w, None, False) == plain
    assert fused_ops._tiles_fit(x, w, None, True) == fused


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


class Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class Function(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("mode", [Dispatch, Function, lambda: FlopCounterMode(display=False)])
def test_modes_see_the_framework(mode):
    x, w = operands()
    with mode():
        assert not fused_ops._tiles_fit(x, w, None)
    assert fused_ops._tiles_fit(x, w, None)


def test_default_device_is_no_transform():
    x, w = operands()
    with torch.device("cpu"):
        assert fused_ops._tiles_fit(x, w, None)


@pytest.mark.parametrize("trace", [
    lambda f, x: torch.jit.trace(f, x, check_trace=False),
    lambda f, x: make_fx(f)(x),
    lambda f, x: make_fx(f, pre_dispatch=True)(x),
    lambda f, x: torch.compile(f, backend="eager", fullgraph=True)(x),
    lambda f, x: torch.export.export(Module(f), (x,))])
def test_traces_hold_the_framework_call(trace):
    """A trace would hold an empty tensor in the place of a kernel's output."""
    x, w = operands()
    seen = []

    def f(a):
        fits = fused_ops._tiles_fit(a, w, None)
        seen.append(fits)
        return torch.nn.functional.linear(a, w)
    trace(f, x)
    assert seen and not any(seen)


class Module(torch.nn.Module):
    def __init__(self, f):
        super().__init__()
        self.f = f

    def forward(self, x):
        return self.f(x)


def test_inference_residual_is_the_frameworks():
    x, _ = operands()
    with torch.inference_mode():
        r = torch.zeros(300, 96)
        assert fused_ops._tiles_resid_fit(r, x, 96)
    assert not fused_ops._tiles_resid_fit(r, x, 96)
    assert fused_ops._tiles_resid_fit(torch.zeros(300, 96), x, 96)


def test_memory_apart():
    buf = torch.zeros(1000)
    out = buf[100:200]
    assert fused_ops._apart(out, None)
    assert fused_ops._apart(out, buf[:100]) and fused_ops._apart(out, buf[200:])
    assert not fused_ops._apart(out, buf[:101]) and not fused_ops._apart(out, buf[199:])
    assert not fused_ops._apart(out, out)
    # rows of 10 every 60 elements, the last ones past out's start
    assert fused_ops._apart(out, buf.as_strided((2, 10), (60, 1)))
    assert not fused_ops._apart(out, buf.as_strided((3, 10), (60, 1)))
    assert fused_ops._apart(out, buf[150:150])
