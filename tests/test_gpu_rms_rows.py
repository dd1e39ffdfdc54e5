"""RMSNorm rows held in registers (csrc/layers.hip, rms_rows_kernel) against the
row kernel, which unaligned rows take: both sum in the canonical order, so the
bits agree (that order is defined for rows of whole 32-element steps: a row of
1000 is summed in another order per access width, by neither of these paths).
Odd row counts, every register count and ranges without steps."""
import pytest
import torch

from serving import _native

pytestmark = pytest.mark.gpu
DEV = "cuda"


def norm(x, w, delta, shift):
    """pkv_rms_norm on copies `shift` elements past an aligned address:
    (y, residual)."""
    def put(t):
        b = torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)[shift:shift + t.numel()]
        return b.view(t.shape).copy_(t)
    xs, y, r = put(x), torch.empty_like(x), torch.empty_like(x)
    d = None if delta is None else put(delta)
    rows, dim = x.shape
    rc = _native.lib().pkv_rms_norm(
        y.data_ptr(), r.data_ptr(), xs.data_ptr(), _native.ptr(d), w.data_ptr(), rows, dim, dim,
        dim, 1e-5, _native.DTYPE_CODES[x.dtype], _native.stream_ptr(x.device))
    _native.check(rc, "rms_norm")
    return y, r


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,dim", [(1, 32), (3, 64), (2, 256), (5, 288), (7, 512), (4, 992),
                                      (9, 960), (1025, 1024), (3, 1056), (2, 2048), (2, 2080),
                                      (1024, 1056), (1025, 2048)])
@pytest.mark.parametrize("add", [False, True])
def test_bits_of_the_row_kernel(dtype, rows, dim, add):
    g = torch.Generator(device=DEV).manual_seed(rows * dim)
    mk = lambda *s: torch.randn(s, generator=g, device=DEV).to(dtype)  # noqa: E731
    x, w, d = mk(rows, dim), mk(dim), mk(rows, dim) if add else None
    y, r = norm(x, w, d, 0)
    y1, r1 = norm(x, w, d, 1)  # x no longer 16-byte aligned
    assert torch.equal(y, y1)
    if add:
        assert torch.equal(r, r1) and torch.equal(r, x + d)
