"""The fp32 many-row projections (csrc/linear_tiles.hip) at the edges of their
tiles, against float64 products and the stand-alone RoPE / SwiGLU kernels.

Tolerance: an fp32 sum of k products of N(0, 1) x N(0, 1/k) values errs by
less than k 2^-24 max|partial sum| ~ 512 * 6e-8 * 4 = 1.2e-4 in the worst case
and sqrt(k) of that in practice; 2e-5 is twice the practical figure."""
import pytest
import torch

from serving import _native, fused_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = dict(rtol=2e-5, atol=2e-5)
# weights of variance 1 in the place of 1/128: sqrt(128) times the sums
WIDE = {False: TOL, True: dict(rtol=2.4e-4, atol=2.4e-4)}


def mk(seed, *shape, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV) * std


def tiles(x, w, bias, epilogue, out):
    n = out.shape[1]
    rc = _native.lib().pkv_linear_tiles(
        out.data_ptr(), x.data_ptr(), w.data_ptr(), _native.ptr(bias), x.shape[0], n, x.shape[1],
        x.stride(0), epilogue, 0, _native.stream_ptr(x.device))
    _native.check(rc, "pkv_linear_tiles")
    return out


@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (63, 33, 64), (64, 64, 32), (65, 130, 96),
                                   (300, 47, 512), (2146, 512, 512), (1025, 640, 128)])
@pytest.mark.parametrize("bias", [False, True])
def test_plain_swiglu_residual(m, n, k, bias):
    x = mk(1, m, k + 8)[:, :k]  # row stride past k
    w = mk(2, 2 * n, k, std=k ** -0.5)
    b = mk(3, 2 * n) if bias else None
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    full = tiles(x, w, b, _native.EPILOGUE_NONE, torch.empty(m, 2 * n, device=DEV))
    torch.testing.assert_close(full.double(), want, **TOL)
    # the epilogues are those of the same sums, bit for bit
    sw = tiles(x, w, b, _native.EPILOGUE_SWIGLU, torch.empty(m, n, device=DEV))
    assert torch.equal(sw, fused_ops.silu_mul(full[:, :n], full[:, n:]))
    r = mk(4, m, 2 * n)
    got = tiles(x, w, b, _native.EPILOGUE_RESIDUAL, r.clone())
    assert torch.equal(got, r + full)


@pytest.mark.parametrize("m,hq,hkv,d,k", [(65, 8, 1, 64, 512), (257, 4, 1, 32, 128),
                                          (100, 3, 1, 10, 64), (1100, 8, 2, 64, 512)])
def test_rope_qkv(m, hq, hkv, d, k):
    x = mk(1, m, k)
    w = mk(2, (hq + 2 * hkv) * d, k, std=k ** -0.5)
    pos = torch.randint(0, 50, (m,), device=DEV, dtype=torch.int32)
    pos[m // 2] = 77  # outside the tables: angle 0 and a status bit
    ang = mk(3, 50, d // 2)
    cos, sin = ang.cos().contiguous(), ang.sin().contiguous()
    full = tiles(x, w, None, _native.EPILOGUE_NONE, torch.empty(m, w.shape[0], device=DEV))
    nq, nk = hq * d, hkv * d
    want = fused_ops.rope(full[:, :nq], full[:, nq:nq + nk], pos, cos, sin, v=full[:, nq + nk:],
                          hq=hq, hkv=hkv, d=d)
    got = [torch.empty_like(t) for t in want]
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    rc = _native.lib().pkv_linear_tiles_rope_qkv(
        *(t.data_ptr() for t in got), x.data_ptr(), w.data_ptr(), None, m, k, k, pos.data_ptr(),
        cos.data_ptr(), sin.data_ptr(), 50, hq, hkv, d, 0, status.data_ptr(),
        _native.stream_ptr(x.device))
    _native.check(rc, "pkv_linear_tiles_rope_qkv")
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert int(status.item()) == _native.PKV_STATUS_BAD_POS


def test_wrappers_take_it_and_gradients_do_not(monkeypatch):
    x, w = mk(1, 1100, 128), mk(2, 96, 128, std=128 ** -0.5)
    calls = []
    real = fused_ops._tiles
    monkeypatch.setattr(fused_ops, "_tiles", lambda *a: calls.append(1) or real(*a))
    y = fused_ops.linear(x, w)
    assert calls
    torch.testing.assert_close(y.double(), x.double() @ w.double().t(), **TOL)
    wg = w.clone().requires_grad_()
    fused_ops.linear(x, wg).sum().backward()
    assert len(calls) == 1 and wg.grad is not None


@pytest.mark.parametrize("k", [32, 64, 96, 128, 160, 192, 224, 256, 1024])
@pytest.mark.parametrize("m,n", [(257, 40), (4090, 250)])
def test_slab_counts(k, m, n):
    """Every remainder of the loop's rounds of four slabs, on the narrow and the
    wide tiles. Tolerance: as above, for 1024 products sqrt(2) of 512's."""
    x, w = mk(1, m, k), mk(2, n, k, std=k ** -0.5)
    got = tiles(x, w, None, _native.EPILOGUE_NONE, torch.empty(m, n, device=DEV))
    torch.testing.assert_close(got.double(), x.double() @ w.double().t(), rtol=3e-5, atol=3e-5)


def test_transformed_calls_stay_with_the_framework():
    """Autocast, forward-mode AD and torch.func see the projection as they see
    F.linear; an x that is the residual itself is read before it is written."""
    x, w, t = mk(1, 1100, 128), mk(2, 128, 128, std=128 ** -0.5), mk(3, 1100, 128)
    with torch.no_grad():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert fused_ops.linear(x, w).dtype == torch.bfloat16
        tangent = torch.func.jvp(lambda a: fused_ops.linear(a, w), (x,), (t,))[1]
        torch.testing.assert_close(tangent.double(), t.double() @ w.double().t(), **TOL)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x, t)
            out = torch.autograd.forward_ad.unpack_dual(fused_ops.linear(dual, w))
        assert out.tangent is not None
        both = torch.func.vmap(lambda a: fused_ops.linear(a, w))(torch.stack([x, t]))
        torch.testing.assert_close(both[1], fused_ops.linear(t, w), **TOL)
        want = x.double() + x.double() @ w.double().t()
        torch.testing.assert_close(fused_ops.linear_residual_(x, x, w).double(), want, **TOL)


@pytest.mark.parametrize("shape", [(1,), (96,), (300, 96), (1, 96)])
def test_bias_forms_of_the_framework(shape):
    """A bias of one value per feature is the kernel's; one that broadcasts is
    added as F.linear adds it. F.linear's sums differ by rounding only."""
    x, w, b = mk(1, 300, 128), mk(2, 96, 128, std=128 ** -0.5), mk(3, *shape)
    want = x.double() @ w.double().t() + b.double()
    with torch.no_grad():
        torch.testing.assert_close(fused_ops.linear(x, w, b).double(), want, **TOL)
        r = mk(4, 300, 96)
        got = fused_ops.linear_residual_(r.clone(), x, w, b)
        torch.testing.assert_close(got.double(), r.double() + want, **TOL)
        # products of two such sums of up to ~5 in size: 5 times their tolerance
        gate, up = want[:, :48], want[:, 48:]
        torch.testing.assert_close(fused_ops.linear_swiglu(x, w, b).double(),
                                   torch.nn.functional.silu(gate) * up, rtol=1e-4, atol=1e-4)
        pos = torch.zeros(300, dtype=torch.int32, device=DEV)  # angle 0: no rotation
        cos, sin = torch.ones(4, 16, device=DEV), torch.zeros(4, 16, device=DEV)
        q, k, v = fused_ops.linear_rope_qkv(x, w, b, pos, cos, sin, 1, 1, 32)
        torch.testing.assert_close(torch.cat([q, k, v], 1).view(300, 96).double(), want, **TOL)


@pytest.mark.parametrize("features", [95, 97])
def test_wrong_bias_is_an_error(features):
    x, w = mk(1, 300, 128), mk(2, 96, 128)
    with torch.no_grad(), pytest.raises(RuntimeError):
        fused_ops.linear(x, w, mk(3, features))


def test_residual_update_is_seen_by_autograd():
    """A backward whose graph saved the residual raises, as after add_; an
    inference tensor outside inference mode is refused."""
    x, w, r = mk(1, 300, 128), mk(2, 96, 128, std=128 ** -0.5), mk(3, 300, 96)
    p = torch.ones(300, 96, device=DEV, requires_grad=True)
    y = (p * r).sum()  # saves r
    with torch.no_grad():
        before = r._version
        fused_ops.linear_residual_(r, x, w)
    assert r._version == before + 1
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()
    with torch.inference_mode():
        q = torch.zeros(300, 96, device=DEV)
        fused_ops.linear_residual_(q, x, w)
    with torch.no_grad(), pytest.raises(RuntimeError, match="inference"):
        fused_ops.linear_residual_(q, x, w)


@pytest.mark.parametrize("shared", ["x", "weight", "bias", "rows of x"])
def test_residual_sharing_memory_is_read_first(shared):
    """resid may be an operand itself: every operand is read before it changes."""
    x, w, b = mk(1, 1024, 128), mk(2, 128, 128, std=128 ** -0.5), mk(3, 128)
    r = mk(4, 1024, 128)
    if shared == "x":
        r = x
    elif shared == "weight":
        w = r[300:428]
    elif shared == "bias":
        b = r[700]
    else:
        buf = mk(5, 2048, 128)
        x, r = buf[:1024], buf[1023:2047]
    want = r.double() + x.double() @ w.double().t() + b.double()
    with torch.no_grad():
        got = fused_ops.linear_residual_(r, x, w, b)
    torch.testing.assert_close(got.double(), want, **WIDE[shared == "weight"])


def test_forms_of_the_framework():
    """A vector as the weight, no features, empty sums, negated views."""
    x, w, b = mk(1, 300, 128), mk(2, 96, 128, std=128 ** -0.5), mk(3, 96)
    with torch.no_grad():
        torch.testing.assert_close(fused_ops.linear(x, w[0]).double(), x.double() @ w[0].double(),
                                   **TOL)
        assert fused_ops.linear(x, w[:0]).shape == (300, 0)
        assert torch.equal(fused_ops.linear(x[:, :0], w[:, :0], b), b.expand(300, 96))
        got = fused_ops.linear(torch._neg_view(x), w)
        torch.testing.assert_close(got.double(), -(x.double() @ w.double().t()), **TOL)


def test_trace_records_the_product():
    """A traced projection answers for other inputs than the traced one."""
    x, x1, w = mk(1, 300, 128), mk(3, 300, 128), mk(2, 96, 128, std=128 ** -0.5)
    with torch.no_grad():
        traced = torch.jit.trace(lambda a: fused_ops.linear(a, w), x, check_trace=False)
        torch.testing.assert_close(traced(x1).double(), x1.double() @ w.double().t(), **TOL)


@pytest.mark.parametrize("rows", [40, 300])
def test_rotary_tables_of_different_length(rows):
    """An error for a prompt, as in rope(); few rows at positions inside both
    tables are rotated."""
    x, w = mk(1, rows, 128), mk(2, 96, 128, std=128 ** -0.5)
    pos = torch.arange(rows, dtype=torch.int32, device=DEV) % 30
    cos, sin = torch.rand(50, 16, device=DEV), torch.rand(30, 16, device=DEV)
    with torch.no_grad():
        if rows > 256:
            with pytest.raises(ValueError, match="equal shape"):
                fused_ops.linear_rope_qkv(x, w, None, pos, cos, sin, 1, 1, 32)
            return
        got = fused_ops.linear_rope_qkv(x, w, None, pos, cos, sin, 1, 1, 32)
        want = fused_ops.linear_rope_qkv(x, w, None, pos, cos[:30].contiguous(), sin, 1, 1, 32)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_refusals():
    L = _native.lib()
    x, w, out = mk(1, 64, 48), mk(2, 16, 48), torch.empty(64, 16, device=DEV)
    st = _native.stream_ptr(x.device)
    args = lambda k, epi, dt: (out.data_ptr(), x.data_ptr(), w.data_ptr(), None, 64, 16, k,  # noqa: E731
                               48, epi, dt, st)
    assert L.pkv_linear_tiles(*args(48, 0, 0)) == _native.PKV_ERR_UNSUPPORTED  # k % 32
    assert L.pkv_linear_tiles(*args(32, 0, 2)) == _native.PKV_ERR_UNSUPPORTED  # bf16
    assert L.pkv_linear_tiles(*args(32, 9, 0)) == _native.PKV_ERR_INVALID
    assert L.pkv_linear_tiles(*args(64, 0, 0)) == _native.PKV_ERR_INVALID  # stride below k
