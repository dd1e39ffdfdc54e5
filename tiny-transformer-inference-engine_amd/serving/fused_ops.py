"""Host wrappers of the decoder block's kernels around the paged attention in
libpagedkv.so: RMSNorm with a fused residual add, RoPE on token-major Q/K
rows, and the SwiGLU gate (csrc/layers.hip); the few-row projections with
those ops fused into their epilogues (csrc/linear.hip); the greedy argmax
(csrc/sampling.hip).

Every function requires ROCm device tensors and the library (RuntimeError
otherwise). The projections hand fp32 prompts to the tile kernel
(csrc/linear_tiles.hip, _tiles_ok) and other shapes their kernel does not take
(k not a multiple of 32, more than LINEAR_MAX_ROWS rows or LINEAR_MAX_FEATURES
features) to the library GEMM. Outputs are allocated with
torch on the input's device and the current stream, so the calls can be
captured in a HIP graph.
"""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from . import _native


def _rows(x: torch.Tensor, what: str):
    """x viewed as [rows, dim] with unit column stride: (tensor, rows, stride)."""
    if x.dim() == 0:
        raise ValueError(f"{what}: expected at least one dimension")
    dim = x.shape[-1]
    x2 = x.reshape(-1, dim) if x.dim() != 2 else x
    if x2.stride(-1) != 1 or (x2.shape[0] > 1 and x2.stride(0) < dim):
        x2 = x2.contiguous()
    return x2, x2.shape[0], (x2.stride(0) if x2.shape[0] > 1 else dim)


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """RMSNorm of the last dimension: (x * rsqrt(mean(x^2) + eps)) * weight in
    fp32, rounded to x.dtype (models/rmsnorm.py:12-18)."""
    _native.require_device(x, weight, what="rms_norm")
    w = weight if weight.dtype == x.dtype else weight.to(x.dtype)
    w = w.contiguous()
    if w.numel() != x.shape[-1]:
        raise ValueError(f"rms_norm: weight has {w.numel()} elements, rows have {x.shape[-1]}")
    x2, rows, stride = _rows(x, "rms_norm")
    y = x.new_empty(x.shape)
    rc = _native.calls().pkv_rms_norm(
        y.data_ptr(), None, x2.data_ptr(), None, w.data_ptr(), rows, x.shape[-1], stride,
        0, float(eps), _native.dtype_code(x.dtype), _native.stream_ptr(x.device))
    _native.check(rc, "rms_norm")
    return y


def add_rms_norm_(x: torch.Tensor, delta: torch.Tensor, weight: torch.Tensor,
                  eps: float) -> torch.Tensor:
    """x += delta (rounded to x.dtype, in place), then return rms_norm(x):
    the residual add of a decoder block fused with the next norm
    (serving/paged_model.py:20-29). x must be contiguous."""
    _native.require_device(x, delta, weight, what="add_rms_norm_")
    if not x.is_contiguous():
        raise ValueError("add_rms_norm_: x must be contiguous (it is updated in place)")
    if delta.shape != x.shape or delta.dtype != x.dtype:
        raise ValueError(f"add_rms_norm_: delta {tuple(delta.shape)} {delta.dtype} vs x "
                         f"{tuple(x.shape)} {x.dtype}")
    w = weight if weight.dtype == x.dtype else weight.to(x.dtype)
    w = w.contiguous()
    dim = x.shape[-1]
    if w.numel() != dim:
        raise ValueError(f"add_rms_norm_: weight has {w.numel()} elements, rows have {dim}")
    d2, rows, dstride = _rows(delta, "add_rms_norm_")
    y = torch.empty_like(x)
    rc = _native.calls().pkv_rms_norm(
        y.data_ptr(), x.data_ptr(), x.data_ptr(), d2.data_ptr(), w.data_ptr(), rows, dim, dim,
        dstride, float(eps), _native.dtype_code(x.dtype), _native.stream_ptr(x.device))
    _native.check(rc, "add_rms_norm_")
    return y


def _tok_rows(t: torch.Tensor, heads: int, d: int, what: str):
    """[T, heads, d] or [T, heads*d] rows with contiguous heads: (tensor, row stride)."""
    if t.dim() == 3:
        if t.shape[1] != heads or t.shape[2] != d:
            raise ValueError(f"{what}: expected [T, {heads}, {d}], got {tuple(t.shape)}")
        ok = t.stride(2) == 1 and t.stride(1) == d
        if not ok:
            t = t.contiguous()
        return t, (t.stride(0) if t.shape[0] > 1 else heads * d)
    if t.dim() == 2 and t.shape[1] == heads * d:
        if t.stride(1) != 1:
            t = t.contiguous()
        return t, (t.stride(0) if t.shape[0] > 1 else heads * d)
    raise ValueError(f"{what}: expected [T, {heads}, {d}], got {tuple(t.shape)}")


def rope(q: torch.Tensor, k: torch.Tensor, positions: torch.Tensor, cos: torch.Tensor,
         sin: torch.Tensor, v: torch.Tensor | None = None, hq: int | None = None,
         hkv: int | None = None, d: int | None = None):
    """Rotary embedding of q [T, Hq, D] and k [T, Hkv, D] at positions [T]
    with fp32 tables cos/sin [max_pos, D/2] (models/rope.py:21-47, values and
    intermediate products rounded to q.dtype). q, k (and v) may be strided
    column ranges of one projection output, given as [T, H*D] slices with
    hq/hkv/d. Returns contiguous (q_rot, k_rot) or, with v, (q_rot, k_rot,
    v_contiguous)."""
    if q.dim() == 3:
        hq, d = q.shape[1], q.shape[2]
    if k.dim() == 3:
        hkv = k.shape[1]
    if hq is None or hkv is None or d is None:
        raise ValueError("rope: pass hq, hkv and d for 2-D q / k")
    tensors = [q, k, positions, cos, sin] + ([v] if v is not None else [])
    _native.require_device(*tensors, what="rope")
    if k.dtype != q.dtype or (v is not None and v.dtype != q.dtype):
        raise ValueError("rope: q, k, v must share a dtype")
    T = q.shape[0]
    if k.shape[0] != T or (v is not None and v.shape[0] != T) or positions.numel() != T:
        raise ValueError("rope: q, k, v and positions disagree on the token count")
    cos2 = cos.reshape(-1, d // 2)
    sin2 = sin.reshape(-1, d // 2)
    if cos2.dtype != torch.float32 or sin2.dtype != torch.float32 or cos2.shape != sin2.shape:
        raise ValueError("rope: cos / sin must be fp32 tables of equal shape [max_pos, D/2]")
    cos2, sin2 = cos2.contiguous(), sin2.contiguous()
    pos = positions if positions.dtype == torch.int32 else positions.to(torch.int32)
    pos = pos.contiguous()
    qs, q_stride = _tok_rows(q, hq, d, "rope q")
    ks, k_stride = _tok_rows(k, hkv, d, "rope k")
    q_out = q.new_empty((T, hq, d))
    k_out = q.new_empty((T, hkv, d))
    if v is not None:
        vs, v_stride = _tok_rows(v, hkv, d, "rope v")
        v_out = q.new_empty((T, hkv, d))
    else:
        vs, v_stride, v_out = None, 0, None
    rc = _native.calls().pkv_rope(
        q_out.data_ptr(), k_out.data_ptr(), _native.ptr(v_out), qs.data_ptr(), ks.data_ptr(),
        _native.ptr(vs), q_stride, k_stride, v_stride, pos.data_ptr(), cos2.data_ptr(),
        sin2.data_ptr(), cos2.shape[0], T, hq, hkv, d, _native.dtype_code(q.dtype), None,
        _native.stream_ptr(q.device))
    _native.check(rc, "rope")
    return (q_out, k_out) if v is None else (q_out, k_out, v_out)


def _rope_tables(cos, sin, d, what, equal):
    """The fp32 tables as contiguous [max_pos, d/2] and the positions both hold.
    equal: tables of different length are an error, as in rope()."""
    if cos.dtype != torch.float32 or sin.dtype != torch.float32:
        raise ValueError(f"{what}: cos / sin must be fp32 tables")
    cos2, sin2 = cos.reshape(-1, d // 2).contiguous(), sin.reshape(-1, d // 2).contiguous()
    shape = cos2.shape
    if shape == sin2.shape:
        return cos2, sin2, shape[0]
    if equal:
        raise ValueError(f"{what}: cos / sin must be tables of equal shape [max_pos, D/2]")
    return cos2, sin2, min(shape[0], sin2.shape[0])


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """gate * sigmoid(gate) * up in fp32, rounded once
    (kernels/fused_swiglu/kernel.py:6-19). gate and up may be strided column
    ranges of one [rows, 2H] projection output; the result is contiguous."""
    _native.require_device(gate, up, what="silu_mul")
    if gate.shape != up.shape or gate.dtype != up.dtype:
        raise ValueError("silu_mul: gate and up must have the same shape and dtype")
    g2, rows, gs = _rows(gate, "silu_mul")
    u2, _, us = _rows(up, "silu_mul")
    cols = gate.shape[-1]
    out = gate.new_empty(gate.shape)
    rc = _native.calls().pkv_silu_mul(out.data_ptr(), g2.data_ptr(), u2.data_ptr(), rows, cols,
                                    gs, us, _native.dtype_code(gate.dtype),
                                    _native.stream_ptr(gate.device))
    _native.check(rc, "silu_mul")
    return out


# the few-row projection kernels (csrc/linear.hip) take decode-sized row
# counts; fp32 prompts go to the tile kernel (_tiles_ok), other wider problems
# (16-bit prefill chunks, the vocabulary projection) to the library GEMM
LINEAR_MAX_ROWS = 256
LINEAR_MAX_FEATURES = 16384


def _as_rows(x: torch.Tensor) -> torch.Tensor:
    x2 = x.reshape(-1, x.shape[-1]) if x.dim() != 2 else x
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    return x2


def _linear_ok(x2: torch.Tensor, w: torch.Tensor, bias, n_features: int) -> bool:
    rows, k = x2.shape
    return (x2.is_cuda and 0 < rows <= LINEAR_MAX_ROWS
            and x2.dtype in (torch.bfloat16, torch.float16, torch.float32)
            and w.dtype == x2.dtype and w.is_cuda
            and k % 32 == 0 and n_features <= LINEAR_MAX_FEATURES
            and _weights_hold(w, n_features, k)
            # one value per weight row; any other bias is the framework's
            and (bias is None or (bias.dtype == x2.dtype and bias.is_contiguous()
                                  and bias.shape == w.shape[:1] and bias.is_cuda))
            and w.is_contiguous()
            and (rows == 1 or x2.stride(0) % 8 == 0)
            and x2.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def _weights_hold(w: torch.Tensor, n: int, k: int) -> bool:
    """Whether w has n rows of k values, as the kernel will read it."""
    shape = w.shape
    return len(shape) == 2 and shape[1] == k and shape[0] >= n


# Projections of more than 256 fp32 rows that pkv_linear_tiles takes, by what it
# was measured to be no slower at than the library GEMM and the element-wise
# launch of its own (library / tiles, us of GPU time, 257 to 8192 rows):
#  - without a fused op it saves no launch: k <= TILES_PLAIN_K and up to
#    TILES_PLAIN_N features (300 x 128, k 128 4.4 / 4.0; but 2481 x 512, k 512
#    14.9 / 19.0, 257 x 512 6.4 / 8.6);
#  - fused, k <= TILES_ANY_K: every size (k 128, 2481 rows, gate/up 10.1 / 5.6; at
#    k 384 1.0 to 1.9 times as fast);
#  - k <= TILES_SMALL_K: more tiles than half the CUs (2481 rows, k 512: q/k/v
#    25.4 / 22.9, gate/up 46.8 / 29.3, out 19.0 / 18.7; but q/k/v of 257 rows 9.5 /
#    10.1);
#  - k <= TILES_MAX_K: more than TILES_MIN_ROWS rows and four and a half rounds of
#    tiles over the CUs (k 1024: 2481 rows, gate/up 109 / 87, 8192 rows, out 141 /
#    135; but 1025 rows, out 27.4 / 30.7, 1600 rows 37.4 / 38.8).
# Of 1580 shapes inside the lines five are slower by more than 1%, one by 8%.
TILES_PLAIN_K, TILES_PLAIN_N = 128, 512
TILES_ANY_K = 384
TILES_SMALL_K = 512
TILES_MAX_K = 1024
TILES_MIN_ROWS = 1024
CUS = 256


def _tiles_faster(rows: int, n: int, k: int, fused: bool) -> bool:
    """The measured line above; n weight rows in tiles of 64 rows x 32."""
    if not fused:
        return k <= TILES_PLAIN_K and n <= TILES_PLAIN_N
    if k <= TILES_ANY_K:
        return True
    tiles = -(-rows // 64) * -(-n // 32)
    if k <= TILES_SMALL_K:
        return 2 * tiles > CUS
    return k <= TILES_MAX_K and rows > TILES_MIN_ROWS and 2 * tiles >= 9 * CUS


def _mode_active() -> bool:
    """Whether a dispatch or function mode is to see the framework's calls. The
    one behind torch.set_default_device only places new tensors."""
    if (torch._C._len_torch_dispatch_stack() != 0
            or torch._ops._len_torch_dispatch_stack_pre_dispatch() != 0):
        return True
    return any(type(torch._C._get_function_stack_at(i)) is not DeviceContext
               for i in range(torch._C._len_torch_function_stack()))


def _transformed(ts) -> bool:
    """Whether a call records, transforms or casts these tensors: compilation
    and tracing (where the tensors can be plain ones: torch.jit.trace, make_fx),
    modes, gradients, torch.func and forward-mode AD, autocast, tensor
    subclasses. A kernel call would be missing from what they record."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing() or _mode_active()
            or (torch.is_grad_enabled() and any(t.requires_grad for t in ts))
            or torch.is_autocast_enabled() or forward_ad._current_level >= 0
            or torch._C._functorch.peek_interpreter_stack() is not None
            or any(type(t) not in (torch.Tensor, torch.nn.Parameter) for t in ts))


def _tiles_fit(x2: torch.Tensor, w: torch.Tensor, bias, fused: bool = False) -> bool:
    """Whether pkv_linear_tiles takes a projection of these operands (fused:
    with an element-wise op in its epilogue). Calls the
    framework has to see stay on its GEMM, and so do forms that only it takes: a
    bias of any other shape than one value per weight row (all the kernel reads),
    a weight that is a vector, sparse or empty, and lazily negated values."""
    ts = (x2, w) if bias is None else (x2, w, bias)
    rows, k = x2.shape
    return (rows > LINEAR_MAX_ROWS and 0 < k <= TILES_MAX_K
            and all(t.dtype == torch.float32 and t.device == x2.device
                    and t.layout is torch.strided for t in ts)
            and not _transformed(ts) and not any(t.is_neg() for t in ts)
            and w.dim() == 2 and w.shape[1] == k and k % 32 == 0
            and 0 < w.shape[0] <= LINEAR_MAX_FEATURES and w.is_contiguous()
            and _tiles_faster(rows, w.shape[0], k, fused)
            and (bias is None or (bias.shape == w.shape[:1] and bias.is_contiguous()))
            and x2.stride(0) >= k and x2.stride(0) % 4 == 0
            and rows * x2.stride(0) < 1 << 29 and w.numel() < 1 << 29
            and x2.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def _tiles_ok(x2: torch.Tensor, w: torch.Tensor, bias, fused: bool = False) -> bool:
    return x2.is_cuda and _tiles_fit(x2, w, bias, fused)


def _tiles(out, x2, w, bias, n, epilogue, what):
    rc = _native.calls().pkv_linear_tiles(
        out.data_ptr(), x2.data_ptr(), w.data_ptr(), _native.ptr(bias), x2.shape[0], n,
        x2.shape[1], x2.stride(0), epilogue, _native.dtype_code(x2.dtype),
        _native.stream_ptr(x2.device))
    _native.check(rc, what)
    return out


def _x_stride(x2):
    return x2.stride(0) if x2.shape[0] > 1 else x2.shape[1]


def linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None):
    """x W^T + b. Few-row bf16/fp16/fp32 problems run on the split-K MFMA
    kernel (pkv_linear); others on the library GEMM (F.linear)."""
    x2 = _as_rows(x)
    n = weight.shape[0]
    if not _linear_ok(x2, weight, bias, n):
        if _tiles_ok(x2, weight, bias):
            out = x.new_empty((x2.shape[0], n))
            _tiles(out, x2, weight, bias, n, _native.EPILOGUE_NONE, "linear")
            return out.view(*x.shape[:-1], n)
        return F.linear(x, weight, bias)
    out = x.new_empty((x2.shape[0], n))
    rc = _native.calls().pkv_linear(out.data_ptr(), x2.data_ptr(), weight.data_ptr(),
                                  _native.ptr(bias), x2.shape[0], n, x2.shape[1], _x_stride(x2),
                                  _native.dtype_code(x.dtype), _native.stream_ptr(x.device))
    _native.check(rc, "linear")
    return out.view(*x.shape[:-1], n)


def linear_swiglu(x: torch.Tensor, w_gate_up: torch.Tensor, b_gate_up: torch.Tensor | None):
    """silu(x Wg^T + bg) * (x Wu^T + bu) with W = [Wg; Wu] (models/mlp.py:24-30
    with the reference's fused_swiglu arithmetic)."""
    x2 = _as_rows(x)
    h = w_gate_up.shape[0] // 2
    if not _linear_ok(x2, w_gate_up, b_gate_up, 2 * h):
        if w_gate_up.shape[0] == 2 * h and _tiles_ok(x2, w_gate_up, b_gate_up, True):
            out = x.new_empty((x2.shape[0], h))
            _tiles(out, x2, w_gate_up, b_gate_up, h, _native.EPILOGUE_SWIGLU, "linear_swiglu")
            return out.view(*x.shape[:-1], h)
        gu = F.linear(x, w_gate_up, b_gate_up)
        return silu_mul(gu[..., :h], gu[..., h:])
    _native.require_device(x2, w_gate_up, what="linear_swiglu")
    out = x.new_empty((x2.shape[0], h))
    rc = _native.calls().pkv_linear_swiglu(
        out.data_ptr(), x2.data_ptr(), w_gate_up.data_ptr(), _native.ptr(b_gate_up),
        x2.shape[0], h, x2.shape[1], _x_stride(x2), _native.dtype_code(x.dtype),
        _native.stream_ptr(x.device))
    _native.check(rc, "linear_swiglu")
    return out.view(*x.shape[:-1], h)


def linear_rope_qkv(x: torch.Tensor, w_qkv: torch.Tensor, b_qkv: torch.Tensor | None,
                    positions: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, hq: int,
                    hkv: int, d: int):
    """q, k, v projections of x [T, d_model] with W = [Wq; Wk; Wv], q and k
    rotated at positions (fp32 tables cos / sin [max_pos, d/2]): contiguous
    q [T, hq, d], k [T, hkv, d], v [T, hkv, d] (serving/paged_mqa.py:76-85)."""
    x2 = _as_rows(x)
    T = x2.shape[0]
    nq, nk = hq * d, hkv * d
    few = _linear_ok(x2, w_qkv, b_qkv, nq + 2 * nk)
    if not few and not (_tiles_ok(x2, w_qkv, b_qkv, True) and w_qkv.shape[0] == nq + 2 * nk
                        and d % 2 == 0):
        qkv = F.linear(x2, w_qkv, b_qkv)
        return rope(qkv[:, :nq], qkv[:, nq:nq + nk], positions, cos, sin, v=qkv[:, nq + nk:],
                    hq=hq, hkv=hkv, d=d)
    _native.require_device(x2, w_qkv, positions, cos, sin, what="linear_rope_qkv")
    cos2, sin2, max_pos = _rope_tables(cos, sin, d, "linear_rope_qkv", not few)
    pos = positions if positions.dtype == torch.int32 else positions.to(torch.int32)
    pos = pos.contiguous()
    if pos.numel() != T:
        raise ValueError("linear_rope_qkv: positions and x disagree on the token count")
    q = x.new_empty((T, hq, d))
    k = x.new_empty((T, hkv, d))
    v = x.new_empty((T, hkv, d))
    fn = _native.calls().pkv_linear_rope_qkv if few else _native.calls().pkv_linear_tiles_rope_qkv
    rc = fn(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), x2.data_ptr(), w_qkv.data_ptr(),
        _native.ptr(b_qkv), T, x2.shape[1], _x_stride(x2), pos.data_ptr(), cos2.data_ptr(),
        sin2.data_ptr(), max_pos, hq, hkv, d, _native.dtype_code(x.dtype), None,
        _native.stream_ptr(x.device))
    _native.check(rc, "linear_rope_qkv")
    return q, k, v


# the projection kernels normalise rows of at most this many features in
# their prologue (pkv_linear_*_rmsnorm); wider rows take rms_norm first
LINEAR_NORM_MAX_K = 1024


def _norm_ok(x2: torch.Tensor, norm_weight: torch.Tensor) -> bool:
    return (x2.shape[1] <= LINEAR_NORM_MAX_K and norm_weight.dtype == x2.dtype
            and norm_weight.is_contiguous() and norm_weight.numel() == x2.shape[1]
            and norm_weight.data_ptr() % 16 == 0)


def _tiles_resid_fit(resid: torch.Tensor, x2: torch.Tensor, n: int) -> bool:
    """Whether the tile kernel may update resid in place where add_ did: an
    inference tensor outside inference mode is add_'s error."""
    return (resid.is_contiguous() and resid.dtype == x2.dtype and resid.device == x2.device
            and resid.numel() == x2.shape[0] * n
            and (not resid.is_inference() or torch.is_inference_mode_enabled())
            and not _transformed((resid,)) and not resid.is_neg()
            and resid.data_ptr() % 16 == 0)


def _apart(out: torch.Tensor, t) -> bool:
    """Whether the memory of t (None, or a tensor without negative strides) lies
    outside the contiguous out's: workgroups write out while others read t."""
    if t is None or t.numel() == 0:
        return True
    last = sum((n - 1) * s for n, s in zip(t.shape, t.stride()))
    a, b = out.data_ptr(), t.data_ptr()
    return (b + (last + 1) * t.element_size() <= a
            or a + out.numel() * out.element_size() <= b)


def linear_residual_(resid: torch.Tensor, x: torch.Tensor, weight: torch.Tensor,
                     bias: torch.Tensor | None = None) -> torch.Tensor:
    """resid += x W^T + b in place, the projection rounded to resid.dtype
    before the add (the residual adds of serving/paged_model.py:20-29, one
    kernel for the projection and the add). resid must be contiguous with
    x's rows. Returns resid."""
    x2 = _as_rows(x)
    n = weight.shape[0]
    if (not _linear_ok(x2, weight, bias, n) or not resid.is_contiguous() or not resid.is_cuda
            or resid.dtype != x.dtype or resid.numel() != x2.shape[0] * n):
        if (_tiles_resid_fit(resid, x2, n) and _tiles_ok(x2, weight, bias, True)
                and _apart(resid, x2) and _apart(resid, weight) and _apart(resid, bias)):
            _tiles(resid, x2, weight, bias, n, _native.EPILOGUE_RESIDUAL, "linear_residual_")
            # as add_ does: a graph that saved resid finds it changed
            torch.autograd.graph.increment_version(resid)
            return resid
        return resid.add_(linear(x, weight, bias).view(resid.shape))
    rc = _native.calls().pkv_linear_residual(
        resid.data_ptr(), x2.data_ptr(), weight.data_ptr(), _native.ptr(bias), x2.shape[0], n,
        x2.shape[1], _x_stride(x2), _native.dtype_code(x.dtype), _native.stream_ptr(x.device))
    _native.check(rc, "linear_residual_")
    return resid


def linear_swiglu_rmsnorm(x: torch.Tensor, norm_weight: torch.Tensor, eps: float,
                          w_gate_up: torch.Tensor, b_gate_up: torch.Tensor | None):
    """linear_swiglu(rms_norm(x, norm_weight, eps), ...) with the norm taken
    in the projection kernel's prologue (bit-identical to the two calls)."""
    x2 = _as_rows(x)
    h = w_gate_up.shape[0] // 2
    if not (_linear_ok(x2, w_gate_up, b_gate_up, 2 * h) and _norm_ok(x2, norm_weight)):
        return linear_swiglu(rms_norm(x, norm_weight, eps), w_gate_up, b_gate_up)
    _native.require_device(x2, norm_weight, w_gate_up, what="linear_swiglu_rmsnorm")
    out = x.new_empty((x2.shape[0], h))
    rc = _native.calls().pkv_linear_swiglu_rmsnorm(
        out.data_ptr(), x2.data_ptr(), norm_weight.data_ptr(), float(eps), w_gate_up.data_ptr(),
        _native.ptr(b_gate_up), x2.shape[0], h, x2.shape[1], _x_stride(x2),
        _native.dtype_code(x.dtype), _native.stream_ptr(x.device))
    _native.check(rc, "linear_swiglu_rmsnorm")
    return out.view(*x.shape[:-1], h)


def linear_rope_qkv_rmsnorm(x: torch.Tensor, norm_weight: torch.Tensor, eps: float,
                            w_qkv: torch.Tensor, b_qkv: torch.Tensor | None,
                            positions: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                            hq: int, hkv: int, d: int):
    """linear_rope_qkv(rms_norm(x, norm_weight, eps), ...) with the norm
    taken in the projection kernel's prologue (bit-identical to the two
    calls)."""
    x2 = _as_rows(x)
    T = x2.shape[0]
    nq, nk = hq * d, hkv * d
    if not (_linear_ok(x2, w_qkv, b_qkv, nq + 2 * nk) and _norm_ok(x2, norm_weight)):
        return linear_rope_qkv(rms_norm(x, norm_weight, eps), w_qkv, b_qkv, positions, cos, sin,
                               hq, hkv, d)
    _native.require_device(x2, norm_weight, w_qkv, positions, cos, sin,
                           what="linear_rope_qkv_rmsnorm")
    cos2, sin2, max_pos = _rope_tables(cos, sin, d, "linear_rope_qkv_rmsnorm", False)
    pos = positions if positions.dtype == torch.int32 else positions.to(torch.int32)
    pos = pos.contiguous()
    if pos.numel() != T:
        raise ValueError("linear_rope_qkv_rmsnorm: positions and x disagree on the token count")
    q = x.new_empty((T, hq, d))
    k = x.new_empty((T, hkv, d))
    v = x.new_empty((T, hkv, d))
    rc = _native.calls().pkv_linear_rope_qkv_rmsnorm(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), x2.data_ptr(), norm_weight.data_ptr(),
        float(eps), w_qkv.data_ptr(), _native.ptr(b_qkv), T, x2.shape[1], _x_stride(x2),
        pos.data_ptr(), cos2.data_ptr(), sin2.data_ptr(), max_pos, hq, hkv, d,
        _native.dtype_code(x.dtype), None, _native.stream_ptr(x.device))
    _native.check(rc, "linear_rope_qkv_rmsnorm")
    return q, k, v


def argmax_rows(logits: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """Index of the largest logit of every row of [rows, vocab] logits as
    int64 [rows] (pkv_argmax_rows; the framework's argmax result: first
    maximum, NaN above every number). With `out`, the ids are written there
    (an int64 device tensor of rows elements)."""
    _native.require_device(logits, what="argmax_rows")
    if logits.dim() != 2:
        raise ValueError(f"argmax_rows: expected [rows, vocab], got {tuple(logits.shape)}")
    lg = logits if logits.stride(1) == 1 else logits.contiguous()
    rows, vocab = lg.shape
    if out is None:
        out = torch.empty(rows, dtype=torch.long, device=logits.device)
    elif (out.dtype != torch.long or out.numel() != rows or not out.is_contiguous()
          or out.device != logits.device):
        raise ValueError("argmax_rows: out must be a contiguous int64 tensor of rows elements")
    stride = lg.stride(0) if rows > 1 else vocab
    ws, wsb = _argmax_workspace(lg)
    rc = _native.calls().pkv_argmax_rows(out.data_ptr(), lg.data_ptr(), rows, vocab, stride,
                                       _native.dtype_code(lg.dtype), _native.ptr(ws), wsb,
                                       _native.stream_ptr(logits.device))
    _native.check(rc, "argmax_rows")
    return out


def _argmax_workspace(lg):
    """The split-row argmax's counters and key words: the "argmax" slot of
    the current workspace (a graph step's own workspace under its scope)."""
    rows, vocab = lg.shape
    wsb = int(_native.calls().pkv_argmax_workspace_bytes(rows, vocab, _native.dtype_code(lg.dtype)))
    if wsb == 0:
        return None, 0
    return _native.current_workspace().get(lg.device, wsb, slot="argmax"), wsb


def sample_rows(logits: torch.Tensor, temperature: float, top_k: int, top_p: float,
                uniforms: torch.Tensor):
    """One draw per row of [rows, vocab] logits with temperature, top-k
    (1..64, ties at the threshold kept) and top-p, by inverse CDF at the
    row's uniform in [0, 1) (pkv_sample_rows). Returns (ids int64 [rows],
    status int32 [1]: PKV_STATUS_* bits; a flagged row's id is -1)."""
    _native.require_device(logits, uniforms, what="sample_rows")
    if logits.dim() != 2:
        raise ValueError(f"sample_rows: expected [rows, vocab], got {tuple(logits.shape)}")
    lg = logits if logits.stride(1) == 1 else logits.contiguous()
    rows, vocab = lg.shape
    u = uniforms.to(torch.float32).contiguous()
    if u.numel() != rows:
        raise ValueError("sample_rows: one uniform per row")
    ids = torch.empty(rows, dtype=torch.long, device=logits.device)
    status = torch.zeros(1, dtype=torch.int32, device=logits.device)
    stride = lg.stride(0) if rows > 1 else vocab
    rc = _native.calls().pkv_sample_rows(ids.data_ptr(), lg.data_ptr(), rows, vocab, stride,
                                       float(temperature), int(top_k), float(top_p),
                                       u.data_ptr(), _native.dtype_code(lg.dtype),
                                       status.data_ptr(), _native.stream_ptr(logits.device))
    _native.check(rc, "sample_rows")
    return ids, status


# module classes known to have no class attribute in the place of a parameter,
# buffer or submodule (a subclass may, and is read by its own rules)
PLAIN_MODULES = {torch.nn.Linear}


def module_attr(mod, name: str):
    """mod.<name> for a parameter, buffer or submodule. Of PLAIN_MODULES it is
    read from its dict where it is there: nn.Module's own lookup goes through a
    failed attribute access first (0.25 us each, some thirty a layer)."""
    if type(mod) in PLAIN_MODULES:
        own = mod.__dict__
        d = own["_parameters"]
        if name in d:
            return d[name]
        d = own["_modules"]
        if name in d:
            return d[name]
        d = own["_buffers"]
        if name in d:
            return d[name]
    return getattr(mod, name)


class FusedRows:
    """Row-concatenated weights (and biases) of several nn.Linear modules
    sharing an input, so one GEMM computes all of their outputs. The
    modules' parameters are re-pointed to views of the concatenation, so
    they stay the state-dict entries, in-place updates (load_state_dict,
    optimiser steps) reach the fused storage, and no copy is kept. When a
    parameter has been replaced (module.to(...), assignment) the
    concatenation is rebuilt on the next call."""

    def __init__(self, *linears: torch.nn.Linear):
        self.linears = linears
        self.weight = None
        self.bias = None

    def _views_intact(self) -> bool:
        if self.weight is None:
            return False
        off = 0
        base = self.weight.data_ptr()
        es = self.weight.element_size()
        dev, dt = self.weight.device, self.weight.dtype
        for lin in self.linears:
            w = module_attr(lin, "weight")
            if (w.device != dev or w.dtype != dt
                    or w.data_ptr() != base + off * es or not w.is_contiguous()):
                return False
            off += w.numel()
        if self.bias is not None:
            off, base, es = 0, self.bias.data_ptr(), self.bias.element_size()
            for lin in self.linears:
                b = module_attr(lin, "bias")
                if b is None or b.data_ptr() != base + off * es or b.dtype != self.bias.dtype:
                    return False
                off += b.numel()
        elif any(module_attr(lin, "bias") is not None for lin in self.linears):
            return False
        return True

    def get(self):
        """(weight [sum(out), in], bias or None) of the concatenation."""
        if not self._views_intact():
            with torch.no_grad():
                w = torch.cat([lin.weight.detach() for lin in self.linears], 0)
                has_b = [lin.bias is not None for lin in self.linears]
                if any(has_b) and not all(has_b):
                    raise ValueError("FusedRows: either every linear has a bias or none")
                b = (torch.cat([lin.bias.detach() for lin in self.linears], 0)
                     if all(has_b) else None)
                off = 0
                for lin in self.linears:
                    n = lin.weight.shape[0]
                    lin.weight.data = w[off:off + n]
                    if b is not None:
                        lin.bias.data = b[off:off + n]
                    off += n
            self.weight, self.bias = w, b
        return self.weight, self.bias
