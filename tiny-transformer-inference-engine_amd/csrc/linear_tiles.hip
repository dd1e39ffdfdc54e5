// Projections of many fp32 rows (prefill), y = x W^T (+ bias), on
// v_mfma_f32_16x16x4_f32, with the element-wise op that follows the projection
// in a decoder block as the epilogue: plain, SwiGLU, q/k/v RoPE or the residual
// add, the same arithmetic as the few-row projections' (linear.hip).
//
// What bounds it: the fp32 matrix pipe (155 TFLOP/s on this machine), which
// vector instructions of the same SIMD overlap little; at k = 512 it is busy for
// little more than half the time (gate/up of 2481 rows: 89 TFLOP/s with 97% of
// the places in five rounds of workgroups filled), the rest is each workgroup's
// first round trips, its epilogue and the fragment reads. A workgroup owns 64
// rows x 32 (or 64) weight rows; k is walked in slabs of 32, loaded in whole
// 128-byte lines through buffer resources whose scalar offset moves along k (no
// address arithmetic in the loop), four slabs ahead in registers, staged in two
// LDS buffers, one barrier a slab. One slab ahead covered 512 to 1024 cycles of
// matrix work against a longer round trip to memory: at 2146 rows x 1024 the
// three fused forms took 191 us together, then 171; at 512 66 and 60. (Operands
// loaded straight from memory in matrix layout, without LDS, took 1.5 times as
// long: sixteen 16-byte pieces of sixteen lines per instruction fill the L1.
// Slabs of 64, and LDS padding that bounds the workgroups per CU, measured the
// same.)
// Measured for a layer of 2481 rows (eight prompts), 512 wide, GPU time of the
// library GEMM with its separate element-wise kernel against this one, us:
// q/k/v + RoPE 25.4 / 22.9, gate/up + SwiGLU 46.8 / 29.3, out + residual 19.0 /
// 18.7; 4096 rows x 1024: 98.9 / 83.0, 134 / 133 (129 TFLOP/s), 73.4 / 70.7. The
// callers' size rule (serving/fused_ops.py) has the other side.
#include "mfma_decode_common.h"

namespace pkv {
namespace {

using namespace mfma;

enum { kTilePlain = 0, kTileSwiglu = 1, kTileRope = 2, kTileResid = 3 };

struct TileArgs {
  float* out;  // plain / swiglu / resid: [m, n] contiguous
  const float* x;
  const float* w;
  const float* bias;  // nullable, one per weight row
  unsigned x_stride;
  int m;
  int n;  // output features (swiglu: per half)
  int k;
  // rope epilogue
  float* q_out;
  float* k_out;
  float* v_out;
  const int32_t* positions;
  const float* cos;
  const float* sin;
  int max_pos;
  int qn;  // hq * d
  int kn;  // hkv * d
  int d;
  int* status;
};

constexpr int kSlab = 32;          // k per staged slab
constexpr int kAhead = 4;          // slabs in flight; even: slab s sits in LDS buffer s % 2
constexpr int kSPitch = kSlab + 4;  // floats: 16 rows of one fragment read hit distinct banks

template <int EPI, int XM>
__global__ __launch_bounds__(256, 3) void linear_tiles_kernel(TileArgs a) {
#pragma clang fp contract(off)
  constexpr int WM = XM == 2 ? 2 : 4;  // wavefronts along the rows
  constexpr int WN = 4 / WM;           // and along the weight rows
  constexpr int ROWS = 16 * XM * WM;   // 64
  constexpr int LROWS = ROWS + 32 * WN;
  constexpr int NL = LROWS / 32;       // 16-byte pieces per thread and slab
  constexpr int FW = EPI == kTileSwiglu ? 16 : 32;  // output features per wavefront
  __shared__ __attribute__((aligned(16))) float lds[2][LROWS * kSPitch];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane >> 4;
  const int l16 = lane & 15;
  const int wm = w % WM;
  const int wn = w / WM;
  const int mb = (int)blockIdx.x * ROWS;
  const int m0 = mb + 16 * XM * wm;
  const int f0 = ((int)blockIdx.y * WN + wn) * FW;

  // This thread's pieces of a slab: staged rows tid / 8 + 32 j (the x rows,
  // then 32 weight rows per wavefront column), 16 bytes at 4 (tid % 8). Rows
  // past the end re-read the last one (their results are not stored).
  unsigned off[NL];
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int r = tid / 8 + 32 * j;
    if (32 * j < ROWS) {
      off[j] = ((unsigned)min(mb + r, a.m - 1) * a.x_stride + 4 * (tid % 8)) * 4;
    } else {
      const int q = r - ROWS;
      const int c = (int)blockIdx.y * WN + q / 32;
      const int f = EPI == kTileSwiglu ? min(c * 16 + q % 16, a.n - 1) + (q % 32) / 16 * a.n
                                       : min(c * 32 + q % 32, a.n - 1);
      off[j] = ((unsigned)f * (unsigned)a.k + 4 * (tid % 8)) * 4;
    }
  }
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.x), (short)0, -1, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.w), (short)0, -1, kRsrcWord3);
  floatx4 g[kAhead][NL];  // the slabs in flight
  auto fetch = [&](floatx4 (&r)[NL], int slab) {
#pragma unroll
    for (int j = 0; j < NL; ++j)
      r[j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                             32 * j < ROWS ? xr : wr, off[j], slab * 128, 0));
  };
  auto stage = [&](const floatx4 (&r)[NL], int b) {
#pragma unroll
    for (int j = 0; j < NL; ++j)
      *reinterpret_cast<floatx4*>(&lds[b][(tid / 8 + 32 * j) * kSPitch + 4 * (tid % 8)]) = r[j];
  };

  floatx4 acc[2][XM];  // [weight tile][row tile]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < XM; ++t) acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int slabs = a.k / kSlab;
  auto multiply = [&](int b) {
    const float* xl = &lds[b][(16 * XM * wm + l16) * kSPitch + 4 * grp];
    const float* wl = &lds[b][(ROWS + 32 * wn + l16) * kSPitch + 4 * grp];
    // product e of half h takes k = 16 h + 4 grp + e of every lane's row
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      floatx4 xf[XM], wf[2];
#pragma unroll
      for (int t = 0; t < XM; ++t)
        xf[t] = *reinterpret_cast<const floatx4*>(xl + 16 * t * kSPitch + 16 * h);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        wf[i] = *reinterpret_cast<const floatx4*>(wl + 16 * i * kSPitch + 16 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < XM; ++t)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][e], xf[t][e], acc[i][t], 0, 0, 0);
    }
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(g[i], min(i, slabs - 1));
  stage(g[0], 0);
  __syncthreads();
  // Whole rounds of kAhead slabs have no branch, which keeps the wait counts
  // exact: slab s + 1 is waited for with kAhead - 2 younger ones in flight.
  // Past the last slab its loads repeat, and what they stage is not read.
  int s = 0;
  for (; s + kAhead <= slabs; s += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      fetch(g[i], min(s + i + kAhead, slabs - 1));
      multiply(i & 1);
      stage(g[(i + 1) % kAhead], (i + 1) & 1);  // its readers passed the previous barrier
      __syncthreads();
    }
  }
#pragma unroll
  for (int i = 0; i < kAhead - 1; ++i) {
    if (s + i >= slabs) break;
    multiply(i & 1);
    stage(g[i + 1], (i + 1) & 1);
    __syncthreads();
  }

  // lane: rows m0 + 16 t + l16, features f0 + 16 i + 4 grp + 0..3 (swiglu:
  // features f0 + 4 grp + 0..3, gate in tile 0 and up in tile 1)
  const bool quad = (a.n & 3) == 0;  // 16-byte rows: whole quads, aligned
#pragma unroll
  for (int t = 0; t < XM; ++t) {
    const int m = m0 + 16 * t + l16;
    if (m >= a.m) continue;
    int pos = 0;
    bool bad_pos = false;
    if constexpr (EPI == kTileRope) {
      pos = a.positions[m];
      bad_pos = (unsigned)pos >= (unsigned)a.max_pos;
      if (bad_pos) pos = 0;
    }
#pragma unroll
    for (int i = 0; i < (EPI == kTileSwiglu ? 1 : 2); ++i) {
      const int f = f0 + 16 * i + 4 * grp;
      if (f >= a.n) continue;
      floatx4 y = acc[i][t];
      floatx4 u = acc[1][t];
      if (a.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int fe = min(f + e, a.n - 1);
          y[e] = y[e] + a.bias[fe];
          if constexpr (EPI == kTileSwiglu) u[e] = u[e] + a.bias[a.n + fe];
        }
      }
      if constexpr (EPI == kTileRope) {
        // every region ([q | k | v], d even) starts at an even feature: the
        // pairs (f, f + 1) and (f + 2, f + 3) are rotation pairs of one head
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int n = f + 2 * h;
          if (n >= a.n) continue;
          const float xe = y[2 * h];
          const float xd = y[2 * h + 1];
          float* o;
          float r0 = xe, r1 = xd;
          if (n < a.qn + a.kn) {
            const int c = (n < a.qn ? n : n - a.qn) % a.d;
            const int64_t tix = (int64_t)pos * (a.d >> 1) + (c >> 1);
            const float cj = a.cos[tix];
            const float sj = a.sin[tix];
            if (bad_pos && a.status && n == 0) atomicOr(a.status, PKV_STATUS_BAD_POS);
            r0 = fp32_value(xe * cj) - fp32_value(xd * sj);
            r1 = fp32_value(xe * sj) + fp32_value(xd * cj);
            o = n < a.qn ? a.q_out + (int64_t)m * a.qn + n
                         : a.k_out + (int64_t)m * a.kn + (n - a.qn);
          } else {
            o = a.v_out + (int64_t)m * a.kn + (n - a.qn - a.kn);
          }
          o[0] = r0;
          o[1] = r1;
        }
      } else {
        if constexpr (EPI == kTileSwiglu) {
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = swiglu_gate(y[e], u[e]);
        }
        float* o = a.out + (int64_t)m * a.n + f;
        if (quad) {
          if constexpr (EPI == kTileResid) y = *reinterpret_cast<const floatx4*>(o) + y;
          *reinterpret_cast<floatx4*>(o) = y;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (f + e < a.n) o[e] = EPI == kTileResid ? o[e] + y[e] : y[e];
        }
      }
    }
  }
}

// A workgroup owns 64 rows x 32 weight rows, or x 64 (the sum order is the same):
// a round of wide tiles over the CUs takes as long as 1.9 narrow ones, so wide ones
// run where their rounds cost less, but not below two and a half, where the
// emptier CUs count more than the fewer operand loads. Wide / narrow, us: 1025
// rows x 512, k 512 14.2 / 13.0; 1400 x 4096, k 1024 102 / 95; 3000 x 1024, k 1024
// 55.5 / 60.9; 2481 x 8192, k 1024 328 / 403. Over 330 shapes of 257-8192 rows
// this costs 0.25% on average against the better one of the two.
template <int EPI>
int launch(const TileArgs& a, int64_t weight_rows, hipStream_t stream) {
  const int64_t cus = device_cu_count();
  auto up = [](int64_t x, int64_t y) { return (x + y - 1) / y; };
  const int64_t mt = up(a.m, 64);
  const int64_t wides = mt * up(weight_rows, 64);
  const bool wide = 2 * wides >= 5 * cus &&
                    15 * up(wides, cus) <= 8 * up(mt * up(weight_rows, 32), cus);
  const int64_t ny = up(weight_rows, wide ? 64 : 32);
  if (ny > 65535) return fail(PKV_ERR_UNSUPPORTED, "linear_tiles: %lld tiles", (long long)ny);
  const dim3 grid((unsigned)mt, (unsigned)ny);
  if (wide)
    hipLaunchKernelGGL((linear_tiles_kernel<EPI, 2>), grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((linear_tiles_kernel<EPI, 1>), grid, dim3(256), 0, stream, a);
  return check_launch("linear_tiles_kernel");
}

int check(const void* out, const void* x, const void* w, int64_t m, int64_t weight_rows, int64_t k,
          int64_t x_stride, int dtype) {
  if (dtype != PKV_DTYPE_F32)
    return fail(PKV_ERR_UNSUPPORTED, "linear_tiles: dtype %d (fp32 only)", dtype);
  if (m < 0 || weight_rows <= 0 || k <= 0 || x_stride < k)
    return fail(PKV_ERR_INVALID, "linear_tiles: bad sizes m=%lld rows=%lld k=%lld stride=%lld",
                (long long)m, (long long)weight_rows, (long long)k, (long long)x_stride);
  if (!out || !x || !w) return fail(PKV_ERR_INVALID, "linear_tiles: null pointer argument");
  if (k % 32 != 0 || x_stride % 4 != 0 || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) ||
      ((uintptr_t)out & 15))
    return fail(PKV_ERR_UNSUPPORTED,
                "linear_tiles: k (%lld) must be a multiple of 32, x rows, weights and out "
                "16-byte aligned", (long long)k);
  // operands are addressed by 32-bit byte offsets
  if (m > (1 << 29) || weight_rows > (1 << 29) || m * x_stride >= (1 << 29) ||
      weight_rows * k >= (1 << 29))
    return fail(PKV_ERR_UNSUPPORTED, "linear_tiles: operand of 2 GiB or more");
  return PKV_OK;
}

TileArgs args(const void* x, const void* w, const void* bias, int64_t m, int64_t n, int64_t k,
              int64_t x_stride) {
  TileArgs a{};
  a.x = static_cast<const float*>(x);
  a.w = static_cast<const float*>(w);
  a.bias = static_cast<const float*>(bias);
  a.x_stride = (unsigned)x_stride;
  a.m = (int)m;
  a.n = (int)n;
  a.k = (int)k;
  return a;
}

}  // namespace
}  // namespace pkv

using namespace pkv;

extern "C" {

int pkv_linear_tiles(void* out, const void* x, const void* w, const void* bias, int64_t m,
                     int64_t n, int64_t k, int64_t x_stride, int epilogue, int dtype,
                     void* stream) {
  const int64_t rows = epilogue == PKV_EPILOGUE_SWIGLU ? 2 * n : n;
  const int rc = check(out, x, w, m, rows, k, x_stride, dtype);
  if (rc != PKV_OK || m == 0) return rc;
  TileArgs a = args(x, w, bias, m, n, k, x_stride);
  a.out = static_cast<float*>(out);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (epilogue == PKV_EPILOGUE_NONE) return launch<kTilePlain>(a, rows, st);
  if (epilogue == PKV_EPILOGUE_SWIGLU) return launch<kTileSwiglu>(a, rows, st);
  if (epilogue == PKV_EPILOGUE_RESIDUAL) return launch<kTileResid>(a, rows, st);
  return fail(PKV_ERR_INVALID, "linear_tiles: epilogue %d", epilogue);
}

int pkv_linear_tiles_rope_qkv(void* q_out, void* k_out, void* v_out, const void* x,
                              const void* w_qkv, const void* bias, int64_t m, int64_t k,
                              int64_t x_stride, const int32_t* positions,
                              const float* cos_table, const float* sin_table, int max_pos, int hq,
                              int hkv, int d, int dtype, int* status, void* stream) {
  if (hq <= 0 || hkv <= 0 || d <= 0 || (d & 1) || max_pos <= 0)
    return fail(PKV_ERR_INVALID, "linear_tiles_rope_qkv: bad sizes hq=%d hkv=%d d=%d max_pos=%d",
                hq, hkv, d, max_pos);
  const int64_t n = ((int64_t)hq + 2 * (int64_t)hkv) * d;
  const int rc = check(q_out, x, w_qkv, m, n, k, x_stride, dtype);
  if (rc != PKV_OK) return rc;
  if (!k_out || !v_out || !positions || !cos_table || !sin_table)
    return fail(PKV_ERR_INVALID, "linear_tiles_rope_qkv: null pointer argument");
  if (m == 0) return PKV_OK;
  TileArgs a = args(x, w_qkv, bias, m, n, k, x_stride);
  a.q_out = static_cast<float*>(q_out);
  a.k_out = static_cast<float*>(k_out);
  a.v_out = static_cast<float*>(v_out);
  a.positions = positions;
  a.cos = cos_table;
  a.sin = sin_table;
  a.max_pos = max_pos;
  a.qn = hq * d;
  a.kn = hkv * d;
  a.d = d;
  a.status = status;
  return launch<kTileRope>(a, n, static_cast<hipStream_t>(stream));
}

}  // extern "C"
