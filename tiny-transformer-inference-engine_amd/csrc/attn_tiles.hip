// Paged attention over tiles of (query token, head) rows on the fp32 matrix
// cores: the shapes the 16-head MFMA kernels do not take. That is prefill and
// mixed batches with fewer than 16 query heads per kv head or in fp32 (the
// default model: 8 heads of 64, fp32), and decode with group sizes the
// small-group kernel has no form for. Any group size, head dim 32 / 64 /
// 128, fp32 / bf16 / fp16 pools. Semantics are those of pagedattn.forward
// (kernels/pagedattn/pagedattn.cu:142-447), see attention.hip.
//
// Precision. Every operand is fp32: 16-bit values are widened exactly in
// registers, the products and sums are v_mfma_f32_16x16x4_f32's (fp32 fused
// multiply-adds), and the probabilities stay fp32, as in the row kernel this
// one stands in for.
//
// Work split. A workgroup owns 32 rows (NT = 2 MFMA tiles of 16, so each K and
// V^T operand feeds two products) or 16 of one (sequence, kv head), held by
// every wavefront, and its 4 wavefronts share the keys: wavefront w takes
// chunks w, w + 4, ... of C tokens, so no barrier sits in the chunk loop and
// the longest causal row of a prompt is a chain a quarter as long as with one
// wavefront per row tile. The four online-softmax states are combined through
// LDS at the end, in wavefront order.
//
// Operands straight from the pool. S^T = K Q^T wants, per lane, dims of one
// token (A: token l % 16, k-group l / 16), and O^T += V^T P^T one token's value
// of dim row l % 16 of each 16-row tile dt. Which dims the k-groups and which
// dims the rows (dt, l % 16) stand for is free, so they are chosen to make a
// lane's values contiguous: k-group g of step pair kp holds dims
// 32 kp + 8 g ... + 7, and row (dt, m) is dim DT m + dt. A lane then loads its
// operands with whole 8 to 32-byte pieces, sixteen lanes cover a V row, four
// lanes 64 or 128 bytes of a K row, and K and V need no LDS: the registers that
// hold the loads in flight are the operands. K of the next chunk is requested
// when the scores are done, V when its products are.
//
// What bounds it: the fp32 matrix pipe and, on short prompts, the dependent
// round trips ahead of the first chunk (length, table, rows).
#include "mfma_decode_common.h"

#include <type_traits>

namespace pkv {
namespace {

using namespace mfma;

constexpr int kTW = 4;             // wavefronts per workgroup
constexpr int kTBlock = 64 * kTW;  // threads
constexpr int kCuLds = 160 * 1024;  // LDS of a CU
static_assert(kTBlock == kTblCap, "one table entry per thread and window");

template <int D>
struct TileGeo {
  static constexpr int C = D == 32 ? 32 : 16;   // tokens per chunk
  static constexpr int HT = C / 16;             // 16-token MFMA tiles
  static constexpr int KP = D / 32;             // 32-dim step pairs
  static constexpr int DT = D / 16;             // 16-dim output tiles
  static constexpr int PITCH = D + 4;           // floats per staged output row
};

// N values of T as loaded (N * sizeof(T) bytes), and their fp32 values.
template <typename T, int N>
struct Piece {
  static constexpr int W = N * (int)sizeof(T) / 4;  // 32-bit words
  unsigned w[W];
  __device__ __forceinline__ void load(const char* p) {
    if constexpr (W == 1) {
      w[0] = *reinterpret_cast<const unsigned*>(p);
    } else if constexpr (W == 2) {
      const u32x2 x = *reinterpret_cast<const u32x2*>(p);
      w[0] = x[0];
      w[1] = x[1];
    } else {
#pragma unroll
      for (int i = 0; i < W; i += 4) {
        const u32x4 x = *reinterpret_cast<const u32x4*>(p + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[i + e] = x[e];
      }
    }
  }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, unsigned off) {
    if constexpr (W == 1) {
      w[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0);
    } else if constexpr (W == 2) {
      const u32x2 x =
          __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
      w[0] = x[0];
      w[1] = x[1];
    } else {
#pragma unroll
      for (int i = 0; i < W; i += 4) {
        const u32x4 x = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 4 * i, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) w[i + e] = x[e];
      }
    }
  }
  __device__ __forceinline__ void keep_if(bool ok) {
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = ok ? w[i] : 0u;
  }
  __device__ __forceinline__ float get(int i) const {
    if constexpr (sizeof(T) == 4) {
      return __uint_as_float(w[i]);
    } else {
      const unsigned short h = (unsigned short)(w[i / 2] >> (16 * (i % 2)));
      return (float)__builtin_bit_cast(T, h);
    }
  }
};
// Keys [kv_lo, kv_hi) of one (sequence, kv head) for the first N of NT row tiles:
// this wavefront's chunks into st. tfirst: this thread's entry of the first
// table window; whole_lim: keys every row of the tile sees. Returns whether a
// table entry was outside the pool.
//
// WHOLE (block size >= 16: each 16-token tile of a chunk lies in one block):
// the tile is read through a buffer resource of its own, base its first row
// and size its rows below kv_hi (0 for a bad table entry), so rows that do not
// exist read as zeros and every lane's offsets are the same for every tile.
// The addresses are then scalar work, which matters here: fp32 matrix and vector
// instructions of one SIMD overlap little on this machine (a loop of both takes
// 82 to 88% of the sum of the two alone, 1 to 4 wavefronts), so the per-row
// addresses cost 1.6 us of every 3.1 us step. Smaller blocks keep them.
template <typename T, int D, int NT, int N, bool WHOLE>
__device__ __forceinline__ bool tile_chunks(const AttnArgs& a, const int32_t* __restrict__ table,
                                            int tfirst, int kvh, int kv_lo, int kv_hi, int whole_lim,
                                            const int (&lim)[NT],
                                            const float (&qf)[NT][D / 32][8],
                                            WaveState<NT, D / 16>& st, int* tbl, int w,
                                            int tid) {
  using Geo = TileGeo<D>;
  constexpr int C = Geo::C;
  constexpr int HT = Geo::HT;
  constexpr int KP = Geo::KP;
  constexpr int DT = Geo::DT;
  constexpr int ES = (int)sizeof(T);
  const int lane = tid & 63;
  const int grp = lane >> 4;
  const int l16 = lane & 15;
  const int64_t row_stride = (int64_t)a.hkv * D * ES;
  const char* kbase = static_cast<const char*>(a.k_pool) + ((int64_t)kvh * D + 8 * grp) * ES;
  const char* vbase = static_cast<const char*>(a.v_pool) + ((int64_t)kvh * D + DT * l16) * ES;
  const int bs_mask = (1 << a.bs_shift) - 1;
  // WHOLE: this lane's offsets in a 16-token tile
  const unsigned koff = (unsigned)l16 * (unsigned)row_stride + 8 * grp * ES;
  const unsigned voff = 4 * grp * (unsigned)row_stride + DT * l16 * ES;
  const float sc = a.scale_log2;
  bool bad_block = false;

  // kTblCap - 1 blocks of tokens per window: one that starts inside a block
  // still touches at most kTblCap table entries. In whole chunks, so that a
  // chunk reaches past its window's end only where that is kv_hi: scores are
  // masked from lim (<= kv_hi) on, and a chunk across an inner window end would
  // leave the next window's tokens in twice (block sizes below 16, and 32-token
  // chunks with blocks of 16). Blocks past 2^20 tokens take smaller windows.
  const int win = ((kTblCap - 1) << min(a.bs_shift, 20)) & ~(C - 1);
  static_assert((C & (C - 1)) == 0 && C < kTblCap && kChunk % C == 0,
                "windows and partitions start at whole chunks");
  for (int lo = kv_lo; lo < kv_hi; lo += win) {
    const int hi = min(lo + win, kv_hi);
    const int blk_lo = lo >> a.bs_shift;
    const int nblk = ((hi - 1) >> a.bs_shift) + 1 - blk_lo;
    __syncthreads();  // the previous window's entries are no longer read
    if (tid < nblk) tbl[tid] = lo == kv_lo ? tfirst : table[blk_lo + tid];
    __syncthreads();
    const int nch = (hi - lo + C - 1) / C;

    // Rows past hi re-read the window's last row (hi is kv_hi then, see win:
    // their scores are masked);
    // rows whose table entry is outside the pool read block 0 and are zeroed
    // before use. off: byte offset of position pos's row.
    auto row_off = [&](int pos, bool& ok) {
      pos = min(pos, hi - 1);
      const int phys = tbl[(pos >> a.bs_shift) - blk_lo];
      ok = phys >= 0 && phys < a.num_blocks;
      return (((int64_t)(ok ? phys : 0) << a.bs_shift) + (pos & bs_mask)) * row_stride;
    };
    Piece<T, 8> kr[HT][KP];
    Piece<T, DT> vr[HT][4];
    unsigned bad_k = 0, bad_v = 0;
    // WHOLE: the table entries of the chunk to request next (read from LDS a
    // chunk ahead), and the resource of tile h of chunk c
    int ent[HT];
    auto read_ent = [&](int c) {
#pragma unroll
      for (int h = 0; h < HT; ++h)
        ent[h] = tbl[(min(lo + c * C + 16 * h, hi - 1) >> a.bs_shift) - blk_lo];
    };
    auto tile_rsrc = [&](const void* pool, int c, int h) {
      const int pos = lo + c * C + 16 * h;
      const int phys = __builtin_amdgcn_readfirstlane(ent[h]);
      const bool ok = phys >= 0 && phys < a.num_blocks;
      bad_block |= !ok;
      const int rows = min(16, hi - pos);
      const int64_t base =
          (((int64_t)(ok ? phys : 0) << a.bs_shift) + (pos & bs_mask)) * row_stride +
          (int64_t)kvh * D * ES;
      const int extent = ok && rows > 0 ? (rows - 1) * (int)row_stride + D * ES : 0;
      return __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char*>(static_cast<const char*>(pool) + base), (short)0, extent,
          kRsrcWord3);
    };
    auto load_k = [&](int c) {
      if constexpr (WHOLE) {
#pragma unroll
        for (int h = 0; h < HT; ++h) {
          const __amdgpu_buffer_rsrc_t rs = tile_rsrc(a.k_pool, c, h);
#pragma unroll
          for (int kp = 0; kp < KP; ++kp) kr[h][kp].load(rs, koff + 32 * kp * ES);
        }
        return;
      }
      bad_k = 0;
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        bool ok;
        const char* p = kbase + row_off(lo + c * C + 16 * h + l16, ok);
        bad_k |= (unsigned)!ok << h;
#pragma unroll
        for (int kp = 0; kp < KP; ++kp) kr[h][kp].load(p + 32 * kp * ES);
      }
    };
    auto load_v = [&](int c) {
      if constexpr (WHOLE) {
#pragma unroll
        for (int h = 0; h < HT; ++h) {
          const __amdgpu_buffer_rsrc_t rs = tile_rsrc(a.v_pool, c, h);
#pragma unroll
          for (int j = 0; j < 4; ++j) vr[h][j].load(rs, voff + j * (unsigned)row_stride);
        }
        read_ent(c + kTW);
        return;
      }
      bad_v = 0;
#pragma unroll
      for (int h = 0; h < HT; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          bool ok;
          const char* p = vbase + row_off(lo + c * C + 16 * h + 4 * grp + j, ok);
          bad_v |= (unsigned)!ok << (4 * h + j);
          vr[h][j].load(p);
        }
    };
    // one chunk; MORE: the wavefront's next one is requested, K when the
    // scores are done and V when its products are, in that order, so that the
    // waits count exactly the loads issued after the ones they need (a branch
    // around the requests made every wait drain all of them)
    auto step = [&](int c, auto more) {
      constexpr bool MORE = decltype(more)::value;
      if (!WHOLE && __builtin_amdgcn_ballot_w64(bad_k != 0) != 0) {
        bad_block = true;
#pragma unroll
        for (int h = 0; h < HT; ++h)
#pragma unroll
          for (int kp = 0; kp < KP; ++kp) kr[h][kp].keep_if(!((bad_k >> h) & 1));
      }
      // S^T = K Q^T: product j of step pair kp takes dim 32 kp + 8 grp + j of
      // every lane's token / row
      floatx4 sacc[N][HT];
#pragma unroll
      for (int nt = 0; nt < N; ++nt)
#pragma unroll
        for (int h = 0; h < HT; ++h) sacc[nt][h] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kp = 0; kp < KP; ++kp)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int h = 0; h < HT; ++h) {
            const float kf = kr[h][kp].get(j);
#pragma unroll
            for (int nt = 0; nt < N; ++nt)
              sacc[nt][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf, qf[nt][kp][j], sacc[nt][h],
                                                                 0, 0, 0);
          }
      if constexpr (MORE) load_k(c + kTW);

      // online softmax in base 2 with a lazily moved reference, as in
      // chunk_update_sub (mfma_decode_common.h): the scale is applied inside
      // the exponent's fma
      const int cb = lo + c * C;
      if (cb + C > whole_lim) {  // uniform: some row does not see the whole chunk
#pragma unroll
        for (int nt = 0; nt < N; ++nt) {
          const int left = lim[nt] - cb - 4 * grp;
#pragma unroll
          for (int h = 0; h < HT; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (16 * h + j >= left) sacc[nt][h][j] = -INFINITY;
        }
      }
      bool move = false;
#pragma unroll
      for (int nt = 0; nt < N; ++nt) {
        float mx = -INFINITY;
#pragma unroll
        for (int h = 0; h < HT; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) mx = fmaxf(mx, sacc[nt][h][j]);
        move |= mx * sc > st.m[nt] + kLazy;
      }
      if (__builtin_amdgcn_ballot_w64(move) != 0) {
#pragma unroll
        for (int nt = 0; nt < N; ++nt) {
          float mx = -INFINITY;
#pragma unroll
          for (int h = 0; h < HT; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) mx = fmaxf(mx, sacc[nt][h][j]);
          mx = head_lanes_max(mx) * sc;
          const float m_new = fmaxf(st.m[nt], mx);
          const float alpha = m_new == -INFINITY ? 1.f : exp2_fast(st.m[nt] - m_new);
          st.l[nt] *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) st.o[nt][dt] *= alpha;
          st.m[nt] = m_new;
        }
      }
#pragma unroll
      for (int nt = 0; nt < N; ++nt) {
        const float nref = st.m[nt] == -INFINITY ? 0.f : -st.m[nt];
        float ps = 0.f;
#pragma unroll
        for (int h = 0; h < HT; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            sacc[nt][h][j] = exp2_fast(__builtin_fmaf(sacc[nt][h][j], sc, nref));
            ps += sacc[nt][h][j];
          }
        st.l[nt] += ps;
      }

      // O^T += V^T P^T: product (h, j) takes token 16 h + 4 grp + j of every lane
      if (!WHOLE && __builtin_amdgcn_ballot_w64(bad_v != 0) != 0) {
        bad_block = true;
#pragma unroll
        for (int h = 0; h < HT; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) vr[h][j].keep_if(!((bad_v >> (4 * h + j)) & 1));
      }
#pragma unroll
      for (int h = 0; h < HT; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const float vf = vr[h][j].get(dt);
#pragma unroll
            for (int nt = 0; nt < N; ++nt)
              st.o[nt][dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf, sacc[nt][h][j],
                                                                  st.o[nt][dt], 0, 0, 0);
          }
      if constexpr (MORE) load_v(c + kTW);
    };
    if (w < nch) {
      int c = w;
      if constexpr (WHOLE) read_ent(c);
      load_k(c);
      asm volatile("" ::: "memory");
      load_v(c);
      asm volatile("" ::: "memory");
      for (; c + kTW < nch; c += kTW) step(c, std::true_type{});
      step(c, std::false_type{});
    }
  }
  return bad_block;
}

template <int D, int NT>
struct TileLds {
  __attribute__((aligned(16))) float ob[kTW][16 * NT * TileGeo<D>::PITCH];  // O of each wavefront
  float ml[kTW][16 * NT][2];                                               // and its (max, sum)
  int tbl[kTblCap];
  int found[2];
};

// Tile `tile` of (sequence s, kv head kvh), key partition blockIdx.z.
template <typename T, int D, int NT, bool WHOLE>
__device__ __forceinline__ void tile_body(const AttnArgs& a, int s, int kvh, int tile,
                                          TileLds<D, NT>& sm) {
  constexpr int PITCH = TileGeo<D>::PITCH;
  constexpr int DT = TileGeo<D>::DT;
  constexpr int R = 16 * NT;  // rows per workgroup
  // opaque, so that nothing derived from it is kept across the packed grid's
  // loop (32 registers, and the third workgroup of a CU, at D = 64)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane >> 4;
  const int l16 = lane & 15;
  const int part = blockIdx.z;
  const int32_t* __restrict__ table = a.block_tables + (int64_t)s * a.max_blk;
  // the first window's entries, requested ahead of the sequence's length when
  // they start at entry 0
  int tfirst = 0;
  if (part == 0 && a.max_blk > 0) tfirst = table[min(tid, a.max_blk - 1)];
  TileGeom g;
  if (!tile_geom(a, s, tile, R, g)) return;
  if (part >= g.nparts) return;
  const int G = a.group;
  const int r0 = tile * R;
  const int kv_lo = part * g.part_len;
  const int kv_hi = min(kv_lo + g.part_len, g.kv_limit);
  if (part > 0) tfirst = table[min((kv_lo >> a.bs_shift) + tid, a.max_blk - 1)];

  // this lane's row of each tile: its key limit and its Q dims
  int lim[NT];
  float qf[NT][D / 32][8];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int rg = r0 + min(16 * nt + l16, g.rows_here - 1);
    const int i = rg / G;
    const int64_t qrow = (int64_t)(g.q_begin + i) * a.hq + kvh * G + (rg - i * G);
    lim[nt] = a.causal ? min(kv_hi, g.ctx + i + 1) : kv_hi;
    const char* qp = static_cast<const char*>(a.q) + (qrow * D + 8 * grp) * (int)sizeof(T);
#pragma unroll
    for (int kp = 0; kp < D / 32; ++kp) {
      Piece<T, 8> p;
      p.load(qp + 32 * kp * (int)sizeof(T));
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[nt][kp][j] = p.get(j);
    }
  }
  WaveState<NT, DT> st;
  st.reset();
  // a single row tile (a decode row's group, a short prompt's end) skips the
  // second one's products
  const int whole_lim = a.causal ? min(kv_hi, g.ctx + r0 / G + 1) : kv_hi;
  bool bad_block;
  if (NT == 1 || g.rows_here > 16)
    bad_block = tile_chunks<T, D, NT, NT, WHOLE>(a, table, tfirst, kvh, kv_lo, kv_hi, whole_lim,
                                                 lim, qf, st, sm.tbl, w, tid);
  else
    bad_block = tile_chunks<T, D, NT, 1, WHOLE>(a, table, tfirst, kvh, kv_lo, kv_hi, whole_lim,
                                                lim, qf, st, sm.tbl, w, tid);
  if (bad_block && a.status) atomicOr(a.status, PKV_STATUS_BAD_BLOCK);

  // ---- the four wavefronts' states through LDS. Lane (l16, grp) holds, of
  // row l16, dims DT (4 grp + e) + dt
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const float l = head_lanes_sum(st.l[nt]);
    const int r = 16 * nt + l16;
    float v[4 * DT];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) v[DT * e + dt] = st.o[nt][dt][e];
#pragma unroll
    for (int k = 0; k < DT; ++k)
      *reinterpret_cast<floatx4*>(&sm.ob[w][r * PITCH + 4 * DT * grp + 4 * k]) =
          floatx4{v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]};
    if (grp == 0) {
      sm.ml[w][r][0] = st.m[nt];
      sm.ml[w][r][1] = l;
    }
  }
  __syncthreads();
  constexpr int TPR = kTBlock / R < D / 4 ? kTBlock / R : D / 4;  // threads per row
  const int r = tid / TPR;
  if (r >= g.rows_here) return;
  float M = -INFINITY;
#pragma unroll
  for (int ww = 0; ww < kTW; ++ww) M = fmaxf(M, sm.ml[ww][r][0]);
  float wt[kTW], L = 0.f;
#pragma unroll
  for (int ww = 0; ww < kTW; ++ww) {
    wt[ww] = M == -INFINITY ? 0.f : exp2f(sm.ml[ww][r][0] - M);
    L += sm.ml[ww][r][1] * wt[ww];
  }
  const int rg = r0 + r;
  const int i = rg / G;
  const int64_t orow = (int64_t)(g.q_begin + i) * a.hq + kvh * G + (rg - i * G);
  const int64_t unit = (((int64_t)s * a.hkv + kvh) * a.tiles_max + tile) * a.parts_max + part;
  const float inv = g.nparts > 1 ? 1.f : L > 0.f ? 1.f / L : 0.f;
#pragma unroll
  for (int k = 0; k < D / (4 * TPR); ++k) {
    const int col = 4 * (tid % TPR + TPR * k);
    floatx4 o = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ww = 0; ww < kTW; ++ww)
      o += wt[ww] * *reinterpret_cast<const floatx4*>(&sm.ob[ww][r * PITCH + col]);
    if (g.nparts > 1) {
      *reinterpret_cast<floatx4*>(a.ws_o + (unit * R + r) * D + col) = o;
    } else if constexpr (sizeof(T) == 4) {
      *reinterpret_cast<floatx4*>(static_cast<float*>(a.out) + orow * D + col) = o * inv;
    } else {
      *reinterpret_cast<uint64_t*>(static_cast<T*>(a.out) + orow * D + col) = pack4<T>(o, inv);
    }
  }
  if (tid % TPR != 0) return;
  if (g.nparts > 1) {
    a.ws_ml[(unit * R + r) * 2] = M;
    a.ws_ml[(unit * R + r) * 2 + 1] = L;
  } else if (a.lse) {
    a.lse[orow] = L > 0.f ? (M + log2f(L)) * kLn2f : INFINITY;
  }
}

template <typename T, int D, int NT, bool WHOLE>
__global__ __launch_bounds__(kTBlock, 2) void attn_tiles_kernel(AttnArgs a, int packed) {
  constexpr int R = 16 * NT;  // rows per workgroup
  __shared__ TileLds<D, NT> sm;
  const int tid = threadIdx.x;
  // Tiles in falling order (the last tile of a prompt sees the most keys and
  // starts first), sequences fastest, rotated by the tile index: with the
  // plain order a sequence's tiles would all fall on one XCD whenever the
  // sequence count is a multiple of 8, and the longest prompt's XCD would
  // finish alone.
  // packed: one workgroup per tile that has rows (blockIdx.x) of kv head
  // blockIdx.y, found by a scan of the sequences' tile counts. The grid is the
  // bound for a cumulative query_start_loc; overlapping query ranges only make
  // the workgroups take more than one tile.
  int slot = blockIdx.x;
  do {
    int s, kvh, tile;
    if (!packed) {
      tile = (int)gridDim.y - 1 - (int)blockIdx.y;
      const int x = (int)((blockIdx.x + (unsigned)tile) % gridDim.x);
      s = x / a.hkv;
      kvh = x - s * a.hkv;
    } else {
      if (tid == 0) sm.found[0] = -1;
      int run = 0;
      for (int base = 0; base < a.n_seq && run <= slot; base += kTBlock) {
        const int sq = base + tid;
        int nt = 0, ex;
        if (sq < a.n_seq) {
          const int qb = a.qloc ? a.qloc[sq] : sq;
          const int ql = a.qloc ? a.qloc[sq + 1] - qb : 1;
          const bool bad = ql > 0 && (qb < 0 || qb + ql > a.n_tokens);
          if (bad && a.status && blockIdx.y == 0) atomicOr(a.status, PKV_STATUS_BAD_QLOC);
          if (ql > 0 && !bad) nt = min((ql * a.group + R - 1) / R, a.tiles_max);
        }
        const int tot = block_scan<kTW>(nt, sm.tbl, ex);
        if (nt > 0 && run + ex <= slot && slot < run + ex + nt) {
          sm.found[0] = sq;
          sm.found[1] = nt - 1 - (slot - run - ex);
        }
        run += tot;
        __syncthreads();
      }
      s = __builtin_amdgcn_readfirstlane(sm.found[0]);
      if (s < 0) return;
      tile = __builtin_amdgcn_readfirstlane(sm.found[1]);
      kvh = blockIdx.y;
    }
    tile_body<T, D, NT, WHOLE>(a, s, kvh, tile, sm);
    __syncthreads();  // sm is written again
    slot += gridDim.x;
  } while (packed);
}

// Launch shape, by the number of 32-row tiles that have rows (tiles_max bounds
// the longest sequence's, n_tokens all of them together; measured at D = 64,
// fp32, 8 heads, us with the table append's 5. Other head dims and 16-bit pools
// take the same lines, which were not measured for them; on both sides of them
// the kernel is 1.3 to 8 times as fast there as the row kernel):
//  - up to kHalfWgs of them leave CUs idle: 16-row tiles (one prompt of 500
//    tokens 12.3 against 17.1);
//  - up to kOneWgs, the longest first, are balanced best one at a time per CU:
//    the dispatcher packs the first ones it can place (500 workgroups at three
//    per CU: 114 CUs took three, 127 one; one prompt of 2000 tokens 53 against
//    60 at two and 75 at three per CU), so a larger LDS request bounds how many
//    fit. Batches that are mostly decode rows wait for memory instead and keep
//    two;
//  - beyond, two or three per CU hide each other's round trips (4 prompts of
//    1000-2000 tokens: 174 one, 151 two, 148 three).
constexpr int kHalfWgs = 256;
constexpr int kOneWgs = 512;
template <typename T, int D>
int launch_d(const AttnArgs& a0, const AttnPlan& p, hipStream_t stream) {
  AttnArgs a = a0;
  const int64_t rows = (int64_t)a.n_tokens * a.group;
  const int64_t wgs = (rows / 32 + a.n_seq) * a.hkv * p.parts_max;
  const bool half = p.parts_max == 1 && wgs <= kHalfWgs;
  if (half) a.tiles_max = (int)(((int64_t)p.tiles_max * kGenRows + 15) / 16);
  const int resident = wgs > kOneWgs ? 3 : half || rows < 128 * (int64_t)a.n_seq ? 2 : 1;
  const int have = (int)(half ? sizeof(TileLds<D, 1>) : sizeof(TileLds<D, 2>));
  const int want = kCuLds / (resident + 1) + 1024;
  const unsigned pad = want > have ? (unsigned)(want - have) : 0u;
  // a ragged batch (one long prompt among decode rows) has mostly empty tiles
  // in the dense (sequence, tile) grid, each a workgroup that waits for its
  // sequence's length before it leaves: 200 decodes + 2 prompts 39 us dense,
  // 17 packed; the scan costs a round trip, so batches below 4 stay dense
  const int64_t slots = rows / (half ? 16 : 32) + a.n_seq;
  const int packed = (int64_t)a.n_seq * a.tiles_max > 4 * slots;
  const dim3 grid = packed ? dim3((unsigned)slots, a.hkv, p.parts_max)
                           : dim3(a.n_seq * a.hkv, a.tiles_max, p.parts_max);
  // a tile's rows are addressed by 32-bit offsets from its first one
  const bool whole = a.bs_shift >= 4 && (int64_t)a.hkv * D * (int)sizeof(T) * 16 < (1 << 30);
  const dim3 block(kTBlock);
  if (half && whole)
    hipLaunchKernelGGL((attn_tiles_kernel<T, D, 1, true>), grid, block, pad, stream, a, packed);
  else if (half)
    hipLaunchKernelGGL((attn_tiles_kernel<T, D, 1, false>), grid, block, pad, stream, a, packed);
  else if (whole)
    hipLaunchKernelGGL((attn_tiles_kernel<T, D, 2, true>), grid, block, pad, stream, a, packed);
  else
    hipLaunchKernelGGL((attn_tiles_kernel<T, D, 2, false>), grid, block, pad, stream, a, packed);
  return check_launch("attn_tiles_kernel");
}

template <typename T>
int launch_t(const AttnArgs& a, const AttnPlan& p, hipStream_t stream) {
  if (a.d == 32) return launch_d<T, 32>(a, p, stream);
  if (a.d == 64) return launch_d<T, 64>(a, p, stream);
  if (a.d == 128) return launch_d<T, 128>(a, p, stream);
  return fail(PKV_ERR_UNSUPPORTED, "attn_tiles: d=%d", a.d);
}

}  // namespace

bool attn_tiles_aligned(const void* q, const void* out, const void* k_pool, const void* v_pool) {
  // every row is a multiple of 64 bytes
  return ((uintptr_t)q | (uintptr_t)out | (uintptr_t)k_pool | (uintptr_t)v_pool) % 16 == 0;
}

bool attn_tiles_supported(const AttnArgs& a, int dtype) {
  // the row kernel takes what is left: other head dims, and a pool, q or out
  // that is not 16-byte aligned
  return (dtype == PKV_DTYPE_F32 || dtype == PKV_DTYPE_BF16 || dtype == PKV_DTYPE_F16) &&
         !a.kv8 && (a.d == 32 || a.d == 64 || a.d == 128) &&
         attn_tiles_aligned(a.q, a.out, a.k_pool, a.v_pool);
}

int launch_attn_tiles(const AttnArgs& a, const AttnPlan& p, int dtype, hipStream_t stream) {
  if (dtype == PKV_DTYPE_F32) return launch_t<float>(a, p, stream);
  if (dtype == PKV_DTYPE_BF16) return launch_t<bf16>(a, p, stream);
  return launch_t<f16>(a, p, stream);
}

}  // namespace pkv
