// Quad decode of (K,N) codes (the layout pack_quad_layer returns, quad_kernels.py:35-37) for 1 to
// 32 tokens with fp16 tables: out_m[j, n] = fp16(s_m * sum_k x[j, k] * W_m[k, n])
// (quad_kernels.py:103-134).
//
// A workgroup of 8 wavefronts takes a strip of columns and a slice of K, an eighth of the slice's
// rows per wavefront, and the wavefronts' sums meet in LDS: 1/8 of the partial sums that slices
// of one wavefront leave.  What bounds the kernels is the code stream and, at 2 to 32 tokens,
// the decode's ~12 instructions a word; so
//  * the tables hold (cos, sin) as the two fp16 the caller gave, in 4 bytes: a word takes four
//    4-byte LDS reads (8 LDS clocks a wavefront; 14 with the float32 tables of quad_lds.h) and
//    the products read them as mixed-precision operands;
//  * a strip is 64 or 32 columns (strip_plan), 256 or 128 contiguous bytes of every row.  16
//    columns (64 bytes) would need no slices for 4096 of them, but read from HBM they took 28.3
//    us at 16 tokens and 4096 x 4096 where this takes 24.5;
//  * a lane's load is 16 (8) bytes of one row, whose words belong to 4 (2) matrix tiles: tile j
//    takes columns 4i + j, so the operands need no transpose.
// Per call in a graph, weights in the last-level cache / from HBM, against quad_kn_kernel (1 token)
// and quad_big_kernel, whose slices are one wavefront's: 4096 x 4096 at 1 token 22.5 / 23.9 ->
// 18.9 / 22.3 us, 16 tokens 29.5 /
// 31.0 -> 23.4 / 24.5, 32 tokens 35.4 / 37.3 -> 24.8 / 26.3; 2048 x 2048 at 1 / 16 / 32 tokens 14.4
// / 16.5 / 20.5 -> 10.7 / 11.7 / 13.9; N x K = 2048 x 11008 at 16 tokens 34.7 -> 27.2, 11008 x 2048
// 46.0 -> 26.4.
#include "rows_common.h"
#include "slice_sums.h"

#include <algorithm>

namespace pp {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int QS_WAVES = 8, QS_NT = 64 * QS_WAVES;
constexpr int64_t QS_MAX_M = 32;
// Code words to which one token takes the strips: above, quad_kn_kernel reads the codes faster (a
// wavefront 1 KiB of a row at a time, where a strip takes 256 bytes).  Strips / row kernel at K x N of 13 M
// words 19.4 / 22.4 us, 24 M 28.0 / 28.4, 25 M 25.7-27.7 / 27.3-27.8, 28 M 34.3 / 31.9, 45 M 41.5 / 40.0,
// 67 M 59.1 / 53.0, 89 M 82.9 / 72.5.
constexpr int64_t QS_GEMV_WORDS = 25ll << 20;

struct QuadStripArgs {
  const uint32_t* codes;   // code of (row 0, column 0); row k at codes + k*ldk
  int64_t ldk;
  const f16* x;            // (M, K), row stride x_sm
  int64_t x_sm;
  f16* out[4];             // (M, N): element (j, n) at out + j*o_sm + n*o_sn
  int64_t o_sm, o_sn;
  int N, K, M;
  int strips, slices;
  int vec_out;             // o_sn == 1, outputs 8-byte aligned, o_sm % 4 == 0: 4 columns per store
  QuadLuts luts;           // fp16
  float s[4];
  float* part;             // slices > 1: float32 sums, [slice][model][token][np]
  int64_t np;              // N rounded up to whole strips
  uint32_t* count;         // one token, slices > 1: slices of each strip that are done, zero between launches
};

// ------------------------------------------------------------------ tables
// The tables of fp16 LUTs in 128 KiB, whatever their values: 256-byte rows, one per code byte,
// [norm (float32) x 32 | (cos3, sin3) x 32] and, 64 KiB on, [(cos1, sin1) x 32 | (cos2, sin2) x
// 32], a (cos, sin) pair being two fp16 in 4 bytes.  Lane l reads replica l % 32: every lookup is
// a conflict-free 4-byte read whose address is one v_perm_b32 of the code word and a lane
// constant.
constexpr uint32_t QS_TABLES = 0x20000;

struct HalfLane {
  uint32_t r, c1, c2, c3;
};
__device__ __forceinline__ HalfLane half_lane(int l) {
  const uint32_t o = 4u * (l & 31);
  return HalfLane{o, 0x10000u | o, 0x10000u | 128u | o, 128u | o};
}

// Table row address of code byte B (3 = norm, 2 = t1, 1 = t2, 0 = t3).
template <int B>
__device__ __forceinline__ uint32_t half_addr(uint32_t cw, uint32_t lane_off) {
  return __builtin_amdgcn_perm(cw, lane_off, 0x0C020000u | ((4u + B) << 8));
}

struct HalfWord {
  float r;
  f16x2 a, b, c;           // (cos, sin) of the three angles
};
__device__ __forceinline__ HalfWord half_lookup(const char* lds, uint32_t cw, const HalfLane& o) {
  HalfWord w;
  w.r = *reinterpret_cast<const float*>(lds + half_addr<3>(cw, o.r));
  w.a = *reinterpret_cast<const f16x2*>(lds + half_addr<2>(cw, o.c1));
  w.b = *reinterpret_cast<const f16x2*>(lds + half_addr<1>(cw, o.c2));
  w.c = *reinterpret_cast<const f16x2*>(lds + half_addr<0>(cw, o.c3));
  return w;
}

// Two threads an entry, 8 of the 16 units of 16 bytes of each of its rows a thread, neighbouring lanes
// starting at different units (distinct banks).  7 loads a thread; with a unit's own values loaded by
// the thread that writes it (32 loads) 4096 x 4096 took 19.5 us a call at 1 token (19.2 this way) and
// the same at 32.
struct HalfTables {
  static_assert(QS_NT == 512, "two threads an entry");
  uint32_t norm, t1, t2, t3;   // norm as float32, the (cos, sin) pairs
  __device__ __forceinline__ void load(const QuadLuts& L) {
    const int e = threadIdx.x & 255;
    uint32_t v[7];
#pragma unroll
    for (int i = 0; i < 7; ++i) v[i] = reinterpret_cast<const uint16_t*>(L.p[i])[e];
    norm = v[0];
    t1 = v[1] | (v[2] << 16);
    t2 = v[3] | (v[4] << 16);
    t3 = v[5] | (v[6] << 16);
  }
  __device__ __forceinline__ void store(char* lds) const {
    const int e = threadIdx.x & 255;
    const uint32_t n = __float_as_uint(h2f(norm));
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int u = (k + 8 * (threadIdx.x >> 8) + e) & 15;
      const uint32_t a = u < 8 ? n : t3, b = u < 8 ? t1 : t2;
      char* p = lds + 256 * e + 16 * u;
      *reinterpret_cast<u32x4*>(p) = u32x4{a, a, a, a};
      *reinterpret_cast<u32x4*>(p + 0x10000) = u32x4{b, b, b, b};
    }
  }
};

// ------------------------------------------------------------------ items
// Item (strip, slice) of round r: neighbouring items on the workgroups of one XCD (block b on XCD
// b % 8).
__device__ __forceinline__ int strip_item(int r) {
  const int g = gridDim.x, b = blockIdx.x;
  const int p = g % 8 == 0 ? (b & 7) * (g >> 3) + (b >> 3) : b;
  return r * g + p;
}

// Rows [k0, k1) of a wave: its share of the slice, in units of U rows.
template <int U>
__device__ __forceinline__ void strip_rows(const QuadStripArgs& A, int slice, int wave, int& k0, int& k1) {
  const int64_t units = A.K / U, parts = (int64_t)QS_WAVES * A.slices, p = (int64_t)slice * QS_WAVES + wave;
  k0 = (int)(p * units / parts) * U;
  k1 = (int)((p + 1) * units / parts) * U;
}

__device__ __forceinline__ float model_scale(const QuadStripArgs& A, int m) {
  return m == 0 ? A.s[0] : m == 1 ? A.s[1] : m == 2 ? A.s[2] : A.s[3];
}
__device__ __forceinline__ f16* model_out(const QuadStripArgs& A, int m) {
  return m == 0 ? A.out[0] : m == 1 ? A.out[1] : m == 2 ? A.out[2] : A.out[3];
}

// ------------------------------------------------------------------ one token
// float32 weights and sums.  Lane l owns columns 4 (l % 16) .. +3 of the 64 and, of each 32 rows,
// rows 8 (l / 16) .. +7: one 16-byte code load per row, one of the 8 activations.
constexpr int QG_COLS = 64, QG_ROWS = 32;

struct GemvChunk {
  u32x4 q[8];
  u32x4 x;
};

__device__ __forceinline__ void gemv_issue(const QuadStripArgs& A, int n0, int k, int kend, uint32_t voff, int lane,
                                           GemvChunk& S) {
  const int rows = max(0, kend - k), kc = min(k, A.K - 1);
  const rsrc_t rc = make_rsrc(A.codes + (int64_t)kc * A.ldk + n0,
                              rows > 0 ? 4u * (uint32_t)((int64_t)(rows - 1) * A.ldk + min(A.N - n0, QG_COLS)) : 0u);
  const rsrc_t rx = make_rsrc(A.x + kc, 2u * (uint32_t)rows);
  vload128c(S.x, 16u * (uint32_t)(lane >> 4), rx);
#pragma unroll
  for (int i = 0; i < 8; ++i) vload128(S.q[i], voff + 4u * (uint32_t)(i * A.ldk), rc);
}

// `in`: the lane's 8 rows lie in the wave's (its rows come in eights).  Rows past them are left out, not
// multiplied as zeros: the tables' first entries need not be finite.
__device__ __forceinline__ void gemv_compute(const char* lds, const HalfLane& hl, const GemvChunk& S, bool in,
                                             float (&acc)[16]) {
  if (!in) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t xw = i < 2 ? S.x.x : i < 4 ? S.x.y : i < 6 ? S.x.z : S.x.w;
    const float x = h2f((i & 1) ? xw >> 16 : xw & 0xFFFFu);
    const uint32_t cw[4] = {S.q[i].x, S.q[i].y, S.q[i].z, S.q[i].w};
    HalfWord w[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = half_lookup(lds, cw[c], hl);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float t0 = w[c].r * x;
      acc[c] = fmaf(t0, (float)w[c].a.x, acc[c]);
      const float t1 = fmaf(t0, (float)w[c].a.y, 0.f);
      acc[4 + c] = fmaf(t1, (float)w[c].b.x, acc[4 + c]);
      const float t2 = fmaf(t1, (float)w[c].b.y, 0.f);
      acc[8 + c] = fmaf(t2, (float)w[c].c.x, acc[8 + c]);
      acc[12 + c] = fmaf(t2, (float)w[c].c.y, acc[12 + c]);
    }
  }
}

__global__ __launch_bounds__(QS_NT) void quad_strip_gemv_kernel(const QuadStripArgs A) {
  __shared__ __attribute__((aligned(16))) char lds[QS_TABLES + 2 * QS_WAVES * 256 * 4 + 16];
  float* red = reinterpret_cast<float*>(lds + QS_TABLES);
  uint32_t* done = reinterpret_cast<uint32_t*>(lds + QS_TABLES + 2 * QS_WAVES * 256 * 4);
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const HalfLane hl = half_lane(lane);
  const int items = A.strips * A.slices;
  int n0, kb, ke;
  uint32_t vo;
  GemvChunk s0, s1;
  auto start = [&](int it) {
    if (it >= items) return;
    n0 = it / A.slices * QG_COLS;
    strip_rows<8>(A, it % A.slices, wave, kb, ke);
    vo = n0 + 4 * (lane & 15) < A.N ? 4u * (uint32_t)(8 * (lane >> 4) * A.ldk + 4 * (lane & 15)) : OOB;
    gemv_issue(A, n0, kb, ke, vo, lane, s0);
  };
  HalfTables tb;
  tb.load(A.luts);
  start(strip_item(0));
  tb.store(lds);
  __syncthreads();
  for (int r = 0; r * (int)gridDim.x < items; ++r) {
    const int it = strip_item(r);
    float acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if (it < items) {
      for (int k = kb; k < ke; k += 2 * QG_ROWS) {
        gemv_issue(A, n0, k + QG_ROWS, ke, vo, lane, s1);
        __builtin_amdgcn_sched_barrier(0);
        gemv_compute(lds, hl, s0, k + 8 * (lane >> 4) < ke, acc);
        __builtin_amdgcn_sched_barrier(0);
        if (k + QG_ROWS >= ke) break;
        gemv_issue(A, n0, k + 2 * QG_ROWS, ke, vo, lane, s0);
        __builtin_amdgcn_sched_barrier(0);
        gemv_compute(lds, hl, s1, k + QG_ROWS + 8 * (lane >> 4) < ke, acc);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const int n = n0;
    start(strip_item(r + 1));
    // sums over the 4 row groups (lane bits 5 and 4): lane l keeps model l / 16, its 4 columns
    halve<5, 16>(acc, lane);
    halve<4, 8>(acc, lane);
    // two buffers in turn: a buffer is written again only after the next round's barrier
    float* rb = red + (r & 1) * QS_WAVES * 256;
    *reinterpret_cast<float4*>(rb + wave * 256 + 4 * lane) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    __syncthreads();
    const bool owner = threadIdx.x < 256 && it < items;      // thread t: model t / 64, column t % 64
    const int m = threadIdx.x >> 6 & 3, col = n + (threadIdx.x & 63);
    float v = 0.f;
    if (owner) {
#pragma unroll
      for (int w = 0; w < QS_WAVES; ++w) v += rb[w * 256 + threadIdx.x];
      v *= model_scale(A, m);
    }
    if (A.slices > 1) {
      // The slice's sums go to memory by exchanges whose results every thread waits for, so they
      // are there before the strip's count goes up; the workgroup that counts last reads all the
      // slices' sums (in slice order: the result does not depend on who is last).
      const int strip = it / A.slices;
      const int64_t at = ((int64_t)m) * A.np + col;
      if (owner) {
        const uint32_t was = __hip_atomic_exchange(reinterpret_cast<uint32_t*>(A.part) + (int64_t)(it % A.slices) * 4 * A.np + at,
                                                   __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" : : "v"(was) : "memory");
      }
      __syncthreads();
      if (threadIdx.x == 0 && it < items)
        *done = __hip_atomic_fetch_add(A.count + strip, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (it >= items || *done != (uint32_t)(A.slices - 1)) continue;
      if (threadIdx.x == 0)
        __hip_atomic_store(A.count + strip, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (owner) {
        v = 0.f;
#pragma unroll 8
        for (int sl = 0; sl < A.slices; ++sl)
          v += __uint_as_float(__hip_atomic_load(reinterpret_cast<uint32_t*>(A.part) + (int64_t)sl * 4 * A.np + at,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      }
    }
    if (owner && col < A.N) model_out(A, m)[(int64_t)col * A.o_sn] = (f16)v;
  }
}

// ------------------------------------------------------------------ 2 to 32 tokens
// v_mfma_f32_16x16x32_f16 per 32 rows and 16 columns.  Lane l: row group q = l / 16 (rows 8q .. +7 of
// the step), columns CT i .. + CT - 1 of the strip's 16 CT (i = l % 16); its CT words of a row
// belong to CT tiles, tile j holding columns CT p + j (p the tile's row of A operands).  x is the
// B operand as stored: token 16 t + i, the same rows.
template <int CT> struct StripVec;
template <> struct StripVec<4> { typedef u32x4 T; };
template <> struct StripVec<2> { typedef u32x2 T; };

template <int CT>
struct StripCodes {
  typename StripVec<CT>::T c[8];
};
template <int TT>
struct StripX {
  u32x4 t[TT];
};

template <int CT, int TT>
struct StripWalk {
  const QuadStripArgs& A;
  const char* lds;
  HalfLane hl;
  int n0, kb, ke;
  uint32_t voc, vox[TT];

  // Codes of the step at row k; past the wave's rows they read 0 and so does x.
  __device__ __forceinline__ void codes(int k, StripCodes<CT>& S) const {
    const int rows = max(0, ke - k), kc = min(k, A.K - 32);
    const rsrc_t rc = make_rsrc(A.codes + (int64_t)kc * A.ldk + n0,
                                rows > 0 ? 4u * (uint32_t)(31 * A.ldk + min(A.N - n0, 16 * CT)) : 0u);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int o = (int)(voc + 4u * (uint32_t)(e * A.ldk));
      if constexpr (CT == 4) S.c[e] = __builtin_amdgcn_raw_buffer_load_b128(rc, o, 0, NT_AUX);
      else S.c[e] = __builtin_amdgcn_raw_buffer_load_b64(rc, o, 0, NT_AUX);
    }
  }
  __device__ __forceinline__ void xs(int k, StripX<TT>& X) const {
    const rsrc_t rx = make_rsrc(A.x + min(k, A.K - 32),
                                k < ke ? 2u * (uint32_t)((int64_t)(A.M - 1) * A.x_sm + 32) : 0u);
#pragma unroll
    for (int t = 0; t < TT; ++t) vload128c(X.t[t], vox[t], rx);
  }
  __device__ __forceinline__ void look(const StripCodes<CT>& S, int j, HalfWord (&w)[8]) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = half_lookup(lds, S.c[e][j], hl);
  }
  // One step: x and codes of the next step issued, then tile by tile the lookups of the tile after
  // it, its arithmetic and its products (the fences keep the loads ahead of the decode and one
  // tile's lookups ahead of the arithmetic).
  __device__ __forceinline__ void step(int k, const StripCodes<CT>& cur, StripCodes<CT>& nxt, const StripX<TT>& xc,
                                       StripX<TT>& xn, f4 (&C)[CT][4][TT]) const {
    xs(k + 32, xn);
    codes(k + 32, nxt);
    __builtin_amdgcn_sched_barrier(0);
    if (k >= ke) return;               // no step of zeros: the tables' first entries need not be finite
    HalfWord w[2][8];
    look(cur, 0, w[0]);
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      if (j + 1 < CT) look(cur, j + 1, w[(j + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      h8 a[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float v[4][2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const HalfWord& h = w[j & 1][e + u];
          const float rs = fmaf(h.r, (float)h.a.y, 0.f), rss = fmaf(rs, (float)h.b.y, 0.f);
          v[0][u] = fmaf(h.r, (float)h.a.x, 0.f);
          v[1][u] = fmaf(rs, (float)h.b.x, 0.f);
          v[2][u] = fmaf(rss, (float)h.c.x, 0.f);
          v[3][u] = fmaf(rss, (float)h.c.y, 0.f);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          // the float32 product, then fp16, as the reference rounds it: not one rounding of both
          asm volatile("" : "+v"(v[m][0]), "+v"(v[m][1]));
          const f16x2 p = __builtin_convertvector((f2{v[m][0], v[m][1]}), f16x2);
          a[m][e] = p.x;
          a[m][e + 1] = p.y;
        }
      }
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const h8 b = __builtin_bit_cast(h8, xc.t[t]);
#pragma unroll
        for (int m = 0; m < 4; ++m) C[j][m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[m], b, C[j][m][t], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};

// Columns n .. n + 4 CT - 1 of token j, model m: v[p][jj] is column n + CT p + jj.
template <int CT>
__device__ __forceinline__ void strip_store(const QuadStripArgs& A, int slice, int m, int j, int n, const f4 (&v)[CT]) {
  if (j >= A.M || n >= A.N) return;
  const float s = model_scale(A, m);
  float o[4 * CT];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int jj = 0; jj < CT; ++jj) o[CT * p + jj] = v[jj][p] * s;
  if (A.slices > 1) {
    float* d = A.part + (((int64_t)slice * 4 + m) * A.M + j) * A.np + n;
#pragma unroll
    for (int c = 0; c < CT; ++c) *reinterpret_cast<float4*>(d + 4 * c) = make_float4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
    return;
  }
  f16* d = model_out(A, m) + (int64_t)j * A.o_sm + (int64_t)n * A.o_sn;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    if (A.vec_out && n + 4 * c + 3 < A.N) {
      *reinterpret_cast<f16x4*>(d + 4 * c) = f16x4{(f16)o[4 * c], (f16)o[4 * c + 1], (f16)o[4 * c + 2], (f16)o[4 * c + 3]};
    } else {
#pragma unroll
      for (int e = 4 * c; e < 4 * c + 4; ++e)
        if (n + e < A.N) d[e * A.o_sn] = (f16)o[e];
    }
  }
}

template <int CT, int TT>
__global__ __launch_bounds__(QS_NT) void quad_strip_kernel(const QuadStripArgs A) {
  // the waves' sums, [wave][block of 4 tiles x models][lane] float4: MP models x CT tiles at a time beside
  // the tables, all of them over the tables once the last item is decoded
  constexpr int MP = 4 / CT, PHASES = 4 * TT / MP;
  static_assert(PHASES <= 4, "all sums must fit where the tables were");
  __shared__ __attribute__((aligned(16))) char lds[QS_TABLES + QS_WAVES * 4 * 64 * 16];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), i = lane & 15, q = lane >> 4;
  const int items = A.strips * A.slices;
  StripWalk<CT, TT> W{A, lds, half_lane(lane)};
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    const int j = 16 * t + i;
    W.vox[t] = j < A.M ? 2u * (uint32_t)(j * A.x_sm + 8 * q) : OOB;
  }
  StripCodes<CT> C0, C1;
  StripX<TT> X0, X1;
  auto start = [&](int it) {
    if (it >= items) return;
    W.n0 = 16 * CT * (it / A.slices);
    strip_rows<32>(A, it % A.slices, wave, W.kb, W.ke);
    W.voc = W.n0 + CT * i < A.N ? 4u * (uint32_t)(8 * q * A.ldk + CT * i) : OOB;
    W.xs(W.kb, X0);
    W.codes(W.kb, C0);
  };
  HalfTables tb;
  tb.load(A.luts);
  start(strip_item(0));
  tb.store(lds);
  __syncthreads();
  for (int r = 0; r * (int)gridDim.x < items; ++r) {
    const int it = strip_item(r);
    const bool last = (r + 1) * (int)gridDim.x >= items;
    f4 acc[CT][4][TT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[c][m][t] = f4{0.f, 0.f, 0.f, 0.f};
    if (it < items) {
      // the loads of both steps with no exit between them, so that each load stays in its step
      for (int k = W.kb; k < W.ke; k += 64) {
        W.step(k, C0, C1, X0, X1, acc);
        W.step(k + 32, C1, C0, X1, X0, acc);
      }
    }
    const int n0 = W.n0, slice = it % A.slices;
    start(strip_item(r + 1));          // travels under the sums
    f4* red = reinterpret_cast<f4*>(last ? lds : lds + QS_TABLES);
    if (last) __syncthreads();         // every wave is done with the tables
#pragma unroll
    for (int p = 0; p < PHASES; ++p) {
      const int t = p * MP / 4, m0 = p * MP % 4;
      f4* rp = last ? red + p * QS_WAVES * 256 : red;
#pragma unroll
      for (int u = 0; u < MP; ++u)
#pragma unroll
        for (int c = 0; c < CT; ++c) rp[(wave * 4 + u * CT + c) * 64 + lane] = acc[c][m0 + u][t];
      if (last && p + 1 < PHASES) continue;
      __syncthreads();
      // wave w sums phase and model w / MP, w % MP of those in LDS
      const int pw = last ? wave / MP : p;
      if (last ? wave < PHASES * MP : wave < MP) {
        const int u = wave % MP, m = pw * MP % 4 + u, tt = pw * MP / 4;
        const f4* src = last ? red + pw * QS_WAVES * 256 : red;
        f4 v[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) v[c] = src[(u * CT + c) * 64 + lane];
#pragma unroll
        for (int w = 1; w < QS_WAVES; ++w)
#pragma unroll
          for (int c = 0; c < CT; ++c) v[c] += src[(w * 4 + u * CT + c) * 64 + lane];
        if (it < items) strip_store<CT>(A, slice, m, 16 * tt + i, n0 + 4 * CT * q, v);
      }
      if (!last) __syncthreads();
    }
  }
}

// ------------------------------------------------------------------ host side
struct StripPlan {
  int cols, strips, slices;
};

// Columns of a strip (64 or 32; 64 at one token, 32 from 17, whose sums would not fit in registers)
// and slices of K: the pair with the least cost, in steps of 32 rows x 32 columns - rounds of
// workgroups x (the longest wave's steps + 2 for an item's first loads and sums, 3 with 64
// columns), and 5 for a second pass over the slices' sums (2 at one token, where the last slice
// adds them).  At 16 tokens, 64 against 32 columns: 4096 x 4096 23.8 / 21.5 us, 2048 x 2048 (N x K)
// 16.4 / 11.9, 2048 x 11008 28.2 / 27.5, 11008 x 2048 27.5 / 32.8.
static StripPlan strip_plan(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = device_cu_count(), steps = (K + 31) / 32, most = std::max<int64_t>(1, steps / QS_WAVES);
  StripPlan best = {};
  int64_t least = INT64_MAX;
  for (int cols = M == 1 ? 64 : 32; cols <= (M <= 16 ? 64 : 32); cols += 32) {
    const int64_t strips = (N + cols - 1) / cols, wide = cols / 32;
    for (int64_t s = 1; s <= std::min<int64_t>(most, 32); ++s) {
      const int64_t rounds = (strips * s + cus - 1) / cus, per = (steps + QS_WAVES * s - 1) / (QS_WAVES * s);
      const int64_t cost = rounds * (per * wide + 1 + wide) + (s == 1 ? 0 : M == 1 ? 2 : 5);
      if (cost < least) {
        least = cost;
        best = {cols, (int)strips, (int)s};
      }
    }
  }
  return best;
}

static bool strip_reads(const void* codes, int64_t ldk, const void* a, int64_t a_sm, int lut_dtype, int64_t M, int64_t N,
                        int64_t K) {
  if (lut_dtype != PP_F16 || M < 1 || M > QS_MAX_M || N < 1 || K < 32 || ldk < N) return false;
  if (K * ldk >= (1ll << 29) || !aligned(a, 16) || (M > 1 && (a_sm < K || a_sm % 8 != 0))) return false;
  if (M * (M > 1 ? a_sm : K) >= (1ll << 29)) return false;
  // 16-byte code loads to 16 tokens, 8-byte ones above
  const int unit = M <= 16 ? 4 : 2;
  return K % (M == 1 ? 8 : 32) == 0 && N % unit == 0 && ldk % unit == 0 && aligned(codes, 4 * unit);
}

}  // namespace pp

using namespace pp;

extern "C" int pp_quad_strip_ok(const void* codes, int64_t ldk, const void* a, int64_t a_sm, int lut_dtype, int64_t M,
                                int64_t N, int64_t K) {
  return strip_reads(codes, ldk, a, a_sm, lut_dtype, M, N, K) && (M > 1 || K * N < QS_GEMV_WORDS);
}

extern "C" int64_t pp_quad_strip_counts(int64_t M, int64_t N, int64_t K) {
  if (M != 1 || N < 1 || K < 1) return 0;
  const StripPlan p = strip_plan(M, N, K);
  return p.slices > 1 ? 4 * (int64_t)p.strips : 0;
}

extern "C" int64_t pp_quad_strip_workspace_size(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 1) return 0;
  const StripPlan p = strip_plan(M, N, K);
  return p.slices > 1 ? (int64_t)p.slices * 4 * M * p.strips * p.cols * (int64_t)sizeof(float) : 0;
}

extern "C" int pp_quad_strip(const uint32_t* codes, int64_t ldk, const void* a, int64_t a_sm, const void* const* luts,
                             int lut_dtype, const float* scales, void* const* out, int64_t o_sm, int64_t o_sn, int64_t M,
                             int64_t N, int64_t K, void* workspace, int64_t workspace_bytes, void* counts,
                             int64_t counts_bytes, void* stream) {
  PP_REQUIRE(codes != nullptr && a != nullptr && out != nullptr && luts != nullptr && scales != nullptr,
             "null pointer argument");
  PP_REQUIRE(strip_reads(codes, ldk, a, a_sm, lut_dtype, M, N, K), "operands the strip kernel does not read");
  for (int m = 0; m < 4; ++m) PP_REQUIRE(out[m] != nullptr, "out[%d] is null", m);
  for (int i = 0; i < 7; ++i) PP_REQUIRE(luts[i] != nullptr, "lut %d is null", i);
  const StripPlan p = strip_plan(M, N, K);
  const int64_t need = pp_quad_strip_workspace_size(M, N, K), need_counts = pp_quad_strip_counts(M, N, K);
  PP_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && aligned(workspace, 16)),
             "workspace too small or misaligned: need %lld bytes", (long long)need);
  PP_REQUIRE(need_counts == 0 || (counts != nullptr && counts_bytes >= need_counts && aligned(counts, 4)),
             "counts too small: need %lld bytes", (long long)need_counts);
  QuadStripArgs A = {};
  A.codes = codes;
  A.ldk = ldk;
  A.x = reinterpret_cast<const f16*>(a);
  A.x_sm = M > 1 ? a_sm : K;
  bool vec = o_sn == 1 && (M == 1 || o_sm % 4 == 0);
  for (int m = 0; m < 4; ++m) {
    A.out[m] = reinterpret_cast<f16*>(out[m]);
    A.s[m] = scales[m];
    vec = vec && aligned(out[m], 8);
  }
  A.vec_out = vec;
  A.o_sm = o_sm;
  A.o_sn = o_sn;
  A.N = (int)N;
  A.K = (int)K;
  A.M = (int)M;
  A.strips = p.strips;
  A.slices = p.slices;
  for (int i = 0; i < 7; ++i) A.luts.p[i] = luts[i];
  A.luts.dtype = lut_dtype;
  A.part = reinterpret_cast<float*>(workspace);
  A.np = (int64_t)p.strips * p.cols;
  A.count = reinterpret_cast<uint32_t*>(counts);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)std::min<int64_t>(device_cu_count(), (int64_t)p.strips * p.slices)), block(QS_NT);
  if (M == 1) hipLaunchKernelGGL(quad_strip_gemv_kernel, grid, block, 0, st, A);
  else if (p.cols == 64) hipLaunchKernelGGL((quad_strip_kernel<4, 1>), grid, block, 0, st, A);
  else if (M <= 16) hipLaunchKernelGGL((quad_strip_kernel<2, 1>), grid, block, 0, st, A);
  else hipLaunchKernelGGL((quad_strip_kernel<2, 2>), grid, block, 0, st, A);
  PP_LAUNCH_CHECK();
  if (M > 1 && p.slices > 1) {
    SliceSums<4> F = {};
    F.part = A.part;
    F.np = A.np;
    for (int m = 0; m < 4; ++m) F.out[m] = A.out[m];
    F.o_sm = o_sm;
    F.o_sn = o_sn;
    F.N = A.N;
    F.M = A.M;
    F.slices = A.slices;
    F.vec_out = A.vec_out;
    launch_slice_sums(F, st);
    PP_LAUNCH_CHECK();
  }
  return PP_OK;
}
