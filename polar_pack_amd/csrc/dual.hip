// Dual-pack fused decode GEMV/GEMM for gfx950.
//
// One 16-bit code per pair of weights: (amp_q << 10) | phase  (polar_bitpack.py:130,
// polar_kernels.py:9-11), decoded as
//   amp = amp_lut[amp_q] * scale[group],  w1 = amp cos_lut[phase],  w2 = amp sin_lut[phase]
// (polar_kernels.py:64-79, polar_bitpack.py:228-247).  Codes are either the kernel
// layout (native int16 = code - 32768) or the .dualpack file layout (big-endian uint16).
//
// Kernels:
//   dual_rows_kernel   -- batch <= 4 decode over the .dualpack stream layout ((N,K)
//                         row-major positions, groups of 32 that restart every chunk).
//                         A lane streams 8 pairs per 16-byte load; the 8 pairs share one
//                         group scale, so the scale multiplies a per-lane partial sum once
//                         per 8 pairs (x * amp_lut, then 2 fma per pair).  Plug entries
//                         replace the amplitude as exact corrections.
//   dual_kn_gemm       -- (dual_kn.hip) codes (K,N) with unit column stride, the layout
//                         quantize_polar_bitpacked returns, in blocks of up to 8 tokens.
//   dual_dequant_kernel / dual_plug_scatter_kernel / dual_ws_gemm_kernel -- generic path
//                         and parity export (any strides, both group-index modes).
#include "dequant_t.h"
#include "dual_kn.h"
#include "dual_lds.h"
#include "rows_common.h"

#include <algorithm>

namespace pp {

struct DualGroup {
  int64_t gs, chunk;  // chunk == 0: logical (k*N + n) // gs of a (K,N) matrix
  int64_t per_chunk;  // ceil(chunk / gs)
  int log2gs;         // fast path: gs is a power of two
  __device__ __forceinline__ int64_t of_pos(int64_t p) const {
    const int64_t c = p / chunk;
    return c * per_chunk + (p - c * chunk) / gs;
  }
};

// Batch 1..4 decode over the .dualpack stream layout.  A task is RG rows x one of `parts`
// runs of 512-pair chunks of K; a task's parts are neighbouring waves of one workgroup, whose
// sums meet in LDS, so the launch needs no workspace and no atomics.
//
// What bounds it: a Linear of a few million pairs is read in less time than a launch, a table
// build and a reduction take, so the kernel is shaped around one round trip: the first chunk
// and the task's place in the plug table (a 64-way search by the whole wave: three dependent
// loads for 262,144 entries, in place of a search kernel of its own) travel while the tables
// are built, and the host picks the parts that leave the fewest chunk times (dual_rows_plan).
// Measured with 1 % plug entries, per call in a graph, against one to four rows a task without
// look-ahead and a search kernel before it: 1531 x 4104 at 3 tokens 24.7 -> 11.9 us, 11008 x
// 2048 at 1 / 2 tokens 30.4 / 36.9 -> 23.4 / 25.7, 2048 x 11016 at 2 tokens 99.7 -> 23.0, 256 x
// 264 at 2 tokens 11.0 -> 6.5.  The large ones are bound by the decode's instructions (~12 a
// pair and token) and table reads at two wavefronts a SIMD.
constexpr int DR_NT = 512;       // threads per workgroup (one per CU: the tables take most of LDS)
constexpr int DR_WAVES = DR_NT / 64;
constexpr int DR_CHUNK = 512;    // pairs per wave, row and step: 8 per lane
// Row strides from here on (a task's 8 rows then span 2^29 pairs, past which 32-bit byte offsets end)
// take the form with a base a row.
constexpr int64_t DR_WIDE = 1ll << 26;

struct DualRowsArgs {
  const uint16_t* codes;   // code of (row 0, k 0)
  int64_t ldc;             // row stride (elements)
  int64_t pos0;            // stream position of (row 0, 0)
  const f16* x;
  int64_t x_sm;
  f16* out[2];
  int64_t o_sm, o_sn;
  int N, K, M;
  int tasks, parts, rounds;
  const f16* scales;
  DualGroup grp;
  DualLuts luts;
  const uint32_t* plug_idx;
  const f16* plug_amp;
  int64_t plug_n;
};

// A wave's task.  Its pairs are addressed by o = their offset from a row's first pair + low, low
// being that pair's place in its group: pair o is in group o / gs of `scales` up to the next chunk
// boundary, where the groups restart.  The offsets are 32 bits: where a task's rows span more (WIDE)
// each row has a base of its own, else row 0's serves them all (one division by the chunk size a task).
template <int RG, bool WIDE>
struct DrTask {
  static constexpr int NB = WIDE ? RG : 1;
  int row0, nrows, k0, k1;
  rsrc_t codes[NB];        // the rows from k0 (past the last row's k1 it reads 0)
  const f16* scales[NB];   // the first pair's group scale
  uint32_t low[NB];
  uint32_t edge[NB];       // o of the next chunk boundary, 0xFFFFFFFF if past the base's rows
  uint32_t edge_group[NB]; // its group
};

template <int RG, bool WIDE>
__device__ __forceinline__ DrTask<RG, WIDE> dr_task(const DualRowsArgs& A, int t, int part) {
  DrTask<RG, WIDE> T;
  const int chunks = (A.K + DR_CHUNK - 1) / DR_CHUNK;
  T.row0 = min(t * RG, A.N);
  T.nrows = t < A.tasks ? min(RG, A.N - T.row0) : 0;
  T.k0 = (int)((int64_t)part * chunks / A.parts) * DR_CHUNK;
  T.k1 = min(A.K, (int)((int64_t)(part + 1) * chunks / A.parts) * DR_CHUNK);
  const bool any = T.nrows > 0 && T.k1 > T.k0;
#pragma unroll
  for (int b = 0; b < DrTask<RG, WIDE>::NB; ++b) {
    const int64_t at = (int64_t)(WIDE ? min(T.row0 + b, A.N - 1) : T.row0) * A.ldc;
    const int64_t span = WIDE ? T.k1 - T.k0 : (T.nrows - 1) * A.ldc + T.k1 - T.k0;
    T.codes[b] = make_rsrc(A.codes + at + T.k0, any && b < T.nrows ? 2u * (uint32_t)span : 0u);
    const int64_t p = A.pos0 + at;
    const int64_t c = p / A.grp.chunk, rem = p - c * A.grp.chunk, g = rem >> A.grp.log2gs;
    T.scales[b] = uniform_ptr(A.scales + c * A.grp.per_chunk + g);
    T.low[b] = (uint32_t)uniform((int)(rem & (A.grp.gs - 1)));
    const int64_t edge = A.grp.chunk - (g << A.grp.log2gs);
    const bool reaches = edge < (int64_t)T.low[b] + (WIDE ? A.K : RG * A.ldc);     // RG * ldc < 2^29, K < 2^30
    T.edge[b] = (uint32_t)uniform(reaches ? (int)edge : -1);
    T.edge_group[b] = (uint32_t)uniform((int)(A.grp.per_chunk - g));
  }
  return T;
}

// Group of pair o of base b.  Past the first boundary within the task a pair is d = o - edge pairs into
// the following chunks; there are several only if a chunk is shorter than the base's rows.
template <int RG, bool WIDE>
__device__ __forceinline__ uint32_t dr_group(const DualRowsArgs& A, const DrTask<RG, WIDE>& T, int b, uint32_t o) {
  if (T.edge[b] == 0xFFFFFFFFu) return o >> A.grp.log2gs;
  if (o < T.edge[b]) return o >> A.grp.log2gs;
  uint32_t d = o - T.edge[b], g = T.edge_group[b];
  if (d >= A.grp.chunk) {
    const uint32_t q = d / (uint32_t)A.grp.chunk;
    d -= q * (uint32_t)A.grp.chunk;
    g += q * (uint32_t)A.grp.per_chunk;
  }
  return g + (d >> A.grp.log2gs);
}

template <int MT>
struct DrX {
  rsrc_t r[MT];
};

template <int MT, int RG>
struct DrStep {
  u32x4 q[RG];
  f16 sc[RG];
  u32x4 x[MT];
};

// A lane past the part's columns reads 0 for its pairs and activations, and the scale of the
// part's last pairs (not used: dr_compute).
template <int MT, int RG, bool WIDE>
__device__ __forceinline__ void dr_issue(const DualRowsArgs& A, const DrTask<RG, WIDE>& T, const DrX<MT>& X, int k, int lane,
                                         DrStep<MT, RG>& S) {
  const int kk = k + 8 * lane, ld = (int)A.ldc;
  const bool in = kk < T.k1;
  const uint32_t voff = 2u * (uint32_t)(kk - T.k0);
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    if constexpr (WIDE) vload128(S.q[r], in ? voff : OOB, T.codes[r]);
    else vload128(S.q[r], in ? voff + 2u * (uint32_t)(r * ld) : OOB, T.codes[0]);
  }
  const uint32_t k8 = (uint32_t)max(0, min(kk, T.k1 - 8));
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    if constexpr (WIDE) {
      S.sc[r] = T.scales[r][dr_group(A, T, r, T.low[r] + k8)];
    } else {
      const int row = max(0, min(r, T.nrows - 1));
      S.sc[r] = T.scales[0][dr_group(A, T, 0, T.low[0] + k8 + (uint32_t)(row * ld))];
    }
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) vload128c(S.x[j], in ? 2u * (uint32_t)kk : OOB, X.r[j]);
}

__device__ __forceinline__ f16 dr_x(const u32x4& x, int e) {
  const uint32_t w = e < 2 ? x.x : e < 4 ? x.y : e < 6 ? x.z : x.w;
  return __builtin_bit_cast(f16, (unsigned short)((e & 1) ? (w >> 16) : w));
}

// A lane's 8 pairs of a row share one group scale (8 | gs, 8 | chunk, 8 | positions), which
// multiplies their partial sum once.  From 3 tokens on the amplitude goes into (cos, sin)
// rather than into every token's activation.
template <int MT, int RG, int LAYOUT>
__device__ __forceinline__ void dr_compute(const char* lds, const DualLane& dl, const DrStep<MT, RG>& S, bool valid,
                                           float (&acc)[RG][2][MT]) {
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    const uint32_t d4[4] = {S.q[r].x, S.q[r].y, S.q[r].z, S.q[r].w};
    float l1[MT], l2[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) l1[j] = l2[j] = 0.f;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float an[2];
      float2 cs[2];
      dual_lookup2<LAYOUT>(lds, d4[h], dl, an, cs);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float wc = an[u] * cs[u].x, ws = an[u] * cs[u].y;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          const float x = (float)dr_x(S.x[j], 2 * h + u);
          if constexpr (MT < 3) {
            l1[j] = fmaf(an[u] * x, cs[u].x, l1[j]);
            l2[j] = fmaf(an[u] * x, cs[u].y, l2[j]);
          } else {
            l1[j] = fmaf(x, wc, l1[j]);
            l2[j] = fmaf(x, ws, l2[j]);
          }
        }
      }
    }
    const float sc = valid ? (float)S.sc[r] : 0.f;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      acc[r][0][j] = fmaf(sc, l1[j], acc[r][0][j]);
      acc[r][1][j] = fmaf(sc, l2[j], acc[r][1][j]);
    }
  }
}

// One window of 64 plug entries: entry e of the lane, if it lies in the task's rows, with what
// its correction x * (plug - amp_lut * scale) * (cos, sin) needs.
template <int MT>
struct DrPlug {
  int row;                 // row in the task, -1 for none
  uint32_t code;
  f16 sc, amp;
  f16 x[MT];
};

template <int MT, int RG, bool WIDE>
__device__ __forceinline__ bool dr_plug_issue(const DualRowsArgs& A, const DrTask<RG, WIDE>& T, int64_t e, uint32_t idx,
                                              DrPlug<MT>& P) {
  const int64_t pos = A.pos0 + (int64_t)T.row0 * A.ldc;
  const int64_t off = e < A.plug_n ? (int64_t)idx - pos : -1;
  const bool in = e < A.plug_n && off < (int64_t)T.nrows * A.ldc;       // ascending: the window ends past the rows
  P.row = -1;
  if (in && off >= 0) {
    int row = 0;
#pragma unroll
    for (int r = 1; r < RG; ++r) row += off >= (int64_t)r * A.ldc ? 1 : 0;
    const int64_t k = off - (int64_t)row * A.ldc;
    if (k < A.K) {
      P.row = row;
      P.code = A.codes[(int64_t)(T.row0 + row) * A.ldc + k];
      if constexpr (WIDE) {
#pragma unroll
        for (int r = 0; r < RG; ++r)
          if (r == row) P.sc = T.scales[r][dr_group(A, T, r, T.low[r] + (uint32_t)k)];
      } else {
        P.sc = T.scales[0][dr_group(A, T, 0, T.low[0] + (uint32_t)off)];
      }
      P.amp = A.plug_amp[e];
#pragma unroll
      for (int j = 0; j < MT; ++j) P.x[j] = j < A.M ? A.x[(int64_t)j * A.x_sm + k] : (f16)0.f;
    }
  }
  return __ballot(in) != 0;
}

template <int MT, int RG, int LAYOUT>
__device__ __forceinline__ void dr_plug_apply(const char* lds, const DualLane& dl, const DrPlug<MT>& P,
                                              float (&acc)[RG][2][MT]) {
  if (P.row < 0) return;
  float an;
  float2 cs;
  dual_lookup1(lds, dual_half<LAYOUT>(P.code), dl, an, cs);
  const float d = (float)P.amp - an * (float)P.sc;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const float xd = (float)P.x[j] * d;
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      acc[r][0][j] = r == P.row ? fmaf(xd, cs.x, acc[r][0][j]) : acc[r][0][j];
      acc[r][1][j] = r == P.row ? fmaf(xd, cs.y, acc[r][1][j]) : acc[r][1][j];
    }
  }
}

template <int MT, int RG, int LAYOUT, bool WIDE>
__global__ __launch_bounds__(DR_NT) void dual_rows_kernel(const DualRowsArgs A) {
  constexpr int MP = MT == 3 ? 4 : MT;              // the reduction takes a power of two
  constexpr int NV = RG * 2 * MP, LNV = Log2<NV>::v;
  __shared__ __attribute__((aligned(16))) char lds[DLDS_BYTES + 2 * DR_WAVES * NV * 4];
  float* red = reinterpret_cast<float*>(lds + DLDS_BYTES);
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const int parts = uniform(A.parts), groups = DR_WAVES / parts;
  const int part = wave % parts;
  const DualLane dl = dual_lane(lane);
  DrX<MT> X;
#pragma unroll
  for (int j = 0; j < MT; ++j) X.r[j] = make_rsrc(A.x + (int64_t)min(j, A.M - 1) * A.x_sm, j < A.M ? 2u * (uint32_t)A.K : 0u);
  DrTask<RG, WIDE> T;
  DrStep<MT, RG> s0, s1;
  int64_t e0 = 0;          // the lane's entry in the part's first window
  uint32_t idx0 = 0;
  auto task = [&](int round) {
    T = dr_task<RG, WIDE>(A, (int)blockIdx.x + (int)gridDim.x * (wave / parts + groups * round), part);
    if (T.nrows > 0) dr_issue<MT, RG, WIDE>(A, T, X, T.k0, lane, s0);
  };
  auto window = [&]() {
    if (A.plug_n == 0 || T.nrows == 0) return;
    e0 = wave_lower_bound(A.plug_idx, A.plug_n, A.pos0 + (int64_t)T.row0 * A.ldc, lane) + 64 * part + lane;
    idx0 = A.plug_idx[min(e0, A.plug_n - 1)];
  };
  // the first chunk, then the LUTs, then the search: their round trips overlap
  task(0);
  if (A.luts.dtype == PP_F16) {
    DualTables<DR_NT, LAYOUT, f16> tb;
    tb.load(A.luts);
    window();
    tb.store(lds);
  } else {
    DualTables<DR_NT, LAYOUT, float> tb;
    tb.load(A.luts);
    window();
    tb.store(lds);
  }
  for (int round = 0; round < A.rounds; ++round) {
    if (round > 0) {
      task(round);
      window();
    }
    float acc[RG][2][MT];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[r][0][j] = acc[r][1][j] = 0.f;
    if (T.nrows > 0) {
      // the task's entries, 64 a window, the windows dealt over its parts
      DrPlug<MT> P;
      bool more = A.plug_n > 0 && dr_plug_issue<MT, RG, WIDE>(A, T, e0, idx0, P);
      for (int k = T.k0; k < T.k1; k += 2 * DR_CHUNK) {
        dr_issue<MT, RG, WIDE>(A, T, X, k + DR_CHUNK, lane, s1);
        dr_compute<MT, RG, LAYOUT>(lds, dl, s0, k + 8 * lane < T.k1, acc);
        if (k + DR_CHUNK >= T.k1) break;
        dr_issue<MT, RG, WIDE>(A, T, X, k + 2 * DR_CHUNK, lane, s0);
        dr_compute<MT, RG, LAYOUT>(lds, dl, s1, k + DR_CHUNK + 8 * lane < T.k1, acc);
      }
      for (int64_t e = e0; more;) {
        dr_plug_apply<MT, RG, LAYOUT>(lds, dl, P, acc);
        e += 64 * parts;
        more = dr_plug_issue<MT, RG, WIDE>(A, T, e, A.plug_idx[min(e, A.plug_n - 1)], P);
      }
    }
    float v[NV];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int j = 0; j < MP; ++j) v[(r * 2 + m) * MP + j] = j < MT ? acc[r][m][j] : 0.f;
    float y = wave_transpose_reduce<LNV>(v, lane);
    constexpr int LOW = 6 - LNV;
    const bool owns = (lane & ((1 << LOW) - 1)) == 0;
    const int i = lane >> LOW;
    auto store = [&](int t, int vi, float val) {
      const int r = vi / (2 * MP), m = vi / MP % 2, j = vi % MP, row = t * RG + r;
      if (t < A.tasks && row < A.N && j < A.M)
        (m == 0 ? A.out[0] : A.out[1])[(int64_t)j * A.o_sm + (int64_t)row * A.o_sn] = (f16)val;
    };
    if (parts == 1) {
      if (owns) store((int)blockIdx.x + (int)gridDim.x * (wave + groups * round), i, y);
      continue;
    }
    // two buffers in turn: a wave writes a buffer again only after the next round's barrier,
    // which every reader of this round has passed
    float* rb = red + (round & 1) * DR_WAVES * NV;
    if (owns) rb[wave * NV + i] = y;
    __syncthreads();
    if ((int)threadIdx.x < groups * NV) {
      const int g = threadIdx.x / NV, vi = threadIdx.x % NV;
      float s = 0.f;
      for (int p = 0; p < parts; ++p) s += rb[(g * parts + p) * NV + vi];
      store((int)blockIdx.x + (int)gridDim.x * (g + groups * round), vi, s);
    }
  }
}

// ------------------------------------------------------------------------------------------
// generic path
struct DualDequantArgs {
  const void* codes;
  int layout;
  int64_t c_sk, c_sn, elem_base;
  const f16* scales;
  DualGroup grp;
  DualLuts luts;
  void* out[2];   // O[K*N] each
  int64_t N, K;
};

// Small decode tables for the element-wise kernel: a wave's random reads conflict in a
// few banks, which costs less than the three global gathers per element they replace.
struct DualDqLds {
  float amp[64];
  float2 cs[1024];
};

template <typename O>
__device__ __forceinline__ void dual_dequant_at(const DualDqLds& T, const DualDequantArgs& A, int64_t e, int64_t k,
                                                int64_t n, int64_t g) {
  const int64_t off = k * A.c_sk + n * A.c_sn;
  const uint32_t raw = reinterpret_cast<const uint16_t*>(A.codes)[off];
  const uint32_t code = A.layout == PP_DUAL_U16_BE ? (((raw & 0xFFu) << 8) | (raw >> 8)) : (raw ^ 0x8000u);
  if (g < 0) g = A.grp.of_pos(A.elem_base + off);
  const float amp = T.amp[(code >> 10) & 63u] * (float)A.scales[g];
  const float2 cs = T.cs[code & 1023u];
  reinterpret_cast<O*>(A.out[0])[e] = (O)(amp * cs.x);
  reinterpret_cast<O*>(A.out[1])[e] = (O)(amp * cs.y);
}

template <typename O>
__global__ __launch_bounds__(256) void dual_dequant_kernel(const DualDequantArgs A) {
  __shared__ DualDqLds T;
  const DualLuts& L = A.luts;
  for (int i = threadIdx.x; i < 1024; i += blockDim.x) {
    T.cs[i] = i < L.phase_n ? make_float2(lut_at(L.cs[0], L.dtype, i), lut_at(L.cs[1], L.dtype, i))
                            : make_float2(0.f, 0.f);
    if (i < 64) T.amp[i] = i < L.amp_n ? lut_at(L.amp, L.dtype, i) : 0.f;
  }
  __syncthreads();
  const int64_t total = A.N * A.K;
  if (total < (1ll << 32) && A.grp.chunk == 0 && (A.grp.gs & (A.grp.gs - 1)) == 0) {
    // 32-bit index arithmetic (a 64-bit division per element costs more than the decode)
    const uint32_t N = (uint32_t)A.N, tot = (uint32_t)total;
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += gridDim.x * blockDim.x)
      dual_dequant_at<O>(T, A, e, e / N, e % N, e >> A.grp.log2gs);
  } else {
    // e = k*N + n: the kernel rule's group is e / gs; g < 0 asks for the chunked rule
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x)
      dual_dequant_at<O>(T, A, e, e / A.N, e % A.N, A.grp.chunk == 0 ? e / A.grp.gs : -1);
  }
}

// Rows contiguous across columns (c_sn == 1, N % 8 == 0, 16-byte aligned rows) and the
// kernel's group rule with gs a power of two >= 8: a thread decodes 8 consecutive
// columns of one row (one 16-byte code load, one group scale, two stores of 8 values).
template <typename O>
__global__ __launch_bounds__(256) void dual_dequant_vec_kernel(const DualDequantArgs A) {
  __shared__ DualDqLds T;
  const DualLuts& L = A.luts;
  for (int i = threadIdx.x; i < 1024; i += blockDim.x) {
    T.cs[i] = i < L.phase_n ? make_float2(lut_at(L.cs[0], L.dtype, i), lut_at(L.cs[1], L.dtype, i))
                            : make_float2(0.f, 0.f);
    if (i < 64) T.amp[i] = i < L.amp_n ? lut_at(L.amp, L.dtype, i) : 0.f;
  }
  __syncthreads();
  const uint32_t N8 = (uint32_t)(A.N / 8), tot8 = (uint32_t)(A.N * A.K / 8);
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < tot8; v += gridDim.x * blockDim.x) {
    const uint32_t k = v / N8, n = 8u * (v - k * N8), e = 8u * v;
    const u32x4 q = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(A.codes) +
                                                    (int64_t)k * A.c_sk + n);
    const float sc = (float)A.scales[e >> A.grp.log2gs];
    const uint32_t w4[4] = {q.x, q.y, q.z, q.w};
    float o1[8], o2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t raw = (w4[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
      const uint32_t code = A.layout == PP_DUAL_U16_BE ? (((raw & 0xFFu) << 8) | (raw >> 8)) : (raw ^ 0x8000u);
      const float amp = T.amp[(code >> 10) & 63u] * sc;
      const float2 cs = T.cs[code & 1023u];
      o1[i] = amp * cs.x;
      o2[i] = amp * cs.y;
    }
    if constexpr (sizeof(O) == 2) {
      // 8 fp16 values as one 16-byte store per output
      u32x4 h1, h2;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t a = __builtin_bit_cast(unsigned short, (f16)o1[2 * i]);
        const uint32_t b = __builtin_bit_cast(unsigned short, (f16)o1[2 * i + 1]);
        const uint32_t c = __builtin_bit_cast(unsigned short, (f16)o2[2 * i]);
        const uint32_t d = __builtin_bit_cast(unsigned short, (f16)o2[2 * i + 1]);
        h1[i] = a | (b << 16);
        h2[i] = c | (d << 16);
      }
      *reinterpret_cast<u32x4*>(reinterpret_cast<O*>(A.out[0]) + e) = h1;
      *reinterpret_cast<u32x4*>(reinterpret_cast<O*>(A.out[1]) + e) = h2;
    } else {
      float4* d1 = reinterpret_cast<float4*>(reinterpret_cast<O*>(A.out[0]) + e);
      float4* d2 = reinterpret_cast<float4*>(reinterpret_cast<O*>(A.out[1]) + e);
      d1[0] = make_float4(o1[0], o1[1], o1[2], o1[3]);
      d1[1] = make_float4(o1[4], o1[5], o1[6], o1[7]);
      d2[0] = make_float4(o2[0], o2[1], o2[2], o2[3]);
      d2[1] = make_float4(o2[4], o2[5], o2[6], o2[7]);
    }
  }
}

struct DualPlugScatterArgs {
  const void* codes;
  int layout;
  int64_t c_sk, c_sn, elem_base;
  const uint32_t* plug_idx;
  const f16* plug_amp;
  int64_t plug_n;
  DualLuts luts;
  void* out[2];
  int64_t N, K;
  int64_t o_k, o_n;   // output element of (k, n): k*o_k + n*o_n
};

template <typename O>
__global__ void dual_plug_scatter_kernel(const DualPlugScatterArgs A) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= A.plug_n) return;
  const int64_t off = (int64_t)A.plug_idx[j] - A.elem_base;
  if (off < 0) return;
  int64_t k, n;
  if (A.c_sk == 1) {
    n = off / A.c_sn;
    k = off - n * A.c_sn;
  } else {
    k = off / A.c_sk;
    n = off - k * A.c_sk;
  }
  if (k >= A.K || n >= A.N) return;
  const uint32_t raw = reinterpret_cast<const uint16_t*>(A.codes)[off];
  const uint32_t code = A.layout == PP_DUAL_U16_BE ? (((raw & 0xFFu) << 8) | (raw >> 8)) : (raw ^ 0x8000u);
  const int ph = (int)(code & 1023u);
  const float amp = (float)A.plug_amp[j];
  const float c = ph < A.luts.phase_n ? lut_at(A.luts.cs[0], A.luts.dtype, ph) : 0.f;
  const float s = ph < A.luts.phase_n ? lut_at(A.luts.cs[1], A.luts.dtype, ph) : 0.f;
  reinterpret_cast<O*>(A.out[0])[k * A.o_k + n * A.o_n] = (O)(amp * c);
  reinterpret_cast<O*>(A.out[1])[k * A.o_k + n * A.o_n] = (O)(amp * s);
}

// Transposed decode (dequant_t.h): int16 / big-endian codes (K,N), row stride c_sk (unit
// column stride), the kernel group rule (k*N + n) / gs with gs a power of two >= 8 ->
// out_m (N,K) row-major fp16.  8 codes of a row share one group scale.
struct DualDequantTArgs {
  const void* codes;
  int layout;
  int64_t c_sk;
  const f16* scales;
  int log2gs;
  DualLuts luts;
  f16* out[2];
  int64_t N, K;
};

struct DualDecT {
  const DualDqLds& T;
  const DualDequantTArgs& A;
  struct Raw {
    u32x4 q;
    float sc;
  };
  __device__ __forceinline__ Raw load(int64_t k, int64_t n) const {
    return Raw{*reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(A.codes) + k * A.c_sk + n),
               (float)A.scales[(k * A.N + n) >> A.log2gs]};
  }
  __device__ __forceinline__ void decode(const Raw& r, float (&v)[2][8]) const {
    const uint32_t w4[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t raw = (w4[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
      const uint32_t code = A.layout == PP_DUAL_U16_BE ? (((raw & 0xFFu) << 8) | (raw >> 8)) : (raw ^ 0x8000u);
      const float amp = T.amp[(code >> 10) & 63u] * r.sc;
      const float2 cs = T.cs[code & 1023u];
      v[0][i] = amp * cs.x;
      v[1][i] = amp * cs.y;
    }
  }
};

__global__ __launch_bounds__(DQT_NT) void dual_dequant_t_kernel(const DualDequantTArgs A) {
  __shared__ DualDqLds T;
  __shared__ __attribute__((aligned(16))) char tile[2 * DQT_T * 128];
  const DualLuts& L = A.luts;
  for (int i = threadIdx.x; i < 1024; i += blockDim.x) {
    T.cs[i] = i < L.phase_n ? make_float2(lut_at(L.cs[0], L.dtype, i), lut_at(L.cs[1], L.dtype, i))
                            : make_float2(0.f, 0.f);
    if (i < 64) T.amp[i] = i < L.amp_n ? lut_at(L.amp, L.dtype, i) : 0.f;
  }
  __syncthreads();
  f16* const out[2] = {A.out[0], A.out[1]};
  dequant_t_tiles<2>(DualDecT{T, A}, tile, A.N, A.K, out);
}

struct DualWsGemmArgs {
  const f16* a;
  int64_t a_sm, a_sk;
  const float* w[2];
  f16* out[2];
  int64_t o_sm, o_sn;
  int64_t M, N, K;
};

__global__ __launch_bounds__(256) void dual_ws_gemm_kernel(const DualWsGemmArgs A) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = blockIdx.y;
  if (n >= A.N) return;
  float a0 = 0.f, a1 = 0.f;
  const f16* ar = A.a + i * A.a_sm;
  for (int64_t k = 0; k < A.K; ++k) {
    const float av = (float)ar[k * A.a_sk];
    a0 = fmaf(av, A.w[0][k * A.N + n], a0);
    a1 = fmaf(av, A.w[1][k * A.N + n], a1);
  }
  A.out[0][i * A.o_sm + n * A.o_sn] = (f16)a0;
  A.out[1][i * A.o_sm + n * A.o_sn] = (f16)a1;
}

// ------------------------------------------------------------------------------------------
// host side

static bool dual_fast_ok(const void* a, int64_t a_sm, int64_t a_sk, const void* codes, int64_t c_sk, int64_t c_sn,
                         int64_t elem_base, int64_t chunk, int64_t gs, int64_t M, int64_t K) {
  return c_sk == 1 && c_sn % 8 == 0 && c_sn >= K && K % 8 == 0 && K > 0 && aligned(codes, 16) && M >= 1 &&
         M <= 4 && chunk > 0 && chunk % 8 == 0 && gs >= 8 && (gs & (gs - 1)) == 0 && elem_base % 8 == 0 &&
         (a_sk == 1 || K == 1) && (M == 1 || a_sm % 4 == 0) && aligned(a, 8) &&
         K < (1ll << 30);             // 32-bit offsets in a row
}

struct DualRowsPlan {
  int rg, tasks, parts, rounds;
};

// Rows per task (8 or 4, from 3 tokens 4 or 2), parts of K per task (1, 2, 4 or 8 neighbouring
// waves of a workgroup) and rounds of tasks.  Two costs decide, both in rows x chunks: what the
// busiest workgroup decodes (its 8 waves share the CU's units) and what its slowest wave does
// one after another, an item's reduction and stores counted as a chunk of 4 rows.  Wide rows take the
// smaller tasks, whose rows' bases stay in scalar registers.
static DualRowsPlan dual_rows_plan(int mt, int64_t N, int64_t K, bool wide) {
  const int64_t chunks = (K + DR_CHUNK - 1) / DR_CHUNK, cus = device_cu_count();
  DualRowsPlan best = {};
  int64_t least = INT64_MAX;
  for (int rg = (mt <= 2 ? 8 : 4) >> wide; rg >= (mt <= 2 ? 4 : 2); rg /= 2) {
    const int64_t tasks = (N + rg - 1) / rg;
    for (int parts = 1; parts <= DR_WAVES && parts <= chunks; parts *= 2) {
      const int64_t slots = cus * (DR_WAVES / parts), rounds = (tasks + slots - 1) / slots;
      const int64_t wave = rounds * (rg * ((chunks + parts - 1) / parts) + 4);
      const int64_t group = (tasks + cus - 1) / cus * (rg * chunks + 4 * parts);
      const int64_t cost = wave + group / 4;
      if (cost < least) {
        least = cost;
        best = {rg, (int)tasks, parts, (int)rounds};
      }
    }
  }
  return best;
}

template <int MT, int RG, int LAYOUT, bool WIDE = false>
static int launch_dual_rows(const DualRowsArgs& A, hipStream_t st) {
  hipLaunchKernelGGL((dual_rows_kernel<MT, RG, LAYOUT, WIDE>), dim3((unsigned)std::min(device_cu_count(), A.tasks)),
                     dim3(DR_NT), 0, st, A);
  PP_LAUNCH_CHECK();
  return PP_OK;
}

template <int LAYOUT>
static int dispatch_dual_rows(const DualRowsArgs& A, int mt, int rg, bool wide, hipStream_t st) {
  if (wide) {
    switch (mt) {
      case 1: return launch_dual_rows<1, 4, LAYOUT, true>(A, st);
      case 2: return launch_dual_rows<2, 4, LAYOUT, true>(A, st);
      case 3: return launch_dual_rows<3, 2, LAYOUT, true>(A, st);
      default: return launch_dual_rows<4, 2, LAYOUT, true>(A, st);
    }
  }
  switch (mt) {
    case 1: return rg == 8 ? launch_dual_rows<1, 8, LAYOUT>(A, st) : launch_dual_rows<1, 4, LAYOUT>(A, st);
    case 2: return rg == 8 ? launch_dual_rows<2, 8, LAYOUT>(A, st) : launch_dual_rows<2, 4, LAYOUT>(A, st);
    case 3: return rg == 4 ? launch_dual_rows<3, 4, LAYOUT>(A, st) : launch_dual_rows<3, 2, LAYOUT>(A, st);
    default: return rg == 4 ? launch_dual_rows<4, 4, LAYOUT>(A, st) : launch_dual_rows<4, 2, LAYOUT>(A, st);
  }
}

static DualLuts make_dual_luts(const void* amp, int amp_n, const void* c, const void* s, int phase_n, int dtype) {
  DualLuts L;
  L.amp = amp;
  L.cs[0] = c;
  L.cs[1] = s;
  L.amp_n = amp_n;
  L.phase_n = phase_n;
  L.dtype = dtype;
  return L;
}

}  // namespace pp

using namespace pp;

static int dual_common_checks(const void* codes, int code_layout, int64_t group_size, int64_t chunk_size,
                              const void* amp_lut, int amp_lut_n, const void* cos_lut, const void* sin_lut,
                              int phase_n, int lut_dtype, int64_t plug_n, const uint32_t* plug_idx,
                              const void* plug_amp, int64_t c_sk, int64_t c_sn, int64_t N, int64_t K) {
  PP_REQUIRE(code_layout == PP_DUAL_I16_OFFSET || code_layout == PP_DUAL_U16_BE, "bad code_layout");
  PP_REQUIRE(lut_dtype == PP_F16 || lut_dtype == PP_F32, "bad lut_dtype");
  PP_REQUIRE(amp_lut && cos_lut && sin_lut, "lut pointers are null");
  PP_REQUIRE(amp_lut_n >= 1 && amp_lut_n <= 64, "amp_lut_n must be 1..64 (6 amplitude bits)");
  PP_REQUIRE(phase_n >= 1 && phase_n <= 1024, "phase_n must be 1..1024 (10 phase bits)");
  PP_REQUIRE(group_size >= 1 && chunk_size >= 0, "bad group_size / chunk_size");
  PP_REQUIRE(plug_n >= 0 && (plug_n == 0 || (plug_idx && plug_amp)), "plug arrays are null");
  PP_REQUIRE(plug_n == 0 || (c_sk == 1 && c_sn >= K) || (c_sn == 1 && c_sk >= N),
             "plug entries need a unit-stride (K,N) view");
  PP_REQUIRE(codes != nullptr || N * K == 0, "codes is null");
  return PP_OK;
}

extern "C" int64_t pp_dual_gemm_workspace_size(const void* a, int64_t a_sm, int64_t a_sk, const void* codes,
                                               int64_t c_sk, int64_t c_sn, int64_t group_size, int64_t chunk_size,
                                               int64_t elem_base, int64_t plug_n, int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0) return 0;
  if (dual_fast_ok(a, a_sm, a_sk, codes, c_sk, c_sn, elem_base, chunk_size, group_size, M, K))
    return 0;
  // (K,N) codes: blocks of up to 8 tokens, one after another, sharing the workspace (the
  // last block may have 1..7 tokens: the larger of the 4- and 8-token needs covers it)
  if (dual_kn_ok(a, a_sm, a_sk, codes, c_sk, c_sn, group_size, chunk_size, std::min<int64_t>(M, 8), N, K))
    return std::max(dual_kn_workspace(std::min<int64_t>(M, 8), N, K, plug_n),
                    dual_kn_workspace(std::min<int64_t>(M, 4), N, K, plug_n));
  return 2 * N * K * (int64_t)sizeof(float);
}

template <typename O>
static int dual_dequant_to(const void* codes, int code_layout, int64_t c_sk, int64_t c_sn, const void* bmax,
                               int64_t group_size, int64_t chunk_size, const void* amp_lut, int amp_lut_n,
                               const void* cos_lut, const void* sin_lut, int phase_n, int lut_dtype,
                               const uint32_t* plug_idx, const void* plug_amp, int64_t plug_n, int64_t elem_base,
                               void* out1, void* out2, int64_t N, int64_t K, void* stream) {
  if (int rc = dual_common_checks(codes, code_layout, group_size, chunk_size, amp_lut, amp_lut_n, cos_lut, sin_lut,
                                  phase_n, lut_dtype, plug_n, plug_idx, plug_amp, c_sk, c_sn, N, K))
    return rc;
  PP_REQUIRE(out1 && out2 && bmax, "out / bmax pointers are null");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (N * K == 0) return PP_OK;
  DualDequantArgs A;
  A.codes = codes;
  A.layout = code_layout;
  A.c_sk = c_sk;
  A.c_sn = c_sn;
  A.elem_base = elem_base;
  A.scales = reinterpret_cast<const f16*>(bmax);
  A.grp.gs = group_size;
  A.grp.chunk = chunk_size;
  A.grp.per_chunk = chunk_size > 0 ? (chunk_size + group_size - 1) / group_size : 0;
  A.grp.log2gs = 0;
  while ((1ll << A.grp.log2gs) < group_size) ++A.grp.log2gs;
  A.luts = make_dual_luts(amp_lut, amp_lut_n, cos_lut, sin_lut, phase_n, lut_dtype);
  A.out[0] = out1;
  A.out[1] = out2;
  A.N = N;
  A.K = K;
  const bool vec = c_sn == 1 && c_sk % 8 == 0 && N % 8 == 0 && aligned(codes, 16) && chunk_size == 0 &&
                   group_size >= 8 && (group_size & (group_size - 1)) == 0 && N * K < (1ll << 32) &&
                   aligned(out1, 16) && aligned(out2, 16);
  if (vec) {
    const int64_t blocks = std::min<int64_t>((N * K / 8 + 255) / 256, (int64_t)device_cu_count() * 8);
    hipLaunchKernelGGL(dual_dequant_vec_kernel<O>, dim3((unsigned)blocks), dim3(256), 0, st, A);
  } else {
    const int64_t blocks = std::min<int64_t>((N * K + 255) / 256, (int64_t)device_cu_count() * 16);
    hipLaunchKernelGGL(dual_dequant_kernel<O>, dim3((unsigned)blocks), dim3(256), 0, st, A);
  }
  PP_LAUNCH_CHECK();
  if (plug_n > 0) {
    DualPlugScatterArgs P;
    P.codes = codes;
    P.layout = code_layout;
    P.c_sk = c_sk;
    P.c_sn = c_sn;
    P.elem_base = elem_base;
    P.plug_idx = plug_idx;
    P.plug_amp = reinterpret_cast<const f16*>(plug_amp);
    P.plug_n = plug_n;
    P.luts = A.luts;
    P.out[0] = out1;
    P.out[1] = out2;
    P.N = N;
    P.K = K;
    P.o_k = N;
    P.o_n = 1;
    hipLaunchKernelGGL(dual_plug_scatter_kernel<O>, dim3((unsigned)((plug_n + 255) / 256)), dim3(256), 0, st, P);
    PP_LAUNCH_CHECK();
  }
  return PP_OK;
}

extern "C" int pp_dual_dequant(const void* codes, int code_layout, int64_t c_sk, int64_t c_sn, const void* bmax,
                               int64_t group_size, int64_t chunk_size, const void* amp_lut, int amp_lut_n,
                               const void* cos_lut, const void* sin_lut, int phase_n, int lut_dtype,
                               const uint32_t* plug_idx, const void* plug_amp, int64_t plug_n, int64_t elem_base,
                               float* out1, float* out2, int64_t N, int64_t K, void* stream) {
  return dual_dequant_to<float>(codes, code_layout, c_sk, c_sn, bmax, group_size, chunk_size, amp_lut, amp_lut_n,
                                cos_lut, sin_lut, phase_n, lut_dtype, plug_idx, plug_amp, plug_n, elem_base, out1,
                                out2, N, K, stream);
}

extern "C" int pp_dual_dequant_f16(const void* codes, int code_layout, int64_t c_sk, int64_t c_sn,
                                   const void* bmax, int64_t group_size, int64_t chunk_size, const void* amp_lut,
                                   int amp_lut_n, const void* cos_lut, const void* sin_lut, int phase_n,
                                   int lut_dtype, const uint32_t* plug_idx, const void* plug_amp, int64_t plug_n,
                                   int64_t elem_base, void* out1, void* out2, int64_t N, int64_t K, void* stream) {
  return dual_dequant_to<f16>(codes, code_layout, c_sk, c_sn, bmax, group_size, chunk_size, amp_lut, amp_lut_n,
                              cos_lut, sin_lut, phase_n, lut_dtype, plug_idx, plug_amp, plug_n, elem_base, out1,
                              out2, N, K, stream);
}

extern "C" int pp_dual_dequant_f16_t(const void* codes, int code_layout, int64_t c_sk, const void* bmax,
                                     int64_t group_size, const void* amp_lut, int amp_lut_n, const void* cos_lut,
                                     const void* sin_lut, int phase_n, int lut_dtype, const uint32_t* plug_idx,
                                     const void* plug_amp, int64_t plug_n, int64_t elem_base, void* out1,
                                     void* out2, int64_t N, int64_t K, void* stream) {
  if (int rc = dual_common_checks(codes, code_layout, group_size, 0, amp_lut, amp_lut_n, cos_lut, sin_lut, phase_n,
                                  lut_dtype, plug_n, plug_idx, plug_amp, c_sk, 1, N, K))
    return rc;
  PP_REQUIRE(out1 && out2 && bmax, "out / bmax pointers are null");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (N * K == 0) return PP_OK;
  PP_REQUIRE(N % 8 == 0 && K % 8 == 0 && c_sk >= N && c_sk % 8 == 0 && aligned(codes, 16),
             "the transposed decode needs N % 8 == 0, K % 8 == 0 and 16-byte aligned code rows "
             "(row stride >= N, a multiple of 8)");
  PP_REQUIRE(group_size >= 8 && (group_size & (group_size - 1)) == 0,
             "the transposed decode needs a power-of-two group_size >= 8");
  PP_REQUIRE(aligned(out1, 16) && aligned(out2, 16), "outputs must be 16-byte aligned");
  DualDequantTArgs A;
  A.codes = codes;
  A.layout = code_layout;
  A.c_sk = c_sk;
  A.scales = reinterpret_cast<const f16*>(bmax);
  A.log2gs = 0;
  while ((1ll << A.log2gs) < group_size) ++A.log2gs;
  A.luts = make_dual_luts(amp_lut, amp_lut_n, cos_lut, sin_lut, phase_n, lut_dtype);
  A.out[0] = reinterpret_cast<f16*>(out1);
  A.out[1] = reinterpret_cast<f16*>(out2);
  A.N = N;
  A.K = K;
  const int64_t tiles = ((N + DQT_T - 1) / DQT_T) * ((K + DQT_T - 1) / DQT_T);
  // 24.3 KiB of LDS a workgroup: six fit a CU (with the next-tile loads, 21.0 against 22.7 us
  // for a 4096 x 4096 pair with four and no prefetch)
  const int64_t blocks = std::min<int64_t>(tiles, (int64_t)device_cu_count() * 6);
  hipLaunchKernelGGL(dual_dequant_t_kernel, dim3((unsigned)blocks), dim3(DQT_NT), 0, st, A);
  PP_LAUNCH_CHECK();
  if (plug_n > 0) {
    DualPlugScatterArgs P;
    P.codes = codes;
    P.layout = code_layout;
    P.c_sk = c_sk;
    P.c_sn = 1;
    P.elem_base = elem_base;
    P.plug_idx = plug_idx;
    P.plug_amp = reinterpret_cast<const f16*>(plug_amp);
    P.plug_n = plug_n;
    P.luts = A.luts;
    P.out[0] = out1;
    P.out[1] = out2;
    P.N = N;
    P.K = K;
    P.o_k = 1;
    P.o_n = K;
    hipLaunchKernelGGL(dual_plug_scatter_kernel<f16>, dim3((unsigned)((plug_n + 255) / 256)), dim3(256), 0, st, P);
    PP_LAUNCH_CHECK();
  }
  return PP_OK;
}

extern "C" int pp_dual_gemm_kernel(const void* a, int64_t a_sm, int64_t a_sk, const void* codes, int64_t c_sk,
                                   int64_t c_sn, int64_t group_size, int64_t chunk_size, int64_t elem_base,
                                   int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (dual_fast_ok(a, a_sm, a_sk, codes, c_sk, c_sn, elem_base, chunk_size, group_size, M, K)) return PP_GEMM_ROWS;
  if (dual_kn_ok(a, a_sm, a_sk, codes, c_sk, c_sn, group_size, chunk_size, std::min<int64_t>(M, 8), N, K))
    return PP_GEMM_KN;
  return PP_GEMM_GENERIC;
}

extern "C" int pp_dual_gemm(const void* a, int64_t a_sm, int64_t a_sk, const void* codes, int code_layout,
                            int64_t c_sk, int64_t c_sn, const void* bmax, int64_t group_size, int64_t chunk_size,
                            const void* amp_lut, int amp_lut_n, const void* cos_lut, const void* sin_lut,
                            int phase_n, int lut_dtype, const uint32_t* plug_idx, const void* plug_amp,
                            int64_t plug_n, int64_t elem_base, void* out1, void* out2, int64_t o_sm, int64_t o_sn,
                            int64_t M, int64_t N, int64_t K, void* workspace, int64_t workspace_bytes,
                            void* stream) {
  if (int rc = dual_common_checks(codes, code_layout, group_size, chunk_size, amp_lut, amp_lut_n, cos_lut, sin_lut,
                                  phase_n, lut_dtype, plug_n, plug_idx, plug_amp, c_sk, c_sn, N, K))
    return rc;
  PP_REQUIRE(M >= 0 && N >= 0 && K >= 0, "negative shape");
  PP_REQUIRE(out1 && out2 && bmax, "out / bmax pointers are null");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (M == 0 || N == 0) return PP_OK;
  PP_REQUIRE(a != nullptr, "a is null");
  PP_REQUIRE(N < (1ll << 31) && K < (1ll << 31), "N and K must be < 2^31");
  const DualLuts L = make_dual_luts(amp_lut, amp_lut_n, cos_lut, sin_lut, phase_n, lut_dtype);
  if (dual_fast_ok(a, a_sm, a_sk, codes, c_sk, c_sn, elem_base, chunk_size, group_size, M, K)) {
    const int mt = (int)M;
    const bool wide = c_sn >= DR_WIDE;
    const DualRowsPlan p = dual_rows_plan(mt, N, K, wide);
    DualRowsArgs A = {};
    A.codes = reinterpret_cast<const uint16_t*>(codes);
    A.ldc = c_sn;
    A.pos0 = elem_base;
    A.x = reinterpret_cast<const f16*>(a);
    A.x_sm = a_sm;
    A.out[0] = reinterpret_cast<f16*>(out1);
    A.out[1] = reinterpret_cast<f16*>(out2);
    A.o_sm = o_sm;
    A.o_sn = o_sn;
    A.N = (int)N;
    A.K = (int)K;
    A.M = (int)M;
    A.tasks = p.tasks;
    A.parts = p.parts;
    A.rounds = p.rounds;
    A.scales = reinterpret_cast<const f16*>(bmax);
    A.grp.gs = group_size;
    A.grp.chunk = chunk_size;
    A.grp.per_chunk = (chunk_size + group_size - 1) / group_size;
    A.grp.log2gs = 0;
    while ((1ll << A.grp.log2gs) < group_size) ++A.grp.log2gs;
    A.luts = L;
    A.plug_idx = plug_idx;
    A.plug_amp = reinterpret_cast<const f16*>(plug_amp);
    A.plug_n = plug_n;
    return code_layout == PP_DUAL_U16_BE ? dispatch_dual_rows<PP_DUAL_U16_BE>(A, mt, p.rg, wide, st)
                                         : dispatch_dual_rows<PP_DUAL_I16_OFFSET>(A, mt, p.rg, wide, st);
  }
  if (dual_kn_ok(a, a_sm, a_sk, codes, c_sk, c_sn, group_size, chunk_size, std::min<int64_t>(M, 8), N, K)) {
    for (int64_t i0 = 0; i0 < M; i0 += 8) {
      void* o[2] = {reinterpret_cast<f16*>(out1) + i0 * o_sm, reinterpret_cast<f16*>(out2) + i0 * o_sm};
      if (int rc = dual_kn_gemm(reinterpret_cast<const f16*>(a) + i0 * a_sm, a_sm, codes, code_layout, c_sk, bmax,
                                group_size, L, plug_idx, plug_amp, plug_n, elem_base, o, o_sm, o_sn,
                                std::min<int64_t>(8, M - i0), N, K, workspace, workspace_bytes, st))
        return rc;
    }
    return PP_OK;
  }
  const int64_t need = 2 * N * K * (int64_t)sizeof(float);
  PP_REQUIRE(workspace != nullptr && workspace_bytes >= need, "workspace too small: need %lld bytes",
             (long long)need);
  float* w0 = reinterpret_cast<float*>(workspace);
  float* w1 = w0 + N * K;
  if (int rc = pp_dual_dequant(codes, code_layout, c_sk, c_sn, bmax, group_size, chunk_size, amp_lut, amp_lut_n,
                               cos_lut, sin_lut, phase_n, lut_dtype, plug_idx, plug_amp, plug_n, elem_base, w0, w1,
                               N, K, stream))
    return rc;
  DualWsGemmArgs G;
  G.a = reinterpret_cast<const f16*>(a);
  G.a_sm = a_sm;
  G.a_sk = a_sk;
  G.w[0] = w0;
  G.w[1] = w1;
  G.out[0] = reinterpret_cast<f16*>(out1);
  G.out[1] = reinterpret_cast<f16*>(out2);
  G.o_sm = o_sm;
  G.o_sn = o_sn;
  G.M = M;
  G.N = N;
  G.K = K;
  hipLaunchKernelGGL(dual_ws_gemm_kernel, dim3((unsigned)((N + 255) / 256), (unsigned)M), dim3(256), 0, st, G);
  PP_LAUNCH_CHECK();
  return PP_OK;
}
