// Dual decode of container (N,K) rows (.dualpack layout) for 1 to 32 tokens on the matrix cores:
// out_m[j, n] = fp16(sum_k x[j, k] * W_m[n, k]), each weight rounded to fp16, plug amplitudes
// substituted (polar_kernels.py:60-86, polar_bitpack.py:240-243).
//
// The work is split as in quad_tile.hip: `group` tiles of 16 rows (x a slice of K) a workgroup, cut
// into 8 equal runs of 32-column steps, a run in at most two tiles, the runs' sums meeting in LDS
// over the tables.  At the format's 1 % of plug entries almost every step of 16 x 32 pairs holds
// some, so a wavefront finds its run's entries while the LUTs travel and keeps them in LDS, row by
// row (from the table itself where they do not fit): dual_nk_mfma_kernel reloads windows of 4 from
// the table and waits for them nearly every step, and needs a launch before it to find the rows'
// entries and one after it to read the atomics' sums.  Per call in a graph (1 % plug), against it:
// 11008 x 2048 at 3 / 16 / 32 tokens 78.1 / 79.9 / 83.3 -> 34.3 / 35.5 / 36.2 us; 2048 x 11008 at 1 / 16
// 58.0 / 59.3 -> 34.5 / 36.2; 4096 x 4096 at 16 46.5 -> 28.4; 1000 x 512 at 5 17.8 -> 11.7.
#include "dual_lds.h"
#include "row_tiles.h"
#include "rows_common.h"
#include "slice_sums.h"

namespace pp {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int DT_NT = 64 * RT_WAVES;
constexpr int64_t DT_MAX_M = 32;
constexpr int DT_CAP = 960;                               // a wavefront's plug entries in LDS
template <int T> constexpr int DT_SUB = T == 1 ? 4 : 2;   // steps a load stage
static_assert(DLDS_BYTES + RT_WAVES * DT_CAP * 4 <= 160 * 1024, "tables and entries must fit a CU's LDS");

struct DualTileArgs {
  const uint16_t* codes;   // row n at codes + n*ldc
  int64_t ldc;
  int64_t pos0;            // stream position of (row 0, column 0)
  const f16* x;            // (M, K), row stride x_sm
  int64_t x_sm;
  f16* out[2];             // (M, N), row stride o_sm
  int64_t o_sm;
  int N, K, M;
  int tiles, group, slices;
  int vec_out;             // outputs 8-byte aligned, o_sm % 4 == 0
  const f16* scales;       // the stream's group scales
  int64_t n_groups;
  int chunk, log2gs;       // chunk size (>= 32, a multiple of 8), log2 of the group size
  int64_t gpc;             // groups a chunk
  DualLuts luts;
  const uint32_t* plug_idx;
  const f16* plug_amp;
  int64_t plug_n;
  float* part;             // slices > 1: float32 sums, [slice][model][token][16 tiles]
};

// The chunk index and offset of a lane's next load position (no division but at a segment's start).
struct DtPos {
  int64_t c;
  int r;
  __device__ __forceinline__ void set(int64_t p, int chunk) {
    c = p / chunk;
    r = (int)(p - c * chunk);
  }
  __device__ __forceinline__ void advance32(int chunk) {   // chunk >= 32
    r += 32;
    const bool w = r >= chunk;
    r = w ? r - chunk : r;
    c += w ? 1 : 0;
  }
};

template <int T>
struct DtStage {
  u32x4 c[DT_SUB<T>];      // per step: 8 stored codes of the lane's row
  uint32_t sc[DT_SUB<T>];  // their group scale
  u32x4 xb[DT_SUB<T>][T];  // 8 fp16 x of token 16t + l%16
};

// The stage at column k of segment S, `pos` the lane's position there.  Steps past the segment's end
// have resources of no bytes; rows past N lie past the resource's end.  Neighbouring steps share the
// codes' lines, so the loads keep the caches' policy.
template <int T>
__device__ __forceinline__ void dt_issue(const DualTileArgs& A, const RowSeg& S, int k, DtPos& pos, uint32_t voc,
                                         const uint32_t (&vox)[T], DtStage<T>& D) {
  const int nrows = min(16, A.N - 16 * S.tile);
#pragma unroll
  for (int u = 0; u < DT_SUB<T>; ++u) {
    const bool in = k + 32 * u < S.ke;
    const int kc = in ? k + 32 * u : 0;
    const rsrc_t rc = make_rsrc(A.codes + (int64_t)S.tile * 16 * A.ldc + kc,
                                in ? 2u * (uint32_t)((int64_t)(nrows - 1) * A.ldc + (A.K - kc)) : 0u);
    vload128c(D.c[u], voc, rc);
    const int64_t g = pos.c * A.gpc + (pos.r >> A.log2gs);
    vload16(D.sc[u], g < A.n_groups ? 2u * (uint32_t)g : OOB, make_rsrc(A.scales, in ? 2u * (uint32_t)A.n_groups : 0u));
    pos.advance32(A.chunk);
    const rsrc_t rx = make_rsrc(A.x + kc, in ? 2u * (uint32_t)((int64_t)(A.M - 1) * A.x_sm + (A.K - kc)) : 0u);
#pragma unroll
    for (int t = 0; t < T; ++t) vload128c(D.xb[u][t], vox[t], rx);
  }
}

// A wavefront's plug entries: lists 16 s + i, row i of its segment s.
struct DtPlugs {
  int64_t from = 0;        // first entry of the wave's rows in the table
  int at = 0;              // lane 16 a + i: place (from `from`) of row i's start / end in segment 0, 1 (a = 0..3)
  int n = 0, base = 0;     // lane l < 32: list l's entries and its first place in LDS
  bool held = true;        // the lists are in LDS

  __device__ __forceinline__ void find(const DualTileArgs& A, const RowSeg (&S)[2], int lane) {
    const int64_t top = A.pos0 + (int64_t)min(A.N, 16 * (S[1].tile + 1)) * A.ldc;
    const int tile = lane >= 32 ? S[1].tile : S[0].tile, row = 16 * tile + (lane & 15);
    const int kb = lane >= 32 ? S[1].kb : S[0].kb, ke = lane >= 32 ? S[1].ke : S[0].ke;
    const int64_t key = A.pos0 + (int64_t)row * A.ldc + ((lane & 16) ? ke : kb);
    from = wave_lower_bound(A.plug_idx, A.plug_n, A.pos0 + (int64_t)S[0].tile * 16 * A.ldc, lane);
    const int all = (int)wave_lower_bound(A.plug_idx + from, A.plug_n - from, top, lane);
    if (all == 0) return;
    // 64 samples of the rows' entries, searched in registers, then the entries between two of them
    const int step = (all + 63) / 64;
    const bool has = lane * step < all;
    const uint32_t mine = has ? A.plug_idx[from + lane * step] : 0u;
    const int samples = __popcll(__ballot(has));
    int c = 0;                                             // samples below the key
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
      const uint32_t probe = (uint32_t)__shfl((int)mine, min(c + s, 64) - 1);
      c += c + s <= samples && (int64_t)probe < key ? s : 0;
    }
    const uint32_t last = (uint32_t)__shfl((int)mine, 63);
    c += c == 63 && samples == 64 && (int64_t)last < key ? 1 : 0;
    int lo = c == 0 ? 0 : (c - 1) * step + 1, hi = c == 0 ? 0 : min(all, c * step);
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      const bool below = (int64_t)A.plug_idx[from + mid] < key;
      lo = below ? mid + 1 : lo;
      hi = below ? hi : mid;
    }
    at = lo;
  }
  // The lists into the wave's part of LDS: (column from the segment's first) << 16 | amplitude.
  __device__ __forceinline__ void keep(const DualTileArgs& A, const RowSeg (&S)[2], int lane, uint32_t* ent) {
    const int s = lane >> 4 & 1, row = 16 * (s ? S[1].tile : S[0].tile) + (lane & 15);
    const int b = __shfl(at, 32 * s + (lane & 15)), e = __shfl(at, 32 * s + 16 + (lane & 15));
    const bool some = s ? S[1].ke > S[1].kb : S[0].ke > S[0].kb;
    n = lane < 32 && row < A.N && some ? e - b : 0;
    int sum = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(sum, o);
      sum += lane >= o ? v : 0;
    }
    base = sum - n;
    const int total = uniform(__shfl(sum, 63));
    held = total <= DT_CAP && max(S[0].ke - S[0].kb, S[1].ke - S[1].kb) <= 65536;
    if (!held) {
      base = b;
      return;
    }
    for (int t0 = 0; t0 < total; t0 += 64) {
      const int t = min(t0 + lane, total - 1);
      int l = 0;                                           // the last list that starts at or before t
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) l += __shfl(base, l + o) <= t ? o : 0;
      const int src = __shfl(b, l) + t - __shfl(base, l);
      const RowSeg g = (l & 16) ? S[1] : S[0];
      const int64_t first = A.pos0 + (int64_t)(16 * g.tile + (l & 15)) * A.ldc + g.kb;
      const uint32_t k = A.plug_idx[from + src] - (uint32_t)first;
      const uint32_t amp = __builtin_bit_cast(unsigned short, A.plug_amp[from + src]);
      if (t0 + lane < total) ent[t] = (k << 16) | amp;
    }
  }
};

template <int T>
struct DtRun {
  const DualTileArgs& A;
  RowSeg S[2];
  int nseg;
  uint32_t voc, vox[T];
  int ri, q;
  DtPos pos;
  // the row's entries still to come: the first one's column and amplitude, and the places of the rest
  const uint32_t* ent;
  int64_t from;
  bool held;
  int near, next, end, next1, end1;
  float amp0;
  f4 C[2][T], H[2][T];     // the segment at hand, and the first one once there is a second

  __device__ __forceinline__ int64_t row_pos(int tile) const { return A.pos0 + (int64_t)(16 * tile + ri) * A.ldc; }

  // The next entry of the row in segment s.
  __device__ __forceinline__ void entry(const RowSeg& s) {
    if (next >= end) {
      near = 0x7FFFFFFF;
    } else if (held) {
      const uint32_t v = ent[next++];
      near = s.kb + (int)(v >> 16);
      amp0 = h2f(v & 0xFFFFu);
    } else {
      near = (int)((int64_t)A.plug_idx[from + next] - row_pos(s.tile));
      amp0 = (float)A.plug_amp[from + next];
      ++next;
    }
  }

  // Stage (sg, k) decoded from `cur` while the next one travels; false after the last.
  template <int LAYOUT>
  __device__ __forceinline__ bool step(const char* lds, const DualLane& dl, const DtStage<T>& cur, DtStage<T>& pre,
                                       int& sg, int& k) {
    constexpr int SUB = DT_SUB<T>;
    const RowSeg s = sg == 0 ? S[0] : S[1];
    int nsg = sg, nk = k + 32 * SUB;
    if (nk >= s.ke) {
      nsg = sg + 1;
      nk = nsg < nseg ? S[1].kb : S[1].ke;            // past the run: an empty stage
      if (nsg < nseg) pos.set(row_pos(S[1].tile) + nk + 8 * q, A.chunk);
    }
    dt_issue<T>(A, nsg == 0 ? S[0] : S[1], nk, pos, voc, vox, pre);
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
      const int ks = k + 32 * u, kk = ks + 8 * q;
      if (ks >= s.ke) break;
      const float sc = h2f(cur.sc[u]);
      const uint32_t w4[4] = {cur.c[u].x, cur.c[u].y, cur.c[u].z, cur.c[u].w};
      float amp[8];
      float2 cs[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float an[2];
        float2 c2[2];
        dual_lookup2<LAYOUT>(lds, w4[e], dl, an, c2);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          amp[2 * e + h] = an[h] * sc;
          cs[2 * e + h] = c2[h];
        }
      }
      while (__ballot(near < ks + 32)) {
        const int e = near - kk;                      // outside 0..7: another lane of the row holds it
#pragma unroll
        for (int ee = 0; ee < 8; ++ee) amp[ee] = e == ee ? amp0 : amp[ee];
        if (near < ks + 32) entry(s);
      }
      h8 a[2];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float v[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          v[0][h] = amp[e + h] * cs[e + h].x;
          v[1][h] = amp[e + h] * cs[e + h].y;
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          // the float32 product, then fp16, as the reference rounds it: not one rounding of both
          asm("" : "+v"(v[m][0]), "+v"(v[m][1]));
          const f16x2 p = __builtin_convertvector((f2{v[m][0], v[m][1]}), f16x2);
          a[m][e] = p.x;
          a[m][e + 1] = p.y;
        }
      }
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const h8 b = __builtin_bit_cast(h8, cur.xb[u][t]);
#pragma unroll
        for (int m = 0; m < 2; ++m) C[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[m], b, C[m][t], 0, 0, 0);
      }
    }
    if (nsg != sg && nsg < nseg) {
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int t = 0; t < T; ++t) {
          H[m][t] = C[m][t];
          C[m][t] = f4{0.f, 0.f, 0.f, 0.f};
        }
      next = next1;
      end = end1;
      entry(S[1]);
    }
    sg = nsg;
    k = nk;
    return nsg < nseg;
  }
};

// Rows n .. n + 3 of token j, model m.
__device__ __forceinline__ void dt_store(const DualTileArgs& A, int slice, int m, int j, int n, f4 v) {
  if (j >= A.M || n >= A.N) return;
  if (A.slices > 1) {
    *reinterpret_cast<f4*>(A.part + (((int64_t)slice * 2 + m) * A.M + j) * (16ll * A.tiles) + n) = v;
    return;
  }
  f16* o = (m == 0 ? A.out[0] : A.out[1]) + (int64_t)j * A.o_sm + n;
  if (A.vec_out && n + 3 < A.N) {
    *reinterpret_cast<f16x4*>(o) = f16x4{(f16)v[0], (f16)v[1], (f16)v[2], (f16)v[3]};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < A.N) o[r] = (f16)v[r];
  }
}

template <int T, int LAYOUT>
__global__ __launch_bounds__(DT_NT) void dual_tile_kernel(const DualTileArgs A) {
  __shared__ __attribute__((aligned(16))) char lds[DLDS_BYTES + RT_WAVES * DT_CAP * 4];
  static_assert(RT_WAVES * 2 * 2 * T * 64 * 16 <= DLDS_BYTES, "the runs' sums must fit where the tables were");
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), ri = lane & 15, q = lane >> 4;
  const RowShare W(A, wave);
  DtRun<T> R{A};
  R.nseg = W.nseg;
  R.S[0] = W.S[0];
  R.S[1] = W.S[1];
  R.ri = ri;
  R.q = q;
  R.voc = 2u * (uint32_t)(ri * A.ldc + 8 * q);
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int j = 16 * t + ri;
    R.vox[t] = j < A.M ? 2u * (uint32_t)(j * A.x_sm + 8 * q) : OOB;
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int t = 0; t < T; ++t) R.C[m][t] = R.H[m][t] = f4{0.f, 0.f, 0.f, 0.f};
  uint32_t* ent = reinterpret_cast<uint32_t*>(lds + DLDS_BYTES) + wave * DT_CAP;
  R.ent = ent;
  R.near = 0x7FFFFFFF;
  DtStage<T> D0, D1;
  // the first stage and the plug entries travel under the table build
  auto early = [&]() {
    if (R.nseg == 0) return;
    R.pos.set(R.row_pos(R.S[0].tile) + R.S[0].kb + 8 * q, A.chunk);
    dt_issue<T>(A, R.S[0], R.S[0].kb, R.pos, R.voc, R.vox, D0);
    DtPlugs F;
    if (A.plug_n > 0) {
      F.find(A, R.S, lane);
      F.keep(A, R.S, lane, ent);
    }
    R.from = F.from;
    R.held = F.held;
    R.next = __shfl(F.base, ri);
    R.end = R.next + __shfl(F.n, ri);
    R.next1 = __shfl(F.base, 16 + ri);
    R.end1 = R.next1 + __shfl(F.n, 16 + ri);
  };
  if (A.luts.dtype == PP_F16) {
    DualTables<DT_NT, LAYOUT, f16> tb;
    tb.load(A.luts);
    early();
    tb.store(lds);
  } else {
    DualTables<DT_NT, LAYOUT, float> tb;
    tb.load(A.luts);
    early();
    tb.store(lds);
  }
  if (R.nseg > 0) {
    const DualLane dl = dual_lane(lane);
    R.entry(R.S[0]);
    int sg = 0, k = R.S[0].kb;
    for (;;) {
      if (!R.template step<LAYOUT>(lds, dl, D0, D1, sg, k)) break;
      if (!R.template step<LAYOUT>(lds, dl, D1, D0, sg, k)) break;
    }
  }
  __syncthreads();         // every wave is done with the tables
  row_sums<2, T>(reinterpret_cast<f4*>(lds), W, R, wave, lane, [&](int tile, int m, int t, f4 v) {
    dt_store(A, W.slice, m, 16 * t + ri, 16 * (W.t0 + tile) + 4 * q, v);
  });
}

// ------------------------------------------------------------------ host side
// A step takes about half as long as the quad kernel's, so a second pass counts 8 of them.
static RowPlan dual_tile_plan(int64_t N, int64_t K) { return row_plan(N, K, 8); }

}  // namespace pp

using namespace pp;

extern "C" int pp_dual_tile_ok(int64_t ldc, int64_t elem_base, int64_t a_sm, int64_t group_size, int64_t chunk_size,
                               int64_t plug_n, int64_t M, int64_t N, int64_t K) {
  if (M < 1 || M > DT_MAX_M || N < 1 || N >= (1ll << 30) || K < 32 || K % 32 != 0 || ldc < K || ldc % 8 != 0) return 0;
  if (elem_base < 0 || elem_base % 8 != 0 || group_size < 8 || (group_size & (group_size - 1)) != 0) return 0;
  if (chunk_size < 32 || chunk_size % 8 != 0 || chunk_size >= (1ll << 30)) return 0;
  if (32 * ldc >= (1ll << 31) || (M > 1 && (a_sm < K || a_sm % 8 != 0)) || (M - 1) * a_sm + K >= (1ll << 30)) return 0;
  return plug_n >= 0 && plug_n < (1ll << 29) && dual_tile_plan(N, K).group > 0;
}

extern "C" int64_t pp_dual_tile_workspace_size(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 32) return 0;
  const RowPlan p = dual_tile_plan(N, K);
  return p.slices > 1 ? (int64_t)p.slices * 2 * M * ((N + 15) / 16 * 16) * (int64_t)sizeof(float) : 0;
}

extern "C" int pp_dual_tile(const void* codes, int code_layout, int64_t ldc, int64_t elem_base, const void* a,
                            int64_t a_sm, const void* scales, int64_t n_groups, int64_t group_size, int64_t chunk_size,
                            const void* amp_lut, int64_t amp_n, const void* cos_lut, const void* sin_lut,
                            int64_t phase_n, int lut_dtype, const uint32_t* plug_idx, const void* plug_amp,
                            int64_t plug_n, void* out1, void* out2, int64_t o_sm, int64_t M, int64_t N, int64_t K,
                            void* workspace, int64_t workspace_bytes, void* stream) {
  PP_REQUIRE(codes && a && scales && amp_lut && cos_lut && sin_lut && out1 && out2, "null pointer argument");
  PP_REQUIRE(code_layout == PP_DUAL_U16_BE || code_layout == PP_DUAL_I16_OFFSET, "bad code_layout");
  PP_REQUIRE(lut_dtype == PP_F16 || lut_dtype == PP_F32, "bad lut_dtype");
  PP_REQUIRE(amp_n >= 1 && amp_n <= 64 && phase_n >= 1 && phase_n <= 1024, "amp_n must be 1..64, phase_n 1..1024");
  PP_REQUIRE(pp_dual_tile_ok(ldc, elem_base, a_sm, group_size, chunk_size, plug_n, M, N, K) && aligned(codes, 16) &&
                 aligned(a, 16), "operands the tile kernel does not read");
  PP_REQUIRE(n_groups >= 1 && n_groups < (1ll << 30), "n_groups must be in [1, 2^30)");
  PP_REQUIRE(o_sm >= N, "o_sm must be >= N");
  PP_REQUIRE(plug_n == 0 || (plug_idx && plug_amp), "plug arrays are null");
  const RowPlan p = dual_tile_plan(N, K);
  const int64_t need = pp_dual_tile_workspace_size(M, N, K);
  PP_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && aligned(workspace, 16)),
             "workspace too small or misaligned: need %lld bytes", (long long)need);
  DualTileArgs A = {};
  A.codes = reinterpret_cast<const uint16_t*>(codes);
  A.ldc = ldc;
  A.pos0 = elem_base;
  A.x = reinterpret_cast<const f16*>(a);
  A.x_sm = M > 1 ? a_sm : K;
  A.out[0] = reinterpret_cast<f16*>(out1);
  A.out[1] = reinterpret_cast<f16*>(out2);
  A.o_sm = o_sm;
  A.vec_out = (M == 1 || o_sm % 4 == 0) && aligned(out1, 8) && aligned(out2, 8);
  A.N = (int)N;
  A.K = (int)K;
  A.M = (int)M;
  A.tiles = (int)((N + 15) / 16);
  A.group = p.group;
  A.slices = p.slices;
  A.scales = reinterpret_cast<const f16*>(scales);
  A.n_groups = n_groups;
  A.chunk = (int)chunk_size;
  A.log2gs = 63 - __builtin_clzll((unsigned long long)group_size);
  A.gpc = (chunk_size + group_size - 1) / group_size;
  A.luts.amp = amp_lut;
  A.luts.cs[0] = cos_lut;
  A.luts.cs[1] = sin_lut;
  A.luts.amp_n = (int)amp_n;
  A.luts.phase_n = (int)phase_n;
  A.luts.dtype = lut_dtype;
  A.plug_idx = plug_idx;
  A.plug_amp = reinterpret_cast<const f16*>(plug_amp);
  A.plug_n = plug_n;
  A.part = reinterpret_cast<float*>(workspace);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)((A.tiles + p.group - 1) / p.group * p.slices)), block(DT_NT);
  const bool be = code_layout == PP_DUAL_U16_BE;
  if (M <= 16 && be) hipLaunchKernelGGL((dual_tile_kernel<1, PP_DUAL_U16_BE>), grid, block, 0, st, A);
  else if (M <= 16) hipLaunchKernelGGL((dual_tile_kernel<1, PP_DUAL_I16_OFFSET>), grid, block, 0, st, A);
  else if (be) hipLaunchKernelGGL((dual_tile_kernel<2, PP_DUAL_U16_BE>), grid, block, 0, st, A);
  else hipLaunchKernelGGL((dual_tile_kernel<2, PP_DUAL_I16_OFFSET>), grid, block, 0, st, A);
  PP_LAUNCH_CHECK();
  if (p.slices > 1) {
    SliceSums<2> F = {};
    F.part = A.part;
    F.np = 16ll * A.tiles;
    F.out[0] = A.out[0];
    F.out[1] = A.out[1];
    F.o_sm = o_sm;
    F.o_sn = 1;
    F.N = A.N;
    F.M = A.M;
    F.slices = p.slices;
    F.vec_out = A.vec_out;
    launch_slice_sums(F, st);
    PP_LAUNCH_CHECK();
  }
  return PP_OK;
}
