// Quad decode of (N,K) rows (a container's layout) for 1 to 32 tokens on the matrix cores:
// out_m[j, n] = fp16(s_m * sum_k x[j, k] * W_m[n, k]) with the plug table patched into the decoded
// weights (quad_kernels.py:103-134, quaternion_packer.py:173-193).
//
// A workgroup of 8 wavefronts takes `group` neighbouring tiles of 16 rows (and, where N alone
// leaves the chip idle, a slice of K); the group's steps of 32 columns are cut into 8 equal runs,
// one a wavefront, each in at most two tiles (group <= 8).  The runs' sums meet in LDS, over the
// tables, once every wavefront is done.  quad_mfma_kernel (more tokens, explicit slices) gives a
// wavefront one tile x slice: 11008 x 2048 made 1,376 items for 2,048 wavefronts, 1.4 million
// atomic adds and launches to find the rows' plug entries and to read the sums back.  Here a
// wavefront finds its rows' entries itself while the LUTs travel, and one slice needs no second
// launch.  The decode takes ~19 vector instructions and 4 LDS reads (14 LDS clocks a wavefront) a
// word; at two wavefronts a SIMD, all the tables leave room for, the vector units are busy 45 % and
// LDS 23 % of the time (SQ counters), so what bounds it is the latency of a step's loads and lookups.
// Per call in a graph (0.1 % plug), against quad_mfma_kernel: 11008 x 2048 at 5 / 16 tokens 46.3 / 49.4
// -> 30.8 / 31.9 us; 4096 x 4096 38.1 / 38.7 -> 24.1 / 24.6; 2048 x 2048 28.5 / 24.7 -> 14.6 / 15.4.
#include "quad_mfma.h"
#include "row_tiles.h"
#include "slice_sums.h"

namespace pp {

typedef float f2 __attribute__((ext_vector_type(2)));

constexpr int QT_NT = 64 * RT_WAVES;
constexpr int64_t QT_MAX_M = 32;
// Steps a load stage (3 fit the registers beside two tiles' sums, and were 1 us slower at 16 tokens).
template <int T> constexpr int QT_SUB = T == 1 ? 2 : 1;

struct QuadTileArgs {
  const uint32_t* codes;   // code of (row 0, col 0); row n at codes + n*ldc
  int64_t ldc;
  int64_t pos0;            // stream position of (row 0, col 0)
  const f16* x;            // (M, K), row stride x_sm
  int64_t x_sm;
  f16* out[4];             // (M, N), row stride o_sm
  int64_t o_sm;
  int N, K, M;
  int tiles, group, slices;
  int vec_out;             // outputs 8-byte aligned, o_sm % 4 == 0
  QuadLuts luts;
  float s[4];
  PlugSrc plug;
  float* part;             // slices > 1: float32 sums, [slice][model][token][16 tiles]
};

template <int T>
struct TileStage {
  u32x4 c[QT_SUB<T>][2];   // per step: 8 code words of the lane's row
  u32x4 xb[QT_SUB<T>][T];  // per step: 8 fp16 x of token 16t + l%16
};

// The stage at column k of segment S.  Steps past the segment's end have resources of no bytes:
// they read 0, cost no traffic and are not used.  Rows past N lie past the resource's end.  Two
// loads share each 128-byte line, so the codes keep the caches' policy: with the streaming one
// 11008 x 2048 at 16 tokens took 35.6 us for 32.3.
template <int T>
__device__ __forceinline__ void tile_issue(const QuadTileArgs& A, const RowSeg& S, int k, uint32_t voc,
                                           const uint32_t (&vox)[T], TileStage<T>& D) {
  const int nrows = min(16, A.N - 16 * S.tile);
#pragma unroll
  for (int u = 0; u < QT_SUB<T>; ++u) {
    const bool in = k + 32 * u < S.ke;
    const int kc = in ? k + 32 * u : 0;
    const rsrc_t rc = make_rsrc(A.codes + (int64_t)S.tile * 16 * A.ldc + kc,
                                in ? 4u * (uint32_t)((int64_t)(nrows - 1) * A.ldc + (A.K - kc)) : 0u);
    vload128c(D.c[u][0], voc, rc);
    vload128c(D.c[u][1], voc + 16u, rc);
    const rsrc_t rx = make_rsrc(A.x + kc, in ? 2u * (uint32_t)((int64_t)(A.M - 1) * A.x_sm + (A.K - kc)) : 0u);
#pragma unroll
    for (int t = 0; t < T; ++t) vload128c(D.xb[u][t], vox[t], rx);
  }
}

// The first entry of each of the wave's rows in both its segments: lane 16 a + i searches the
// entries of the wave's rows for row i's start (a = 0) and end (1) in the first segment, and in
// the second (2, 3).
struct TilePlugs {
  int64_t from = 0;
  int at = 0;              // lane 16 a + i: entry from + at
  __device__ __forceinline__ void find(const QuadTileArgs& A, const RowSeg (&S)[2], int lane) {
    const int64_t top = A.pos0 + (int64_t)min(A.N, 16 * (S[1].tile + 1)) * A.ldc;
    const int tile = lane >= 32 ? S[1].tile : S[0].tile, row = 16 * tile + (lane & 15);
    const int kb = lane >= 32 ? S[1].kb : S[0].kb, ke = lane >= 32 ? S[1].ke : S[0].ke;
    const int64_t key = A.pos0 + (int64_t)row * A.ldc + ((lane & 16) ? ke : kb);
    from = wave_lower_bound(A.plug.idx, A.plug.n, A.pos0 + (int64_t)S[0].tile * 16 * A.ldc, lane);
    // Usually (0.1 % of 2 tiles x 2048) the rows' entries fit one window, searched in registers:
    // 4 memory round trips in all, where a search of memory takes 12.
    const int64_t left = A.plug.n - from;
    const uint32_t mine = lane < left ? A.plug.idx[from + lane] : 0xFFFFFFFFu;
    if (__ballot(lane >= left || (int64_t)mine >= top)) {
#pragma unroll
      for (int step = 32; step > 0; step >>= 1) {
        const uint32_t probe = (uint32_t)__shfl((int)mine, at + step - 1);
        at += (int64_t)probe < key ? step : 0;
      }
      at = min(at, (int)min(left, (int64_t)64));
      return;
    }
    int n = (int)wave_lower_bound(A.plug.idx + from, left, top, lane);
    while (n > 0) {
      const int half = n >> 1;
      const bool below = (int64_t)A.plug.idx[from + at + half] < key;
      at = below ? at + half + 1 : at;
      n = below ? n - half - 1 : half;
    }
  }
  // The row's entries of segment s.
  __device__ __forceinline__ void range(const QuadTileArgs& A, const RowSeg& S, int s, int ri, int64_t& next, int64_t& end) const {
    const int b = __shfl(at, 32 * s + ri), e = __shfl(at, 32 * s + 16 + ri);
    const bool ok = 16 * S.tile + ri < A.N && S.ke > S.kb;
    next = ok ? from + b : 0;
    end = ok ? from + e : 0;
  }
};

// 8 code words as the fp16 operands of the 4 models.
template <class L>
__device__ __forceinline__ void tile_decode(const char* lds, const LaneOff& lo, const u32x4& c0, const u32x4& c1,
                                            h8 (&a)[4]) {
  const uint32_t cw[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    float v[4][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float r;
      float2 ta, tb, tc;
      lookup<L>(lds, cw[e + u], lo, r, ta, tb, tc);
      const float rs = r * ta.y, rss = rs * tb.y;
      v[0][u] = r * ta.x;
      v[1][u] = rs * tb.x;
      v[2][u] = rss * tc.x;
      v[3][u] = rss * tc.y;
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      // the float32 product, then fp16, as the reference rounds it: not one rounding of both
      asm("" : "+v"(v[m][0]), "+v"(v[m][1]));
      const f16x2 p = __builtin_convertvector((f2{v[m][0], v[m][1]}), f16x2);
      a[m][e] = p.x;
      a[m][e + 1] = p.y;
    }
  }
}

// Patch the row's plug entries that lie in the step's columns ks .. ks+31 into the lane's 8 columns
// from kk; `near` is the first entry's column not yet passed, the common step's only test.  An
// entry replaces one half of one register a model (a bit select), where mplug_patch selects over
// all 32 halves: 40 % of the steps hold an entry at 0.1 %, and 11008 x 2048 at 16 tokens spent
// 5.6 us of 38 on its entries, 3.4 of 36 this way.
__device__ __forceinline__ void tile_patch(const PlugSrc& S, MPlug& P, int& near, int64_t rowpos, int kk, int ks,
                                           h8 (&a)[4]) {
  if (!__ballot(near < ks + 32)) return;
  u32x4 w[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) w[m] = __builtin_bit_cast(u32x4, a[m]);
  for (;;) {
#pragma unroll
    for (int i = 0; i < MPW; ++i) {
      const int e = P.k[i] - kk;
      if (!__ballot((unsigned)e < 8u)) continue;
      const uint32_t half = (e & 1) ? 0xFFFF0000u : 0xFFFFu;
      const uint32_t v[4] = {(P.v[i][0] & 0xFFFFu) | (P.v[i][0] << 16), (P.v[i][0] >> 16) | (P.v[i][0] & 0xFFFF0000u),
                             (P.v[i][1] & 0xFFFFu) | (P.v[i][1] << 16), (P.v[i][1] >> 16) | (P.v[i][1] & 0xFFFF0000u)};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t mask = (e >> 1) == d ? half : 0u;
#pragma unroll
        for (int m = 0; m < 4; ++m) w[m][d] = (w[m][d] & ~mask) | (v[m] & mask);
      }
    }
    const bool refill = P.k[MPW - 1] < ks + 32 && P.next < P.end;
    if (!__ballot(refill)) break;
    // rare: load and wait here (see mplug_patch_loop); a lane without a refill patches the same again
    uint32_t idx[MPW];
    MPlug R = P;
    mplug_issue(S, R, idx);
#pragma unroll
    for (int i = 0; i < MPW; ++i) asm volatile("" : : "v"(idx[i]), "v"(R.v[i]));
    mplug_take(R, idx, rowpos);
    if (refill) P = R;
  }
  near = 0x7FFFFFFF;
#pragma unroll
  for (int i = 0; i < MPW; ++i) near = P.k[i] >= ks + 32 ? min(near, P.k[i]) : near;
#pragma unroll
  for (int m = 0; m < 4; ++m) a[m] = __builtin_bit_cast(h8, w[m]);
}

template <int T>
struct TileRun {
  const QuadTileArgs& A;
  RowSeg S[2];
  int nseg;
  uint32_t voc, vox[T];
  int ri, q;
  MPlug P;
  int near;                // tile_patch
  int64_t next1, end1;     // the second segment's entries of the row
  int64_t rowpos;
  f4 C[4][T], H[4][T];     // the segment at hand, and the first one once there is a second

  __device__ __forceinline__ int64_t row_pos(int tile) const { return A.pos0 + (int64_t)(16 * tile + ri) * A.ldc; }

  // The first entries of the row of `tile` (waits for them: once a segment, see mplug_patch_loop).
  __device__ __forceinline__ void window(int tile) {
    uint32_t idx[MPW];
    mplug_issue(A.plug, P, idx);
    rowpos = row_pos(tile);
#pragma unroll
    for (int i = 0; i < MPW; ++i) asm volatile("" : : "v"(idx[i]), "v"(P.v[i]));
    mplug_take(P, idx, rowpos);
    near = P.k[0];
  }

  // Stage (sg, k) decoded from `cur` while the next one travels; false after the last.
  template <class L>
  __device__ __forceinline__ bool step(const char* lds, const LaneOff& lo, const TileStage<T>& cur, TileStage<T>& pre,
                                       int& sg, int& k) {
    constexpr int SUB = QT_SUB<T>;
    const int ke = sg == 0 ? S[0].ke : S[1].ke;
    int nsg = sg, nk = k + 32 * SUB;
    if (nk >= ke) {
      nsg = sg + 1;
      nk = nsg < nseg ? S[1].kb : S[1].ke;            // past the run: an empty stage
    }
    tile_issue<T>(A, nsg == 0 ? S[0] : S[1], nk, voc, vox, pre);
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
      const int ks = k + 32 * u;
      if (ks >= ke) break;
      h8 a[4];
      tile_decode<L>(lds, lo, cur.c[u][0], cur.c[u][1], a);
      tile_patch(A.plug, P, near, rowpos, ks + 8 * q, ks, a);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const h8 b = __builtin_bit_cast(h8, cur.xb[u][t]);
#pragma unroll
        for (int m = 0; m < 4; ++m) C[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[m], b, C[m][t], 0, 0, 0);
      }
    }
    if (nsg != sg && nsg < nseg) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int t = 0; t < T; ++t) {
          H[m][t] = C[m][t];
          C[m][t] = f4{0.f, 0.f, 0.f, 0.f};
        }
      P.next = next1;
      P.end = end1;
      window(S[1].tile);
    }
    sg = nsg;
    k = nk;
    return nsg < nseg;
  }
  template <class L>
  __device__ __forceinline__ void walk(const char* lds, const LaneOff& lo, TileStage<T>& s0) {
    if (nseg == 0) return;
    TileStage<T> s1;
    int sg = 0, k = S[0].kb;
    for (;;) {
      if (!step<L>(lds, lo, s0, s1, sg, k)) break;
      if (!step<L>(lds, lo, s1, s0, sg, k)) break;
    }
  }
};

// Rows n .. n + 3 of token j, model m: their sums, scaled.
__device__ __forceinline__ void tile_store(const QuadTileArgs& A, int slice, int m, int j, int n, f4 v) {
  if (j >= A.M || n >= A.N) return;
  const float s = m == 0 ? A.s[0] : m == 1 ? A.s[1] : m == 2 ? A.s[2] : A.s[3];
  v *= s;
  if (A.slices > 1) {
    *reinterpret_cast<f4*>(A.part + (((int64_t)slice * 4 + m) * A.M + j) * (16ll * A.tiles) + n) = v;
    return;
  }
  f16* o = (m == 0 ? A.out[0] : m == 1 ? A.out[1] : m == 2 ? A.out[2] : A.out[3]) + (int64_t)j * A.o_sm + n;
  if (A.vec_out && n + 3 < A.N) {
    *reinterpret_cast<f16x4*>(o) = f16x4{(f16)v[0], (f16)v[1], (f16)v[2], (f16)v[3]};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < A.N) o[r] = (f16)v[r];
  }
}

template <int T>
__global__ __launch_bounds__(QT_NT) void quad_tile_kernel(const QuadTileArgs A) {
  __shared__ __attribute__((aligned(16))) uint32_t Tb[QLDS_BYTES / 4];
  static_assert(RT_WAVES * 2 * 4 * T * 64 * 16 <= QLDS_BYTES, "the runs' sums must fit where the tables were");
  char* lds = reinterpret_cast<char*>(Tb);
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), ri = lane & 15, q = lane >> 4;
  const RowShare W(A, wave);
  TileRun<T> R{A};
  R.nseg = W.nseg;
  R.S[0] = W.S[0];
  R.S[1] = W.S[1];
  R.ri = ri;
  R.q = q;
  R.voc = 4u * (uint32_t)(ri * A.ldc + 8 * q);
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int j = 16 * t + ri;
    R.vox[t] = j < A.M ? 2u * (uint32_t)(j * A.x_sm + 8 * q) : OOB;
  }
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int t = 0; t < T; ++t) R.C[m][t] = R.H[m][t] = f4{0.f, 0.f, 0.f, 0.f};
  TileStage<T> D;
  // the first stage and the plug entries travel under the table build
  auto early = [&]() {
    if (R.nseg == 0) return;
    tile_issue<T>(A, R.S[0], R.S[0].kb, R.voc, R.vox, D);
    TilePlugs F;
    if (A.plug.n > 0) F.find(A, R.S, lane);
    F.range(A, R.S[0], 0, ri, R.P.next, R.P.end);
    F.range(A, R.S[1], 1, ri, R.next1, R.end1);
    R.window(R.S[0].tile);
  };
  bool shared;
  if (A.luts.dtype == PP_F16) {
    QuadTableBuild<QT_NT, f16> tb;
    tb.load(A.luts);
    early();
    shared = tb.finish(Tb, A.luts);
  } else {
    QuadTableBuild<QT_NT, float> tb;
    tb.load(A.luts);
    early();
    shared = tb.finish(Tb, A.luts);
  }
  if (shared) R.template walk<LayShared>(lds, LayShared::lane(lane), D);
  else R.template walk<LaySplit>(lds, LaySplit::lane(lane), D);
  __syncthreads();         // every wave is done with the tables
  row_sums<4, T>(reinterpret_cast<f4*>(lds), W, R, wave, lane, [&](int tile, int m, int t, f4 v) {
    tile_store(A, W.slice, m, 16 * t + ri, 16 * (W.t0 + tile) + 4 * q, v);
  });
}

// ------------------------------------------------------------------ host side
// A step of 8 wavefronts takes about 1 us, a second pass 4-5.
static RowPlan tile_plan(int64_t N, int64_t K) { return row_plan(N, K, 5); }

}  // namespace pp

using namespace pp;

extern "C" int pp_quad_tile_ok(int64_t ldc, int64_t a_sm, int64_t plug_n, int64_t M, int64_t N, int64_t K) {
  if (M < 1 || M > QT_MAX_M || N < 1 || K < 32 || K % 32 != 0 || ldc < K || ldc % 4 != 0) return 0;
  if (64 * ldc >= (1ll << 31) || (M > 1 && (a_sm < K || a_sm % 8 != 0)) || (M - 1) * a_sm + K >= (1ll << 30)) return 0;
  return plug_n >= 0 && plug_n < (1ll << 28) && tile_plan(N, K).group > 0;
}

extern "C" int64_t pp_quad_tile_workspace_size(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 32) return 0;
  const RowPlan p = tile_plan(N, K);
  return p.slices > 1 ? (int64_t)p.slices * 4 * M * ((N + 15) / 16 * 16) * (int64_t)sizeof(float) : 0;
}

extern "C" int pp_quad_tile(const uint32_t* codes, int64_t ldc, int64_t elem_base, const void* a, int64_t a_sm,
                            const void* const* luts, int lut_dtype, const float* scales, const uint32_t* plug_idx,
                            const void* plug_vals, int64_t plug_n, void* const* out, int64_t o_sm, int64_t M, int64_t N,
                            int64_t K, void* workspace, int64_t workspace_bytes, void* stream) {
  PP_REQUIRE(codes != nullptr && a != nullptr && out != nullptr && luts != nullptr && scales != nullptr,
             "null pointer argument");
  for (int m = 0; m < 4; ++m) PP_REQUIRE(out[m] != nullptr, "out[%d] is null", m);
  for (int i = 0; i < 7; ++i) PP_REQUIRE(luts[i] != nullptr, "lut %d is null", i);
  PP_REQUIRE(lut_dtype == PP_F16 || lut_dtype == PP_F32, "bad lut_dtype");
  PP_REQUIRE(pp_quad_tile_ok(ldc, a_sm, plug_n, M, N, K) && aligned(codes, 16) && aligned(a, 16),
             "operands the tile kernel does not read");
  PP_REQUIRE(o_sm >= N, "o_sm must be >= N");
  PP_REQUIRE(plug_n == 0 || (plug_idx && plug_vals), "plug arrays are null");
  const RowPlan p = tile_plan(N, K);
  const int64_t need = pp_quad_tile_workspace_size(M, N, K);
  PP_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && aligned(workspace, 16)),
             "workspace too small or misaligned: need %lld bytes", (long long)need);
  QuadTileArgs A = {};
  A.codes = codes;
  A.ldc = ldc;
  A.pos0 = elem_base;
  A.x = reinterpret_cast<const f16*>(a);
  A.x_sm = M > 1 ? a_sm : K;
  bool vec = M == 1 || o_sm % 4 == 0;
  for (int m = 0; m < 4; ++m) {
    A.out[m] = reinterpret_cast<f16*>(out[m]);
    A.s[m] = scales[m];
    vec = vec && aligned(out[m], 8);
  }
  A.vec_out = vec;
  A.o_sm = o_sm;
  A.N = (int)N;
  A.K = (int)K;
  A.M = (int)M;
  A.tiles = (int)((N + 15) / 16);
  A.group = p.group;
  A.slices = p.slices;
  for (int i = 0; i < 7; ++i) A.luts.p[i] = luts[i];
  A.luts.dtype = lut_dtype;
  A.plug = PlugSrc{plug_idx, reinterpret_cast<const f16*>(plug_vals), plug_n};
  A.part = reinterpret_cast<float*>(workspace);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)((A.tiles + p.group - 1) / p.group * p.slices)), block(QT_NT);
  if (M <= 16) hipLaunchKernelGGL(quad_tile_kernel<1>, grid, block, 0, st, A);
  else hipLaunchKernelGGL(quad_tile_kernel<2>, grid, block, 0, st, A);
  PP_LAUNCH_CHECK();
  if (p.slices > 1) {
    SliceSums<4> F = {};
    F.part = A.part;
    F.np = 16ll * A.tiles;
    for (int m = 0; m < 4; ++m) F.out[m] = A.out[m];
    F.o_sm = o_sm;
    F.o_sn = 1;
    F.N = A.N;
    F.M = A.M;
    F.slices = p.slices;
    F.vec_out = vec;
    launch_slice_sums(F, st);
    PP_LAUNCH_CHECK();
  }
  return PP_OK;
}
