// Dual decode of int16 (K,N) codes (the layout quantize_polar_bitpacked returns) for 1 to 32 tokens
// on the matrix cores, no plug table: out_m[j, n] = fp16(sum_k x[j, k] * W_m[k, n]), each weight
// rounded to fp16 as the reference's tl.dot takes it (polar_kernels.py:60-86).
//
// A workgroup of 8 wavefronts takes a strip of 64 columns and a slice of K, an eighth of the
// slice's rows per wavefront; the wavefronts' sums meet in LDS, over the tables, once all are done.
// A lane's load is 8 bytes of one row (128 contiguous bytes over 16 lanes), whose 4 codes belong to
// 4 matrix tiles: tile j takes columns 4i + j, so the operands need no transpose.  dual_mfma_kernel
// (plug tables, groups that straddle rows, more tokens) gives a wavefront 16 columns: it transposes
// the weights through LDS and adds every slice's sums to memory by atomics.  What bounds both is
// the decode, ~9 vector instructions and 2 LDS reads a code, and at these sizes the fixed cost of
// a launch with its tables.  Per call in a graph, against dual_mfma_kernel: 4096 x 4096 at 8 / 32 tokens
// 28.8 / 34.5 -> 15.4 / 19.2 us; K x N = 1536 x 11008 at 8 / 32 tokens 33.4 / 42.5 -> 15.6 / 18.2; 512 x
// 512 at 8 tokens 13.9 -> 9.4.  Loads two, three or four steps ahead were slower (16.6 / 17.5 / 18.6 us).
#include "dual_lds.h"
#include "rows_common.h"
#include "slice_sums.h"

#include <algorithm>

namespace pp {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int DS_WAVES = 8, DS_NT = 64 * DS_WAVES, DS_COLS = 64;
constexpr int64_t DS_MAX_M = 32;

struct DualStripArgs {
  const uint16_t* codes;   // row k at codes + k*ldk (stored = code ^ 0x8000)
  int64_t ldk;
  const f16* x;            // (M, K), row stride x_sm
  int64_t x_sm;
  f16* out[2];             // (M, N), row stride o_sm
  int64_t o_sm;
  int N, K, M;
  int slices;
  int vec_out;             // outputs 8-byte aligned, o_sm % 4 == 0
  const f16* scales;       // gcols a row of codes
  int gcols, log2gs;
  DualLuts luts;
  float* part;             // slices > 1: float32 sums, [slice][model][token][np]
  int64_t np;              // N rounded up to whole strips
};

template <int TT>
struct DsStep {
  u32x2 c[8];              // row 8 (l / 16) + e: 4 codes
  uint32_t sc[8];          // their group scale
  u32x4 x[TT];             // token 16 t + l % 16, the same rows
};

template <int TT>
struct DsWalk {
  const DualStripArgs& A;
  const char* lds;
  DualLane dl;
  int n0, ke;
  uint32_t voc, vos, vox[TT];

  // Loads of the step at row k; past the wave's rows they read 0 (x among them) without traffic.
  __device__ __forceinline__ void issue(int k, DsStep<TT>& S) const {
    const bool in = k < ke;
    const int kc = min(k, A.K - 32);
    const rsrc_t rc = make_rsrc(A.codes + (int64_t)kc * A.ldk + n0,
                                in ? 2u * (uint32_t)(31 * A.ldk + min(A.N - n0, DS_COLS)) : 0u);
    const rsrc_t rs = make_rsrc(A.scales + (int64_t)kc * A.gcols, in ? 64u * (uint32_t)A.gcols : 0u);
    const rsrc_t rx = make_rsrc(A.x + kc, in ? 2u * (uint32_t)((int64_t)(A.M - 1) * A.x_sm + 32) : 0u);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      S.c[e] = __builtin_amdgcn_raw_buffer_load_b64(rc, (int)(voc + 2u * (uint32_t)(e * A.ldk)), 0, NT_AUX);
#pragma unroll
    for (int e = 0; e < 8; ++e) vload16(S.sc[e], vos + 2u * (uint32_t)(e * A.gcols), rs);
#pragma unroll
    for (int t = 0; t < TT; ++t) vload128c(S.x[t], vox[t], rx);
  }
  // Tiles 2h and 2h + 1 of a step: the lookups of two rows ahead of the arithmetic of the two before.
  __device__ __forceinline__ void pair(const DsStep<TT>& S, int h, f4 (&C)[4][2][TT]) const {
    h8 a[2][2];
    float an[2][2][2];
    float2 cs[2][2][2];
    auto look = [&](int e, int b) {
#pragma unroll
      for (int u = 0; u < 2; ++u) dual_lookup2<PP_DUAL_I16_OFFSET>(lds, S.c[e + u][h], dl, an[b][u], cs[b][u]);
    };
    look(0, 0);
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const int b = e / 2 & 1;
      if (e + 2 < 8) look(e + 2, b ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      const float sc[2] = {h2f(S.sc[e]), h2f(S.sc[e + 1])};
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float v[2][2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const float amp = an[b][u][j] * sc[u];
          v[0][u] = amp * cs[b][u][j].x;
          v[1][u] = amp * cs[b][u][j].y;
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          // the float32 product, then fp16, as the reference rounds it: not one rounding of both
          asm volatile("" : "+v"(v[m][0]), "+v"(v[m][1]));
          const f16x2 p = __builtin_convertvector((f2{v[m][0], v[m][1]}), f16x2);
          a[j][m][e] = p.x;
          a[j][m][e + 1] = p.y;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const h8 x = __builtin_bit_cast(h8, S.x[t]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int m = 0; m < 2; ++m)
          C[2 * h + j][m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j][m], x, C[2 * h + j][m][t], 0, 0, 0);
    }
  }
  __device__ __forceinline__ void step(int k, const DsStep<TT>& cur, DsStep<TT>& nxt, f4 (&C)[4][2][TT]) const {
    issue(k + 32, nxt);
    __builtin_amdgcn_sched_barrier(0);
    pair(cur, 0, C);
    pair(cur, 1, C);
  }
};

template <int TT>
__global__ __launch_bounds__(DS_NT) void dual_strip_kernel(const DualStripArgs A) {
  __shared__ __attribute__((aligned(16))) char lds[DLDS_BYTES];
  static_assert(DS_WAVES * 8 * TT * 64 * 16 <= DLDS_BYTES, "the waves' sums must fit where the tables were");
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), i = lane & 15, q = lane >> 4;
  const int strip = blockIdx.x / A.slices, slice = blockIdx.x % A.slices, n0 = strip * DS_COLS;
  const int64_t units = A.K / 32, parts = (int64_t)DS_WAVES * A.slices, p = (int64_t)slice * DS_WAVES + wave;
  const int kb = (int)(p * units / parts) * 32, ke = (int)((p + 1) * units / parts) * 32;
  DsWalk<TT> W{A, lds, dual_lane(lane), n0, ke};
  const bool ok = n0 + 4 * i < A.N;
  W.voc = ok ? 2u * (uint32_t)(8 * q * A.ldk + 4 * i) : OOB;
  W.vos = ok ? 2u * (uint32_t)(8 * q * A.gcols + ((n0 + 4 * i) >> A.log2gs)) : OOB;
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    const int j = 16 * t + i;
    W.vox[t] = j < A.M ? 2u * (uint32_t)(j * A.x_sm + 8 * q) : OOB;
  }
  DsStep<TT> S0, S1;
  // the first step travels under the table build
  if (A.luts.dtype == PP_F16) {
    DualTables<DS_NT, PP_DUAL_I16_OFFSET, f16> tb;
    tb.load(A.luts);
    W.issue(kb, S0);
    tb.store(lds);
  } else {
    DualTables<DS_NT, PP_DUAL_I16_OFFSET, float> tb;
    tb.load(A.luts);
    W.issue(kb, S0);
    tb.store(lds);
  }
  f4 C[4][2][TT];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int t = 0; t < TT; ++t) C[j][m][t] = f4{0.f, 0.f, 0.f, 0.f};
  for (int k = kb; k < ke; k += 64) {
    W.step(k, S0, S1, C);
    if (k + 32 >= ke) break;     // no step of zeros: the entries that a stored 0 names need not be finite
    W.step(k + 32, S1, S0, C);
  }
  __syncthreads();         // every wave is done with the tables
  f4* red = reinterpret_cast<f4*>(lds);
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[(((wave * 2 + m) * TT + t) * 4 + j) * 64 + lane] = C[j][m][t];
  __syncthreads();
  if (wave >= 2 * TT) return;
  // wave w: model w / TT, token tile w % TT; row r of the lane's sums of tile j is column 16q + 4r + j
  const int m = wave / TT, tok = 16 * (wave % TT) + i;
  f4 v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = red[(wave * 4 + j) * 64 + lane];
#pragma unroll
  for (int w = 1; w < DS_WAVES; ++w)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += red[((w * 2 * TT + wave) * 4 + j) * 64 + lane];
  if (tok >= A.M) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + 16 * q + 4 * r;
    if (n >= A.N) continue;
    const float o[4] = {v[0][r], v[1][r], v[2][r], v[3][r]};
    if (A.slices > 1) {
      float* d = A.part + (((int64_t)slice * 2 + m) * A.M + tok) * A.np + n;
      *reinterpret_cast<float4*>(d) = make_float4(o[0], o[1], o[2], o[3]);
      continue;
    }
    f16* d = (m == 0 ? A.out[0] : A.out[1]) + (int64_t)tok * A.o_sm + n;       // N % 4 == 0
    if (A.vec_out) {
      *reinterpret_cast<f16x4*>(d) = f16x4{(f16)o[0], (f16)o[1], (f16)o[2], (f16)o[3]};
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) d[c] = (f16)o[c];
    }
  }
}

// ------------------------------------------------------------------ host side
// Slices of K: the least of rounds of workgroups x (the longest wave's steps + 4 for the tables,
// the first loads and the sums), and 4 for a second pass over the slices' sums; about 1 us each.
static int dual_strip_slices(int64_t N, int64_t K) {
  const int64_t cus = device_cu_count(), strips = (N + DS_COLS - 1) / DS_COLS, steps = K / 32;
  int best = 1;
  int64_t least = INT64_MAX;
  for (int64_t s = 1; s <= std::min<int64_t>(32, std::max<int64_t>(1, steps / DS_WAVES)); ++s) {
    const int64_t rounds = (strips * s + cus - 1) / cus, per = (steps + DS_WAVES * s - 1) / (DS_WAVES * s);
    const int64_t cost = rounds * (per + 4) + (s > 1 ? 4 : 0);
    if (cost < least) {
      least = cost;
      best = (int)s;
    }
  }
  return best;
}

static int64_t dual_strip_np(int64_t N) { return (N + DS_COLS - 1) / DS_COLS * DS_COLS; }

}  // namespace pp

using namespace pp;

extern "C" int pp_dual_strip_ok(const void* codes, int64_t ldk, const void* a, int64_t a_sm, int64_t group_size,
                                int64_t M, int64_t N, int64_t K) {
  if (M < 1 || M > DS_MAX_M || N < 1 || K < 32 || K % 32 != 0 || N % 4 != 0 || ldk < N || ldk % 4 != 0) return 0;
  if (group_size < 4 || (group_size & (group_size - 1)) != 0 || N % group_size != 0) return 0;
  if (!aligned(codes, 8) || !aligned(a, 16) || (M > 1 && (a_sm < K || a_sm % 8 != 0))) return 0;
  return K * ldk < (1ll << 29) && M * (M > 1 ? a_sm : K) < (1ll << 29);
}

extern "C" int64_t pp_dual_strip_workspace_size(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 32) return 0;
  const int s = dual_strip_slices(N, K);
  return s > 1 ? (int64_t)s * 2 * M * dual_strip_np(N) * (int64_t)sizeof(float) : 0;
}

extern "C" int pp_dual_strip(const void* codes, int64_t ldk, const void* a, int64_t a_sm, const void* scales,
                             int64_t group_size, const void* amp_lut, int64_t amp_n, const void* cos_lut,
                             const void* sin_lut, int64_t phase_n, int lut_dtype, void* out1, void* out2, int64_t o_sm,
                             int64_t M, int64_t N, int64_t K, void* workspace, int64_t workspace_bytes, void* stream) {
  PP_REQUIRE(codes && a && scales && amp_lut && cos_lut && sin_lut && out1 && out2, "null pointer argument");
  PP_REQUIRE(lut_dtype == PP_F16 || lut_dtype == PP_F32, "bad lut_dtype");
  PP_REQUIRE(amp_n >= 1 && amp_n <= 64 && phase_n >= 1 && phase_n <= 1024, "bad LUT sizes");
  PP_REQUIRE(pp_dual_strip_ok(codes, ldk, a, a_sm, group_size, M, N, K), "operands the strip kernel does not read");
  PP_REQUIRE(o_sm >= N, "o_sm must be >= N");
  const int64_t need = pp_dual_strip_workspace_size(M, N, K);
  PP_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && aligned(workspace, 16)),
             "workspace too small or misaligned: need %lld bytes", (long long)need);
  DualStripArgs A = {};
  A.codes = reinterpret_cast<const uint16_t*>(codes);
  A.ldk = ldk;
  A.x = reinterpret_cast<const f16*>(a);
  A.x_sm = M > 1 ? a_sm : K;
  A.out[0] = reinterpret_cast<f16*>(out1);
  A.out[1] = reinterpret_cast<f16*>(out2);
  A.o_sm = o_sm;
  A.vec_out = (M == 1 || o_sm % 4 == 0) && aligned(out1, 8) && aligned(out2, 8);
  A.N = (int)N;
  A.K = (int)K;
  A.M = (int)M;
  A.slices = dual_strip_slices(N, K);
  A.scales = reinterpret_cast<const f16*>(scales);
  A.gcols = (int)(N / group_size);
  A.log2gs = 63 - __builtin_clzll((unsigned long long)group_size);
  A.luts.amp = amp_lut;
  A.luts.cs[0] = cos_lut;
  A.luts.cs[1] = sin_lut;
  A.luts.amp_n = (int)amp_n;
  A.luts.phase_n = (int)phase_n;
  A.luts.dtype = lut_dtype;
  A.part = reinterpret_cast<float*>(workspace);
  A.np = dual_strip_np(N);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)(A.np / DS_COLS * A.slices)), block(DS_NT);
  if (M <= 16) hipLaunchKernelGGL(dual_strip_kernel<1>, grid, block, 0, st, A);
  else hipLaunchKernelGGL(dual_strip_kernel<2>, grid, block, 0, st, A);
  PP_LAUNCH_CHECK();
  if (A.slices > 1) {
    SliceSums<2> F = {};
    F.part = A.part;
    F.np = A.np;
    F.out[0] = A.out[0];
    F.out[1] = A.out[1];
    F.o_sm = o_sm;
    F.o_sn = 1;
    F.N = A.N;
    F.M = A.M;
    F.slices = A.slices;
    F.vec_out = A.vec_out;
    launch_slice_sums(F, st);
    PP_LAUNCH_CHECK();
  }
  return PP_OK;
}
