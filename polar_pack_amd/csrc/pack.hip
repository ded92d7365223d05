// The layer packers (quad_kernels.py:16-50, polar_kernels.py:118-151) as a few passes over
// the weights.  The codes are those of the elementwise torch expressions, bit for bit: every
// operation is done and rounded as torch's float32 / fp16 device arithmetic does it (no
// contraction; a Python scalar is float32, a division by one a product with its reciprocal,
// formed in float64 and rounded; a division by a tensor an IEEE division; an fp16 tensor holds
// every result rounded to fp16).
//
// What bounds them: the packed layer's bytes are 12 (quad) and 6 (dual) per element, but a
// tuple takes three atan2, a log1p, four divisions and four square roots, ~400 vector
// instructions, so the code pass is bound by instruction issue (158 us for 4096 x 4096 tuples,
// 129 us for 11008 x 2048 pairs).  One fused pass per dependence (squares -> norms -> codes)
// replaces ~60 elementwise launches, each of them a pass over float32 or int64 intermediates:
// a call, its LUTs built on the host under the passes, takes 360 us for 4096 x 4096 tuples (2,311 us
// on the expressions) and 132 us for 11008 x 2048 pairs (1,068 us).  Small layers are bound by the
// host: 256 x 256 136 us (603) and 48 us (266), of which the LUTs take 10 and 20.
#include "pp_common.h"

#include <algorithm>
#include <cstring>

namespace pp {

constexpr int PK_NT = 256;

template <typename T> struct PkVec;
template <> struct PkVec<f16> { typedef f16x4 V4; };
template <> struct PkVec<float> { typedef float4 V4; };

// A value of a torch tensor of type T: rounded to T, kept in float32.
template <typename T>
__device__ __forceinline__ float rnd(float v) { return (float)(T)v; }

// Four elements of w from i (a multiple of 4); past n they read 0.
template <typename T>
__device__ __forceinline__ void load4(const void* w, int64_t i, int64_t n, float (&v)[4]) {
  const T* p = reinterpret_cast<const T*>(w) + i;
  if (i + 4 <= n) {
    const auto q = *reinterpret_cast<const typename PkVec<T>::V4*>(p);
    v[0] = (float)q.x; v[1] = (float)q.y; v[2] = (float)q.z; v[3] = (float)q.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = i + e < n ? (float)p[e] : 0.f;
  }
}

struct Quad4 {
  const void* w[4];
};

// ---------------------------------------------------------------------------- quad
// meta: [0..3] the models' RMS scales, [4] the largest norm.
constexpr int META_S = 0, META_R = 4;

// sq[i] = w[i]^2 in float32; clears the norm's maximum for the next pass.  One model a launch:
// its squares (64 MiB at 4096 x 4096) are still in the last-level cache when their mean reads
// them (16 + 18 us a model; 62 + 4 x 27 us with the four models squared in one launch).
template <typename T>
__global__ __launch_bounds__(PK_NT) void pack_squares_kernel(const void* w, int64_t n, float* sq, float* meta) {
  if (blockIdx.x == 0 && threadIdx.x == 0) meta[META_R] = 0.f;
  for (int64_t i = 4 * ((int64_t)blockIdx.x * PK_NT + threadIdx.x); i < n; i += 4ll * PK_NT * gridDim.x) {
    float v[4];
    load4<T>(w, i, n, v);
    // sq holds a multiple of 4 floats: the last store may write past n, inside it
    *reinterpret_cast<float4*>(sq + i) = make_float4(v[0] * v[0], v[1] * v[1], v[2] * v[2], v[3] * v[3]);
  }
}

struct Means {
  const float* p[4];
};

// Partial sums of the norm: (w_m / s_m)^2 added left to right.
__device__ __forceinline__ float quad_norm(const float (&x)[4]) {
#pragma clang fp contract(off)
  return sqrtf(x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3]);
}

// s_m = sqrt(mean_m) and the largest norm.  A norm is >= +0 or NaN, so its bits order as
// unsigned integers with NaN above everything: the maximum propagates NaN as torch's does.
template <typename T>
__global__ __launch_bounds__(PK_NT) void quad_pack_norm_kernel(const Quad4 W, int64_t n, const Means M, float* meta) {
  float s[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) s[m] = sqrtf(*M.p[m]);
  if (blockIdx.x == 0 && threadIdx.x < 4)
    meta[META_S + threadIdx.x] = threadIdx.x == 0 ? s[0] : threadIdx.x == 1 ? s[1] : threadIdx.x == 2 ? s[2] : s[3];
  uint32_t top = 0;
  for (int64_t i = 4 * ((int64_t)blockIdx.x * PK_NT + threadIdx.x); i < n; i += 4ll * PK_NT * gridDim.x) {
    float v[4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) load4<T>(W.w[m], i, n, v[m]);
    // only the tuples below n: the zeros past it would be 0 / 0 = NaN where a scale is 0, which
    // weights whose squares underflow (a norm of w / 0 = infinity) must not become
    const int left = (int)min<int64_t>(n - i, 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x[4] = {v[0][e] / s[0], v[1][e] / s[1], v[2][e] / s[2], v[3][e] / s[3]};
      const uint32_t norm = __float_as_uint(quad_norm(x)) & 0x7FFFFFFFu;
      top = max(top, e < left ? norm : 0u);
    }
  }
  // one atomic a workgroup: one a wavefront (16,384 on one address) made this pass 200 us long
  __shared__ uint32_t tops[PK_NT / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, o, 64));
  if ((threadIdx.x & 63) == 0) tops[threadIdx.x >> 6] = top;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < PK_NT / 64; ++w) top = max(top, tops[w]);
    atomicMax(reinterpret_cast<uint32_t*>(meta) + META_R, top);
  }
}

// torch's clip(0, 255) of a float: NaN stays NaN.
__device__ __forceinline__ float clip255(float v) { return v != v ? v : fminf(fmaxf(v, 0.f), 255.f); }

struct QuadPackConst {
  float mu, inv_log_mu;
};

// One tuple's code word (quad_kernels.py:23-37).
__device__ __forceinline__ uint32_t quad_pack_word(const float (&x)[4], float inv_r_max, const QuadPackConst& C) {
#pragma clang fp contract(off)
  const float two_pi = (float)6.283185307179586;
  const float inv_pi = (float)(1.0 / 3.141592653589793), inv_two_pi = (float)(1.0 / 6.283185307179586);
  const float r = quad_norm(x);
  const float p1 = x[1] * x[1], p2 = x[2] * x[2], p3 = x[3] * x[3];
  const float t1 = atan2f(sqrtf(p1 + p2 + p3), x[0]);
  const float t2 = atan2f(sqrtf(p2 + p3), x[1]);
  float t3 = atan2f(x[3], x[2]);
  if (t3 < 0.f) t3 = t3 + two_pi;               // remainder by two_pi of an angle in [-pi, pi]
  const float nq = clip255(rintf(log1pf(C.mu * r * inv_r_max) * C.inv_log_mu * 255.f));
  const float q1 = clip255(rintf(t1 * inv_pi * 255.f));
  const float q2 = clip255(rintf(t2 * inv_pi * 255.f));
  const float q3 = clip255(rintf(t3 * inv_two_pi * 255.f));
  const int64_t w = ((int64_t)nq << 24) | ((int64_t)q1 << 16) | ((int64_t)q2 << 8) | (int64_t)q3;
  return (uint32_t)w;
}

template <typename T>
__global__ __launch_bounds__(PK_NT) void quad_pack_codes_kernel(const Quad4 W, int64_t n, const QuadPackConst C,
                                                                const float* meta, uint32_t* codes) {
  float s[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) s[m] = meta[META_S + m];
  const float inv_r_max = (float)(1.0 / ((double)meta[META_R] * 1.001));
  for (int64_t i = 4 * ((int64_t)blockIdx.x * PK_NT + threadIdx.x); i < n; i += 4ll * PK_NT * gridDim.x) {
    float v[4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) load4<T>(W.w[m], i, n, v[m]);
    uint32_t q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x[4] = {v[0][e] / s[0], v[1][e] / s[1], v[2][e] / s[2], v[3][e] / s[3]};
      q[e] = quad_pack_word(x, inv_r_max, C);
    }
    if (i + 4 <= n) {
      u32x4 o = {q[0], q[1], q[2], q[3]};
      *reinterpret_cast<u32x4*>(codes + i) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < n) codes[i + e] = q[e];
    }
  }
}

// ---------------------------------------------------------------------------- dual
struct DualPackConst {
  float num_phases, mu, inv_log_mu, levels;
  int phases, group_log2;
};

// One thread takes 8 consecutive pairs, 2^(group_log2 - 3) neighbouring lanes a group.
template <typename T>
__global__ __launch_bounds__(PK_NT) void dual_pack_kernel(const void* w1, const void* w2, int64_t n,
                                                          const DualPackConst C, int16_t* codes, f16* bmax) {
#pragma clang fp contract(off)
  const float pi = (float)3.141592653589793, inv_two_pi = (float)(1.0 / 6.283185307179586);
  const int lanes = 1 << (C.group_log2 - 3);
  const int64_t end = (n + 511) / 512 * 512;         // whole wavefronts: every lane of a group takes part
  for (int64_t i = 8 * ((int64_t)blockIdx.x * PK_NT + threadIdx.x); i < end; i += 8ll * PK_NT * gridDim.x) {
    float a[8], amp[8];
    uint32_t phase[8];
    uint32_t top = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float x[4], y[4];
      load4<T>(w1, i + 4 * h, n, x);
      load4<T>(w2, i + 4 * h, n, y);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        amp[4 * h + e] = rnd<T>(sqrtf(rnd<T>(rnd<T>(x[e] * x[e]) + rnd<T>(y[e] * y[e]))));
        a[4 * h + e] = rnd<T>(atan2f(y[e], x[e]));
      }
    }
    // polar_kernels.py:122-124: round((phase + pi) / (2 pi) * num_phases) mod num_phases
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t = rnd<T>(rintf(rnd<T>(rnd<T>(rnd<T>(a[e] + pi) * inv_two_pi) * C.num_phases)));
      int v = (int)t;                                 // 0 .. num_phases (NaN: 0)
      if (v >= C.phases) v -= C.phases;
      phase[e] = (uint32_t)v;
      top = max(top, __float_as_uint(amp[e]) & 0x7FFFFFFFu);   // >= 0 or NaN, which orders above
    }
    for (int o = 1; o < lanes; o <<= 1) top = max(top, (uint32_t)__shfl_xor((int)top, o, 64));
    float b = __uint_as_float(top);
    if (!(b > 1e-10f)) b = 1.f;
    uint32_t q[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float nrm = rnd<T>(amp[e] / b);
      const float sg = nrm > 0.f ? 1.f : 0.f;         // >= 0 or NaN
      const float c = rnd<T>(rnd<T>(sg * rnd<T>(log1pf(rnd<T>(C.mu * nrm)))) * C.inv_log_mu);
      const float l = rnd<T>(rintf(rnd<T>(c * C.levels)));
      const float cl = l != l ? l : fminf(fmaxf(l, 0.f), C.levels);
      q[e] = ((((uint32_t)(int)cl & 0x3Fu) << 10) | (phase[e] & 0x3FFu)) ^ 0x8000u;
    }
    if (i + 8 <= n) {
      u32x4 o = {q[0] | (q[1] << 16), q[2] | (q[3] << 16), q[4] | (q[5] << 16), q[6] | (q[7] << 16)};
      *reinterpret_cast<u32x4*>(codes + i) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (i + e < n) codes[i + e] = (int16_t)q[e];
    }
    if (i < n && ((i >> 3) & (lanes - 1)) == 0) bmax[i >> C.group_log2] = (f16)b;
  }
}

// ------------------------------------------------------------------- host bytes to the device
// A few KB of tables carried in the launch's own arguments: no staging buffer, and no wait
// for the work queued before it, as a copy from pageable memory makes.
constexpr int UP_WORDS = 896, UP_PARTS = 8;      // 3.7 KB of the 4 KB that a launch's arguments may take
struct UpBlock {
  uint32_t v[UP_WORDS];
  uint32_t* dst[UP_PARTS];
  int first[UP_PARTS + 1];                       // part p: words first[p] .. first[p + 1] - 1
};
// One walk over the words of all parts, its loads side by side (a loop a part made the launch 5 us longer).
__global__ __launch_bounds__(PK_NT) void upload_kernel(const UpBlock B) {
  uint32_t v[(UP_WORDS + PK_NT - 1) / PK_NT];
#pragma unroll
  for (int k = 0; k * PK_NT < UP_WORDS; ++k) v[k] = B.v[min((int)threadIdx.x + k * PK_NT, UP_WORDS - 1)];
#pragma unroll
  for (int k = 0; k * PK_NT < UP_WORDS; ++k) {
    const int i = threadIdx.x + k * PK_NT;
    uint32_t* dst = B.dst[0];
    int at = i;
#pragma unroll
    for (int p = 1; p < UP_PARTS; ++p) {
      dst = i >= B.first[p] ? B.dst[p] : dst;
      at = i >= B.first[p] ? i - B.first[p] : at;
    }
    if (i < B.first[UP_PARTS]) dst[at] = v[k];
  }
}

static unsigned pack_grid(int64_t n, int per_thread, int per_cu = 16) {
  const int64_t blocks = (n + (int64_t)per_thread * PK_NT - 1) / ((int64_t)per_thread * PK_NT);
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(blocks, (int64_t)per_cu * device_cu_count()));
}

static bool pack_weights_ok(const void* const* w, int count, int dtype) {
  for (int m = 0; m < count; ++m)
    if (w[m] == nullptr || !aligned(w[m], dtype == PP_F16 ? 8 : 16)) return false;
  return true;
}

}  // namespace pp

using namespace pp;

extern "C" int pp_quad_pack_squares(const void* w, int dtype, int64_t n, float* sq, float* meta, void* stream) {
  PP_REQUIRE(dtype == PP_F16 || dtype == PP_F32, "weights must be fp16 or float32");
  PP_REQUIRE(n > 0 && sq != nullptr && meta != nullptr, "null pointer / empty weights");
  PP_REQUIRE(pack_weights_ok(&w, 1, dtype) && aligned(sq, 16), "weights must be aligned to 4 elements, sq to 16 bytes");
  const dim3 grid(pack_grid(n, 4));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == PP_F16) hipLaunchKernelGGL((pack_squares_kernel<f16>), grid, dim3(PK_NT), 0, st, w, n, sq, meta);
  else hipLaunchKernelGGL((pack_squares_kernel<float>), grid, dim3(PK_NT), 0, st, w, n, sq, meta);
  PP_LAUNCH_CHECK();
  return PP_OK;
}

extern "C" int pp_quad_pack_norm(const void* const* w, int dtype, int64_t n, const float* const* means, float* meta,
                                 void* stream) {
  PP_REQUIRE(dtype == PP_F16 || dtype == PP_F32, "weights must be fp16 or float32");
  PP_REQUIRE(n > 0 && w != nullptr && means != nullptr && meta != nullptr, "null pointer / empty weights");
  PP_REQUIRE(pack_weights_ok(w, 4, dtype), "weights must be aligned to 4 elements");
  Quad4 W;
  Means M;
  for (int m = 0; m < 4; ++m) {
    PP_REQUIRE(means[m] != nullptr, "null mean");
    W.w[m] = w[m];
    M.p[m] = means[m];
  }
  const dim3 grid(pack_grid(n, 4, 8));       // 8 workgroups of 4 wavefronts: a CU's 32
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == PP_F16) hipLaunchKernelGGL((quad_pack_norm_kernel<f16>), grid, dim3(PK_NT), 0, st, W, n, M, meta);
  else hipLaunchKernelGGL((quad_pack_norm_kernel<float>), grid, dim3(PK_NT), 0, st, W, n, M, meta);
  PP_LAUNCH_CHECK();
  return PP_OK;
}

extern "C" int pp_quad_pack_codes(const void* const* w, int dtype, int64_t n, double mu, double log_mu,
                                  const float* meta, uint32_t* codes, void* stream) {
  PP_REQUIRE(dtype == PP_F16 || dtype == PP_F32, "weights must be fp16 or float32");
  PP_REQUIRE(n > 0 && w != nullptr && meta != nullptr && codes != nullptr, "null pointer / empty weights");
  PP_REQUIRE(pack_weights_ok(w, 4, dtype) && aligned(codes, 16), "weights must be aligned to 4 elements, codes to 16 bytes");
  Quad4 W;
  for (int m = 0; m < 4; ++m) W.w[m] = w[m];
  QuadPackConst C;
  C.mu = (float)mu;
  C.inv_log_mu = (float)(1.0 / log_mu);
  const dim3 grid(pack_grid(n, 4));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == PP_F16) hipLaunchKernelGGL((quad_pack_codes_kernel<f16>), grid, dim3(PK_NT), 0, st, W, n, C, meta, codes);
  else hipLaunchKernelGGL((quad_pack_codes_kernel<float>), grid, dim3(PK_NT), 0, st, W, n, C, meta, codes);
  PP_LAUNCH_CHECK();
  return PP_OK;
}

extern "C" int pp_dual_pack(const void* w1, const void* w2, int dtype, int64_t n, int64_t group_size, int64_t num_phases,
                            int levels, double mu, double log_mu, int16_t* codes, void* bmax, void* stream) {
  PP_REQUIRE(dtype == PP_F16 || dtype == PP_F32, "weights must be fp16 or float32");
  PP_REQUIRE(group_size >= 8 && group_size <= 512 && (group_size & (group_size - 1)) == 0,
             "group_size must be a power of two in 8..512");
  PP_REQUIRE(num_phases >= 1 && num_phases <= 1024 && levels >= 1 && levels <= 63, "codes are 6-bit amplitude + 10-bit phase");
  PP_REQUIRE(n > 0 && codes != nullptr && bmax != nullptr && aligned(codes, 16), "null pointer / empty weights");
  const void* w[2] = {w1, w2};
  PP_REQUIRE(pack_weights_ok(w, 2, dtype), "weights must be aligned to 4 elements");
  DualPackConst C;
  C.num_phases = (float)num_phases;
  C.phases = (int)num_phases;
  C.levels = (float)levels;
  C.mu = (float)mu;
  C.inv_log_mu = (float)(1.0 / log_mu);
  C.group_log2 = 63 - __builtin_clzll((unsigned long long)group_size);
  const dim3 grid(pack_grid(n, 8));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  f16* b = reinterpret_cast<f16*>(bmax);
  if (dtype == PP_F16) hipLaunchKernelGGL((dual_pack_kernel<f16>), grid, dim3(PK_NT), 0, st, w1, w2, n, C, codes, b);
  else hipLaunchKernelGGL((dual_pack_kernel<float>), grid, dim3(PK_NT), 0, st, w1, w2, n, C, codes, b);
  PP_LAUNCH_CHECK();
  return PP_OK;
}

extern "C" int pp_upload_tables(void* const* dst, const void* const* src, const int64_t* bytes, int count,
                                void* stream) {
  PP_REQUIRE(count >= 0 && (count == 0 || (dst && src && bytes)), "null pointer argument");
  for (int t = 0; t < count; ++t) {
    PP_REQUIRE(bytes[t] >= 0 && bytes[t] % 4 == 0, "bytes must be a multiple of 4");
    PP_REQUIRE(bytes[t] == 0 || (dst[t] != nullptr && src[t] != nullptr && aligned(dst[t], 4)),
               "null or misaligned pointer");
  }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int t = 0;
  int64_t done = 0;                              // words of table t that earlier launches carry
  while (t < count) {
    UpBlock B;
    int used = 0, parts = 0;
    while (t < count && parts < UP_PARTS && used < UP_WORDS) {
      const int64_t left = bytes[t] / 4 - done;
      const int n = (int)std::min<int64_t>(UP_WORDS - used, left);
      if (n > 0) {
        memcpy(B.v + used, reinterpret_cast<const char*>(src[t]) + 4 * done, 4 * (size_t)n);
        B.dst[parts] = reinterpret_cast<uint32_t*>(dst[t]) + done;
        B.first[parts++] = used;
        used += n;
        done += n;
      }
      if (n == left) {
        ++t;
        done = 0;
      }
    }
    if (used == 0) break;
    for (int p = parts; p <= UP_PARTS; ++p) B.first[p] = used;
    for (int p = parts; p < UP_PARTS; ++p) B.dst[p] = nullptr;
    hipLaunchKernelGGL(upload_kernel, dim3(1), dim3(PK_NT), 0, st, B);
    PP_LAUNCH_CHECK();
  }
  return PP_OK;
}

extern "C" int pp_upload(void* dst, const void* src, int64_t bytes, void* stream) {
  return pp_upload_tables(&dst, &src, &bytes, 1, stream);
}
