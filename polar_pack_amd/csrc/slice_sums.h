// The last pass of a decode whose K slices leave float32 sums: out_m[j, n] = fp16(the sum over
// the slices of part[slice][m][j][n]), 4 columns a thread, slices added in order.
#pragma once

#include "pp_common.h"

namespace pp {

template <int MODELS>
struct SliceSums {
  const float* part;       // [slice][model][token][np]
  int64_t np;              // columns a row, a multiple of 4
  f16* out[MODELS];        // (M, N): element (j, n) at out + j*o_sm + n*o_sn
  int64_t o_sm, o_sn;
  int N, M, slices;
  int vec_out;             // o_sn == 1, outputs 8-byte aligned, o_sm % 4 == 0: 4 columns per store
};

template <int MODELS>
__global__ __launch_bounds__(256) void slice_sums_kernel(const SliceSums<MODELS> A) {
  const int64_t q4 = A.np / 4, total = MODELS * A.M * q4, at = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (at >= total) return;
  const int64_t mj = at / q4;
  const int n = (int)(at - mj * q4) * 4, m = (int)(mj / A.M), j = (int)(mj % A.M);
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
  for (int s = 0; s < A.slices; ++s) {
    const float4 p = *reinterpret_cast<const float4*>(A.part + ((int64_t)s * MODELS * A.M + mj) * A.np + n);
    v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
  }
  f16* base = A.out[0];
#pragma unroll
  for (int i = 1; i < MODELS; ++i) base = m == i ? A.out[i] : base;
  f16* o = base + (int64_t)j * A.o_sm + (int64_t)n * A.o_sn;
  if (A.vec_out && n + 3 < A.N) {
    *reinterpret_cast<f16x4*>(o) = f16x4{(f16)v.x, (f16)v.y, (f16)v.z, (f16)v.w};
  } else {
    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (n + c < A.N) o[c * A.o_sn] = (f16)e[c];
  }
}

template <int MODELS>
inline void launch_slice_sums(const SliceSums<MODELS>& A, hipStream_t st) {
  const int64_t threads = (int64_t)MODELS * A.M * (A.np / 4);
  hipLaunchKernelGGL((slice_sums_kernel<MODELS>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, A);
}

}  // namespace pp
