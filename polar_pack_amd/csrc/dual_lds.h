// LDS decode tables of the dual-pack kernels (dual_rows.hip, dual_kn.hip) and their
// lookups.
//
// (cos, sin) of the 1024 phases in 128-byte rows of 16 replicas (lane l reads replica
// l % 16, so a wavefront's 64 reads of 8 bytes spread over the banks), the 64 amplitudes
// one per 4-byte bank (a wave's 64 reads hit distinct banks or share one address, so no
// replicas).  For the int16 layout (stored = code ^ 0x8000, polar_kernels.py:9-11) the
// amplitude entry a holds amp_lut[a ^ 32], so the stored bits index it directly.
#pragma once

#include "pp_common.h"

namespace pp {

// The decode tables as the caller holds them: amp_lut[amp_n], cos_lut / sin_lut[phase_n],
// fp16 or float32 (dtype); indices past amp_n / phase_n decode to 0.
struct DualLuts {
  const void* amp;
  const void* cs[2];  // cos, sin
  int amp_n, phase_n, dtype;
};

constexpr uint32_t DLDS_AMP = 0;               // the 64 amplitudes, 4 bytes each: one per LDS bank
constexpr uint32_t DLDS_CS = 0x400;            // (cos, sin) rows: phase p at DLDS_CS + p*128 + 8*(lane % 16)
constexpr uint32_t DLDS_BYTES = 0x400 + 1024 * 128;

// Stored 32-bit word (two pairs) -> two codes in the table-index form: the file layout is
// byte-swapped per half, the int16 layout is used as stored.
template <int LAYOUT>
__device__ __forceinline__ uint32_t dual_word(uint32_t w) {
  if constexpr (LAYOUT == PP_DUAL_U16_BE) return __builtin_amdgcn_perm(w, w, 0x02030001u);
  else return w;
}
template <int LAYOUT>
__device__ __forceinline__ uint32_t dual_half(uint32_t h16) {
  if constexpr (LAYOUT == PP_DUAL_U16_BE) return ((h16 & 0xFFu) << 8) | ((h16 >> 8) & 0xFFu);
  else return h16 & 0xFFFFu;
}

struct DualLane {
  uint32_t cs;        // the lane's replica inside a (cos, sin) row
};

__device__ __forceinline__ DualLane dual_lane(int l) {
  DualLane o;
  o.cs = 8u * (l & 15);
  return o;
}

// Amplitude and (cos, sin) of both codes of a stored 32-bit word.  The amplitude table
// needs no replicas (a wave's 64 reads hit distinct banks or share one address), so its
// byte offset, 4 * amp bits, comes straight out of the stored word: byte 0 / byte 2 of
// a big-endian word, byte 1 / byte 3 of the int16 layout, masked with 0xFC.
template <int LAYOUT>
__device__ __forceinline__ void dual_lookup2(const char* lds, uint32_t raw, const DualLane& o, float (&an)[2],
                                             float2 (&cs)[2]) {
  const uint32_t a0 = (LAYOUT == PP_DUAL_U16_BE ? raw : raw >> 8) & 0xFCu;
  const uint32_t a1 = (raw >> (LAYOUT == PP_DUAL_U16_BE ? 16 : 24)) & 0xFCu;
  const uint32_t w = dual_word<LAYOUT>(raw);
  const uint32_t c0 = ((w << 7) & 0x1FF80u) | o.cs;
  const uint32_t c1 = ((w >> 9) & 0x1FF80u) | o.cs;
  an[0] = *reinterpret_cast<const float*>(lds + DLDS_AMP + a0);
  an[1] = *reinterpret_cast<const float*>(lds + DLDS_AMP + a1);
  cs[0] = *reinterpret_cast<const float2*>(lds + DLDS_CS + c0);
  cs[1] = *reinterpret_cast<const float2*>(lds + DLDS_CS + c1);
}

// The same for one code in the table-index form (amp bits 10..15, phase 0..9).
__device__ __forceinline__ void dual_lookup1(const char* lds, uint32_t c, const DualLane& o, float& an, float2& cs) {
  an = *reinterpret_cast<const float*>(lds + DLDS_AMP + ((c >> 8) & 0xFCu));
  cs = *reinterpret_cast<const float2*>(lds + DLDS_CS + (((c << 7) & 0x1FF80u) | o.cs));
}

// Build the tables of a workgroup of NT threads (a multiple of 64) from the caller's LUTs
// (entries of type E), in two steps so that a kernel can issue other loads between them:
// load() issues every LUT load of a thread, store() writes the (cos, sin) rows and ends with a
// barrier.  For the int16 layout (stored = code ^ 0x8000) amplitude entry a holds amp_lut[a ^ 32].
// A thread loads whole phases and writes their rows' 8 units of 16 bytes, neighbouring lanes
// starting at different units so that 16 of them fill 256 bytes of distinct banks: 5 loads a
// thread at NT = 512.  With a unit's own entry loaded by the thread that writes it (33 loads) a
// launch of dual_strip_kernel took 2 us more (4096 x 4096 at 8 tokens 17.4 us, 15.4 this way).
template <int NT, int LAYOUT, typename E>
struct DualTables {
  static constexpr int KP = (1024 + NT - 1) / NT;
  E c[KP], s[KP], amp;
  __device__ __forceinline__ void load(const DualLuts& L) {
    const E* cp = reinterpret_cast<const E*>(L.cs[0]);
    const E* sp = reinterpret_cast<const E*>(L.cs[1]);
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      const int p = threadIdx.x + k * NT;
      c[k] = p < L.phase_n ? cp[p] : (E)0.f;
      s[k] = p < L.phase_n ? sp[p] : (E)0.f;
    }
    const int e = LAYOUT == PP_DUAL_I16_OFFSET ? ((threadIdx.x & 63) ^ 32) : (threadIdx.x & 63);
    amp = e < L.amp_n ? reinterpret_cast<const E*>(L.amp)[e] : (E)0.f;
  }
  __device__ __forceinline__ void store(char* lds) const {
    if (threadIdx.x < 64) *reinterpret_cast<float*>(lds + DLDS_AMP + 4 * threadIdx.x) = (float)amp;
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      const int p = threadIdx.x + k * NT;
      if (1024 % NT != 0 && p >= 1024) break;
      const float4 v = make_float4((float)c[k], (float)s[k], (float)c[k], (float)s[k]);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        *reinterpret_cast<float4*>(lds + DLDS_CS + 128 * p + 16 * ((u + (threadIdx.x >> 1)) & 7)) = v;
    }
    __syncthreads();
  }
};

template <int NT, int LAYOUT, typename E>
__device__ __forceinline__ void dual_tables_of(char* lds, const DualLuts& L) {
  DualTables<NT, LAYOUT, E> t;
  t.load(L);
  t.store(lds);
}

}  // namespace pp
