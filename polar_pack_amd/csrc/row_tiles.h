// The split of (N,K) rows over workgroups that quad_tile.hip and dual_tile.hip share: `group`
// neighbouring tiles of 16 rows (x a slice of K) a workgroup, the group's steps of 32 columns cut into
// RT_WAVES equal runs, one a wavefront, each in at most two tiles; the runs' sums meet in LDS.
#pragma once

#include "pp_common.h"

#include <algorithm>

namespace pp {

constexpr int RT_WAVES = 8;
constexpr int64_t RT_MAX_GROUP = 8;      // more tiles and a run could lie in three

// Columns [kb, ke) of a tile, a part of a wavefront's run.
struct RowSeg {
  int tile, kb, ke;
};

// Wave w's run [a, b) of the workgroup's steps.
__device__ __forceinline__ void row_run(int steps, int w, int& a, int& b) {
  a = w * steps / RT_WAVES;
  b = (w + 1) * steps / RT_WAVES;
}

// A wavefront's share of its workgroup's rows.
struct RowShare {
  int slice, t0, ntiles;   // the workgroup's slice of K and tiles
  int per, steps;          // steps of a tile, of the workgroup
  int nseg;                // segments of the run, 0 to 2
  RowSeg S[2];
  template <class Args>
  __device__ __forceinline__ RowShare(const Args& A, int wave) {
    slice = blockIdx.x % A.slices;
    t0 = (int)(blockIdx.x / A.slices) * A.group;
    ntiles = min(A.group, A.tiles - t0);
    const int all = A.K / 32, s0 = (int)((int64_t)slice * all / A.slices);
    const int s1 = (int)((int64_t)(slice + 1) * all / A.slices);
    per = s1 - s0;
    steps = ntiles * per;
    int a, b;
    row_run(steps, wave, a, b);
    const int ta = a / per;
    nseg = b <= a ? 0 : b > (ta + 1) * per ? 2 : 1;
    S[0] = RowSeg{t0 + min(ta, ntiles - 1), 32 * (s0 + a - ta * per), 32 * (s0 + min(b - ta * per, per))};
    S[1] = nseg == 2 ? RowSeg{t0 + ta + 1, 32 * s0, 32 * (s0 + b - (ta + 1) * per)} : RowSeg{S[0].tile, S[0].ke, S[0].ke};
  }
};

// The runs' sums through LDS, [wave][segment][model][token tile][lane] in `red`: R.H the first segment's
// and R.C the last one's of this wave (R.nseg of them); store(tile, model, token tile, sum) for every tile
// of the workgroup.  Every wave must be done with what `red` held before.
template <int MODELS, int T, class V, class Run, class Store>
__device__ __forceinline__ void row_sums(V* red, const RowShare& W, const Run& R, int wave, int lane, Store store) {
  auto slot = [&](int w, int sg, int m, int t) { return red + ((((w * 2 + sg) * MODELS + m) * T + t) << 6) + lane; };
#pragma unroll
  for (int m = 0; m < MODELS; ++m)
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if (R.nseg == 2) *slot(wave, 0, m, t) = R.H[m][t];
      if (R.nseg > 0) *slot(wave, R.nseg - 1, m, t) = R.C[m][t];
    }
  __syncthreads();
  for (int u = wave; u < W.ntiles * MODELS * T; u += RT_WAVES) {
    const int tile = u / (MODELS * T), m = u / T % MODELS, t = u % T;
    V v = V{0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < RT_WAVES; ++w) {
      int wa, wb;
      row_run(W.steps, w, wa, wb);
      if (max(wa, tile * W.per) >= min(wb, (tile + 1) * W.per)) continue;
      v += *slot(w, wa / W.per == tile ? 0 : 1, m, t);
    }
    store(tile, m, t, v);
  }
}

// ------------------------------------------------------------------ host side
struct RowPlan {
  int group, slices;
};

// Slices of K and tiles a workgroup, one round of workgroups on the chip: the least of the longest
// wave's steps, with `second` steps for a second pass over the slices' sums.  No plan (group 0) past
// RT_MAX_GROUP tiles a workgroup.
static inline RowPlan row_plan(int64_t N, int64_t K, int64_t second) {
  const int64_t cus = device_cu_count(), tiles = (N + 15) / 16, steps = K / 32;
  RowPlan best = {};
  int64_t least = INT64_MAX;
  for (int64_t s = 1; s <= std::min<int64_t>({16, cus, std::max<int64_t>(1, steps / RT_WAVES)}); ++s) {
    const int64_t groups = cus / s, group = (tiles + groups - 1) / groups, per = (steps + s - 1) / s;
    if (group > RT_MAX_GROUP) break;
    const int64_t cost = (group * per + RT_WAVES - 1) / RT_WAVES + (s > 1 ? second : 0);
    if (cost < least) {
      least = cost;
      best = {(int)group, (int)s};
    }
  }
  return best;
}

}  // namespace pp
