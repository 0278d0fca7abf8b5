// pairwalk.hpp -- how the waves of an FP64 pair kernel divide a target tile's
// source sets.
//
// A workgroup is S waves on one tile of up to 64 targets: four of them take
// the sets in turn, and S / 4 take consecutive parts of each set, dealt round
// so that an uneven division evens out.  The waves' sums are added in wave
// order through LDS, so a result depends on S and on nothing else; S follows
// from the length of the tile list alone, so members, launch shapes and graph
// replays agree to the bit.
//
// One wave per tile left each SIMD with too few waves to hide the source
// records' scalar loads behind (vector issue busy 55% at 8,190 tiles) and the
// longest tile, run by one wave, set the end of the launch.
#pragma once
#include "device.hpp"

namespace sbslpm {

// Waves per tile.  k_bve64, microseconds per launch with 1 / 4 / 8 / 16 waves:
//     126 tiles  143 / 41 / 27 / 20        8,190 tiles   541 /  407 /  412 /  426
//     636 tiles  250 / 76 / 62 / 58       10,236 tiles   573 /  498 /  507 /  531
//   2,556 tiles  313 / 195 / 183 / 188    40,956 tiles  2538 / 2358 / 2392 / 2534
inline int tile_waves(int ntiles) { return ntiles < 1500 ? 16 : ntiles < 6000 ? 8 : 4; }

// f(set, a, b) for this wave's part [a, b) of each of its source sets.
template <int S, typename F>
__device__ inline void walk_sets(const TargetTile& T, const SourceSet* __restrict__ sets, int wave, F&& f) {
  constexpr int SK = S / 4;  // waves per set
  const int ws = wave & 3, wk = wave >> 2;
  int it = 0;
  for (int e = T.src_begin + ws; e < T.src_end; e += 4, ++it) {
    const SourceSet set = sets[e];
    if (SK == 1) {
      f(set, 0, set.count);
    } else {
      const int per = (set.count + 4 * SK - 1) / (4 * SK) * 4;
      const int a = min(set.count, ((wk + it) & (SK - 1)) * per), b = min(set.count, a + per);
      if (a < b) f(set, a, b);
    }
  }
}

// Sum of v over the S waves of the workgroup in wave order, valid in wave 0
// (every thread of the workgroup calls it).
template <int S, int K>
__device__ inline void tile_sum(double (&v)[K], int wave, int lane) {
  __shared__ double red[S - 1][K][64];
  if (wave > 0)
#pragma unroll
    for (int k = 0; k < K; ++k) red[wave - 1][k][lane] = v[k];
  __syncthreads();
  if (wave == 0)
    for (int w = 0; w < S - 1; ++w)
#pragma unroll
      for (int k = 0; k < K; ++k) v[k] += red[w][k][lane];
}

// Tile of this workgroup under the PairShape mappings (its `waves` plays no part).
__device__ inline int walk_tile(const int* __restrict__ xcd_start, int xcd) {
  const int b = (int)blockIdx.x;
  if (xcd == 2) {
    const int tile = xcd_start[b & 7] + (b >> 3);
    return tile < xcd_start[(b & 7) + 1] ? tile : 0x7fffffff;
  }
  return xcd == 1 ? xcd_remap(b, gridDim.x) : b;
}
inline unsigned walk_grid(int ntiles, const PairShape& shape) {
  return (unsigned)(shape.xcd == 2 && shape.grid1 > 0 ? shape.grid1 : ntiles);
}

}  // namespace sbslpm
