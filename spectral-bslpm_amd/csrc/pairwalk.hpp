// pairwalk.hpp -- how the waves of a pair kernel that share a target tile divide
// its source sets: FP64 with a row per lane, and the lane copies of either
// precision (lanes.hpp).
//
// A workgroup is S waves on one tile of up to 64 targets: four of them take
// the sets in turn, and S / 4 take consecutive parts of each set, dealt round
// so that an uneven division evens out.  The waves' sums are added in wave
// order through LDS, so a result depends on S and on nothing else; S follows
// from the length of the tile list and its rows per tile alone, so members,
// launch shapes and graph replays agree to the bit.
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

// Part [a, b) of a set of `count` records for one of SK waves that share it, `turn`
// rotating the parts from set to set.
template <int SK>
__device__ inline void set_part(int count, int turn, int& a, int& b) {
  a = 0;
  b = count;
  if (SK > 1) {
    const int per = (count + 4 * SK - 1) / (4 * SK) * 4;
    a = min(count, (turn & (SK - 1)) * per);
    b = min(count, a + per);
  }
}

// This wave's share of a tile's source sets, part by part: records [first + a,
// first + b) of set e.
template <int S>
struct SetWalk {
  static constexpr int SS = S < 4 ? S : 4, SK = S / SS;  // sets in turn, waves per set
  const SourceSet* __restrict__ sets;
  int e, end, wk, it = 0, first = 0, a = 0, b = 0;
  __device__ SetWalk(const TargetTile& T, const SourceSet* __restrict__ s, int wave)
      : sets(s), e(T.src_begin + (wave & (SS - 1)) - SS), end(T.src_end), wk(wave / SS) {}
  // Moves to the next part that is not empty; false at the end.
  __device__ bool next() {
    while ((e += SS) < end) {
      first = sets[e].first;
      set_part<SK>(sets[e].count, wk + it++, a, b);
      if (a < b) return true;
    }
    return false;
  }
};

// f(set, a, b) for this wave's part [a, b) of each of its source sets.
template <int S, typename F>
__device__ inline void walk_sets(const TargetTile& T, const SourceSet* __restrict__ sets, int wave, F&& f) {
  constexpr int SS = S < 4 ? S : 4, SK = S / SS;  // sets in turn, waves per set
  const int ws = wave & (SS - 1), wk = wave / SS;
  int it = 0;
  for (int e = T.src_begin + ws; e < T.src_end; e += SS, ++it) {
    const SourceSet set = sets[e];
    int a, b;
    set_part<SK>(set.count, wk + it, a, b);
    if (SK == 1 || a < b) f(set, a, b);
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

// Tile of this workgroup where XCD x (the hardware deals workgroup b to XCD b % 8)
// takes strips x, x + 8, ... of neighbouring tiles: a strip's tiles share sources
// in that XCD's L2, and 32 strips each even out the lists, whose coarse panels
// come first and cost most.  (k_swe64 at 40,956 tiles, 64-byte records: 3.53 ms;
// one contiguous range per XCD 3.84, workgroup b on tile b 4.21.  k_lap64, whose
// coarse tiles evaluate erf: 1.03 ms at 10,236 tiles, one range per XCD 1.45.)
__host__ __device__ inline int strip_length(int ntiles) {
  const int k = ntiles / 256;
  return k < 1 ? 1 : k < 64 ? k : 64;
}
__device__ inline int strip_tile(int ntiles) {
  const int k = strip_length(ntiles), b = (int)blockIdx.x, i = b >> 3;
  return (i / k * 8 + (b & 7)) * k + i % k;
}
// The same over a list that heaviest_first has ordered where it is short: such a
// list is dealt tile by tile.  Microseconds per call in breadth-first strips and
// heaviest first, interpolation degree and leaf grid 8: velocity at 510 panels 76
// and 70 (FP32 66 and 61), at 2,046 panels 191 and 177 (FP32 146 and 128); Poisson
// solve at degree 10 142 and 129, 376 and 362.  Not for k_lap64, whose coarse tiles
// cost more than their pairs (erf) and come first in breadth-first order: with it
// heaviest first the two sums of a shallow-water stage took 368 and 392, 756 and 810.
// Nor for k_swe64, whose 64-byte records (17 MB at 2,046 panels) want the strips'
// locality: 753 and 760.
__device__ inline int dealt_tile(int ntiles) {
  return ntiles < kBalancedTiles ? (int)blockIdx.x : strip_tile(ntiles);
}
inline unsigned strip_grid(int ntiles) {
  const int k = 8 * strip_length(ntiles);
  return (unsigned)((ntiles + k - 1) / k * k);
}

}  // namespace sbslpm
