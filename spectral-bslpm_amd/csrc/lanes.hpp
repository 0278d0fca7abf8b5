// lanes.hpp -- lane copies of a tile's targets for the FP32 pair kernels.
//
// A vector instruction of FP32 operands from vector registers issues in 2.5
// cycles per wave, one with a scalar-register operand in 4.5 (measured with
// eight waves per SIMD), so the source records are read from LDS into vector
// registers rather than as scalar loads.  Each lane then holds NT targets, so
// that one record read (16 LDS cycles for 32 bytes over a wave) serves NT pairs,
// and the tile's ceil(count / NT) lanes are repeated in as many copies as a wave
// holds; copy g takes sources g, g + G, ... of a staged chunk.  The copies' and
// then the waves' sums are added in order through LDS.
#pragma once
#include "pairwalk.hpp"

namespace sbslpm {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kLaneChunk = 64;               // records staged at a time, one per lane
constexpr int kLanePad = 16;                 // copies at most, padding of a chunk at most kLanePad - 1
constexpr int kLaneSlots = kLaneChunk + kLanePad;

struct LaneTile {
  int T, G, g, i;  // lanes per copy, copies, this lane's copy and lane within it
  bool active;
};
template <int NT>
__device__ inline LaneTile lane_tile(int count, int lane) {
  LaneTile l;
  l.T = (count + NT - 1) / NT;
  l.G = min(64 / l.T, kLanePad);
  l.g = lane / l.T;
  l.i = lane - l.g * l.T;
  l.active = l.g < l.G;
  if (!l.active) l.g = 0;
  return l;
}

// Sums w[t][c] over the copies and the S waves into row t T + i of lane
// t T + i of wave 0, valid where the lane is below the tile's count; `stage` is
// each wave's slot of at least 192 doubles (every thread calls it).
template <int NT, int K, int S>
__device__ inline void lane_sum(const LaneTile& l, double (&w)[NT][K], double (*stage)[kLaneSlots * 4], int wave,
                                int lane, double (&out)[K]) {
  double* mine = stage[wave];
  double v[NT][K];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int c = 0; c < K; ++c) mine[c * 64 + lane] = w[t][c];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int c = 0; c < K; ++c) {
      v[t][c] = 0;
      if (lane < l.T)
        for (int g = 0; g < l.G; ++g) v[t][c] += mine[c * 64 + g * l.T + lane];
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  if (lane < l.T)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (t * l.T + lane < 64)
#pragma unroll
        for (int c = 0; c < K; ++c) mine[c * 64 + t * l.T + lane] = v[t][c];
  __syncthreads();
  if (wave == 0)
#pragma unroll
    for (int c = 0; c < K; ++c) {
      out[c] = 0;
      for (int s = 0; s < S; ++s) out[c] += stage[s][c * 64 + lane];
    }
}

}  // namespace sbslpm
