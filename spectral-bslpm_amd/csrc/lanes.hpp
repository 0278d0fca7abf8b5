// lanes.hpp -- lane copies of a tile's targets, for the FP32 pair kernels and for
// the FP64 ones on small or uneven tiles.
//
// A vector instruction of FP32 operands from vector registers issues in 2.7
// cycles per wave, one with a scalar-register operand in 4.8 (probe/issue_rates.hip,
// mixes 10 and 11 with eight waves per SIMD at a nominal 2.4 GHz; FP64 4.8 to 5.1 with
// either), so the source records are read from LDS into vector registers rather
// than as scalar loads.  Each lane then holds NT targets, so that one record read
// (16 LDS cycles for 32 bytes over a wave) serves NT pairs, and the tile's
// ceil(count / NT) lanes are repeated in as many copies as a wave holds; copy g takes
// sources g, g + G, ... of a staged chunk.  The copies' and then the waves' sums are
// added in order through LDS.  In FP64 the gain is the lanes that a row per lane
// leaves idle.
#pragma once
#include "pairwalk.hpp"

namespace sbslpm {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kLaneChunk = 64;               // records staged at a time, one per lane
constexpr int kLanePad = 16;                 // copies at most, padding of a chunk at most kLanePad - 1
constexpr int kLaneSlots = kLaneChunk + kLanePad;

// The FP64 kernels, bound by issue with scalar records at no LDS cost, take lane
// copies where those fill more of the wave: with two rows per lane three or more
// copies of at most 42 rows (36 rows use 54 lanes' worth twice over against 36 of
// 64).  Vortex velocity on the 1 degree lat-lon grid's tree, a row per lane and here:
// mean 28 rows 140 and 126 us, 35 rows 157 and 147, 40 rows 358 and 317; 46 rows (degree
// 6) 186 and 196, 48 rows 190 and 206.
inline bool lanes64(const DevTree& t) { return t.rows <= 42; }

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

// Stages N 16-byte words of each of the records [0, cn) of `src` from lane to slot,
// and a record of zeros but for the first float, `first`, in the slots up to 64;
// slots 64 .. 79 are filled once by lane_pads.  (Word by word: a record selected as
// a whole is first stored as padding and then again.)
template <int N>
__device__ inline void lane_stage(v4f* mine, const v4f* __restrict__ src, int cn, float first, int lane) {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  v4f v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = v4f{i == 0 ? first : 0.f, 0.f, 0.f, 0.f};
  if (lane < cn) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = src[N * lane + i];
  }
#pragma unroll
  for (int i = 0; i < N; ++i) mine[N * lane + i] = v[i];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}
template <int N>
__device__ inline void lane_pads(v4f* mine, float first, int lane) {
  if (lane < kLanePad)
#pragma unroll
    for (int i = 0; i < N; ++i)
      mine[N * (kLaneChunk + lane) + i] = v4f{i == 0 ? first : 0.f, 0.f, 0.f, 0.f};
}

// Waves per tile of the lane-copy kernels.  (The FP32 kernels' times stand beside them.
// FP64 shallow-water velocity at degree 4, microseconds per call with 2 / 4 / 8 waves:
// 510 tiles 50 / 36 / 36, 2,046 78 / 76 / 91, 8,190 211 / 209 / 282.)
inline int lane_waves(int ntiles) { return ntiles < 1000 ? 8 : 4; }
// The FP64 kernels on long lists of tiles of at most 16 rows: one wave, whose walk of
// short sets costs less than adding the sums of four.  (Shallow-water velocity at
// degree 2, 3 x 3 points a leaf, with 4 waves and one: 6 x 96^2 148 and 121 us, 6 x
// 192^2 454 and 315; at 6 x 48^2, 2,046 tiles, 66 and 67.  The Laplacian kernel puts
// eight such tiles behind one copy of its 30 KB table: 401 and 271 us at 6 x 192^2.)
inline int lane_waves64(const DevTree& t, int ntiles) {
  return t.rows <= 16 && ntiles >= 6000 ? 1 : lane_waves(ntiles);
}

// Walks a wave's share of the source sets of a tile: begin(set) and flush(set)
// around each part of a set, add(r) for each trip, r the lane's record (N 16-byte
// words) in LDS; `first` as in lane_stage.
template <int S, int N, int UNROLL, typename Begin, typename Add, typename Flush>
__device__ inline void lane_walk(const TargetTile& T, const SourceSet* __restrict__ sets, const v4f* __restrict__ rec,
                                 const LaneTile& l, v4f* mine, float first, int wave, int lane, Begin&& begin,
                                 Add&& add, Flush&& flush) {
  lane_pads<N>(mine, first, lane);
  walk_sets<S>(T, sets, wave, [&](const SourceSet& set, int a, int b) {
    begin(set);
    for (int c = a; c < b; c += kLaneChunk) {
      const int cn = min(kLaneChunk, b - c), trips = (cn + l.G - 1) / l.G;
      lane_stage<N>(mine, rec + N * ((int64_t)set.first + c), cn, first, lane);
      const v4f* r = mine + N * l.g;
#pragma unroll UNROLL
      for (int k = 0; k < trips; ++k, r += N * l.G) add(r);
    }
    flush(set);
  });
}

// lane_walk for the FP64 kernels, whose sums run on from set to set: a chunk is
// filled with as many sets' records as make whole pairs of trips (up to 64), so that
// only a wave's last chunk is padded.  (One set at a time, a set of 9 records gave 12
// copies one trip and a padded one: the shallow-water velocity at degree 2, 24,576
// leaves of 3 x 3, took 620 us and takes 454; at degree 4, 5 x 5, 867 and 737; the
// vortex velocity at degree 8, 6 x 6, 411 and 408 at 6 x 192^2.)  add(r0, r1) takes two trips, so that two rows
// of two records share a reciprocal; an odd last trip is paired with a padding record
// (slot 79, which no trip reaches).  REPEAT (N = 2, the charge in the last eight bytes):
// padding repeats the chunk's last record without its charge, for a kernel that takes
// another form where a pair is far away.
template <int S, int N, bool REPEAT = false, typename Add>
__device__ inline void lane_walk2(const TargetTile& T, const SourceSet* __restrict__ sets, const v4f* __restrict__ rec,
                                  const LaneTile& l, v4f* mine, int wave, int lane, Add&& add) {
  static_assert(!REPEAT || N == 2, "lane_walk2: REPEAT knows the layout of two-word records");
  if (!REPEAT) lane_pads<N>(mine, 0.f, lane);
  const int full = kLaneChunk / (2 * l.G) * (2 * l.G);
  SetWalk<S> part(T, sets, wave);
  bool more = part.next();
  while (more) {
    int src = 0, fill = 0;  // this lane's record, records in the chunk
    do {
      const int n = min(full - fill, part.b - part.a), from = part.first + part.a - fill;
      src = lane >= fill ? from + lane : src;
      part.a += n;
      fill += n;
      if (part.a == part.b) more = part.next();
    } while (more && fill < full);
    const int trips = (fill + l.G - 1) / l.G;
    if (REPEAT) src = lane < fill ? src : __builtin_amdgcn_readlane(src, fill - 1);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    v4f v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = v4f{0.f, 0.f, 0.f, 0.f};
    if (REPEAT || lane < fill) {
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = rec[N * (int64_t)src + i];
    }
    if constexpr (REPEAT) {
      if (lane >= fill) v[N - 1].z = v[N - 1].w = 0.f;
      if (lane < kLanePad) {
        const int last = __builtin_amdgcn_readlane(src, fill - 1);
        const v4f l0 = rec[N * (int64_t)last], l1 = rec[N * (int64_t)last + 1];
        mine[N * (kLaneChunk + lane)] = l0;
        mine[N * (kLaneChunk + lane) + 1] = v4f{l1.x, l1.y, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) mine[N * lane + i] = v[i];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const v4f* r = mine + N * l.g;
    for (int k = 0; k < trips; k += 2, r += 2 * N * l.G)
      add(r, k + 1 < trips ? r + N * l.G : mine + N * (kLaneSlots - 1));
  }
}

// Sums w[t][c] over the copies and the S waves into row t T + i of lane
// t T + i of wave 0, valid where the lane is below the tile's count; `stage` is
// each wave's slot of SLOT >= 64 K doubles (every thread calls it).
template <int NT, int K, int S, int SLOT>
__device__ inline void lane_sum(const LaneTile& l, double (&w)[NT][K], double (*stage)[SLOT], int wave,
                                int lane, double (&out)[K]) {
  static_assert(SLOT >= 64 * K, "lane_sum: slot too small");
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
  if constexpr (S > 1)
    __syncthreads();
  else
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  if (wave == 0)
#pragma unroll
    for (int c = 0; c < K; ++c) {
      out[c] = 0;
      for (int s = 0; s < S; ++s) out[c] += stage[s][c * 64 + lane];
    }
}

}  // namespace sbslpm
