// fmm_interact.hip -- pair kernels over the target-major interaction lists.
//
// Reference: bve_vel_panel_interaction (fmm_interactions/bve_vel_impl.hpp:34-70)
// and poisson_panel_interaction (inverse_poisson_impl.hpp:23-52) run one
// thread per interaction, recompute every source node's map per pair and
// scatter three atomics per pair.  Here:
//   * a tile of up to 64 target points of one target panel belongs to one
//     workgroup, whose waves share that panel's source sets; a target is
//     accumulated in registers and the waves' sums are added in order (no
//     atomics, fixed summation order);
//   * displaced, re-projected source positions and scaled charges are built
//     once per evaluation into a record array (SrcRec64 / SrcRec32);
//   * on FP64 tiles of more than 42 rows every lane of a wave reads the same
//     source record, a wave-uniform load through the scalar cache
//     (pairwalk.hpp); on smaller tiles and in FP32 a wave stages the records
//     in LDS and copies of the tile, two targets per lane, take its sources in
//     turn (lanes.hpp);
//   * u = sum_j g_j q_j (x cross y_j) is accumulated as x cross (sum_j g_j q_j y_j),
//     saving the per-pair cross product (six multiplies) of the reference form.
// A list in breadth-first panel order is dealt in strips, so that neighbouring tiles
// (adjacent target panels sharing sources) land on the same XCD and its L2; a short
// one runs heaviest first (dealt_tile, PairShape).  The matrix-core kernels and
// k_bve_mixed run one wave per tile.
#include <cmath>

#include "device.hpp"
#include "lanes.hpp"
#include "lapkernel.hpp"

namespace sbslpm {
namespace {

struct Ptr3 {
  double* p[3];
};
struct CPtr3 {
  const double* p[3];
};

// Member slices of a batched launch (gridDim.y members): charges and
// displacements of the sources, outputs of the targets.
__device__ inline void member_sources(const DevTree& t, const double* __restrict__& q_part,
                                      const double* __restrict__& q_proxy, CPtr3& dpart,
                                      CPtr3& dprox) {
  const int64_t mp = member_part(t), mx = member_proxy(t);
  q_part += mp;
  q_proxy += mx;
  for (int f = 0; f < 3; ++f) {
    if (dpart.p[f]) dpart.p[f] += mp;
    if (dprox.p[f]) dprox.p[f] += mx;
  }
}
__device__ inline void member_targets(const DevTree& t, Ptr3& part, Ptr3& proxy) {
  const int64_t mp = member_part(t), mx = member_proxy(t);
  for (int f = 0; f < 3; ++f) {
    if (part.p[f]) part.p[f] += mp;
    if (proxy.p[f]) proxy.p[f] += mx;
  }
}

// Target-major ownership: every target point is written by exactly one lane,
// so `assign` may replace the accumulate of the reference functors.
__device__ inline void store_u(const DevTree& t, int64_t u, Ptr3 part, Ptr3 proxy, double a, double b, double c,
                               int assign) {
  double* o[3];
  int64_t v = u;
  if (u < t.npart) {
    o[0] = part.p[0]; o[1] = part.p[1]; o[2] = part.p[2];
  } else {
    v = u - t.npart;
    o[0] = proxy.p[0]; o[1] = proxy.p[1]; o[2] = proxy.p[2];
  }
  if (assign) {
    o[0][v] = a; o[1][v] = b; o[2][v] = c;
  } else {
    o[0][v] += a; o[1][v] += b; o[2][v] += c;
  }
}

__device__ inline void store_s(const DevTree& t, int64_t u, double* part, double* proxy, double a, int assign) {
  double* o = u < t.npart ? part + u : proxy + (u - t.npart);
  *o = assign ? a : *o + a;
}

// Source records, FP64: y = P(node + disp) (bve_vel_impl.hpp:54-60), q' = -q/(4 pi).
// Leaf proxy rows are never sources and are left untouched.
__global__ void k_src64(DevTree t, const double* __restrict__ q_part, const double* __restrict__ q_proxy,
                        CPtr3 dpart, CPtr3 dprox, int project, SrcRec64* __restrict__ rec) {
  int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.U) return;
  member_sources(t, q_part, q_proxy, dpart, dprox);
  rec += (int64_t)blockIdx.y * t.U;
  double x = t.px[u], y = t.py[u], z = t.pz[u], q;
  if (u < t.npart) {
    if (dpart.p[0]) { x += dpart.p[0][u]; y += dpart.p[1][u]; z += dpart.p[2][u]; }
    q = q_part[u];
  } else {
    int64_t v = u - t.npart;
    if (v / t.n >= t.offset) return;
    if (dprox.p[0]) { x += dprox.p[0][v]; y += dprox.p[1][v]; z += dprox.p[2][v]; }
    q = q_proxy[v];
  }
  if (project) project_to_sphere(x, y, z);
  rec[u] = SrcRec64{x, y, z, kNegInv4Pi * q};
}

// Source records, FP32: position relative to the owning panel's centre.
__global__ void k_src32(DevTree t, const double* __restrict__ q_part, const double* __restrict__ q_proxy,
                        CPtr3 dpart, CPtr3 dprox, int project, SrcRec32* __restrict__ rec) {
  int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.U) return;
  member_sources(t, q_part, q_proxy, dpart, dprox);
  rec += (int64_t)blockIdx.y * t.U;
  double x = t.px[u], y = t.py[u], z = t.pz[u], q;
  int panel;
  if (u < t.npart) {
    if (dpart.p[0]) { x += dpart.p[0][u]; y += dpart.p[1][u]; z += dpart.p[2][u]; }
    q = q_part[u];
    panel = t.offset + (int)(u / t.m2);
  } else {
    int64_t v = u - t.npart;
    panel = (int)(v / t.n);
    if (panel >= t.offset) return;
    if (dprox.p[0]) { x += dprox.p[0][v]; y += dprox.p[1][v]; z += dprox.p[2][v]; }
    q = q_proxy[v];
  }
  if (project) project_to_sphere(x, y, z);
  const DevPanel& P = t.panels[panel];
  rec[u] = SrcRec32{(float)(x - P.cx), (float)(y - P.cy), (float)(z - P.cz), (float)(kNegInv4Pi * q)};
}

// FP64 Biot-Savart pair kernel: g = -q/(4 pi (1 - x.y + eps)).  S waves share a
// tile (pairwalk.hpp) and take the sources in batches of four with one shared
// reciprocal (rcp4).
// Bound: FP64 vector issue, 12.25 slots per pair against 15 with a reciprocal
// each, at the 2.1 GHz the chip holds under this load.  Microseconds per launch
// before (one wave per tile, one source at a time) and now: 6 x 28^2 180 -> 20,
// 6 x 64^2 303 -> 58, 6 x 224^2 642 -> 407, 6 x 512^2 2945 -> 2358 (2326 is the
// issue time of its pairs alone).
template <int S>
__global__ __launch_bounds__(64 * S) void k_bve64(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                  const SourceSet* __restrict__ sets,
                                                  const SrcRec64* __restrict__ rec, double eps, Ptr3 part, Ptr3 proxy,
                                                  int assign, int xcd) {
  member_targets(t, part, proxy);
  rec += (int64_t)blockIdx.y * t.U;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = walk_tile(t.xcd_start ? t.xcd_start + 9 : nullptr, xcd);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const int64_t u = (int64_t)T.first + (lane < T.count ? lane : T.count - 1);
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  double w[3] = {0, 0, 0};
  walk_sets<S>(T, sets, wave, [&](const SourceSet& set, int a, int b) {
    const SrcRec64* __restrict__ r = rec + set.first;
    int k = a;
    for (; k + 4 <= b; k += 4) {
      double d[4], g[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = one_minus_dot(x, y, z, r[k + i].x, r[k + i].y, r[k + i].z) + eps;
      rcp4(d, g);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double gq = g[i] * r[k + i].q;
        w[0] = fma(gq, r[k + i].x, w[0]);
        w[1] = fma(gq, r[k + i].y, w[1]);
        w[2] = fma(gq, r[k + i].z, w[2]);
      }
    }
    for (; k < b; ++k) {
      const SrcRec64 s = r[k];
      const double g = rcp64_pair(one_minus_dot(x, y, z, s.x, s.y, s.z) + eps) * s.q;
      w[0] = fma(g, s.x, w[0]);
      w[1] = fma(g, s.y, w[1]);
      w[2] = fma(g, s.z, w[2]);
    }
  });
  tile_sum<S>(w, wave, lane);
  if (wave == 0 && lane < T.count)
    store_u(t, u, part, proxy, y * w[2] - z * w[1], z * w[0] - x * w[2], x * w[1] - y * w[0], assign);
}

// The same in lane copies (lanes.hpp) of two targets, for tiles of at most 42 rows
// (lanes64), whose rows fill 36 of 64 lanes one per lane.  Microseconds per pair call
// (records included), one wave per tile with a row per lane and here: 6 x 96^2 (degree
// 8) 265 -> 117, 6 x 192^2 665 -> 400 (a row per lane and waves sharing the tile: 499 a
// launch), degree 5 463 -> 254, 6 x 160^2 (degree 4) 324 -> 157.  At 16 waves per tile
// the short loops gain nothing.
template <int S>
__global__ __launch_bounds__(64 * S) void k_bve64_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                        const SourceSet* __restrict__ sets,
                                                        const SrcRec64* __restrict__ rec, double eps, Ptr3 part,
                                                        Ptr3 proxy, int assign, int xcd) {
  constexpr int NT = 2;
  __shared__ __align__(16) double stage[S][kLaneSlots * 4];
  member_targets(t, part, proxy);
  rec += (int64_t)blockIdx.y * t.U;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = walk_tile(t.xcd_start ? t.xcd_start + 9 : nullptr, xcd);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  double x[NT], y[NT], z[NT], w[NT][3];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    x[q] = t.px[u]; y[q] = t.py[u]; z[q] = t.pz[u];
  }
  shared_sums(w, [&](auto shared) {
#pragma unroll
    for (int q = 0; q < NT; ++q) w[q][0] = w[q][1] = w[q][2] = 0;
    lane_walk2<S, 2>(T, sets, reinterpret_cast<const v4f*>(rec), l, reinterpret_cast<v4f*>(stage[wave]), wave, lane,
                     [&](const v4f* r0, const v4f* r1) {
      const SrcRec64 R[2] = {*reinterpret_cast<const SrcRec64*>(r0), *reinterpret_cast<const SrcRec64*>(r1)};
      double d[4], g[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = i & 1;
        d[i] = one_minus_dot(x[q], y[q], z[q], R[i >> 1].x, R[i >> 1].y, R[i >> 1].z) + eps;
      }
      rcps<decltype(shared)::value>(d, g);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = i & 1;
        const SrcRec64& P = R[i >> 1];
        const double gq = g[i] * P.q;
        w[q][0] = fma(gq, P.x, w[q][0]);
        w[q][1] = fma(gq, P.y, w[q][1]);
        w[q][2] = fma(gq, P.z, w[q][2]);
      }
    });
  });
  double s[3];
  lane_sum<NT, 3, S>(l, w, stage, wave, lane, s);
  if (wave > 0 || lane >= T.count) return;
  const int64_t u = (int64_t)T.first + lane;
  const double X = t.px[u], Y = t.py[u], Z = t.pz[u];
  store_u(t, u, part, proxy, Y * s[2] - Z * s[1], Z * s[0] - X * s[2], X * s[1] - Y * s[0], assign);
}

// FP64 log pair kernel: psi += -1/(4 pi) log(1 - x.y) q, pairs with
// x.y >= 1 - 1e-15 skipped (inverse_poisson_impl.hpp:46-49).  S waves share a
// tile (pairwalk.hpp); the logarithm is log_wide (fasttab.hpp) on the context's
// table, staged in LDS.  A pair outside its range (a source that coincides with
// a target: the target's own node, or a node on a shared leaf edge; or one
// closer than 4e-5 rad) is rare, so the wave tests four sources at once (one
// ballot) and only a batch holding such a pair takes the guarded form, with
// log_tab for the close ones.
// Bound: FP64 vector issue, 16 instructions per pair (23 with log_tab and a
// compare on every pair), at the 1.9 GHz the chip holds under this load: issue is
// busy 88% of the time, the gathers from the table (9 LDS cycles each, bank
// conflicts included) half of it.  Microseconds per launch with log_tab, one
// wave per tile, and now: 6 x 28^2 281 -> 25, 6 x 64^2 494 -> 97, degree 10 at
// 6 x 256^2 (theta 0.7) 1751 -> 1033, 6 x 512^2 4890 -> 3632.
constexpr double kSkipOneMinusDot = 1.0 - (1.0 - 1e-15);

// The logarithms of N values any of which may be outside log_wide's range; zero
// at a skipped pair.
template <int N>
__device__ inline void log_guarded(double (&d)[N], double (&l)[N], const LogTabEntry* __restrict__ wide,
                                   const LogTabEntry* __restrict__ tab, double c7) {
  bool skip[N];
  uint32_t h[N], far = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    skip[i] = d[i] <= kSkipOneMinusDot;
    d[i] = skip[i] ? 1.0 : d[i];
    h[i] = log_wide_cell(d[i]);
    far = h[i] > far ? h[i] : far;
  }
  if (__builtin_amdgcn_ballot_w64(far >= kLogWideSpan) != 0) {
#pragma unroll 1
    for (int i = 0; i < N; ++i) l[i] = log_tab(d[i], tab);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) l[i] = log_wide(d[i], h[i], wide, c7);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) l[i] = skip[i] ? 0.0 : l[i];
}

// Waves per tile of the log kernel, whose table (32 KB of LDS) holds a compute
// unit to four workgroups: at 126 tiles 62 / 38 / 27 us with 4 / 8 / 16 waves, at
// 636 122 / 105 / 112, at 2,556 316 / 280 / 346, at 40,956 4160 / 3843 / 5155.
inline int log_waves(int ntiles) { return ntiles < 400 ? 16 : 8; }

template <int S>
__global__ __launch_bounds__(64 * S) void k_log64(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                  const SourceSet* __restrict__ sets,
                                                  const SrcRec64* __restrict__ rec, double* __restrict__ part,
                                                  double* __restrict__ proxy, int assign) {
  __shared__ LogTabEntry wide[kLogWideSize];
  for (int i = threadIdx.x; i < kLogWideSize; i += 64 * S) wide[i] = t.logwide[i];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const int64_t u = (int64_t)T.first + (lane < T.count ? lane : T.count - 1);
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  const double c7 = in_vgpr(1.0 / 7.0);
  double acc[1] = {0};
  walk_sets<S>(T, sets, wave, [&](const SourceSet& set, int a, int b) {
    const SrcRec64* __restrict__ r = rec + set.first;
    int k = a;
    for (; k + 4 <= b; k += 4) {
      double d[4];
      uint32_t h[4], far = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d[i] = one_minus_dot(x, y, z, r[k + i].x, r[k + i].y, r[k + i].z);
        h[i] = log_wide_cell(d[i]);
        far = h[i] > far ? h[i] : far;
      }
      loaded(r[k].q, r[k + 1].q, r[k + 2].q, r[k + 3].q);
      double l[4];
      if (__builtin_amdgcn_ballot_w64(far >= kLogWideSpan) != 0) {
        log_guarded(d, l, wide, t.logtab, c7);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) l[i] = log_wide(d[i], h[i], wide, c7);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[0] = fma(l[i], r[k + i].q, acc[0]);
    }
    for (; k < b; ++k) {
      const SrcRec64 s = r[k];
      double d[1] = {one_minus_dot(x, y, z, s.x, s.y, s.z)}, l[1];
      log_guarded(d, l, wide, t.logtab, c7);
      acc[0] = fma(l[0], s.q, acc[0]);
    }
  });
  tile_sum<S>(acc, wave, lane);
  if (wave == 0 && lane < T.count) store_s(t, u, part, proxy, acc[0], assign);
}

// The same in lane copies (lanes.hpp) of two targets, for tiles of at most 42 rows
// (lanes64).  Microseconds per pair call, one wave per tile and here: 6 x 96^2 (degree
// 8) 459 -> 155, 6 x 192^2 1109 -> 548 (a row per lane and waves sharing the tile: 672 a
// launch), degree 5 725 -> 342, 6 x 160^2 (degree 4) 502 -> 232.
template <int S>
__global__ __launch_bounds__(64 * S) void k_log64_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                        const SourceSet* __restrict__ sets,
                                                        const SrcRec64* __restrict__ rec, double* __restrict__ part,
                                                        double* __restrict__ proxy, int assign) {
  constexpr int NT = 2;
  __shared__ LogTabEntry wide[kLogWideSize];
  __shared__ __align__(16) double stage[S][kLaneSlots * 4];
  for (int i = threadIdx.x; i < kLogWideSize; i += 64 * S) wide[i] = t.logwide[i];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  const double c7 = in_vgpr(1.0 / 7.0);
  double x[NT], y[NT], z[NT], w[NT][1];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    x[q] = t.px[u]; y[q] = t.py[u]; z[q] = t.pz[u];
    w[q][0] = 0;
  }
  lane_walk2<S, 2>(T, sets, reinterpret_cast<const v4f*>(rec), l, reinterpret_cast<v4f*>(stage[wave]), wave, lane,
                   [&](const v4f* r0, const v4f* r1) {
    const SrcRec64 R[2] = {*reinterpret_cast<const SrcRec64*>(r0), *reinterpret_cast<const SrcRec64*>(r1)};
    double d[4], lg[4];
    uint32_t h[4], far = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = i & 1;
      d[i] = one_minus_dot(x[q], y[q], z[q], R[i >> 1].x, R[i >> 1].y, R[i >> 1].z);
      h[i] = log_wide_cell(d[i]);
      far = h[i] > far ? h[i] : far;
    }
    if (__builtin_amdgcn_ballot_w64(far >= kLogWideSpan) != 0) {
      log_guarded(d, lg, wide, t.logtab, c7);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) lg[i] = log_wide(d[i], h[i], wide, c7);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i & 1][0] = fma(lg[i], R[i >> 1].q, w[i & 1][0]);
  });
  double s[1];
  lane_sum<NT, 1, S>(l, w, stage, wave, lane, s);
  if (wave == 0 && lane < T.count) store_s(t, (int64_t)T.first + lane, part, proxy, s[0], assign);
}

// Horner multipliers of the FP64 regularised-Laplacian kernel in vector registers.
struct LapV64 {
  double a1, b2, c24;
};

// K(t) of k_lap64 where t >= t_sat (erf factor exactly 1): A + E B.
__device__ inline double lap_pair(double dp, const LapCoef64& kp, const LapV64& kv, const double* etab) {
  const double t2 = dp * dp;
  const double A = dp * fma(kv.a1, t2, kp.a0);
  const double B = fma(fma(kv.b2, t2, kp.b1), t2, kp.b0);
  return fma(exp_neg(fma(t2, kp.inv_eps, -kp.inv_eps), etab, kv.c24), B, A);
}
// K(t) for any t: A + f E B, zero at or below the cut.
__device__ inline double lap_pair_slow(double dp, const LapCoef64& kp, const LapV64& kv, const double* etab) {
  const double t2 = dp * dp;
  const double A = dp * fma(kv.a1, t2, kp.a0);
  const double B = fma(fma(kv.b2, t2, kp.b1), t2, kp.b0);
  const double sv = dp * kp.inv_eps;
  const double f = sv >= 6.0 ? 1.0 : (sv <= -6.0 ? 0.0 : 0.5 * (1.0 + erf(sv)));
  const double K = fma(exp_neg(fma(t2, kp.inv_eps, -kp.inv_eps), etab, kv.c24) * f, B, A);
  return dp > kp.cut ? K : 0.0;
}

// Regularised-Laplacian pair kernel (lap_panel_interaction,
// laplacian_impl.hpp:46-66, eps = 0.1): phi += K(x.y) q with K in the folded
// form of lapkernel.hpp (A + E B where t >= 6 eps, erf only below).  Sources
// are displaced and projected; the records hold q' = -q/(4 pi), so the
// coefficients arrive multiplied by -4 pi / eps^{5/2}.  Over 99% of the pair
// work has t > 0.6, so a wave tests four sources at once (a ballot) and
// evaluates erf only when one of its pairs needs it.  The exponential is
// exp_neg (fasttab.hpp: its argument lies in [-1/eps, 0]) on the context's
// table, staged in LDS.  S waves share a tile (pairwalk.hpp).
// Bound: FP64 vector issue, 22 instructions per pair.  Microseconds per launch
// with one wave per tile (two sub-tiles of 18 rows in lane groups at m = 6) and
// now: 6 x 28^2 321 -> 98, 6 x 64^2 612 -> 223, 6 x 192^2 (degree 8) 1176 -> 1028,
// degree 10 at 6 x 256^2 2366 -> 1673.
template <int S>
__global__ __launch_bounds__(64 * S) void k_lap64(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                  const SourceSet* __restrict__ sets,
                                                  const SrcRec64* __restrict__ rec, LapCoef64 kp,
                                                  double* __restrict__ part, double* __restrict__ proxy, int assign) {
  __shared__ double etab[kExpNegTabSize];
  for (int i = threadIdx.x; i < kExpNegTabSize; i += 64 * S) etab[i] = t.expnegtab[i];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = strip_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const int64_t u = (int64_t)T.first + (lane < T.count ? lane : T.count - 1);
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  // every pair passes the cut when 1 - 30 eps < -1 (eps = 0.1); else every pair takes the slow form
  const double fast_from = kp.cut < -1.0 ? kp.t_sat : 4.0;
  const LapV64 kv{in_vgpr(kp.a1), in_vgpr(kp.b2), in_vgpr(1.0 / 24.0)};
  double acc[1] = {0};
  walk_sets<S>(T, sets, wave, [&](const SourceSet& set, int a, int b) {
    const SrcRec64* __restrict__ r = rec + set.first;
    int k = a;
    for (; k + 4 <= b; k += 4) {
      double dp[4], K[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) dp[i] = x * r[k + i].x + y * r[k + i].y + z * r[k + i].z;
      loaded(r[k].q, r[k + 1].q, r[k + 2].q, r[k + 3].q);
      if (__builtin_amdgcn_ballot_w64(fmin(fmin(dp[0], dp[1]), fmin(dp[2], dp[3])) < fast_from) != 0) {
#pragma unroll 1
        for (int i = 0; i < 4; ++i) {
          const SrcRec64 s = r[k + i];
          acc[0] = fma(lap_pair_slow(x * s.x + y * s.y + z * s.z, kp, kv, etab), s.q, acc[0]);
        }
        continue;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) K[i] = lap_pair(dp[i], kp, kv, etab);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[0] = fma(K[i], r[k + i].q, acc[0]);
    }
    for (; k < b; ++k) {
      const SrcRec64 s = r[k];
      const double dp = x * s.x + y * s.y + z * s.z;
      const bool slow = __builtin_amdgcn_ballot_w64(dp < fast_from) != 0;
      acc[0] = fma(slow ? lap_pair_slow(dp, kp, kv, etab) : lap_pair(dp, kp, kv, etab), s.q, acc[0]);
    }
  });
  tile_sum<S>(acc, wave, lane);
  if (wave == 0 && lane < T.count) store_s(t, u, part, proxy, acc[0], assign);
}

// The same in lane copies (lanes.hpp) of two targets, for tiles of at most 42 rows
// (lanes64), W tiles to a workgroup.  Microseconds per pair call in lane groups of one
// target and here: 6 x 96^2 (degree 8) 445 -> 247, 6 x 192^2 1167 -> 762 (a row per lane:
// 1010 a launch), degree 5 586 -> 437, 6 x 160^2 (degree 4) 360 -> 262 (419).
template <int S, int W>
__global__ __launch_bounds__(64 * S * W) void k_lap64_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                        const SourceSet* __restrict__ sets,
                                                        const SrcRec64* __restrict__ rec, LapCoef64 kp,
                                                        double* __restrict__ part, double* __restrict__ proxy,
                                                        int assign) {
  constexpr int NT = 2;
  __shared__ double etab[kExpNegTabSize];
  __shared__ __align__(16) double stage[W][S][kLaneSlots * 4];
  for (int i = threadIdx.x; i < kExpNegTabSize; i += 64 * S * W) etab[i] = t.expnegtab[i];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % S;
  const int sub = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / S;
  const int lane = threadIdx.x & 63;
  static_assert(S == 1 || W == 1, "waves that share a tile meet at barriers: one tile per workgroup");
  const int tile = strip_tile((ntiles + W - 1) / W) * W + sub;
  if (tile >= ntiles) return;  // all waves of the tile
  const TargetTile T = tiles[tile];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  const double fast_from = kp.cut < -1.0 ? kp.t_sat : 4.0;
  const LapV64 kv{in_vgpr(kp.a1), in_vgpr(kp.b2), in_vgpr(1.0 / 24.0)};
  double x[NT], y[NT], z[NT], w[NT][1];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    x[q] = t.px[u]; y[q] = t.py[u]; z[q] = t.pz[u];
    w[q][0] = 0;
  }
  lane_walk2<S, 2, true>(T, sets, reinterpret_cast<const v4f*>(rec), l, reinterpret_cast<v4f*>(stage[sub][wave]), wave, lane,
                         [&](const v4f* r0, const v4f* r1) {
    const SrcRec64 R[2] = {*reinterpret_cast<const SrcRec64*>(r0), *reinterpret_cast<const SrcRec64*>(r1)};
    double dp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = i & 1;
      dp[i] = x[q] * R[i >> 1].x + y[q] * R[i >> 1].y + z[q] * R[i >> 1].z;
    }
    if (__builtin_amdgcn_ballot_w64(fmin(fmin(dp[0], dp[1]), fmin(dp[2], dp[3])) < fast_from) != 0) {
#pragma unroll 1
      for (int i = 0; i < 2; ++i) {
        const SrcRec64 s = *reinterpret_cast<const SrcRec64*>(i ? r1 : r0);
#pragma unroll
        for (int q = 0; q < NT; ++q)
          w[q][0] = fma(lap_pair_slow(x[q] * s.x + y[q] * s.y + z[q] * s.z, kp, kv, etab), s.q, w[q][0]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i & 1][0] = fma(lap_pair(dp[i], kp, kv, etab), R[i >> 1].q, w[i & 1][0]);
    }
  });
  double s[1];
  lane_sum<NT, 1, S>(l, w, stage[sub], wave, lane, s);
  if (wave == 0 && lane < T.count) store_s(t, (int64_t)T.first + lane, part, proxy, s[0], assign);
}

// Mixed-precision regularised-Laplacian pairs in the folded form of
// lapkernel.hpp: the squared chord h2 = |x - y|^2 = 2(1 - t) in FP32 from
// panel-centred coordinates, t^2 - 1 = h2 (h2/4 - 1) (no cancellation), the
// exponential on the hardware base-2 exponential of u = (t^2 - 1) log2(e)/eps
// (u in [-2/(eps ln 2), 0]), the polynomials in u; erf only when a wave-wide
// ballot finds a pair with t < 0.6 (elsewhere it is +-1 in FP32 too).  FP32
// sums per source set; c3 (times -4 pi, undoing the record's -1/(4 pi))
// applied per set in FP64.
__device__ inline float lap32_K_slow(float h2, const LapCoef32& kp, float a1v, float b2v) {
  const float tt = fmaf(h2, -0.5f, 1.0f);
  const float u = h2 * fmaf(h2, 0.25f * kp.k, -kp.k);
  const float A = tt * fmaf(a1v, u, kp.a0);
  const float B = fmaf(fmaf(b2v, u, kp.b1), u, kp.b0);
  const float sv = tt * kp.inv_eps;
  const float f = sv >= 6.0f ? 1.0f : (sv <= -6.0f ? 0.0f : 0.5f * (1.0f + erff(sv)));
  const float K = fmaf(__builtin_amdgcn_exp2f(u) * f, B, A);
  return tt > kp.cut ? K : 0.0f;
}

// Lane copies (lanes.hpp) of two targets.
// Bound: FP32 vector issue, 16 instructions and a base-2 exponential per pair.
// Microseconds per launch before and with 2 / 4 / 8 waves per tile: 126 tiles 217,
// 162 / 88 / 56; 636 352, 153 / 97 / 90; 2,556 (36 rows) 202, 148 / 123 / 124; 10,236
// 502, 356 / 345 / 363; 40,956 2522, 2073 / 2032 / 2068.
template <int S>
__global__ __launch_bounds__(64 * S) void k_lap_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                      const SourceSet* __restrict__ sets,
                                                      const SrcRec32* __restrict__ rec, LapCoef32 kp, double c3,
                                                      double* __restrict__ part, double* __restrict__ proxy,
                                                      int assign) {
  constexpr int NT = 2;
  __shared__ __align__(16) double stage[S][kLaneSlots * 2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const DevPanel& PT = t.panels[T.panel];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  // t < t_sat  <=>  h2 > h_sat; every pair passes the cut when 1 - 30 eps < -1 (eps = 0.1), else every pair is slow
  const float h_sat = kp.cut < -1.0f ? 2.0f * (1.0f - kp.t_sat) : -1.0f;
  LapCoef32 kv = kp;  // the fast form's coefficients in vector registers
  kv.a1 = in_vgpr_f(kp.a1); kv.a0 = in_vgpr_f(kp.a0);
  kv.b2 = in_vgpr_f(kp.b2); kv.b1 = in_vgpr_f(kp.b1); kv.b0 = in_vgpr_f(kp.b0);
  const float k4 = in_vgpr_f(0.25f * kp.k), km = in_vgpr_f(-kp.k);
  float ax[NT], ay[NT], az[NT], px[NT], py[NT], pz[NT], v[NT];
  double w[NT][1];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    ax[q] = (float)(t.px[u] - PT.cx);
    ay[q] = (float)(t.py[u] - PT.cy);
    az[q] = (float)(t.pz[u] - PT.cz);
    w[q][0] = 0;
  }
  lane_walk<S, 1, 1>(
      T, sets, reinterpret_cast<const v4f*>(rec), l, reinterpret_cast<v4f*>(stage[wave]), 0.f, wave, lane,
      [&](const SourceSet& set) {
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          px[q] = ax[q] + set.ox;
          py[q] = ay[q] + set.oy;
          pz[q] = az[q] + set.oz;
          v[q] = 0.f;
        }
      },
      [&](const v4f* r) {
        const v4f s = r[0];
        float h2[NT], K[NT];
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          const float d0 = s.x - px[q], d1 = s.y - py[q], d2 = s.z - pz[q];
          h2[q] = fmaf(d0, d0, fmaf(d1, d1, d2 * d2));
          const float u = h2[q] * fmaf(h2[q], k4, km);
          const float A = fmaf(h2[q], -0.5f, 1.0f) * fmaf(kv.a1, u, kv.a0);
          const float B = fmaf(fmaf(kv.b2, u, kv.b1), u, kv.b0);
          K[q] = fmaf(__builtin_amdgcn_exp2f(u), B, A);
        }
        if (__builtin_amdgcn_ballot_w64(fmaxf(h2[0], h2[1]) > h_sat) != 0) {
          // a real branch (the empty asm keeps the compiler from evaluating erf on every pair)
          __asm__ volatile("");
#pragma unroll
          for (int q = 0; q < NT; ++q) K[q] = lap32_K_slow(h2[q], kp, kp.a1, kp.b2);
        }
#pragma unroll
        for (int q = 0; q < NT; ++q) v[q] = fmaf(K[q], s.w, v[q]);
      },
      [&](const SourceSet&) {
#pragma unroll
        for (int q = 0; q < NT; ++q) w[q][0] += c3 * (double)v[q];
      });
  double s[1];
  lane_sum<NT, 1, S>(l, w, stage, wave, lane, s);
  if (wave == 0 && lane < T.count) store_s(t, (int64_t)T.first + lane, part, proxy, s[0], assign);
}

// Mixed precision Biot-Savart: FP32 pair arithmetic in panel-centred
// coordinates with 1 - x.y computed as |x - y|^2 / 2, FP32 partial sums per
// source set flushed into FP64 accumulators, cross product in FP64.
__global__ __launch_bounds__(256) void k_bve_mixed(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                   const SourceSet* __restrict__ sets,
                                                   const SrcRec32* __restrict__ rec, float eps, Ptr3 part,
                                                   Ptr3 proxy, int assign, int xcd) {
  member_targets(t, part, proxy);
  rec += (int64_t)blockIdx.y * t.U;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = shaped_tile(t.xcd_start ? t.xcd_start + 9 : nullptr, wave, xcd);
  if (tile >= ntiles) return;
  const TargetTile T = tiles[tile];
  const DevPanel& PT = t.panels[T.panel];
  const int64_t u = (int64_t)T.first + (lane < T.count ? lane : T.count - 1);
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  const float ax = (float)(x - PT.cx), ay = (float)(y - PT.cy), az = (float)(z - PT.cz);
  double w0 = 0, w1 = 0, w2 = 0;
  for (int e = T.src_begin; e < T.src_end; ++e) {
    const SourceSet S = sets[e];
    // target relative to the source panel centre: a + (c_t - c_s)
    const float px = ax + S.ox, py = ay + S.oy, pz = az + S.oz;
    const SrcRec32* __restrict__ r = rec + S.first;
    float v0 = 0.f, v1 = 0.f, v2 = 0.f;
#pragma unroll 4
    for (int k = 0; k < S.count; ++k) {
      const SrcRec32 s = r[k];
      const float d0 = s.x - px, d1 = s.y - py, d2 = s.z - pz;
      const float h = fmaf(0.5f, fmaf(d0, d0, fmaf(d1, d1, d2 * d2)), eps);
      const float g = __builtin_amdgcn_rcpf(h) * s.q;
      v0 = fmaf(g, d0, v0);
      v1 = fmaf(g, d1, v1);
      v2 = fmaf(g, d2, v2);
    }
    w0 += v0; w1 += v1; w2 += v2;
  }
  if (lane < T.count) store_u(t, u, part, proxy, y * w2 - z * w1, z * w0 - x * w2, x * w1 - y * w0, assign);
}

// Mixed precision log kernel: log(|x - y|^2 / 2) in FP32, same guard.  The
// pair takes the hardware base-2 logarithm (v_log_f32; h >= 1e-15 is far from
// the denormal range, so the library's range scaling is not needed) and the
// factor ln 2 is applied once per source set in FP64.
// Lane copies (lanes.hpp) of two targets.
// Bound: FP32 vector issue, 10 instructions and a logarithm per pair.
// Microseconds per launch before and with 2 / 4 / 8 waves per tile: 126 tiles 125,
// 40 / 23 / 18; 636 202, 77 / 47 / 45; 2,556 (36 rows) 203, 89 / 78 / 81; 10,236 510,
// 258 / 258 / 270; 40,956 2039, 1537 / 1531 / 1565.
template <int S>
__global__ __launch_bounds__(64 * S) void k_log_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                      const SourceSet* __restrict__ sets,
                                                      const SrcRec32* __restrict__ rec, double* __restrict__ part,
                                                      double* __restrict__ proxy, int assign) {
  constexpr int NT = 2;
  __shared__ __align__(16) double stage[S][kLaneSlots * 2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const DevPanel& PT = t.panels[T.panel];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  float ax[NT], ay[NT], az[NT], px[NT], py[NT], pz[NT], v[NT];
  double w[NT][1];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    ax[q] = (float)(t.px[u] - PT.cx);
    ay[q] = (float)(t.py[u] - PT.cy);
    az[q] = (float)(t.pz[u] - PT.cz);
    w[q][0] = 0;
  }
  lane_walk<S, 1, 2>(
      T, sets, reinterpret_cast<const v4f*>(rec), l, reinterpret_cast<v4f*>(stage[wave]), 4.f, wave, lane,
      [&](const SourceSet& set) {
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          px[q] = ax[q] + set.ox;
          py[q] = ay[q] + set.oy;
          pz[q] = az[q] + set.oz;
          v[q] = 0.f;
        }
      },
      [&](const v4f* r) {
        const v4f s = r[0];
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          const float d0 = s.x - px[q], d1 = s.y - py[q], d2 = s.z - pz[q];
          const float h = 0.5f * fmaf(d0, d0, fmaf(d1, d1, d2 * d2));
          const float l2 = __builtin_amdgcn_logf(h);
          v[q] = fmaf(h > 1e-15f ? l2 : 0.f, s.w, v[q]);
        }
      },
      [&](const SourceSet&) {
#pragma unroll
        for (int q = 0; q < NT; ++q) w[q][0] += 0.69314718055994530942 * (double)v[q];
      });
  double s[1];
  lane_sum<NT, 1, S>(l, w, stage, wave, lane, s);
  if (wave == 0 && lane < T.count) store_s(t, (int64_t)T.first + lane, part, proxy, s[0], assign);
}

typedef __bf16 v4bf __attribute__((ext_vector_type(4)));

// The kernel products of NTT 16 x 16 tiles, D_ij = beta_i - p_j.b_i: FP32
// (v_mfma_f32_16x16x4_f32, lane i + 16 k holding component k), or, for an M2L
// set on a context with bf16 M2L, bf16 operands with FP32 accumulation
// (v_mfma_f32_16x16x16_bf16: lane i + 16 k holds K slots 4k..4k+3, the
// component in the first and zeros in the others, the same pairing of A and B).
// One branch for all NTT products.
template <int NTT>
__device__ inline void kernel_products(float a1, const float (&b1)[NTT], bool lowp, v4f (&d)[NTT]) {
  if (lowp) {
    const v4bf a = v4bf{(__bf16)a1, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt)
      d[tt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
          a, v4bf{(__bf16)b1[tt], (__bf16)0.f, (__bf16)0.f, (__bf16)0.f}, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  } else {
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt)
      d[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1[tt], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  }
}

// Records of the MFMA kernel (16-padded per source set; padding slots zero).
__global__ void k_src_mfma(DevTree t, const double* __restrict__ q_part, const double* __restrict__ q_proxy,
                           CPtr3 dpart, CPtr3 dprox, SrcRecMfma* __restrict__ rec) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= t.U16) return;
  member_sources(t, q_part, q_proxy, dpart, dprox);
  rec += (int64_t)blockIdx.y * t.U16;
  const int64_t lp = (int64_t)t.Pl * t.m2p;
  int panel, k;
  int64_t u;
  bool valid;
  if (s < lp) {
    const int leaf = (int)(s / t.m2p);
    k = (int)(s % t.m2p);
    panel = t.offset + leaf;
    valid = k < t.m2;
    u = (int64_t)leaf * t.m2 + k;
  } else {
    const int64_t v = s - lp;
    panel = (int)(v / t.np16);
    k = (int)(v % t.np16);
    valid = k < t.n;
    u = t.npart + (int64_t)panel * t.n + k;
  }
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (valid) {
    double x = t.px[u], y = t.py[u], z = t.pz[u], q;
    if (u < t.npart) {
      if (dpart.p[0]) { x += dpart.p[0][u]; y += dpart.p[1][u]; z += dpart.p[2][u]; }
      q = q_part[u];
    } else {
      const int64_t w = u - t.npart;
      if (dprox.p[0]) { x += dprox.p[0][w]; y += dprox.p[1][w]; z += dprox.p[2][w]; }
      q = q_proxy[w];
    }
    project_to_sphere(x, y, z);
    const DevPanel& P = t.panels[panel];
    const float bx = (float)(x - P.cx), by = (float)(y - P.cy), bz = (float)(z - P.cz);
    const double qq = kNegInv4Pi * q;
    v[0] = bx; v[1] = by; v[2] = bz;
    v[3] = (float)(0.5 * ((double)bx * bx + (double)by * by + (double)bz * bz));
    v[4] = (float)(qq * bx); v[5] = (float)(qq * by); v[6] = (float)(qq * bz); v[7] = (float)qq;
  }
  float* tile = reinterpret_cast<float*>(rec) + (s >> 4) * 128;
  const int i = (int)(s & 15);
#pragma unroll
  for (int k = 0; k < 4; ++k) tile[k * 16 + i] = v[k];
#pragma unroll
  for (int c = 0; c < 4; ++c) tile[64 + ((i >> 2) * 4 + c) * 4 + (i & 3)] = v[4 + c];
}

// Mixed-precision Biot-Savart pair kernel on the matrix cores, for contexts with
// bf16 M2L products (k_bve_lanes takes the others).
//
// Per wave: NTT (1..4) target tiles of 16 (up to 64 targets of one panel).
// For every source set, coordinates are taken relative to the source-panel
// centre c_s: target p = (x - c_t) + (c_t - c_s), source b (record).  For a
// 16 x 16 tile
//   D = alpha_j + beta_i - p_j.b_i = eps + |p_j - b_i|^2 / 2  (= 1 - x.y + eps)
// is one v_mfma_f32_16x16x4_f32 (A = (b, beta) per source, B = (-p, 1) per
// target) plus alpha per target column; R = 1/D on the vector unit; then four
// v_mfma_f32_4x4x1_16b_f32 accumulate W_j = sum_i R_ij (q b_i, q), 4
// components x 16 targets per quarter of the source tile.  After each source
// set every lane adds its quarter's w_j += W_xyz - p_j W_q into FP64; the four
// quarters are summed across lanes once at the end, and u = x cross w in FP64
// (x cross y = x cross (y - x)).
// Lane layouts: A[i][k] from lane i + 16 k, B[k][j] from lane j + 16 k,
// D[i][j] in lane j + 16 (i / 4), register i % 4 (16x16x4); block b of the
// 4x4x1 form uses lanes 4 b .. 4 b + 3 (A row / B column = lane % 4, D row =
// register).  The next source tile's operands are loaded before the current
// tile's arithmetic (every index stays inside the set's padded records).
template <int NTT>
__device__ inline void bve_mfma_tiles(const DevTree& t, const TargetTile& T, const SourceSet* __restrict__ sets,
                                      const float* __restrict__ rec, float eps, int lane, double (&w)[4][3]) {
  const int col = lane & 15, grp = lane >> 4;
  const DevPanel& PT = t.panels[T.panel];
  float ax[NTT], ay[NTT], az[NTT];
#pragma unroll
  for (int tt = 0; tt < NTT; ++tt) {
    const int j = min(tt * 16 + col, T.count - 1);
    const int64_t u = (int64_t)T.first + j;
    ax[tt] = (float)(t.px[u] - PT.cx);
    ay[tt] = (float)(t.py[u] - PT.cy);
    az[tt] = (float)(t.pz[u] - PT.cz);
  }
  const int off_b = 64 + 4 * (grp * 4 + (lane & 3));  // float4: (q b, q)[lane % 4] of sources 4 grp + 0..3
  if (T.src_begin >= T.src_end) return;
  // b1 = (-p_x, -p_y, -p_z, 1)[lane / 16] without branches
  const float sx = grp == 0 ? -1.f : 0.f, sy = grp == 1 ? -1.f : 0.f, sz = grp == 2 ? -1.f : 0.f;
  const float s1 = grp == 3 ? 1.f : 0.f;
  float px[NTT], py[NTT], pz[NTT], b1[NTT], alpha[NTT];
  v4f acc[NTT];
  auto begin_set = [&](const SourceSet& S) {
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt) {
      px[tt] = ax[tt] + S.ox;
      py[tt] = ay[tt] + S.oy;
      pz[tt] = az[tt] + S.oz;
      alpha[tt] = fmaf(0.5f, fmaf(px[tt], px[tt], fmaf(py[tt], py[tt], pz[tt] * pz[tt])), eps);
      b1[tt] = fmaf(sx, px[tt], fmaf(sy, py[tt], fmaf(sz, pz[tt], s1)));
      acc[tt] = v4f{0.f, 0.f, 0.f, 0.f};
    }
  };
  // One flat loop over the 16-source tiles of all source sets, so that the
  // operands of the next tile are loaded one tile ahead across set boundaries
  // and the set records two sets ahead (the loads stay in the loop body).
  const int last = T.src_end - 1;
  int e = T.src_begin;
  SourceSet S = sets[e], Sn = sets[min(e + 1, last)], Snn = sets[min(e + 2, last)];
  begin_set(S);
  int nst = (S.count + 15) >> 4, st = 0;
  const float* __restrict__ r = rec + (int64_t)S.first16 * 8;
  float a1 = r[lane];
  v4f bq = *reinterpret_cast<const v4f*>(r + off_b);
  while (true) {
    const float* __restrict__ rn = st + 1 < nst ? r + 128 * (st + 1) : rec + (int64_t)Sn.first16 * 8;
    const float na1 = rn[lane];
    const v4f nbq = *reinterpret_cast<const v4f*>(rn + off_b);
    v4f d[NTT];
    kernel_products<NTT>(a1, b1, S.m2l, d);
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
      for (int q = 0; q < 4; ++q) d[tt][q] = __builtin_amdgcn_rcpf(d[tt][q] + alpha[tt]);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int tt = 0; tt < NTT; ++tt)
        acc[tt] = __builtin_amdgcn_mfma_f32_4x4x1f32(bq[q], d[tt][q], acc[tt], 0, 0, 0);
    a1 = na1;
    bq = nbq;
    if (++st == nst) {
#pragma unroll
      for (int tt = 0; tt < NTT; ++tt) {
        w[tt][0] += (double)fmaf(-px[tt], acc[tt][3], acc[tt][0]);
        w[tt][1] += (double)fmaf(-py[tt], acc[tt][3], acc[tt][1]);
        w[tt][2] += (double)fmaf(-pz[tt], acc[tt][3], acc[tt][2]);
      }
      if (++e > last) break;
      S = Sn;
      Sn = Snn;
      Snn = sets[min(e + 2, last)];
      begin_set(S);
      r = rec + (int64_t)S.first16 * 8;
      nst = (S.count + 15) >> 4;
      st = 0;
    }
  }
}

__global__ __launch_bounds__(256) void k_bve_mfma(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                  const SourceSet* __restrict__ sets,
                                                  const float* __restrict__ rec, float eps, Ptr3 part,
                                                  Ptr3 proxy, int assign, int xcd) {
  member_targets(t, part, proxy);
  rec += (int64_t)blockIdx.y * t.U16 * 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;
  const int tile = shaped_tile(t.xcd_start, wave, xcd);
  if (tile >= ntiles) return;
  const TargetTile T = tiles[tile];
  const int ntt = (T.count + 15) >> 4;
  double w[4][3];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) w[tt][0] = w[tt][1] = w[tt][2] = 0.0;
  switch (ntt) {
    case 4: bve_mfma_tiles<4>(t, T, sets, rec, eps, lane, w); break;
    case 3: bve_mfma_tiles<3>(t, T, sets, rec, eps, lane, w); break;
    case 2: bve_mfma_tiles<2>(t, T, sets, rec, eps, lane, w); break;
    default: bve_mfma_tiles<1>(t, T, sets, rec, eps, lane, w); break;
  }
  // sum the four source quarters (lanes col, col+16, col+32, col+48)
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      w[tt][k] += __shfl_xor(w[tt][k], 16);
      w[tt][k] += __shfl_xor(w[tt][k], 32);
    }
  // lane group g stores target tile g
  const int j = grp * 16 + col;
  if (grp < ntt && j < T.count) {
    const double w0 = grp == 0 ? w[0][0] : grp == 1 ? w[1][0] : grp == 2 ? w[2][0] : w[3][0];
    const double w1 = grp == 0 ? w[0][1] : grp == 1 ? w[1][1] : grp == 2 ? w[2][1] : w[3][1];
    const double w2 = grp == 0 ? w[0][2] : grp == 1 ? w[1][2] : grp == 2 ? w[2][2] : w[3][2];
    const int64_t u = (int64_t)T.first + j;
    const double x = t.px[u], y = t.py[u], z = t.pz[u];
    store_u(t, u, part, proxy, y * w2 - z * w1, z * w0 - x * w2, x * w1 - y * w0, assign);
  }
}

// ---- multi-right-hand-side form (ensembles with shared positions)
//
// When every member of an ensemble has its sources and targets at the same
// positions (the undisplaced first RK4 stage), R_ij = 1/(eps + |p_j - b_i|^2/2)
// is the same matrix for all members and the pair sums are the product
// W[j][n] = sum_i R_ij Q[i][n] with one column n per member and component
// (q b_x, q b_y, q b_z, q).  R comes from the 16x16x4 product of the
// single-member kernel once per wave and is used again as the A operand of
// 16x16x4 products against 16 charge columns (four members): register r of
// lane l holds R[4 (l/16) + r][l % 16], i.e. A[j][a] = R[4 a + r][j], so
// product r takes sources {4 a + r}, and its B operand is Q[4 a + r][n] from
// lane n + 16 a.  The result W[j][n] lands in lane n + 16 (j/4), register
// j % 4.
//
// Charge columns: for 16-source tile g and chunk k of four members, 64 lanes x
// float4,  qcol[((g * nchunk + k) * 64 + n + 16 a) * 4 + r] = Q[4 a + r][n],
// n = 4 * (member % 4) + c.  Members beyond the ensemble (padding of the last
// chunk group) have zero columns.
__global__ void k_src_mrhs(DevTree t, const double* __restrict__ q_part, const double* __restrict__ q_proxy,
                           const float* __restrict__ geo, int nmem, int nchunk, float* __restrict__ qcol) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= t.U16) return;
  const int mem = (int)blockIdx.y;
  const int64_t lp = (int64_t)t.Pl * t.m2p;
  int64_t u;
  bool valid;
  if (s < lp) {
    const int k = (int)(s % t.m2p);
    valid = k < t.m2;
    u = (s / t.m2p) * t.m2 + k;
  } else {
    const int64_t v = s - lp;
    const int k = (int)(v % t.np16);
    valid = k < t.n;
    u = t.npart + (v / t.np16) * t.n + k;
  }
  double q = 0.0;
  if (valid && mem < nmem)
    q = u < t.npart ? q_part[(int64_t)mem * t.npart + u]
                    : q_proxy[(int64_t)mem * t.P * t.n + (u - t.npart)];
  const int64_t g = s >> 4;
  const int i = (int)(s & 15);
  const float* tile = geo + g * 128;  // (b_x, b_y, b_z) of source i at [16 k + i]
  const double qq = kNegInv4Pi * q;
  const float v[4] = {(float)(qq * tile[i]), (float)(qq * tile[16 + i]), (float)(qq * tile[32 + i]), (float)qq};
  float* o = qcol + ((g * nchunk + (mem >> 2)) * 64 + 16 * (i >> 2) + 4 * (mem & 3)) * 4 + (i & 3);
#pragma unroll
  for (int c = 0; c < 4; ++c) o[4 * c] = v[c];
}

// Lane SEL of each quad of lanes (DPP quad_perm, all four lanes read SEL).
template <int SEL>
__device__ inline float quad_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), SEL * 0x55, 0xF, 0xF, false));
}
template <int SEL>
__device__ inline double quad_bcast(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), SEL * 0x55, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), SEL * 0x55, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// Pair sums of NTT target tiles of 16 for CB chunks of four members.  Lane l
// accumulates, per source set, w[tt][cb][r] += W_c - p_c W_q for target
// tt*16 + 4 (l/16) + r, member 4 (chunk0 + cb) + (l%16)/4, component c = l % 4
// (lanes with c = 3 carry W_q and are discarded).
template <int NTT, int CB, bool M2L>
__device__ inline void bve_mrhs_tiles(const DevTree& t, const TargetTile& T, const SourceSet* __restrict__ sets,
                                      const float* __restrict__ geo, const float* __restrict__ qcol, int nchunk,
                                      int chunk0, float eps, int lane, double (&w)[4][CB][4]) {
  const int col = lane & 15, grp = lane >> 4, comp = lane & 3;
  const DevPanel& PT = t.panels[T.panel];
  const double* __restrict__ pc_arr = comp == 0 ? t.px : comp == 1 ? t.py : t.pz;
  const double pc_ctr = comp == 0 ? PT.cx : comp == 1 ? PT.cy : PT.cz;
  float ax[NTT], ay[NTT], az[NTT], ac[NTT][4];
#pragma unroll
  for (int tt = 0; tt < NTT; ++tt) {
    const int j = min(tt * 16 + col, T.count - 1);
    const int64_t u = (int64_t)T.first + j;
    ax[tt] = (float)(t.px[u] - PT.cx);
    ay[tt] = (float)(t.py[u] - PT.cy);
    az[tt] = (float)(t.pz[u] - PT.cz);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int jj = min(tt * 16 + 4 * grp + r, T.count - 1);
      ac[tt][r] = comp == 3 ? 0.f : (float)(pc_arr[(int64_t)T.first + jj] - pc_ctr);
    }
  }
  if (T.src_begin >= T.src_end) return;
  const float sx = grp == 0 ? -1.f : 0.f, sy = grp == 1 ? -1.f : 0.f, sz = grp == 2 ? -1.f : 0.f;
  const float s1 = grp == 3 ? 1.f : 0.f;
  float b1[NTT], alpha[NTT], pc[NTT][4];
  v4f acc[NTT][CB];
  auto begin_set = [&](const SourceSet& S) {
    const float so = comp == 0 ? S.ox : comp == 1 ? S.oy : comp == 2 ? S.oz : 0.f;
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt) {
      const float px = ax[tt] + S.ox, py = ay[tt] + S.oy, pz = az[tt] + S.oz;
      alpha[tt] = fmaf(0.5f, fmaf(px, px, fmaf(py, py, pz * pz)), eps);
      b1[tt] = fmaf(sx, px, fmaf(sy, py, fmaf(sz, pz, s1)));
#pragma unroll
      for (int r = 0; r < 4; ++r) pc[tt][r] = comp == 3 ? 0.f : ac[tt][r] + so;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[tt][cb] = v4f{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto qptr = [&](int64_t g) { return qcol + ((g * nchunk + chunk0) * 64 + lane) * 4; };
  const int last = T.src_end - 1;
  int e = T.src_begin;
  SourceSet S = sets[e], Sn = sets[min(e + 1, last)], Snn = sets[min(e + 2, last)];
  begin_set(S);
  int nst = (S.count + 15) >> 4, st = 0;
  int64_t g = S.first16 >> 4;
  float a1 = geo[g * 128 + lane];
  v4f qv[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) qv[cb] = *reinterpret_cast<const v4f*>(qptr(g) + cb * 256);
  while (true) {
    const int64_t gn = st + 1 < nst ? g + 1 : (int64_t)(Sn.first16 >> 4);
    const float na1 = geo[gn * 128 + lane];
    v4f nqv[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) nqv[cb] = *reinterpret_cast<const v4f*>(qptr(gn) + cb * 256);
    v4f d[NTT];
    kernel_products<NTT>(a1, b1, M2L && S.m2l, d);
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) d[tt][r] = __builtin_amdgcn_rcpf(d[tt][r] + alpha[tt]);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
          acc[tt][cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(d[tt][r], qv[cb][r], acc[tt][cb], 0, 0, 0);
    a1 = na1;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) qv[cb] = nqv[cb];
    g = gn;
    if (++st == nst) {
#pragma unroll
      for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float wq = quad_bcast<3>(acc[tt][cb][r]);
            w[tt][cb][r] += (double)fmaf(-pc[tt][r], wq, acc[tt][cb][r]);
          }
      if (++e > last) break;
      S = Sn;
      Sn = Snn;
      Snn = sets[min(e + 2, last)];
      begin_set(S);
      nst = (S.count + 15) >> 4;
      st = 0;
    }
  }
}

// One wave per target tile and group of CB member chunks (blockIdx.y).  Every
// (target, member, component) is written by exactly one lane.
template <int CB, bool M2L>
__global__ __launch_bounds__(256) void k_bve_mrhs(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                  const SourceSet* __restrict__ sets, const float* __restrict__ geo,
                                                  const float* __restrict__ qcol, int nchunk, int nmem, float eps,
                                                  Ptr3 part, Ptr3 proxy, int assign, int xcd) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4, comp = lane & 3;
  const int tile = shaped_tile(t.xcd_start, wave, xcd);
  if (tile >= ntiles) return;
  const TargetTile T = tiles[tile];
  const int ntt = (T.count + 15) >> 4;
  const int chunk0 = (int)blockIdx.y * CB;
  double w[4][CB][4];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int r = 0; r < 4; ++r) w[tt][cb][r] = 0.0;
  switch (ntt) {
    case 4: bve_mrhs_tiles<4, CB, M2L>(t, T, sets, geo, qcol, nchunk, chunk0, eps, lane, w); break;
    case 3: bve_mrhs_tiles<3, CB, M2L>(t, T, sets, geo, qcol, nchunk, chunk0, eps, lane, w); break;
    case 2: bve_mrhs_tiles<2, CB, M2L>(t, T, sets, geo, qcol, nchunk, chunk0, eps, lane, w); break;
    default: bve_mrhs_tiles<1, CB, M2L>(t, T, sets, geo, qcol, nchunk, chunk0, eps, lane, w); break;
  }
  // u = x cross w: the three components of one (target, member) sit in one quad
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    if (tt >= ntt) break;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double w0 = quad_bcast<0>(w[tt][cb][r]), w1 = quad_bcast<1>(w[tt][cb][r]),
                     w2 = quad_bcast<2>(w[tt][cb][r]);
        const int j = tt * 16 + 4 * grp + r;
        const int mem = 4 * (chunk0 + cb) + (col >> 2);
        if (comp < 3 && j < T.count && mem < nmem) {
          const int64_t u = (int64_t)T.first + j;
          const double x = t.px[u], y = t.py[u], z = t.pz[u];
          const double val = comp == 0 ? y * w2 - z * w1 : comp == 1 ? z * w0 - x * w2 : x * w1 - y * w0;
          double* o = u < t.npart ? part.p[comp] + (int64_t)mem * t.npart + u
                                  : proxy.p[comp] + (int64_t)mem * t.P * t.n + (u - t.npart);
          if (assign) *o = val;
          else *o += val;
        }
      }
  }
}

inline unsigned blocks_for(int64_t count, int bs) { return (unsigned)((count + bs - 1) / bs); }

inline CPtr3 cptr3(const double* const* a) {
  CPtr3 r{};
  if (a)
    for (int f = 0; f < 3; ++f) r.p[f] = a[f];
  return r;
}
inline Ptr3 ptr3(double* const* a) {
  Ptr3 r{};
  for (int f = 0; f < 3; ++f) r.p[f] = a[f];
  return r;
}

}  // namespace

// The multi-right-hand-side kernel in its FP32 form or with bf16 M2L products.
template <int CB>
static auto mrhs_kernel(const DevTree& t) { return t.bf16_m2l ? k_bve_mrhs<CB, true> : k_bve_mrhs<CB, false>; }

// Mapping 2 needs the tree's XCD ranges and the grid the context computed for
// its full list; otherwise the launch uses mapping 0.
static PairShape checked_shape(const DevTree& t, PairShape shape) {
  if (shape.xcd == 2 && (!t.xcd_start || shape.grid <= 0)) shape.xcd = 0;
  return shape;
}

void launch_source_records64(const DevTree& t, const double* q_part, const double* q_proxy,
                             const double* const* disp_part, const double* const* disp_proxy, bool project,
                             SrcRec64* rec, hipStream_t s, int nmem) {
  hipLaunchKernelGGL(k_src64, dim3(blocks_for(t.U, 256), nmem), dim3(256), 0, s, t, q_part, q_proxy, cptr3(disp_part),
                     cptr3(disp_proxy), project ? 1 : 0, rec);
}

void launch_source_records32(const DevTree& t, const double* q_part, const double* q_proxy,
                             const double* const* disp_part, const double* const* disp_proxy, SrcRec32* rec,
                             hipStream_t s, int nmem) {
  hipLaunchKernelGGL(k_src32, dim3(blocks_for(t.U, 256), nmem), dim3(256), 0, s, t, q_part, q_proxy, cptr3(disp_part),
                     cptr3(disp_proxy), 1, rec);
}

void launch_bve_interact64(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                           const SrcRec64* rec, double eps, double* const* out_part, double* const* out_proxy,
                           hipStream_t s, bool assign, int nmem, PairShape shape) {
  if (ntiles == 0) return;
  shape = checked_shape(t, shape);
  int S = tile_waves(ntiles);
  auto kernel = S == 16 ? k_bve64<16> : S == 8 ? k_bve64<8> : k_bve64<4>;
  if ((lanes64(t) && S < 16) || !rcp4_in_range(eps)) {
    S = lane_waves64(t, ntiles);
    if (S == 1) S = 2;  // velocity at degree 3 with 4 / 2 / 1: 8,190 tiles 96 / 92 / 100 us, 32,766 287 / 263 / 260
    kernel = S == 8 ? k_bve64_lanes<8> : S == 4 ? k_bve64_lanes<4> : k_bve64_lanes<2>;
  }
  hipLaunchKernelGGL(kernel, dim3(walk_grid(ntiles, shape), nmem), dim3(64 * S), 0, s, t, tiles, ntiles, sets, rec, eps,
                     ptr3(out_part), ptr3(out_proxy), assign ? 1 : 0, shape.xcd);
}

void launch_poisson_interact64(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                               const SrcRec64* rec, double* out_part, double* out_proxy, hipStream_t s,
                               bool assign) {
  if (ntiles == 0) return;
  int S = log_waves(ntiles);
  auto kernel = S == 16 ? k_log64<16> : k_log64<8>;
  if (lanes64(t) && S < 16) {
    S = lane_waves(ntiles);
    kernel = S == 8 ? k_log64_lanes<8> : k_log64_lanes<4>;
  }
  hipLaunchKernelGGL(kernel, dim3(strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, sets, rec, out_part, out_proxy,
                     assign ? 1 : 0);
}

void launch_laplacian_interact64(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                                 const SrcRec64* rec, double* out_part, double* out_proxy, hipStream_t s,
                                 bool assign) {
  if (ntiles == 0) return;
  const double eps = 0.1, pi = 3.14159265358979323846;
  // the records carry -q/(4 pi): undo it with the kernel's eps^{-5/2}
  const LapCoef64 kp = lap_coef64(eps, -4.0 * pi / std::pow(eps, 2.5));
  // us per launch with 4 / 8 / 16 waves: 126 tiles 181 / 116 / 98, 636 223 / 219 / 230, 10,236 1028 / 1088 / 1373
  int S = ntiles < 400 ? 16 : 4;
  auto kernel = S == 16 ? k_lap64<16> : k_lap64<4>;
  if (lanes64(t) && S < 16) {
    S = lane_waves64(t, ntiles);
    kernel = S == 8 ? k_lap64_lanes<8, 1> : S == 4 ? k_lap64_lanes<4, 1> : k_lap64_lanes<1, 8>;
  }
  const int per = S > 1 ? 1 : 8;  // tiles per workgroup
  hipLaunchKernelGGL(kernel, dim3(strip_grid((ntiles + per - 1) / per)), dim3(64 * S * per), 0, s, t, tiles, ntiles,
                     sets, rec, kp, out_part, out_proxy, assign ? 1 : 0);
}

void launch_laplacian_interact_mixed(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                                     const SrcRec32* rec, double* out_part, double* out_proxy, hipStream_t s,
                                     bool assign) {
  if (ntiles == 0) return;
  const double eps = 0.1, pi = 3.14159265358979323846;
  const double c3 = -4.0 * pi / std::pow(eps, 2.5);
  const int S = lane_waves(ntiles);
  hipLaunchKernelGGL(S == 8 ? k_lap_lanes<8> : k_lap_lanes<4>, dim3(strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, sets, rec,
                     lap_coef32(eps, 1.0), c3, out_part, out_proxy, assign ? 1 : 0);
}

void launch_bve_interact_mixed(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                               const SrcRec32* rec, double eps, double* const* out_part,
                               double* const* out_proxy, hipStream_t s, bool assign, int nmem, PairShape shape) {
  if (ntiles == 0) return;
  shape = checked_shape(t, shape);
  hipLaunchKernelGGL(k_bve_mixed, dim3(pair_grid(ntiles, shape), nmem), dim3(64 * shape.waves), 0, s, t,
                     tiles, ntiles, sets, rec, (float)eps, ptr3(out_part), ptr3(out_proxy), assign ? 1 : 0, shape.xcd);
}

void launch_source_records_mfma(const DevTree& t, const double* q_part, const double* q_proxy,
                                const double* const* disp_part, const double* const* disp_proxy, SrcRecMfma* rec,
                                hipStream_t s, int nmem) {
  hipLaunchKernelGGL(k_src_mfma, dim3(blocks_for(t.U16, 256), nmem), dim3(256), 0, s, t, q_part, q_proxy,
                     cptr3(disp_part), cptr3(disp_proxy), rec);
}

void launch_bve_interact_mfma(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                              const SrcRecMfma* rec, double eps, double* const* out_part, double* const* out_proxy,
                              hipStream_t s, bool assign, int nmem, PairShape shape) {
  if (ntiles == 0) return;
  shape = checked_shape(t, shape);
  hipLaunchKernelGGL(k_bve_mfma, dim3(pair_grid(ntiles, shape), nmem), dim3(64 * shape.waves), 0, s, t,
                     tiles, ntiles, sets, (const float*)rec, (float)eps, ptr3(out_part), ptr3(out_proxy),
                     assign ? 1 : 0, shape.xcd);
}

void launch_source_columns_mrhs(const DevTree& t, const double* q_part, const double* q_proxy,
                                const SrcRecMfma* geo, int nmem, int cb, float* qcol, hipStream_t s) {
  const int nchunk = mrhs_chunks(nmem, cb);
  hipLaunchKernelGGL(k_src_mrhs, dim3(blocks_for(t.U16, 256), 4 * nchunk), dim3(256), 0, s, t, q_part, q_proxy,
                     (const float*)geo, nmem, nchunk, qcol);
}

void launch_bve_interact_mrhs(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                              const SrcRecMfma* geo, const float* qcol, int nmem, int cb, double eps,
                              double* const* out_part, double* const* out_proxy, hipStream_t s, bool assign,
                              PairShape shape) {
  if (ntiles == 0) return;
  const int nchunk = mrhs_chunks(nmem, cb);
  shape = checked_shape(t, shape);
  const dim3 grid(pair_grid(ntiles, shape), nchunk / cb), block(64 * shape.waves);
  if (cb == 2)
    hipLaunchKernelGGL(mrhs_kernel<2>(t), grid, block, 0, s, t, tiles, ntiles, sets, (const float*)geo, qcol, nchunk,
                       nmem, (float)eps, ptr3(out_part), ptr3(out_proxy), assign ? 1 : 0, shape.xcd);
  else
    hipLaunchKernelGGL(mrhs_kernel<1>(t), grid, block, 0, s, t, tiles, ntiles, sets, (const float*)geo, qcol, nchunk,
                       nmem, (float)eps, ptr3(out_part), ptr3(out_proxy), assign ? 1 : 0, shape.xcd);
}

void launch_poisson_interact_mixed(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                                   const SrcRec32* rec, double* out_part, double* out_proxy, hipStream_t s,
                                   bool assign) {
  if (ntiles == 0) return;
  const int S = lane_waves(ntiles);
  hipLaunchKernelGGL(S == 8 ? k_log_lanes<8> : k_log_lanes<4>, dim3(strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, sets, rec, out_part,
                     out_proxy, assign ? 1 : 0);
}

}  // namespace sbslpm
