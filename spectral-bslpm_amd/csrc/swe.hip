// swe.hip -- shallow-water velocity pair sums (fmm_interactions/swe_vel.cpp:9-67,
// swe_vel_impl.hpp:12-147), FP64, on the same target-major tiles as the
// Biot-Savart kernels.
//
// Per pair, with x the target, y = P(node + disp) the displaced source and
// y0 the undisplaced node:
//   variant 1 (swe_vel_panel_interaction):
//     u += g qz (x cross y) + g qd (y - x (x.y)),      g = -1/(4 pi (1 - x.y + eps))
//   variant 2 (swe_vel_panel_interaction_2):
//     u += g qz (x cross y) + g0 qd (y0 - x (x.y0)),   g0 = +1/(4 pi (1 - x.y0 + eps))
//   variant 3 (swe_vel_panel_interaction_ll, swe_vel_impl.hpp:265-276, no displacement):
//     u += g qz (x cross y) - g qd (y - x (x.y)),      g = -1/(4 pi (1 - x.y + eps))
// The kernels accumulate W = sum g qz y and D = sum gd y' (y' = y or y0) and form
// u = x cross W + D - x (x.D) once per target, the same sums regrouped.
#include "device.hpp"
#include "lanes.hpp"

namespace sbslpm {
namespace {

struct CPtr3 {
  const double* p[3];
};
struct Ptr3 {
  double* p[3];
};

// Source records: displaced re-projected position, undisplaced node, and the
// charges pre-multiplied by the variant's constants.
__global__ void k_src_swe(DevTree t, const double* __restrict__ qz_part, const double* __restrict__ qz_proxy,
                          const double* __restrict__ qd_part, const double* __restrict__ qd_proxy, CPtr3 dpart,
                          CPtr3 dprox, double qd_scale, SrcRecSwe* __restrict__ rec) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.U) return;
  const double x0 = t.px[u], y0 = t.py[u], z0 = t.pz[u];
  double x = x0, y = y0, z = z0, qz, qd;
  if (u < t.npart) {
    if (dpart.p[0]) { x += dpart.p[0][u]; y += dpart.p[1][u]; z += dpart.p[2][u]; }
    qz = qz_part[u];
    qd = qd_part[u];
  } else {
    const int64_t v = u - t.npart;
    if (v / t.n >= t.offset) return;  // leaf proxy rows are never sources
    if (dprox.p[0]) { x += dprox.p[0][v]; y += dprox.p[1][v]; z += dprox.p[2][v]; }
    qz = qz_proxy[v];
    qd = qd_proxy[v];
  }
  project_to_sphere(x, y, z);
  rec[u] = SrcRecSwe{x, y, z, kNegInv4Pi * qz, x0, y0, z0, qd_scale * qd};
}

// S waves share a tile (pairwalk.hpp), sources in batches of four with one
// shared reciprocal (two in variant 2).  S_t = sum gd (x.y') of the header is
// x.D, formed once per target.  heaviest_first: workgroup b takes tile b, for a
// list sorted by decreasing work (the irregular trees).
// Bound: FP64 vector issue, 16 slots per pair (variant 1; 21 with a reciprocal
// and the x.y' sum on every pair).  Microseconds per launch with one wave per
// tile (in lane groups at m = 6) and now: 6 x 28^2 121 -> 25, 6 x 64^2 443 -> 85,
// 6 x 192^2 (degree 8) 860 -> 694, 6 x 512^2 4365 -> 3525; the 1 degree lat-lon
// tree's whole evaluation 649 -> 555.
template <int VARIANT, int S>
__global__ __launch_bounds__(64 * S) void k_swe64(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                  const SourceSet* __restrict__ sets,
                                                  const SrcRecSwe* __restrict__ rec, double eps, Ptr3 part, Ptr3 proxy,
                                                  int assign, int heaviest_first) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = heaviest_first ? (int)blockIdx.x : strip_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const int64_t u = (int64_t)T.first + (lane < T.count ? lane : T.count - 1);
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  double acc[6] = {0, 0, 0, 0, 0, 0};  // W, D
  auto add = [&](const SrcRecSwe& s, double g, double g0) {
    const double gz = g * s.qz, gd = g0 * s.qd;
    acc[0] = fma(gz, s.x, acc[0]);
    acc[1] = fma(gz, s.y, acc[1]);
    acc[2] = fma(gz, s.z, acc[2]);
    acc[3] = fma(gd, VARIANT == 1 ? s.x : s.x0, acc[3]);
    acc[4] = fma(gd, VARIANT == 1 ? s.y : s.y0, acc[4]);
    acc[5] = fma(gd, VARIANT == 1 ? s.z : s.z0, acc[5]);
  };
  walk_sets<S>(T, sets, wave, [&](const SourceSet& set, int a, int b) {
    const SrcRecSwe* __restrict__ r = rec + set.first;
    int k = a;
    for (; k + 4 <= b; k += 4) {
      double d[4], g[4], g0[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = one_minus_dot(x, y, z, r[k + i].x, r[k + i].y, r[k + i].z) + eps;
      rcp4(d, g);
      if (VARIANT == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = one_minus_dot(x, y, z, r[k + i].x0, r[k + i].y0, r[k + i].z0) + eps;
        rcp4(d, g0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) add(r[k + i], g[i], VARIANT == 1 ? g[i] : g0[i]);
    }
    for (; k < b; ++k) {
      const SrcRecSwe s = r[k];
      const double g = rcp64_pair(one_minus_dot(x, y, z, s.x, s.y, s.z) + eps);
      add(s, g, VARIANT == 1 ? g : rcp64_pair(one_minus_dot(x, y, z, s.x0, s.y0, s.z0) + eps));
    }
  });
  tile_sum<S>(acc, wave, lane);
  if (wave > 0 || lane >= T.count) return;
  const double sd = x * acc[3] + y * acc[4] + z * acc[5];
  const double a = (y * acc[2] - z * acc[1]) + (acc[3] - x * sd);
  const double b = (z * acc[0] - x * acc[2]) + (acc[4] - y * sd);
  const double c = (x * acc[1] - y * acc[0]) + (acc[5] - z * sd);
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

// The same in lane copies (lanes.hpp) of two targets, for tiles of at most 42 rows
// (lanes64) and for irregular trees.  Microseconds per pair call in lane groups of one
// target and here: 6 x 96^2 (degree 8) 272 -> 150, 6 x 192^2 838 -> 530 (a row per lane:
// 686 a launch), degree 5 478 -> 325 (423), 6 x 160^2 (degree 4, 25 rows) 267 -> 198
// (294).  Variant 2, velocity calls in lane groups, with a row per lane and
// here: 6 x 96^2 (degree 8) 366, 258, 223; 6 x 192^2 1120, 909, 772; 6 x 160^2 (degree
// 4) 366, 381, 278; 6 x 320^2 1201, 1396, 1013.
template <int VARIANT, int S>
__global__ __launch_bounds__(64 * S) void k_swe64_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                        const SourceSet* __restrict__ sets,
                                                        const SrcRecSwe* __restrict__ rec, double eps, Ptr3 part,
                                                        Ptr3 proxy, int assign, int heaviest_first) {
  constexpr int NT = 2, K = 6;
  __shared__ __align__(16) double stage[S][kLaneSlots * 8];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = heaviest_first ? (int)blockIdx.x : strip_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  double x[NT], y[NT], z[NT], w[NT][K];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    x[q] = t.px[u]; y[q] = t.py[u]; z[q] = t.pz[u];
  }
  shared_sums(w, [&](auto shared) {
#pragma unroll
    for (int q = 0; q < NT; ++q)
#pragma unroll
      for (int k = 0; k < K; ++k) w[q][k] = 0;
    lane_walk2<S, 4>(T, sets, reinterpret_cast<const v4f*>(rec), l, reinterpret_cast<v4f*>(stage[wave]), wave, lane,
                     [&](const v4f* r0, const v4f* r1) {
      const SrcRecSwe* R[2] = {reinterpret_cast<const SrcRecSwe*>(r0), reinterpret_cast<const SrcRecSwe*>(r1)};
      double d[4], g[4], a[2], b[2], c[2], qz[2], qd[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i] = R[i]->x; b[i] = R[i]->y; c[i] = R[i]->z; qz[i] = R[i]->qz; qd[i] = R[i]->qd;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = one_minus_dot(x[i & 1], y[i & 1], z[i & 1], a[i >> 1], b[i >> 1], c[i >> 1]) + eps;
      rcps<decltype(shared)::value>(d, g);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = i & 1, k = i >> 1;
        const double gz = g[i] * qz[k];
        w[q][0] = fma(gz, a[k], w[q][0]);
        w[q][1] = fma(gz, b[k], w[q][1]);
        w[q][2] = fma(gz, c[k], w[q][2]);
      }
      if constexpr (VARIANT == 2) {  // the divergence's pairs are at the undisplaced sources
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[i] = R[i]->x0; b[i] = R[i]->y0; c[i] = R[i]->z0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          d[i] = one_minus_dot(x[i & 1], y[i & 1], z[i & 1], a[i >> 1], b[i >> 1], c[i >> 1]) + eps;
        rcps<decltype(shared)::value>(d, g);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = i & 1, k = i >> 1;
        const double gd = g[i] * qd[k];
        w[q][3] = fma(gd, a[k], w[q][3]);
        w[q][4] = fma(gd, b[k], w[q][4]);
        w[q][5] = fma(gd, c[k], w[q][5]);
      }
    });
  });
  double s[K];
  lane_sum<NT, K, S>(l, w, stage, wave, lane, s);
  if (wave > 0 || lane >= T.count) return;
  const int64_t u = (int64_t)T.first + lane;
  const double X = t.px[u], Y = t.py[u], Z = t.pz[u], sd = X * s[3] + Y * s[4] + Z * s[5];
  const double o[3] = {(Y * s[2] - Z * s[1]) + (s[3] - X * sd), (Z * s[0] - X * s[2]) + (s[4] - Y * sd),
                       (X * s[1] - Y * s[0]) + (s[5] - Z * sd)};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double* p = u < t.npart ? part.p[k] + u : proxy.p[k] + (u - t.npart);
    *p = assign ? o[k] : *p + o[k];
  }
}

// Mixed-precision records: position relative to the source panel centre (FP32)
// and the two charges with the variant's constants, FP32.
__global__ void k_src_swe32(DevTree t, const double* __restrict__ qz_part, const double* __restrict__ qz_proxy,
                            const double* __restrict__ qd_part, const double* __restrict__ qd_proxy, CPtr3 dpart,
                            CPtr3 dprox, double qd_scale, SrcRecSwe32* __restrict__ rec) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.U) return;
  double x = t.px[u], y = t.py[u], z = t.pz[u], qz, qd;
  int panel;
  if (u < t.npart) {
    if (dpart.p[0]) { x += dpart.p[0][u]; y += dpart.p[1][u]; z += dpart.p[2][u]; }
    qz = qz_part[u];
    qd = qd_part[u];
    panel = t.offset + (int)(u / t.m2);
  } else {
    const int64_t v = u - t.npart;
    panel = (int)(v / t.n);
    if (panel >= t.offset) return;  // leaf proxy rows are never sources
    if (dprox.p[0]) { x += dprox.p[0][v]; y += dprox.p[1][v]; z += dprox.p[2][v]; }
    qz = qz_proxy[v];
    qd = qd_proxy[v];
  }
  project_to_sphere(x, y, z);
  const DevPanel& P = t.panels[panel];
  rec[u] = SrcRecSwe32{(float)(x - P.cx), (float)(y - P.cy), (float)(z - P.cz), (float)(kNegInv4Pi * qz),
                       (float)(qd_scale * qd), 0.f, 0.f, 0.f};
}

// Mixed-precision shallow-water pairs (variants 1 and 3): with d = y - x and
// h = |d|^2 / 2 = 1 - x.y computed in FP32 from panel-centred coordinates,
// x cross y = x cross d and y - x (x.y) = d - x (x.d), so
//   u = x cross sum(g qz d) + E - x (x.E),   E = sum(g qd d),   g = 1/(h + eps).
// FP32 partial sums per source set are added into FP64; the cross product, the
// projection and the output are FP64.  Lane copies (lanes.hpp) of two targets, or of
// one whose trips feed two sums in turn.
// Bound: FP32 vector issue, 15 instructions and a reciprocal per pair.
// Microseconds per launch before (one wave per tile with scalar records, or lane
// groups of one target) and with 2 / 4 / 8 waves per tile: 126 tiles 115, 53 / 32 /
// 25; 636 380, 106 / 67 / 65; 2,556 (36 rows) 187, 130 / 117 / 123; 10,236 543, 387 /
// 390 / 432; 40,956 2931, 2268 / 2231 / 2318.
template <int S, int NT>
__global__ __launch_bounds__(64 * S) void k_swe_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                      const SourceSet* __restrict__ sets,
                                                      const SrcRecSwe32* __restrict__ rec, float eps, Ptr3 part,
                                                      Ptr3 proxy, int assign) {
  constexpr int K = 6;
  __shared__ __align__(16) double stage[S][64 * K];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const DevPanel& PT = t.panels[T.panel];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  float ax[NT], ay[NT], az[NT], px[NT], py[NT], pz[NT], v[2][K];
  double w[NT][K];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    ax[q] = (float)(t.px[u] - PT.cx);
    ay[q] = (float)(t.py[u] - PT.cy);
    az[q] = (float)(t.pz[u] - PT.cz);
#pragma unroll
    for (int k = 0; k < K; ++k) w[q][k] = 0;
  }
  lane_walk<S, 2, 2>(
      T, sets, reinterpret_cast<const v4f*>(rec), l, reinterpret_cast<v4f*>(stage[wave]), 4.f, wave, lane,
      [&](const SourceSet& set) {
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          px[q] = ax[q] + set.ox;
          py[q] = ay[q] + set.oy;
          pz[q] = az[q] + set.oz;
        }
#pragma unroll
        for (int k = 0; k < K; ++k) v[0][k] = v[1][k] = 0.f;
      },
      [&](const v4f* r) {
        const v4f s = r[0];
        const float qd = r[1].x;
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          const float d0 = s.x - px[q], d1 = s.y - py[q], d2 = s.z - pz[q];
          const float g = __builtin_amdgcn_rcpf(fmaf(0.5f, fmaf(d0, d0, fmaf(d1, d1, d2 * d2)), eps));
          const float gz = g * s.w, gd = g * qd;
          v[q][0] = fmaf(gz, d0, v[q][0]);
          v[q][1] = fmaf(gz, d1, v[q][1]);
          v[q][2] = fmaf(gz, d2, v[q][2]);
          v[q][3] = fmaf(gd, d0, v[q][3]);
          v[q][4] = fmaf(gd, d1, v[q][4]);
          v[q][5] = fmaf(gd, d2, v[q][5]);
        }
        if constexpr (NT == 1)
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const float even = v[0][k];
            v[0][k] = v[1][k];
            v[1][k] = even;
          }
      },
      [&](const SourceSet&) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int k = 0; k < K; ++k) w[q < NT ? q : 0][k] += v[q][k];
      });
  double s[K];
  lane_sum<NT, K, S>(l, w, stage, wave, lane, s);
  if (wave > 0 || lane >= T.count) return;
  const int64_t u = (int64_t)T.first + lane;
  const double x = t.px[u], y = t.py[u], z = t.pz[u], sd = x * s[3] + y * s[4] + z * s[5];
  const double o[3] = {(y * s[2] - z * s[1]) + (s[3] - x * sd), (z * s[0] - x * s[2]) + (s[4] - y * sd),
                       (x * s[1] - y * s[0]) + (s[5] - z * sd)};
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double* p = u < t.npart ? part.p[c] + u : proxy.p[c] + (u - t.npart);
    *p = assign ? o[c] : *p + o[c];
  }
}

}  // namespace

void launch_source_records_swe32(const DevTree& t, int variant, const double* qz_part, const double* qz_proxy,
                                 const double* qd_part, const double* qd_proxy, const double* const* disp_part,
                                 const double* const* disp_proxy, SrcRecSwe32* rec, hipStream_t s) {
  CPtr3 dp{}, dx{};
  for (int f = 0; f < 3; ++f) {
    dp.p[f] = disp_part ? disp_part[f] : nullptr;
    dx.p[f] = disp_proxy ? disp_proxy[f] : nullptr;
  }
  const double qd_scale = variant == 1 ? kNegInv4Pi : -kNegInv4Pi;
  hipLaunchKernelGGL(k_src_swe32, dim3((unsigned)((t.U + 255) / 256)), dim3(256), 0, s, t, qz_part, qz_proxy,
                     qd_part, qd_proxy, dp, dx, qd_scale, rec);
}

void launch_swe_interact_mixed(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                               const SrcRecSwe32* rec, double eps, double* const* out_part,
                               double* const* out_proxy, hipStream_t s, bool assign) {
  if (ntiles == 0) return;
  Ptr3 op{}, ox{};
  for (int f = 0; f < 3; ++f) {
    op.p[f] = out_part[f];
    ox.p[f] = out_proxy[f];
  }
  int S = lane_waves(ntiles);
  auto kernel = S == 8 ? k_swe_lanes<8, 2> : k_swe_lanes<4, 2>;
  // one target per lane as in bve_lanes.hip: velocity at degree 2 with two targets and 4
  // waves, and with one and 4 / 2 / 1: 2,046 tiles 63, 56 / 60 / 72 us; 8,190 135, 115 / 113 /
  // 118; 32,766 409, 321 / 296 / 289
  if (t.rows <= 16) {
    S = ntiles < 6000 ? 4 : 2;
    kernel = S == 4 ? k_swe_lanes<4, 1> : k_swe_lanes<2, 1>;
  }
  hipLaunchKernelGGL(kernel, dim3(strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, sets, rec, (float)eps, op,
                     ox, assign ? 1 : 0);
}

void launch_source_records_swe(const DevTree& t, int variant, const double* qz_part, const double* qz_proxy,
                               const double* qd_part, const double* qd_proxy, const double* const* disp_part,
                               const double* const* disp_proxy, SrcRecSwe* rec, hipStream_t s) {
  CPtr3 dp{}, dx{};
  for (int f = 0; f < 3; ++f) {
    dp.p[f] = disp_part ? disp_part[f] : nullptr;
    dx.p[f] = disp_proxy ? disp_proxy[f] : nullptr;
  }
  // variant 1: g qd with g = -1/(4 pi ...); variants 2 and 3: +1/(4 pi ...)
  const double qd_scale = variant == 1 ? kNegInv4Pi : -kNegInv4Pi;
  hipLaunchKernelGGL(k_src_swe, dim3((unsigned)((t.U + 255) / 256)), dim3(256), 0, s, t, qz_part, qz_proxy, qd_part,
                     qd_proxy, dp, dx, qd_scale, rec);
}

void launch_swe_interact64(const DevTree& t, int variant, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                           const SrcRecSwe* rec, double eps, double* const* out_part, double* const* out_proxy,
                           hipStream_t s, bool assign, bool heaviest_first) {
  if (ntiles == 0) return;
  Ptr3 op{}, ox{};
  for (int f = 0; f < 3; ++f) {
    op.p[f] = out_part[f];
    ox.p[f] = out_proxy[f];
  }
  // us per launch with 4 / 8 / 16 waves: 126 tiles 49 / 31 / 25, 636 102 / 85 / 91, 2,556 202 / 200 / 246,
  // 10,236 694 / 710 / 903, 40,956 3525 / 3691 / 4706
  int S = ntiles < 400 ? 16 : ntiles < 3000 ? 8 : 4;
  auto kernel = variant != 2 ? (S == 16 ? k_swe64<1, 16> : S == 8 ? k_swe64<1, 8> : k_swe64<1, 4>)
                             : (S == 16 ? k_swe64<2, 16> : S == 8 ? k_swe64<2, 8> : k_swe64<2, 4>);
  // An irregular tree's list (heaviest first, tiles of one row to 64, sets of a few points)
  // takes lane copies whatever its rows.  Shallow-water velocity on the 1 degree grid, a
  // row per lane and lane copies: 64 points a leaf at degree 4 185 and 152 us, degree 8 574
  // and 417, degree 10 838 and 751; 324 a leaf at degree 8 278 and 249; 484 at degree 10 359
  // and 359.
  if (((lanes64(t) || heaviest_first) && S < 16) || !rcp4_in_range(eps)) {
    S = lane_waves64(t, ntiles);
    kernel = variant != 2 ? (S == 8 ? k_swe64_lanes<1, 8> : S == 4 ? k_swe64_lanes<1, 4> : k_swe64_lanes<1, 1>)
                          : (S == 8 ? k_swe64_lanes<2, 8> : S == 4 ? k_swe64_lanes<2, 4> : k_swe64_lanes<2, 1>);
  }
  hipLaunchKernelGGL(kernel, dim3(heaviest_first ? ntiles : strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, sets, rec, eps, op, ox,
                     assign ? 1 : 0, heaviest_first ? 1 : 0);
}

}  // namespace sbslpm
