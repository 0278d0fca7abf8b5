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
// The kernel accumulates W = sum g qz y, D = sum gd y', S = sum gd (x.y')
// (y' = y or y0) and forms u = x cross W + D - x S once per target, the same
// sums regrouped.
#include "device.hpp"
#include "pairwalk.hpp"

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
// x cross y = x cross d and y - x (x.y) = d + x h, so
//   u = x cross sum(g qz d) + sum(g qd d) + x sum(g qd h),   g = 1/(h + eps).
// FP32 partial sums per source set are added into FP64; the cross product and
// the output are FP64.
template <bool GR>
__global__ __launch_bounds__(256) void k_swe_mixed(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                   RowGroups gs, const SourceSet* __restrict__ sets,
                                                   const SrcRecSwe32* __restrict__ rec, float eps, Ptr3 part,
                                                   Ptr3 proxy, int assign) {
  __shared__ SrcRecSwe32 stage[GR ? kWavesPerBlock : 1][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tile, row0, cg, ci;
  if (!group_tile<GR>(gs, ntiles, wave, 1, tile, row0, cg, ci)) return;
  const TargetTile T = tiles[tile];
  const DevPanel& PT = t.panels[T.panel];
  const int row = row0 + ci;
  const int64_t u = (int64_t)T.first + (row < T.count ? row : T.count - 1);
  const int ng = GR ? gs.G : 1;
  const bool copy_ok = !GR || cg < ng;
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  const float ax = (float)(x - PT.cx), ay = (float)(y - PT.cy), az = (float)(z - PT.cz);
  double w0 = 0, w1 = 0, w2 = 0, d0 = 0, d1 = 0, d2 = 0, sd = 0;
  for (int e = T.src_begin; e < T.src_end; ++e) {
    const SourceSet S = sets[e];
    const float px = ax + S.ox, py = ay + S.oy, pz = az + S.oz;
    const SrcRecSwe32* __restrict__ r = rec + S.first;
    float v0 = 0.f, v1 = 0.f, v2 = 0.f, e0 = 0.f, e1 = 0.f, e2 = 0.f, eh = 0.f;
    for (int c0 = 0; c0 < S.count; c0 += GR ? 64 : S.count) {
      const int cn = GR ? min(64, S.count - c0) : S.count;
      if (GR) stage_records(stage[wave], r + c0, cn);
      const int trips = GR ? (cn + ng - 1) / ng : cn;
#pragma unroll 4
      for (int kk = 0; kk < trips; ++kk) {
        const int k = GR ? kk * ng + cg : kk;
        if (GR && !(copy_ok && k < cn)) continue;
        const SrcRecSwe32 s = GR ? stage[wave][k] : r[k];
        const float c0f = s.x - px, c1f = s.y - py, c2f = s.z - pz;
        const float h = 0.5f * fmaf(c0f, c0f, fmaf(c1f, c1f, c2f * c2f));
        const float g = __builtin_amdgcn_rcpf(h + eps);
        const float gz = g * s.qz, gd = g * s.qd;
        v0 = fmaf(gz, c0f, v0);
        v1 = fmaf(gz, c1f, v1);
        v2 = fmaf(gz, c2f, v2);
        e0 = fmaf(gd, c0f, e0);
        e1 = fmaf(gd, c1f, e1);
        e2 = fmaf(gd, c2f, e2);
        eh = fmaf(gd, h, eh);
      }
    }
    w0 += v0; w1 += v1; w2 += v2;
    d0 += e0; d1 += e1; d2 += e2;
    sd += eh;
  }
  if (GR) {
    w0 = group_sum(w0, gs, ci); w1 = group_sum(w1, gs, ci); w2 = group_sum(w2, gs, ci);
    d0 = group_sum(d0, gs, ci); d1 = group_sum(d1, gs, ci); d2 = group_sum(d2, gs, ci);
    sd = group_sum(sd, gs, ci);
  }
  if (cg != 0 || row >= T.count) return;
  const double a = (y * w2 - z * w1) + (d0 + x * sd);
  const double b = (z * w0 - x * w2) + (d1 + y * sd);
  const double c = (x * w1 - y * w0) + (d2 + z * sd);
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
  const unsigned blocks = (unsigned)((ntiles + kWavesPerBlock - 1) / kWavesPerBlock);
  const RowGroups gs = row_groups(t);
  if (gs.G > 1)
    hipLaunchKernelGGL(k_swe_mixed<true>, dim3((((int64_t)ntiles * gs.H + kWavesPerBlock - 1) / kWavesPerBlock)),
                       dim3(64 * kWavesPerBlock), 0, s, t, tiles, ntiles, gs, sets, rec, (float)eps, op, ox,
                       assign ? 1 : 0);
  else
    hipLaunchKernelGGL(k_swe_mixed<false>, dim3(blocks), dim3(64 * kWavesPerBlock), 0, s, t, tiles, ntiles, gs, sets,
                       rec, (float)eps, op, ox, assign ? 1 : 0);
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
  const int S = ntiles < 400 ? 16 : ntiles < 3000 ? 8 : 4;
  auto kernel = variant != 2 ? (S == 16 ? k_swe64<1, 16> : S == 8 ? k_swe64<1, 8> : k_swe64<1, 4>)
                             : (S == 16 ? k_swe64<2, 16> : S == 8 ? k_swe64<2, 8> : k_swe64<2, 4>);
  hipLaunchKernelGGL(kernel, dim3(heaviest_first ? ntiles : strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, sets, rec, eps, op, ox,
                     assign ? 1 : 0, heaviest_first ? 1 : 0);
}

}  // namespace sbslpm
