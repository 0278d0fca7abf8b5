// adjoint.hip -- exact transpose of the FP64 Biot-Savart FMM evaluation
// (velocity: upward pass, pair sums, downward pass; bve_vel_impl.hpp:34-70,
// fmm_funcs.cpp:341-392) with respect to the source charges and the source
// displacements.
//
// The forward pass computes, for every target row t of the interaction list
// (leaf particles, proxies of non-leaf target panels),
//   phi_t = x_t cross sum_s g(x_t, y_s) q'_s y_s,  g(x, y) = 1 / (1 - x.y + eps),
// with y_s = P(node_s + d_s) and q'_s = -q_s / (4 pi), and the particle
// velocity u = phi_part + L2P(L2L(phi_proxy)).  For a velocity cotangent ubar:
//   * the target-side cotangent is psi = ubar at particles and its
//     anterpolation (P2M, M2M: the transposes of L2P, L2L) at proxy rows;
//   * since psi_t . (x_t cross y) = y . c_t with c_t = psi_t cross x_t, one
//     pair contributes  g q' (y . c_t)  to the loss, whence
//       qbar'_s = sum_t g (y_s . c_t),
//       ybar_s  = q'_s sum_t g (c_t + g (y_s . c_t) x_t)      (dg/dy = g^2 x);
//   * the source-side cotangents go back through the projection
//     (dbar = (I - y y^T) ybar / |node + d|) and, for proxy sources, through
//     the anterpolation of the charges (downward pass) and the interpolation
//     of their displacements (scattered back to the leaf particles).
// The pair sums run over the interaction list seen from its sources: a
// workgroup per tile of at most 64 source points, every source row written once
// (assigned, no atomics), the targets' records read wave-uniformly (FP64) or from
// LDS in lane copies (FP32).
#include "lanes.hpp"

namespace sbslpm {
namespace {

struct CPtr3 {
  const double* p[3];
};
struct Ptr3 {
  double* p[3];
};

// Target record: undisplaced target node and c = psi cross x (48 bytes, read
// with wave-uniform scalar loads).
struct TgtRec {
  double x, y, z, c0, c1, c2;
};

__global__ void k_tgt_rec(DevTree t, CPtr3 psi_part, CPtr3 psi_prox, TgtRec* __restrict__ rec) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.U) return;
  double a, b, d;
  if (u < t.npart) {
    a = psi_part.p[0][u]; b = psi_part.p[1][u]; d = psi_part.p[2][u];
  } else {
    const int64_t v = u - t.npart;
    if (v / t.n >= t.offset) return;  // leaf proxy rows are never targets
    a = psi_prox.p[0][v]; b = psi_prox.p[1][v]; d = psi_prox.p[2][v];
  }
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  rec[u] = TgtRec{x, y, z, b * z - d * y, d * x - a * z, a * y - b * x};
}

// Source-side finish of one row: the charge cotangent and, with POS, the
// position cotangent through the projection.
template <bool POS>
__device__ inline void store_row(const DevTree& t, int64_t u, const SrcRec64& S, const double* a, CPtr3 dpart,
                                 CPtr3 dprox, double* __restrict__ qbar_part, double* __restrict__ qbar_prox,
                                 Ptr3 dbar_part, Ptr3 dbar_prox) {
  const bool part = u < t.npart;
  const int64_t v = part ? u : u - t.npart;
  (part ? qbar_part : qbar_prox)[v] = kNegInv4Pi * a[0];
  if constexpr (POS) {
    const double w0 = t.px[u] + (part ? dpart.p[0] : dprox.p[0])[v];
    const double w1 = t.py[u] + (part ? dpart.p[1] : dprox.p[1])[v];
    const double w2 = t.pz[u] + (part ? dpart.p[2] : dprox.p[2])[v];
    const double ir = 1.0 / sqrt(w0 * w0 + w1 * w1 + w2 * w2);
    const double yb0 = S.q * a[1], yb1 = S.q * a[2], yb2 = S.q * a[3];
    const double yy = S.x * yb0 + S.y * yb1 + S.z * yb2;
    (part ? dbar_part.p[0] : dbar_prox.p[0])[v] = (yb0 - S.x * yy) * ir;
    (part ? dbar_part.p[1] : dbar_prox.p[1])[v] = (yb1 - S.y * yy) * ir;
    (part ? dbar_part.p[2] : dbar_prox.p[2])[v] = (yb2 - S.z * yy) * ir;
  }
}

// Transposed pair sums.  POS: also the position cotangent (displaced stages).
// S waves share a tile (pairwalk.hpp), targets in batches of four with one
// shared reciprocal.
// Bound: FP64 vector issue, 12 slots per pair (19 with POS).  The step adjoint (three
// evaluations with POS and one without) before (one wave per tile, lane groups where
// they fill more) and now: 6 x 28^2 546 -> 287 us, 6 x 64^2 1473 -> 586, 6 x 128^2
// 2164 -> 1440, 6 x 224^2 3496 -> 2815.
template <bool POS, int S>
__global__ __launch_bounds__(64 * S) void k_bve_adj64(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                      const SourceSet* __restrict__ targets,
                                                      const TgtRec* __restrict__ trec,
                                                      const SrcRec64* __restrict__ srec, double eps, CPtr3 dpart,
                                                      CPtr3 dprox, double* __restrict__ qbar_part,
                                                      double* __restrict__ qbar_prox, Ptr3 dbar_part, Ptr3 dbar_prox) {
  constexpr int K = POS ? 4 : 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const int64_t u = (int64_t)T.first + (lane < T.count ? lane : T.count - 1);
  const SrcRec64 Y = srec[u];
  double acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0;
  auto add = [&](const TgtRec& R, double g) {
    const double dc = Y.x * R.c0 + Y.y * R.c1 + Y.z * R.c2;
    acc[0] = fma(g, dc, acc[0]);
    if constexpr (POS) {
      const double h = g * dc;
      acc[K - 3] = fma(g, fma(h, R.x, R.c0), acc[K - 3]);
      acc[K - 2] = fma(g, fma(h, R.y, R.c1), acc[K - 2]);
      acc[K - 1] = fma(g, fma(h, R.z, R.c2), acc[K - 1]);
    }
  };
  walk_sets<S>(T, targets, wave, [&](const SourceSet& set, int a, int b) {
    const TgtRec* __restrict__ r = trec + set.first;
    int k = a;
    for (; k + 4 <= b; k += 4) {
      double d[4], g[4];
      // the forward kernel's denominator, x = target, y = source
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = one_minus_dot(Y.x, Y.y, Y.z, r[k + i].x, r[k + i].y, r[k + i].z) + eps;
      rcp4(d, g);
#pragma unroll
      for (int i = 0; i < 4; ++i) add(r[k + i], g[i]);
    }
    for (; k < b; ++k) add(r[k], rcp64_pair(one_minus_dot(Y.x, Y.y, Y.z, r[k].x, r[k].y, r[k].z) + eps));
  });
  tile_sum<S>(acc, wave, lane);
  if (wave == 0 && lane < T.count)
    store_row<POS>(t, u, Y, acc, dpart, dprox, qbar_part, qbar_prox, dbar_part, dbar_prox);
}

// The same in lane copies (lanes.hpp), two source rows per lane: for tiles of at
// most 42 rows (lanes64), where 36 of 64 lanes held a row.  Step adjoint at
// 6 x 192^2 (degree 8) 3.08 -> 2.71 ms, 3.21 with a row per lane.
template <bool POS, int S>
__global__ __launch_bounds__(64 * S) void k_bve_adj64_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                            const SourceSet* __restrict__ targets,
                                                            const TgtRec* __restrict__ trec,
                                                            const SrcRec64* __restrict__ srec, double eps, CPtr3 dpart,
                                                            CPtr3 dprox, double* __restrict__ qbar_part,
                                                            double* __restrict__ qbar_prox, Ptr3 dbar_part,
                                                            Ptr3 dbar_prox) {
  constexpr int NT = 2, K = POS ? 4 : 1;
  __shared__ __align__(16) double stage[S][kLaneSlots * 6];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  double x[NT], y[NT], z[NT], w[NT][K];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const SrcRec64 Y = srec[(int64_t)T.first + min(q * l.T + l.i, T.count - 1)];
    x[q] = Y.x; y[q] = Y.y; z[q] = Y.z;
  }
  shared_sums(w, [&](auto shared) {
#pragma unroll
    for (int q = 0; q < NT; ++q)
#pragma unroll
      for (int k = 0; k < K; ++k) w[q][k] = 0;
    lane_walk2<S, 3>(T, targets, reinterpret_cast<const v4f*>(trec), l, reinterpret_cast<v4f*>(stage[wave]), wave, lane,
                     [&](const v4f* r0, const v4f* r1) {
      const TgtRec R[2] = {*reinterpret_cast<const TgtRec*>(r0), *reinterpret_cast<const TgtRec*>(r1)};
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
        const TgtRec& P = R[i >> 1];
        const double dc = x[q] * P.c0 + y[q] * P.c1 + z[q] * P.c2;
        w[q][0] = fma(g[i], dc, w[q][0]);
        if constexpr (POS) {
          const double h = g[i] * dc;
          w[q][K - 3] = fma(g[i], fma(h, P.x, P.c0), w[q][K - 3]);
          w[q][K - 2] = fma(g[i], fma(h, P.y, P.c1), w[q][K - 2]);
          w[q][K - 1] = fma(g[i], fma(h, P.z, P.c2), w[q][K - 1]);
        }
      }
    });
  });
  double out[K];
  lane_sum<NT, K, S>(l, w, stage, wave, lane, out);
  if (wave > 0 || lane >= T.count) return;
  const int64_t u = (int64_t)T.first + lane;
  store_row<POS>(t, u, srec[u], out, dpart, dprox, qbar_part, qbar_prox, dbar_part, dbar_prox);
}

// FP32 target record: node relative to its panel centre and c = psi cross x,
// padded to two 16-byte loads.
struct TgtRec32 {
  v4f a, c;
};

__global__ void k_tgt_rec32(DevTree t, CPtr3 psi_part, CPtr3 psi_prox, TgtRec32* __restrict__ rec) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.U) return;
  double a, b, d;
  int panel;
  if (u < t.npart) {
    a = psi_part.p[0][u]; b = psi_part.p[1][u]; d = psi_part.p[2][u];
    panel = t.offset + (int)(u / t.m2);
  } else {
    const int64_t v = u - t.npart;
    panel = (int)(v / t.n);
    if (panel >= t.offset) return;
    a = psi_prox.p[0][v]; b = psi_prox.p[1][v]; d = psi_prox.p[2][v];
  }
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  const DevPanel& P = t.panels[panel];
  rec[u] = TgtRec32{v4f{(float)(x - P.cx), (float)(y - P.cy), (float)(z - P.cz), 0.f},
                    v4f{(float)(b * z - d * y), (float)(d * x - a * z), (float)(a * y - b * x), 0.f}};
}

// Transposed pair sums in FP32 (mixed-precision contexts): 1 - x.y as
// |x - y|^2 / 2 in panel-centred coordinates, FP32 partial sums per target set
// flushed into FP64 accumulators, the source-side finish in FP64.  With
// x_t = c_t + a_t the position term sum g (c + h x_t), h = g (y . c), is
// sum g (c + h a_t) + c_t sum g h, the second sum times the panel centre once per
// set.  Lane copies (lanes.hpp) of two source rows per lane.
// Bound: FP32 vector issue, 11 instructions and a reciprocal per pair (19 with POS).
// Step adjoint before (lane groups of one row per lane, bound by their LDS reads)
// and now: 6 x 28^2 590 -> 277 us, 6 x 64^2 1341 -> 474, 6 x 96^2 994 -> 720, 6 x 192^2
// 2251 -> 1963, degree 10 at 6 x 256^2 4804 -> 4001.
template <bool POS, int S>
__global__ __launch_bounds__(64 * S) void k_bve_adj32(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                      const SourceSet* __restrict__ targets,
                                                      const TgtRec32* __restrict__ trec,
                                                      const SrcRec64* __restrict__ srec, float eps, CPtr3 dpart,
                                                      CPtr3 dprox, double* __restrict__ qbar_part,
                                                      double* __restrict__ qbar_prox, Ptr3 dbar_part, Ptr3 dbar_prox) {
  constexpr int NT = 2, K = POS ? 4 : 1;
  __shared__ __align__(16) double stage[S][kLaneSlots * 4];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = dealt_tile(ntiles);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  const DevPanel& PS = t.panels[T.panel];
  float bx[NT], by[NT], bz[NT], yx[NT], yy[NT], yz[NT];
  double w[NT][K];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const SrcRec64 Y = srec[(int64_t)T.first + min(q * l.T + l.i, T.count - 1)];
    bx[q] = (float)(Y.x - PS.cx); by[q] = (float)(Y.y - PS.cy); bz[q] = (float)(Y.z - PS.cz);
    yx[q] = (float)Y.x; yy[q] = (float)Y.y; yz[q] = (float)Y.z;
#pragma unroll
    for (int k = 0; k < K; ++k) w[q][k] = 0;
  }
  v4f* mine = reinterpret_cast<v4f*>(stage[wave]);
  lane_pads<2>(mine, 4.f, lane);  // padding: a target four radii away without a cotangent
  walk_sets<S>(T, targets, wave, [&](const SourceSet& set, int a, int b) {
    float qx[NT], qy[NT], qz[NT], sq[NT], s0[NT], s1[NT], s2[NT], sh[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) {  // source relative to the target panel's centre
      qx[q] = bx[q] - set.ox; qy[q] = by[q] - set.oy; qz[q] = bz[q] - set.oz;
      sq[q] = s0[q] = s1[q] = s2[q] = sh[q] = 0.f;
    }
    for (int c = a; c < b; c += kLaneChunk) {
      const int cn = min(kLaneChunk, b - c), trips = (cn + l.G - 1) / l.G;
      lane_stage<2>(mine, reinterpret_cast<const v4f*>(trec + set.first + c), cn, 4.f, lane);
      const TgtRec32* r = reinterpret_cast<const TgtRec32*>(mine) + l.g;
#pragma unroll 2
      for (int k = 0; k < trips; ++k, r += l.G) {
        const v4f A = r->a, C = r->c;
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          const float d0 = A.x - qx[q], d1 = A.y - qy[q], d2 = A.z - qz[q];  // x_t - y_s
          const float g = __builtin_amdgcn_rcpf(fmaf(0.5f, fmaf(d0, d0, fmaf(d1, d1, d2 * d2)), eps));
          const float dc = fmaf(yx[q], C.x, fmaf(yy[q], C.y, yz[q] * C.z));
          if constexpr (POS) {
            const float h = g * dc;
            sq[q] += h;
            sh[q] = fmaf(g, h, sh[q]);
            s0[q] = fmaf(g, fmaf(h, A.x, C.x), s0[q]);
            s1[q] = fmaf(g, fmaf(h, A.y, C.y), s1[q]);
            s2[q] = fmaf(g, fmaf(h, A.z, C.z), s2[q]);
          } else {
            sq[q] = fmaf(g, dc, sq[q]);
          }
        }
      }
    }
    const DevPanel& PT = t.panels[set.panel];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      w[q][0] += sq[q];
      if constexpr (POS) {
        const double hc = sh[q];
        w[q][K - 3] += fma(hc, PT.cx, (double)s0[q]);
        w[q][K - 2] += fma(hc, PT.cy, (double)s1[q]);
        w[q][K - 1] += fma(hc, PT.cz, (double)s2[q]);
      }
    }
  });
  double out[K];
  lane_sum<NT, K, S>(l, w, stage, wave, lane, out);
  if (wave > 0 || lane >= T.count) return;
  const int64_t u = (int64_t)T.first + lane;
  store_row<POS>(t, u, srec[u], out, dpart, dprox, qbar_part, qbar_prox, dbar_part, dbar_prox);
}

// Waves per tile.  Step adjoint (FP64) with 4 / 8 / 16: 126 tiles 359 / 304 / 285 us,
// 636 626 / 591 / 627, 2,556 1469 / 1428 / 1697, 8,190 2835 / 2858 / 3531; FP32
// 126 tiles 307 / 279 / 277, 636 482 / 475 / 526, 2,556 (36 rows) 714 / 745 / 907,
// 10,236 1919 / 2087 / 2807.
inline int adj_waves(int ntiles, int many) { return ntiles < 300 ? 16 : ntiles < many ? 8 : 4; }

}  // namespace

size_t adj_target_record_bytes() { return sizeof(TgtRec) > sizeof(TgtRec32) ? sizeof(TgtRec) : sizeof(TgtRec32); }

void launch_adj_target_records32(const DevTree& t, const double* const* psi_part, const double* const* psi_prox,
                                 void* rec, hipStream_t s) {
  CPtr3 pp{{psi_part[0], psi_part[1], psi_part[2]}}, px{{psi_prox[0], psi_prox[1], psi_prox[2]}};
  hipLaunchKernelGGL(k_tgt_rec32, dim3((unsigned)((t.U + 255) / 256)), dim3(256), 0, s, t, pp, px,
                     static_cast<TgtRec32*>(rec));
}

void launch_bve_adjoint32(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* targets,
                          const void* trec, const SrcRec64* srec, double eps, const double* const* dpart,
                          const double* const* dprox, double* qbar_part, double* qbar_prox, double* const* dbar_part,
                          double* const* dbar_prox, hipStream_t s) {
  if (ntiles == 0) return;
  const TgtRec32* r = static_cast<const TgtRec32*>(trec);
  CPtr3 dp{}, dx{};
  Ptr3 bp{}, bx{};
  if (dpart) {
    dp = CPtr3{{dpart[0], dpart[1], dpart[2]}};
    dx = CPtr3{{dprox[0], dprox[1], dprox[2]}};
    bp = Ptr3{{dbar_part[0], dbar_part[1], dbar_part[2]}};
    bx = Ptr3{{dbar_prox[0], dbar_prox[1], dbar_prox[2]}};
  }
  const int S = adj_waves(ntiles, 1500);
  auto kernel = dpart ? (S == 16 ? k_bve_adj32<true, 16> : S == 8 ? k_bve_adj32<true, 8> : k_bve_adj32<true, 4>)
                      : (S == 16 ? k_bve_adj32<false, 16> : S == 8 ? k_bve_adj32<false, 8> : k_bve_adj32<false, 4>);
  hipLaunchKernelGGL(kernel, dim3(strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, targets, r, srec, (float)eps, dp,
                     dx, qbar_part, qbar_prox, bp, bx);
}

void launch_adj_target_records(const DevTree& t, const double* const* psi_part, const double* const* psi_prox,
                               void* rec, hipStream_t s) {
  CPtr3 pp{{psi_part[0], psi_part[1], psi_part[2]}}, px{{psi_prox[0], psi_prox[1], psi_prox[2]}};
  hipLaunchKernelGGL(k_tgt_rec, dim3((unsigned)((t.U + 255) / 256)), dim3(256), 0, s, t, pp, px,
                     static_cast<TgtRec*>(rec));
}

void launch_bve_adjoint64(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* targets,
                          const void* trec, const SrcRec64* srec, double eps, const double* const* dpart,
                          const double* const* dprox, double* qbar_part, double* qbar_prox, double* const* dbar_part,
                          double* const* dbar_prox, hipStream_t s) {
  if (ntiles == 0) return;
  const TgtRec* r = static_cast<const TgtRec*>(trec);
  CPtr3 dp{}, dx{};
  Ptr3 bp{}, bx{};
  if (dpart) {
    dp = CPtr3{{dpart[0], dpart[1], dpart[2]}};
    dx = CPtr3{{dprox[0], dprox[1], dprox[2]}};
    bp = Ptr3{{dbar_part[0], dbar_part[1], dbar_part[2]}};
    bx = Ptr3{{dbar_prox[0], dbar_prox[1], dbar_prox[2]}};
  }
  int S = adj_waves(ntiles, 6000);
  auto kernel = dpart ? (S == 16 ? k_bve_adj64<true, 16> : S == 8 ? k_bve_adj64<true, 8> : k_bve_adj64<true, 4>)
                      : (S == 16 ? k_bve_adj64<false, 16> : S == 8 ? k_bve_adj64<false, 8> : k_bve_adj64<false, 4>);
  if ((lanes64(t) && S < 16) || !rcp4_in_range(eps)) {
    S = lane_waves64(t, ntiles);
    kernel = dpart ? (S == 8 ? k_bve_adj64_lanes<true, 8> : S == 4 ? k_bve_adj64_lanes<true, 4> : k_bve_adj64_lanes<true, 1>)
                   : (S == 8 ? k_bve_adj64_lanes<false, 8> : S == 4 ? k_bve_adj64_lanes<false, 4> : k_bve_adj64_lanes<false, 1>);
  }
  hipLaunchKernelGGL(kernel, dim3(strip_grid(ntiles)), dim3(64 * S), 0, s, t, tiles, ntiles, targets, r, srec, eps, dp,
                     dx, qbar_part, qbar_prox, bp, bx);
}

}  // namespace sbslpm
