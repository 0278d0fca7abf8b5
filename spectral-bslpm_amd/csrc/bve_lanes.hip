// bve_lanes.hip -- mixed-precision Biot-Savart pair kernel on the vector unit,
// in lane copies (lanes.hpp).
//
// With target p and source b relative to the source-panel centre,
//   D = 1 - x.y + eps = alpha + beta - p.b,  alpha = eps + |p|^2/2,
// and W = sum (q b)/D, Q = sum q/D give sum q (b - p)/D = W - p Q once per
// source set, added in FP64 (x cross y = x cross (y - x)): eight fused
// multiply-adds and one reciprocal per pair.
//
// Even and odd trips keep sums of their own, so that a set's FP32 chains and the
// terms that the flush subtracts are no longer than the four source quarters of
// the matrix-core form: the velocity's distance from FP64 is 2.3e-7 at 6 x 28^2
// and 4.0e-8 at 6 x 512^2 (3.5e-7 and 4.3e-8 there; one sum per copy 3.1e-7 and
// 4.8e-8).
//
// Bound: FP32 vector issue at the 2.0 GHz the chip holds under it (43,500
// two-target iterations of 58 cycles per SIMD at 6 x 512^2 are 1.26 ms; the
// per-set work of loading, centring and flushing adds 15%).  The matrix-core form
// of the same sums took 154 cycles per 256 pairs, 115 here, and padded targets
// and sources to 16.  Microseconds per launch, matrix cores and now: 6 x 28^2
// 62 -> 20, 6 x 64^2 86 -> 47, 6 x 96^2 128 -> 85, 6 x 192^2 367 -> 280, 6 x 224^2
// 413 -> 303, 6 x 512^2 1674 -> 1529.  Four targets per lane halve the LDS reads,
// but 108 registers leave four waves per SIMD: 9% slower.  Records of 20 bytes
// (q b formed per pair): 11% slower.
#include "lanes.hpp"

namespace sbslpm {
namespace {

struct Ptr3 {
  double* p[3];
};
struct CPtr3 {
  const double* p[3];
};

// Source record, 32 bytes: (b_x, b_y, b_z, beta), (q b_x, q b_y, q b_z, q) with
// b the position relative to the source-panel centre, beta = |b|^2 / 2 and
// q = -charge / (4 pi).
__global__ void k_src_lanes(DevTree t, const double* __restrict__ q_part, const double* __restrict__ q_proxy,
                            CPtr3 dpart, CPtr3 dprox, v4f* __restrict__ rec) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.npart + (int64_t)t.offset * t.n) return;  // leaf proxy rows are never sources
  const int64_t mp = member_part(t), mx = member_proxy(t);
  rec += (int64_t)blockIdx.y * t.U16 * 2;
  double x = t.px[u], y = t.py[u], z = t.pz[u], q;
  int panel;
  if (u < t.npart) {
    if (dpart.p[0]) { x += dpart.p[0][mp + u]; y += dpart.p[1][mp + u]; z += dpart.p[2][mp + u]; }
    q = q_part[mp + u];
    panel = t.offset + (int)(u / t.m2);
  } else {
    const int64_t v = u - t.npart;
    if (dprox.p[0]) { x += dprox.p[0][mx + v]; y += dprox.p[1][mx + v]; z += dprox.p[2][mx + v]; }
    q = q_proxy[mx + v];
    panel = (int)(v / t.n);
  }
  project_to_sphere(x, y, z);
  const DevPanel& P = t.panels[panel];
  const float bx = (float)(x - P.cx), by = (float)(y - P.cy), bz = (float)(z - P.cz);
  const double qq = kNegInv4Pi * q;
  rec[2 * u] = v4f{bx, by, bz, (float)(0.5 * ((double)bx * bx + (double)by * by + (double)bz * bz))};
  rec[2 * u + 1] = v4f{(float)(qq * bx), (float)(qq * by), (float)(qq * bz), (float)qq};
}

template <int S, int NT>
__global__ __launch_bounds__(64 * S) void k_bve_lanes(DevTree t, const TargetTile* __restrict__ tiles, int ntiles,
                                                      const SourceSet* __restrict__ sets, const v4f* __restrict__ rec,
                                                      float eps, Ptr3 part, Ptr3 proxy, int assign, int xcd) {
  __shared__ __align__(16) double stage[S][kLaneSlots * 4];
  rec += (int64_t)blockIdx.y * t.U16 * 2;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = walk_tile(t.xcd_start, xcd);
  if (tile >= ntiles) return;  // the whole workgroup
  const TargetTile T = tiles[tile];
  const DevPanel& PT = t.panels[T.panel];
  const LaneTile l = lane_tile<NT>(T.count, lane);
  float ax[NT], ay[NT], az[NT];  // minus the target relative to its panel's centre
  double w[NT][3];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int64_t u = (int64_t)T.first + min(q * l.T + l.i, T.count - 1);
    ax[q] = (float)(PT.cx - t.px[u]);
    ay[q] = (float)(PT.cy - t.py[u]);
    az[q] = (float)(PT.cz - t.pz[u]);
    w[q][0] = w[q][1] = w[q][2] = 0;
  }
  v4f* mine = reinterpret_cast<v4f*>(stage[wave]);
  const v4f pad = v4f{0.f, 0.f, 0.f, 1.f};  // padding record: denominator above 1, no charge
  if (lane < kLanePad) {
    mine[2 * (kLaneChunk + lane)] = pad;
    mine[2 * (kLaneChunk + lane) + 1] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  walk_sets<S>(T, sets, wave, [&](const SourceSet& set, int a, int b) {
    float px[NT], py[NT], pz[NT], alpha[NT];
    v4f acc[NT], odd[NT];  // even and odd trips: the FP32 chains stay half as long
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      px[q] = ax[q] - set.ox;
      py[q] = ay[q] - set.oy;
      pz[q] = az[q] - set.oz;
      alpha[q] = fmaf(0.5f, fmaf(px[q], px[q], fmaf(py[q], py[q], pz[q] * pz[q])), eps);
      acc[q] = odd[q] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    auto add = [&](const v4f r0, const v4f r1, v4f(&sum)[NT]) {
#pragma unroll
      for (int q = 0; q < NT; ++q) {
        float d = fmaf(px[q], r0.x, r0.w);
        d = fmaf(py[q], r0.y, d);
        d = fmaf(pz[q], r0.z, d);
        const float g = __builtin_amdgcn_rcpf(d + alpha[q]);
        sum[q].x = fmaf(g, r1.x, sum[q].x);
        sum[q].y = fmaf(g, r1.y, sum[q].y);
        sum[q].z = fmaf(g, r1.z, sum[q].z);
        sum[q].w = fmaf(g, r1.w, sum[q].w);
      }
    };
    const v4f* __restrict__ src = rec + 2 * (int64_t)set.first;
    for (int c = a; c < b; c += kLaneChunk) {
      const int cn = min(kLaneChunk, b - c), trips = (cn + l.G - 1) / l.G;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      {
        v4f r0 = pad, r1 = v4f{0.f, 0.f, 0.f, 0.f};
        if (lane < cn) {
          r0 = src[2 * (c + lane)];
          r1 = src[2 * (c + lane) + 1];
        }
        mine[2 * lane] = r0;
        mine[2 * lane + 1] = r1;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      const v4f* r = mine + 2 * l.g;
      int k = 0;
      for (; k + 1 < trips; k += 2, r += 4 * l.G) {
        add(r[0], r[1], acc);
        add(r[2 * l.G], r[2 * l.G + 1], odd);
      }
      if (k < trips) add(r[0], r[1], acc);
    }
#pragma unroll
    for (int q = 0; q < NT; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v4f& f = h ? odd[q] : acc[q];
        w[q][0] += (double)fmaf(px[q], f.w, f.x);
        w[q][1] += (double)fmaf(py[q], f.w, f.y);
        w[q][2] += (double)fmaf(pz[q], f.w, f.z);
      }
  });
  double s[3];
  lane_sum<NT, 3, S>(l, w, stage, wave, lane, s);
  if (wave > 0 || lane >= T.count) return;
  const int64_t u = (int64_t)T.first + lane;
  const double x = t.px[u], y = t.py[u], z = t.pz[u];
  const double v[3] = {y * s[2] - z * s[1], z * s[0] - x * s[2], x * s[1] - y * s[0]};
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double* o = u < t.npart ? part.p[c] + member_part(t) + u : proxy.p[c] + member_proxy(t) + (u - t.npart);
    *o = assign ? v[c] : *o + v[c];
  }
}

}  // namespace

void launch_source_records_lanes(const DevTree& t, const double* q_part, const double* q_proxy,
                                 const double* const* disp_part, const double* const* disp_proxy, void* rec,
                                 hipStream_t s, int nmem) {
  CPtr3 dp{}, dx{};
  for (int f = 0; f < 3; ++f) {
    dp.p[f] = disp_part ? disp_part[f] : nullptr;
    dx.p[f] = disp_proxy ? disp_proxy[f] : nullptr;
  }
  const int64_t n = t.npart + (int64_t)t.offset * t.n;
  hipLaunchKernelGGL(k_src_lanes, dim3((unsigned)((n + 255) / 256), nmem), dim3(256), 0, s, t, q_part, q_proxy, dp, dx,
                     static_cast<v4f*>(rec));
}

void launch_bve_interact_lanes(const DevTree& t, const TargetTile* tiles, int ntiles, const SourceSet* sets,
                               const void* rec, double eps, double* const* out_part, double* const* out_proxy,
                               hipStream_t s, bool assign, int nmem, PairShape shape) {
  if (ntiles == 0) return;
  if (shape.xcd == 2 && (!t.xcd_start || shape.grid1 <= 0)) shape.xcd = 0;
  // us per launch with 4 / 8 waves: 126 tiles 25 / 20, 636 47 / 46, 2,556 (36 rows) 83 / 87, 10,236 267 / 302,
  // 40,956 1490 / 1562
  // (with members a short list fills the chip and 8 waves' sums cost more than they gain:
  // 16 members at 510 tiles of 25 rows 747 us a step, 551 with 4 waves, a single step 168 and
  // 166; at 36 rows and more 2% to 3% of a single step, so 8 stay)
  int S = t.rows <= 32 && ntiles >= 400 ? 4 : lane_waves(ntiles);
  auto kernel = S == 8 ? k_bve_lanes<8, 2> : k_bve_lanes<4, 2>;
  // tiles of at most 10 rows: one target per lane halves what a set costs to centre and
  // flush, and sets of 9 records give fewer waves enough.  Velocity at degree 2, 3 x 3
  // points a leaf, with two targets and 4 waves, and with one and 4 / 2 / 1: 2,046 tiles
  // 42, 38 / 42 / 54 us; 8,190 99, 86 / 86 / 91; 32,766 300, 254 / 237 / 231; a step of 16
  // members at 2,046 tiles 1,182, 993 / 927 / 900.  Their six copies or more still give each
  // FP32 sum one record of a set; the four copies of 16 rows would give it two, and 268 us
  // at 32,766 tiles, but 1% to 10% further from FP64: 11 to 16 rows keep two targets.
  // With 4 / 2 / 1 waves there: 2,046 tiles 37 / 38 / 50, 8,190 104 / 104 / 116, 32,766 316 /
  // 299 / 296; a step of 16 members at 510 tiles 411 (8 waves 636) / 408 / 443
  if (t.rows <= 16) {
    S = ntiles < (t.rows <= 10 ? 1000 : 6000) ? 4 : 2;
    kernel = t.rows > 10 ? (S == 4 ? k_bve_lanes<4, 2> : k_bve_lanes<2, 2>)
                         : (S == 4 ? k_bve_lanes<4, 1> : k_bve_lanes<2, 1>);
  }
  Ptr3 op{{out_part[0], out_part[1], out_part[2]}}, ox{{out_proxy[0], out_proxy[1], out_proxy[2]}};
  hipLaunchKernelGGL(kernel, dim3(walk_grid(ntiles, shape), nmem), dim3(64 * S), 0, s, t, tiles, ntiles, sets,
                     static_cast<const v4f*>(rec), (float)eps, op, ox, assign ? 1 : 0, shape.xcd);
}

}  // namespace sbslpm
