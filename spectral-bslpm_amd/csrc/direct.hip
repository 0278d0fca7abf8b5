// direct.hip -- O(N^2) direct sums (direct_sum.cpp:8-15, direct_sum_impl.hpp:18-27)
// and the Biot-Savart direct sum the reference lacks (same pair kernel as
// bve_vel_impl.hpp:54-66).
//
// A workgroup of eight waves owns 64 NT targets (NT per lane) and one source
// chunk per grid row; each wave takes an eighth of the chunk, sources are
// wave-uniform loads taken four at a time, and the waves' sums are added
// in wave order through LDS.  Each (target tile, chunk) writes a partial sum
// and a second kernel adds the chunks in a fixed order, so the result is
// deterministic and needs no atomics (the reference does one atomic per pair).
#include <algorithm>
#include <mutex>

#include "device.hpp"

namespace sbslpm {
namespace {

constexpr int kWaves = 8;

struct Plan {
  int64_t tiles, chunks, chunk_len;
  int nt_lane;
  bool shared;  // waves share a tile; else each wave takes tiles of its own
  dim3 grid;
};

// chunks is bounded by the waves of 64 targets it takes to fill the chip (4096)
// and by 256 sources per chunk; it alone sets the scratch the sums need.
// Two targets per lane halve the source loads and the uniform work per pair:
// taken unless the second target would idle in a list of a few 64-target rows
// (one row of 64 against 400,000 sources: 2x the pairs for nothing).
// A few sources for more targets than fill the chip: eight waves on a tile would each
// start, add up and stage the log table for a few pairs, so a wave takes whole tiles
// instead, a workgroup's waves tile after tile.  Microseconds per call, waves sharing a
// tile and not: log sum, 2,000,000 targets x 1 / 8 / 64 sources 94 / 101 / 141 and 24 / 29 /
// 100, velocity 115 / 122 / 149 and 39 / 40 / 82; 300,000 x 1 / 64 / 128 (two targets per
// lane) log 17 / 27 / 38 and 12 / 28 / 48, velocity 24 / 29 / 37 and 13 / 24 / 37.
Plan plan(int64_t nt, int64_t ns) {
  Plan p;
  const int64_t rows = (nt + 63) / 64;
  int64_t want = (4096 + rows - 1) / rows;
  int64_t maxc = (ns + 255) / 256;
  p.chunks = std::max<int64_t>(1, std::min(want, maxc));
  p.chunk_len = (ns + p.chunks - 1) / p.chunks;
  p.chunks = p.chunk_len > 0 ? (ns + p.chunk_len - 1) / p.chunk_len : 1;
  if (p.chunks < 1) p.chunks = 1;
  p.nt_lane = (rows & 1) && rows < 8 ? 1 : 2;
  p.tiles = (rows + p.nt_lane - 1) / p.nt_lane;
  p.shared = p.chunk_len > 128 || p.tiles < std::max<int64_t>(1500, 25 * p.chunk_len);
  if (!p.shared && rows < 8192) {
    // a target per lane, twice the waves: 300,000 x 64 log 27 -> 25 us, velocity 23 -> 22
    p.nt_lane = 1;
    p.tiles = rows;
  }
  const int64_t groups = p.shared ? p.tiles : std::min<int64_t>((p.tiles + kWaves - 1) / kWaves, 1024);
  p.grid = dim3((unsigned)groups, (unsigned)p.chunks);
  return p;
}

// This wave's part [a, b) of the workgroup's source chunk where W waves share it:
// W-ths rounded up to whole batches of four.
template <int W>
__device__ inline void wave_sources(int64_t ns, int64_t chunk_len, int wave, int64_t& a, int64_t& b) {
  const int64_t j0 = (int64_t)blockIdx.y * chunk_len, j1 = std::min<int64_t>(ns, j0 + chunk_len);
  if (W == 1) {
    a = j0;
    b = j1;
    return;
  }
  const int64_t q = ((j1 - j0 + 4 * W - 1) / (4 * W)) * 4;
  a = std::min<int64_t>(j1, j0 + wave * q);
  b = std::min<int64_t>(j1, a + q);
}

// Sum of v over the workgroup's waves in wave order, valid in wave 0.
template <int K>
__device__ inline void wave_sum(double (&v)[K], int wave, int lane) {
  __shared__ double red[kWaves - 1][K][64];
  if (wave > 0)
#pragma unroll
    for (int k = 0; k < K; ++k) red[wave - 1][k][lane] = v[k];
  __syncthreads();
  if (wave == 0)
#pragma unroll
    for (int w = 0; w < kWaves - 1; ++w)
#pragma unroll
      for (int k = 0; k < K; ++k) v[k] += red[w][k][lane];
}

// A wave's first tile: the workgroup's one (W waves share it), or the first of every
// 8 gridDim.x-th.
template <int W>
__device__ inline int64_t first_tile(int wave) {
  return W > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * kWaves + wave;
}

// guard 0: skip j == self_offset + i (the reference's i != j);
// guard 1: skip x.y >= 1 - 1e-15 (the FMM kernel's coincidence guard).
// The logarithm is log_wide (fasttab.hpp) where 1 - x.y is in its range; a batch
// of sources that holds the targets themselves or a pair outside (closer than
// 4e-5 rad, or skipped) takes the guarded form, with the library's logarithm for
// the close ones (one unsigned maximum per pair and a ballot per batch).
// Bound: FP64 vector issue, 20 instructions per pair (about 90 with the library's
// logarithm on every pair).  24,576 x 24,576 points: 2.13 -> 0.44 ms
// (0.57 with log_tab), vector issue busy 70% of the time.
template <int NT, int W>
__global__ __launch_bounds__(64 * kWaves) void k_direct_log(int64_t nt, const double* __restrict__ tx,
                                                    const double* __restrict__ ty, const double* __restrict__ tz,
                                                    int64_t ns, const double* __restrict__ sx,
                                                    const double* __restrict__ sy, const double* __restrict__ sz,
                                                    const double* __restrict__ area, const double* __restrict__ pots,
                                                    int64_t self_offset, int guard, int64_t chunk_len, int64_t tiles,
                                                    const LogTabEntry* __restrict__ logwide,
                                                    double* __restrict__ partials) {
  // x.y rounded exactly as written in direct_sum_impl.hpp:23 (no fused
  // multiply-add): for nearly coincident points log(1 - x.y) amplifies a
  // one-ulp change of x.y by 1/(1 - x.y).
#pragma clang fp contract(off)
  __shared__ LogTabEntry wide[kLogWideSize];
  for (int i = threadIdx.x; i < kLogWideSize; i += blockDim.x) wide[i] = logwide[i];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  int64_t tile = first_tile<W>(wave);
  if (W == 1 && tile >= tiles) return;
  do {
    const int64_t i0 = tile * (64 * NT);
    double x[NT], y[NT], z[NT], acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int64_t i = std::min<int64_t>(i0 + t * 64 + lane, nt - 1);
      x[t] = tx[i]; y[t] = ty[i]; z[t] = tz[i];
      acc[t] = 0;
    }
    int64_t a, b;
    wave_sources<W>(ns, chunk_len, wave, a, b);
    const int64_t self_lo = self_offset + i0, self_hi = self_lo + 64 * NT;
    const double c7 = in_vgpr(1.0 / 7.0);
    auto guarded = [&](int t, int64_t j) {
      const int64_t i = std::min<int64_t>(i0 + t * 64 + lane, nt - 1);
      const double d = 1.0 - (x[t] * sx[j] + y[t] * sy[j] + z[t] * sz[j]);
      const bool skip = guard ? !(d > 1.0 - (1.0 - 1e-15)) : (j == self_offset + i);
      const double v = skip ? 1.0 : d;
      const uint32_t h = log_wide_cell(v);
      const bool close = h >= kLogWideSpan;
      double l = log_wide(v, close ? 0u : h, wide, c7);
      if (__builtin_amdgcn_ballot_w64(close) != 0) l = close ? log(fmax(v, 1e-300)) : l;
      const double q = area[j] * pots[j];
      acc[t] = skip ? acc[t] : fma(l, q, acc[t]);
    };
    int64_t j = a;
    for (; j + 4 <= b; j += 4) {
      double d[NT][4];
      uint32_t h[NT][4], far = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double s0 = sx[j + k], s1 = sy[j + k], s2 = sz[j + k];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          d[t][k] = 1.0 - (x[t] * s0 + y[t] * s1 + z[t] * s2);
          h[t][k] = log_wide_cell(d[t][k]);
          far = h[t][k] > far ? h[t][k] : far;
        }
      }
      loaded(area[j], area[j + 1], area[j + 2], area[j + 3]);
      loaded(pots[j], pots[j + 1], pots[j + 2], pots[j + 3]);
      const bool own = !guard && j < self_hi && j + 4 > self_lo;
      if (own || __builtin_amdgcn_ballot_w64(far >= kLogWideSpan) != 0) {
#pragma unroll 1
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int t = 0; t < NT; ++t) guarded(t, j + k);
        continue;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double q = area[j + k] * pots[j + k];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = fma(log_wide(d[t][k], h[t][k], wide, c7), q, acc[t]);
      }
    }
    for (; j < b; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t) guarded(t, j);
    if constexpr (W > 1) wave_sum(acc, wave, lane);
    if (W == 1 || wave == 0)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (i0 + t * 64 + lane < nt) partials[(int64_t)blockIdx.y * nt + i0 + t * 64 + lane] = kNegInv4Pi * acc[t];
    tile += (int64_t)gridDim.x * kWaves;
  } while (W == 1 && tile < tiles);
}

// Bound: FP64 vector issue.  The four denominators of a batch share one
// reciprocal (rcp4: 12.5 instruction slots per pair with the loads' share
// against 17 with a reciprocal each), and 1 - x.y is one chain of fused
// multiply-adds from 1.  4,096 targets x 393,216 sources: 4.09 -> 0.77 ms (one
// target per lane and one source per step waited on each source's scalar loads;
// now vector issue is busy 83% of the time, at 2.1 GHz under this load).
template <int NT, int W, bool SHARED>
__global__ __launch_bounds__(64 * kWaves) void k_direct_bs(int64_t nt, const double* __restrict__ tx,
                                                   const double* __restrict__ ty, const double* __restrict__ tz,
                                                   int64_t ns, const double* __restrict__ sx,
                                                   const double* __restrict__ sy, const double* __restrict__ sz,
                                                   const double* __restrict__ area, const double* __restrict__ vor,
                                                   double eps, int64_t chunk_len, int64_t tiles,
                                                   double* __restrict__ partials) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  int64_t tile = first_tile<W>(wave);
  if (W == 1 && tile >= tiles) return;
  do {
    const int64_t i0 = tile * (64 * NT);
    double x[NT], y[NT], z[NT], w[3 * NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int64_t i = std::min<int64_t>(i0 + t * 64 + lane, nt - 1);
      x[t] = tx[i]; y[t] = ty[i]; z[t] = tz[i];
      w[3 * t] = w[3 * t + 1] = w[3 * t + 2] = 0;
    }
    int64_t a, b;
    wave_sources<W>(ns, chunk_len, wave, a, b);
    int64_t j = a;
    for (; j + 4 <= b; j += 4) {
      double s0[4], s1[4], s2[4], q[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        s0[k] = sx[j + k]; s1[k] = sy[j + k]; s2[k] = sz[j + k];
        q[k] = area[j + k] * vor[j + k];
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        double d[4], g[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) d[k] = one_minus_dot(x[t], y[t], z[t], s0[k], s1[k], s2[k]) + eps;
        rcps<SHARED>(d, g);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double gq = g[k] * q[k];
          w[3 * t] = fma(gq, s0[k], w[3 * t]);
          w[3 * t + 1] = fma(gq, s1[k], w[3 * t + 1]);
          w[3 * t + 2] = fma(gq, s2[k], w[3 * t + 2]);
        }
      }
    }
    for (; j < b; ++j) {
      const double s0 = sx[j], s1 = sy[j], s2 = sz[j], q = area[j] * vor[j];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const double g = rcp64(one_minus_dot(x[t], y[t], z[t], s0, s1, s2) + eps) * q;
        w[3 * t] = fma(g, s0, w[3 * t]);
        w[3 * t + 1] = fma(g, s1, w[3 * t + 1]);
        w[3 * t + 2] = fma(g, s2, w[3 * t + 2]);
      }
    }
    if constexpr (W > 1) wave_sum(w, wave, lane);
    if (W > 1 && wave > 0) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int64_t i = i0 + t * 64 + lane;
      if (i >= nt) continue;
      const double *u = w + 3 * t;
      double* p = partials + (int64_t)blockIdx.y * 3 * nt;
      p[i] = kNegInv4Pi * (y[t] * u[2] - z[t] * u[1]);
      p[nt + i] = kNegInv4Pi * (z[t] * u[0] - x[t] * u[2]);
      p[2 * nt + i] = kNegInv4Pi * (x[t] * u[1] - y[t] * u[0]);
    }
    tile += (int64_t)gridDim.x * kWaves;
  } while (W == 1 && tile < tiles);
}

struct Ptr3 {
  double* p[3];
};

// out[blockIdx.y] += the chunks' partial sums: 64 targets per workgroup, wave w
// adds chunks w, w + 8, ..., the waves' sums are added in wave order.  (With one
// thread per target walking every chunk of three components, the 64 chunks of
// 4,096 targets took 52 us, a chain of loads in 64 waves; now 4.9 us.)
__global__ __launch_bounds__(64 * kWaves) void k_reduce(int64_t nt, int ncomp, int64_t chunks,
                                                const double* __restrict__ partials, Ptr3 out) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int f = (int)blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * 64 + lane, ic = std::min<int64_t>(i, nt - 1);
  double s[1] = {0};
#pragma unroll 4
  for (int64_t c = wave; c < chunks; c += kWaves) s[0] += partials[(c * ncomp + f) * nt + ic];
  wave_sum(s, wave, lane);
  if (wave == 0 && i < nt) out.p[f][i] += s[0];
}

// The same for at most three chunks, a thread per target, the chunks' loads together.
__global__ __launch_bounds__(256) void k_reduce_few(int64_t nt, int ncomp, int64_t chunks,
                                                    const double* __restrict__ partials, Ptr3 out) {
  const int f = (int)blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nt) return;
  double v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = c < chunks ? partials[((int64_t)c * ncomp + f) * nt + i] : 0;
  out.p[f][i] += v[0] + v[1] + v[2];
}

void launch_reduce(int64_t nt, int ncomp, int64_t chunks, const double* partials, Ptr3 out, hipStream_t s) {
  if (chunks < 4)
    hipLaunchKernelGGL(k_reduce_few, dim3((unsigned)((nt + 255) / 256), ncomp), dim3(256), 0, s, nt, ncomp, chunks,
                       partials, out);
  else
    hipLaunchKernelGGL(k_reduce, dim3((unsigned)((nt + 63) / 64), ncomp), dim3(64 * kWaves), 0, s, nt, ncomp, chunks,
                       partials, out);
}

// Displaced, re-projected source positions (bve_vel_impl.hpp:57-60).
__global__ void k_displace(int64_t ns, const double* __restrict__ sx, const double* __restrict__ sy,
                           const double* __restrict__ sz, const double* __restrict__ dx,
                           const double* __restrict__ dy, const double* __restrict__ dz, double* __restrict__ out) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ns) return;
  double a = sx[j] + dx[j], b = sy[j] + dy[j], c = sz[j] + dz[j];
  project_to_sphere(a, b, c);
  out[j] = a; out[ns + j] = b; out[2 * ns + j] = c;
}

}  // namespace

// Fixed device scratch of the allocation-free direct sum
// (sbslpm_direct_sum_inv_lap_noalloc): the per-chunk partial sums of
// k_direct_log.  Each device holds its own copy until the process ends.  In
// host code `scratch` only names the symbol; its device address comes from
// hipGetSymbolAddress, once per device, in direct_noalloc_init.
static __device__ __align__(256) double scratch[kNoAllocScratchDoubles];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

int direct_noalloc_init(int device) {
  if (device < 0 || device >= kMaxDevices) return -1;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return 0;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) return (int)(e != hipSuccess ? e : hipErrorInvalidSymbol);
  g_scratch_ptr[device] = static_cast<double*>(p);
  return 0;
}

double* direct_noalloc_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[device];
}

// Scratch doubles needed by a direct sum with nt targets, ns sources.
int64_t direct_partials_size(int64_t nt, int64_t ns, int ncomp) {
  Plan p = plan(nt, ns);
  return p.chunks * ncomp * nt + (ncomp == 3 ? 3 * ns : 0);
}

void launch_direct_inv_lap(int64_t nt, const double* tx, const double* ty, const double* tz, int64_t ns,
                           const double* sx, const double* sy, const double* sz, const double* area,
                           const double* pots, int64_t self_offset, bool guard_coincident,
                           const LogTabEntry* logwide, double* partials, double* soln, hipStream_t s) {
  if (nt <= 0) return;
  const Plan p = plan(nt, ns);
  auto kernel = p.nt_lane == 2 ? (p.shared ? k_direct_log<2, kWaves> : k_direct_log<2, 1>)
                               : (p.shared ? k_direct_log<1, kWaves> : k_direct_log<1, 1>);
  hipLaunchKernelGGL(kernel, p.grid, dim3(64 * kWaves), 0, s, nt, tx, ty, tz, ns, sx, sy, sz, area, pots, self_offset,
                     guard_coincident ? 1 : 0, p.chunk_len, p.tiles, logwide, partials);
  launch_reduce(nt, 1, p.chunks, partials, Ptr3{{soln, nullptr, nullptr}}, s);
}

void launch_direct_bve_vel(int64_t nt, const double* tx, const double* ty, const double* tz, int64_t ns,
                           const double* sx, const double* sy, const double* sz, const double* area,
                           const double* vor, const double* const* disp, double eps, double* partials,
                           double* const* vel, hipStream_t s) {
  if (nt <= 0) return;
  const Plan p = plan(nt, ns);
  const double *ax = sx, *ay = sy, *az = sz;
  if (disp && disp[0]) {
    double* moved = partials + p.chunks * 3 * nt;
    hipLaunchKernelGGL(k_displace, dim3((unsigned)((ns + 255) / 256)), dim3(256), 0, s, ns, sx, sy, sz, disp[0],
                       disp[1], disp[2], moved);
    ax = moved; ay = moved + ns; az = moved + 2 * ns;
  }
  auto kernel = p.nt_lane == 2 ? (p.shared ? k_direct_bs<2, kWaves, true> : k_direct_bs<2, 1, true>)
                               : (p.shared ? k_direct_bs<1, kWaves, true> : k_direct_bs<1, 1, true>);
  if (!rcp4_in_range(eps))
    kernel = p.nt_lane == 2 ? (p.shared ? k_direct_bs<2, kWaves, false> : k_direct_bs<2, 1, false>)
                            : (p.shared ? k_direct_bs<1, kWaves, false> : k_direct_bs<1, 1, false>);
  hipLaunchKernelGGL(kernel, p.grid, dim3(64 * kWaves), 0, s, nt, tx, ty, tz, ns, ax, ay, az, area, vor, eps,
                     p.chunk_len, p.tiles, partials);
  launch_reduce(nt, 3, p.chunks, partials, Ptr3{{vel[0], vel[1], vel[2]}}, s);
}

}  // namespace sbslpm
