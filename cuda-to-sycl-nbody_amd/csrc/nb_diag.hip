// fp64 diagnostics on the GPU (no reference counterpart): the oracle force
// on a sampled subset of targets and the total energy / momentum.  These are
// the only fp64 computations on the device; the step itself stays fp32.
//
//   forces:  F_i = sum_{j != i} r (|r|^2 + eps)^{-3/2} in fp64 from the float
//            positions (r formed in double), for targets idx[0..m).  The
//            sources are split over grid.y chunks; a second kernel adds the
//            chunk partials in chunk order (deterministic).
//   energy:  K = sum |v|^2 / 2,  W = -G sum_{i<j} (|r|^2 + eps)^{-1/2}
//            (the potential whose negative gradient is the step's force),
//            P = sum v (unit masses).  Each pair is visited once; every sum
//            is fp64, in an order that depends on n alone (deterministic).
//
// Both are bound by fp64 issue (4 cycles an instruction), so the powers of d
// are not taken with sqrt and division (some thirty instructions): v_rsq_f64
// cut to 26 bits gives y with y * y exact, so e = 1 - d y^2 carries one
// rounding of its own small size, and a series in e restores the full result
// (|e| <= 2^-23.19 over 10^9 values at each of six scales: the terms left out,
// 0.31 e^3 for d^{-1/2} and 2.19 e^3 for d^{-3/2}, are under 2^-71 and 2^-68).  With u = 2^-53 the relative
// error is u for d^{-1/2} (correctly rounded sqrt and division: 2 u) and 2 u
// for d^{-3/2} (3 u).  d = 0 and d = inf turn the series into NaN: a tile
// whose sum is NaN is summed again with sqrt and division, which give the
// infinities and zeros that belong there.
//
// Measured on MI355X, us a call with its host work, against every ordered
// pair by sqrt and division with one workgroup per 256 targets: energy
// n = 1000 40 (209), 16384 177 (2760), 65536 1337 (10700), 262144 16500
// (105700: 76 cycles a pair and SIMD); forces on 4096 of 65536 188 (498), on
// 100 of 1000 25 (178).  Against 80-bit sums over 120 states of 200 to 4900
// particles the potential is off by 0.55 u in the mean and 1.73 u at most
// (before 0.63 and 1.83); forces over 500 targets by 0.9 to 1.4e-16 in the
// mean (before 3.2 to 7.6e-16).

#include <algorithm>
#include <type_traits>
#include <vector>

#include "nb_internal.hpp"

namespace nb {
namespace {

constexpr int kBlock = 256;
constexpr int kTile = 512;     // sources staged in LDS, as doubles
constexpr int kPerLane = 2;    // energy: targets per lane
constexpr int kETile = kBlock * kPerLane;

struct Sources {
  double x[kTile], y[kTile], z[kTile];
};

__device__ inline void stage(Sources &sm, const float *px, const float *py,
                             const float *pz, int j0, int cnt) {
  for (int l = threadIdx.x; l < cnt; l += kBlock) {
    sm.x[l] = px[j0 + l];
    sm.y[l] = py[j0 + l];
    sm.z[l] = pz[j0 + l];
  }
}

// y near d^{-1/2} in 26 bits and e = 1 - d y^2.
__device__ inline double rsqrt_seed(double d, double &e) {
  const long long cut = ~((1LL << 27) - 1);
  const double y = __longlong_as_double(
      __double_as_longlong(__builtin_amdgcn_rsq(d)) & cut);
  e = fma(-d, y * y, 1.0);
  return y;
}

struct ForceArgs {
  const float *px, *py, *pz;
  const int *idx;
  int m, n, chunk;
  double eps;
  double *part; // [chunks][3][m]
};

__global__ __launch_bounds__(kBlock) void f64_force_partial(ForceArgs a) {
  __shared__ Sources sm;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int raw = a.idx[t < a.m ? t : a.m - 1];
  const bool valid = raw >= 0 && raw < a.n; // an invalid index yields NaN
  const int i = valid ? raw : 0;
  const double xi = a.px[i], yi = a.py[i], zi = a.pz[i];
  const int jbeg = blockIdx.y * a.chunk;
  const int jend = min(jbeg + a.chunk, a.n);
  double fx = 0.0, fy = 0.0, fz = 0.0;
  for (int j0 = jbeg; j0 < jend; j0 += kTile) {
    const int cnt = min(kTile, jend - j0);
    __syncthreads();
    stage(sm, a.px, a.py, a.pz, j0, cnt);
    __syncthreads();
    // the self pair adds r = 0 times a finite power, or makes the sum NaN
    double tx = 0.0, ty = 0.0, tz = 0.0;
#pragma unroll 2
    for (int l = 0; l < cnt; ++l) {
      const double rx = sm.x[l] - xi, ry = sm.y[l] - yi, rz = sm.z[l] - zi;
      const double d = fma(rz, rz, fma(ry, ry, fma(rx, rx, a.eps)));
      double e;
      const double y = rsqrt_seed(d, e);
      const double c = y * y * y;
      const double inv = fma(c, e * fma(1.875, e, 1.5), c);
      tx = fma(rx, inv, tx);
      ty = fma(ry, inv, ty);
      tz = fma(rz, inv, tz);
    }
    if (tx != tx || ty != ty || tz != tz) {
      tx = ty = tz = 0.0;
      for (int l = 0; l < cnt; ++l) {
        if (j0 + l == i) continue;
        const double rx = sm.x[l] - xi, ry = sm.y[l] - yi, rz = sm.z[l] - zi;
        const double d = rx * rx + ry * ry + rz * rz + a.eps;
        const double inv = 1.0 / (d * sqrt(d));
        tx += rx * inv;
        ty += ry * inv;
        tz += rz * inv;
      }
    }
    fx += tx;
    fy += ty;
    fz += tz;
  }
  if (!valid) fx = fy = fz = __builtin_nan("");
  if (t < a.m) {
    const size_t base = (size_t)blockIdx.y * 3 * a.m;
    a.part[base + t] = fx;
    a.part[base + a.m + t] = fy;
    a.part[base + 2 * (size_t)a.m + t] = fz;
  }
}

constexpr int kFinLanes = 8, kFinTargets = kBlock / kFinLanes;

// One component per grid.y, eight threads a target: each adds every eighth
// partial, so up to 1024 of them are a chain of 128 and their rounding is no
// larger than that of a few long chunks.
__global__ __launch_bounds__(kBlock) void f64_force_finish(
    const double *part, int m, int chunks, double *fx, double *fy,
    double *fz) {
  __shared__ double sh[kFinLanes][kFinTargets];
  const int lt = threadIdx.x % kFinTargets, lane = threadIdx.x / kFinTargets;
  const int t = blockIdx.x * kFinTargets + lt, k = blockIdx.y;
  double s = 0.0;
  if (t < m) {
#pragma unroll 8
    for (int c = lane; c < chunks; c += kFinLanes)
      s += part[((size_t)c * 3 + k) * m + t];
  }
  sh[lane][lt] = s;
  __syncthreads();
  if (lane != 0 || t >= m) return;
  (k == 0 ? fx : k == 1 ? fy : fz)[t] =
      ((sh[0][lt] + sh[1][lt]) + (sh[2][lt] + sh[3][lt])) +
      ((sh[4][lt] + sh[5][lt]) + (sh[6][lt] + sh[7][lt]));
}

// Block-wide fp64 sum of `v` as a tree (all threads of the block call it).
template <int WAVES>
__device__ double block_sum(double v, double *sh) {
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) v += __shfl_xor(v, w, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = sh[threadIdx.x % WAVES];
#pragma unroll
  for (int w = WAVES / 2; w > 0; w >>= 1) r += __shfl_xor(r, w, 64);
  return r;
}

struct EnergyArgs {
  const float *px, *py, *pz, *vx, *vy, *vz;
  int n, chunk, tiles, chunks;
  double eps;
  double *part; // [chunks][tiles] potentials, then [4][tiles] K and P
};

// Workgroup (tile, chunk): the tile's targets against the chunk's sources of
// larger index; chunk 0 also adds the tile's kinetic energy and momentum.
__global__ __launch_bounds__(kBlock) void f64_energy_partial(EnergyArgs a) {
  __shared__ Sources sm;
  __shared__ double red[kBlock / 64];
  const int base = blockIdx.x * kETile;
  int idx[kPerLane];
  double xi[kPerLane], yi[kPerLane], zi[kPerLane], w[kPerLane];
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) {
    idx[k] = base + k * kBlock + threadIdx.x;
    const int ic = min(idx[k], a.n - 1);
    xi[k] = a.px[ic];
    yi[k] = a.py[ic];
    zi[k] = a.pz[ic];
    w[k] = 0.0;
  }
  const long long cbeg = (long long)blockIdx.y * a.chunk;
  const int jend = (int)min(cbeg + a.chunk, (long long)a.n);
  const int jbeg = (int)max(cbeg, (long long)base + 1);
  for (int j0 = jbeg; j0 < jend; j0 += kTile) {
    const int cnt = min(kTile, jend - j0);
    __syncthreads();
    stage(sm, a.px, a.py, a.pz, j0, cnt);
    __syncthreads();
    const bool mask = j0 < base + kETile; // some pairs have j <= i
    double tw[kPerLane] = {};
    auto pairs = [&](auto masked) {
#pragma unroll 2
      for (int l = 0; l < cnt; ++l) {
        const double xj = sm.x[l], yj = sm.y[l], zj = sm.z[l];
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) {
          const double rx = xj - xi[k], ry = yj - yi[k], rz = zj - zi[k];
          const double d = fma(rz, rz, fma(ry, ry, fma(rx, rx, a.eps)));
          double e;
          const double y = rsqrt_seed(d, e);
          double inv = fma(y, e * fma(0.375, e, 0.5), y);
          if constexpr (decltype(masked)::value)
            inv = j0 + l > idx[k] ? inv : 0.0;
          tw[k] += inv;
        }
      }
    };
    if (mask)
      pairs(std::true_type{});
    else
      pairs(std::false_type{});
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) {
      if (tw[k] != tw[k]) {
        tw[k] = 0.0;
        for (int l = 0; l < cnt; ++l) {
          if (j0 + l <= idx[k]) continue;
          const double rx = sm.x[l] - xi[k], ry = sm.y[l] - yi[k],
                       rz = sm.z[l] - zi[k];
          tw[k] += 1.0 / sqrt(rx * rx + ry * ry + rz * rz + a.eps);
        }
      }
      w[k] += tw[k];
    }
  }
  double ws = 0.0;
#pragma unroll
  for (int k = 0; k < kPerLane; ++k)
    if (idx[k] < a.n) ws += w[k];
  const double r = block_sum<kBlock / 64>(ws, red);
  if (threadIdx.x == 0)
    a.part[(size_t)blockIdx.y * a.tiles + blockIdx.x] = r;
  if (blockIdx.y != 0) return;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) {
    if (idx[k] >= a.n) continue;
    const double ux = a.vx[idx[k]], uy = a.vy[idx[k]], uz = a.vz[idx[k]];
    s[0] += 0.5 * (ux * ux + uy * uy + uz * uz);
    s[1] += ux;
    s[2] += uy;
    s[3] += uz;
  }
  double *kp = a.part + (size_t)a.chunks * a.tiles;
  for (int c = 0; c < 4; ++c) {
    const double v = block_sum<kBlock / 64>(s[c], red);
    if (threadIdx.x == 0) kp[(size_t)c * a.tiles + blockIdx.x] = v;
  }
}

constexpr int kFinish = 1024;

// One result per workgroup.
__global__ __launch_bounds__(kFinish) void f64_energy_finish(
    const double *part, int tiles, int chunks, double G, double *out) {
  __shared__ double red[kFinish / 64];
  const int c = blockIdx.x; // K, W, Px, Py, Pz
  const size_t pots = (size_t)chunks * tiles;
  const double *p = part;
  size_t count = pots;
  if (c != 1) {
    p += pots + (size_t)(c == 0 ? 0 : c - 1) * tiles;
    count = tiles;
  }
  double s = 0.0;
#pragma unroll 4
  for (size_t b = threadIdx.x; b < count; b += kFinish) s += p[b];
  const double r = block_sum<kFinish / 64>(s, red);
  if (threadIdx.x == 0) out[c] = c == 1 ? -G * r : r;
}

} // namespace
} // namespace nb

using namespace nb;

extern "C" {

int nb_forces_f64_dev(const nb_params *p, const nb_vec3 *pos,
                      const int32_t *idx, size_t m, double *fx, double *fy,
                      double *fz, size_t n, void *stream) {
  if (!p || !pos) return set_error(NB_ERR_INVALID_ARG, "NULL argument");
  if (n > ((size_t)1 << 28) || m > ((size_t)1 << 28))
    return set_error(NB_ERR_INVALID_ARG, "size exceeds 2^28");
  if (m == 0) return NB_OK;
  if (n == 0) return set_error(NB_ERR_INVALID_ARG, "targets need sources");
  if (!pos->x || !pos->y || !pos->z || !idx || !fx || !fy || !fz)
    return set_error(NB_ERR_INVALID_ARG, "device pointer is NULL");
  // Enough source chunks that the grid holds several workgroups per CU, of
  // at least 32 sources each (a workgroup's fixed cost is about that).
  const int tblocks = (int)((m + kBlock - 1) / kBlock);
  int chunks = std::max(1, std::min(1024 / tblocks, (int)((n + 31) / 32)));
  ForceArgs a;
  a.px = pos->x;
  a.py = pos->y;
  a.pz = pos->z;
  a.idx = idx;
  a.m = (int)m;
  a.n = (int)n;
  a.chunk = (int)(((n + chunks - 1) / chunks + 31) / 32 * 32);
  chunks = (int)((n + a.chunk - 1) / a.chunk);
  a.eps = (double)p->dist_eps;
  hipStream_t s = static_cast<hipStream_t>(stream);
  ScratchLease part; // held until both launches are enqueued
  int st = acquire_scratch(sizeof(double) * 3 * m * (size_t)chunks, s, part);
  if (st) return st;
  a.part = reinterpret_cast<double *>(part.get());
  void *args[] = {&a};
  st = hip_check(hipLaunchKernel(reinterpret_cast<const void *>(f64_force_partial),
                                 dim3(tblocks, chunks), dim3(kBlock), args, 0, s),
                 "fp64 force launch");
  if (st) return st;
  hipLaunchKernelGGL(f64_force_finish,
                     dim3((int)((m + kFinTargets - 1) / kFinTargets), 3),
                     dim3(kBlock), 0, s,
                     a.part, a.m, chunks, fx, fy, fz);
  return hip_check(hipGetLastError(), "fp64 force finish launch");
}

int nb_energy_momentum_dev(const nb_params *p, const nb_vec3 *pos,
                           const nb_vec3 *vel, size_t n, double *out,
                           void *stream) {
  if (!p || !pos || !vel || !out)
    return set_error(NB_ERR_INVALID_ARG, "NULL argument");
  if (n > ((size_t)1 << 28)) return set_error(NB_ERR_INVALID_ARG, "n exceeds 2^28");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (n == 0) {
    hipLaunchKernelGGL(f64_energy_finish, dim3(5), dim3(kFinish), 0, s,
                       static_cast<const double *>(nullptr), 0, 0, 0.0, out);
    return hip_check(hipGetLastError(), "energy finish launch");
  }
  if (!pos->x || !pos->y || !pos->z || !vel->x || !vel->y || !vel->z)
    return set_error(NB_ERR_INVALID_ARG, "device pointer is NULL");
  // At 65536: 2048 / 8192 / 16384 / 32768 workgroups 2018 / 1250 / 1232 / 1235
  // us, at 50021 959 / 654 / 627 / 622, at 16384 170 / 159 / 164 / 165.
  // About 16384 workgroups, half of them below the diagonal and empty, of at
  // least 32 sources each; past 2^22 particles one chunk, longest tiles first.
  const int tiles = (int)((n + kETile - 1) / kETile);
  int chunks = std::max(1, std::min(16384 / tiles, (int)((n + 31) / 32)));
  const int chunk = (int)(((n + chunks - 1) / chunks + 31) / 32 * 32);
  chunks = (int)((n + chunk - 1) / chunk);
  EnergyArgs a;
  a.px = pos->x;
  a.py = pos->y;
  a.pz = pos->z;
  a.vx = vel->x;
  a.vy = vel->y;
  a.vz = vel->z;
  a.n = (int)n;
  a.chunk = chunk;
  a.tiles = tiles;
  a.chunks = chunks;
  a.eps = (double)p->dist_eps;
  ScratchLease part; // held until both launches are enqueued
  int st = acquire_scratch(sizeof(double) * (size_t)(chunks + 4) * tiles, s,
                           part);
  if (st) return st;
  a.part = reinterpret_cast<double *>(part.get());
  void *args[] = {&a};
  st = hip_check(hipLaunchKernel(reinterpret_cast<const void *>(f64_energy_partial),
                                 dim3(tiles, chunks), dim3(kBlock), args, 0,
                                 s),
                 "energy launch");
  if (st) return st;
  hipLaunchKernelGGL(f64_energy_finish, dim3(5), dim3(kFinish), 0, s,
                     static_cast<const double *>(a.part), tiles, chunks,
                     (double)p->G, out);
  return hip_check(hipGetLastError(), "energy finish launch");
}

} // extern "C"
