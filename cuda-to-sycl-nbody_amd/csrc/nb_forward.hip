// Forward all-pairs gravity step for gfx950 (MI355X).
//
// Semantics follow particle_interaction<BRANCH|PREDICATED>
// (src/simulator.cu:186-229):
//   F_i = sum_{j != i} r_ij * rsqrt(d^3),  r_ij = x_j - x_i,  d = |r_ij|^2 + eps
//   v_i <- v_i * damping;  v_i <- v_i + (F_i * dt) * G;  x'_i = x_i + v_i * dt
//
// Below 4096 particles one launch does the step (fwd_small_kernel); the
// symmetric shapes above are in nb_sym.hip.  The target-sharded shapes:
// Mapping (one workgroup = BLOCK threads x U targets):
//   * target i's position and force accumulator live in VGPRs, U per thread
//     (i = base + k * BLOCK + lane, so global loads/stores stay coalesced);
//   * sources stream through LDS tiles of TILE particles (nb_pairs.hpp:
//     accumulate_sources), read back as wave-uniform b128 broadcasts;
//   * optional source split (grid.y = S chunks) writes partial forces and a
//     second kernel sums the S partials in chunk order and integrates.
// The pair arithmetic (11 VALU + v_rsq_f32 per interaction) is in
// nb_pairs.hpp.  No matrix cores: the pair loop is not a dense contraction.
//
// Build with -ffp-contract=off: the integrator must round each product and
// sum separately, as written in the reference.

#include "nb_pairs.hpp"
#include "nb_small.hpp"


namespace nb {
namespace {

struct FwdArgs {
  const float *px, *py, *pz;
  float *vx, *vy, *vz;
  float *nx, *ny, *nz;
  float *part; // [split][3][n] partial forces when split > 1
  int n;
  int jchunk; // sources per grid.y chunk (a multiple of the tile length)
  int split;
  StepConsts c;
};

template <int BLOCK, int U, int TILE, int MODE, bool SPLIT>
__global__ __launch_bounds__(BLOCK) void fwd_kernel(FwdArgs a) {
  __shared__ SourceTile<TILE> sm;
  const int n = a.n;
  Targets<U, MODE> T;
  T.load(a.px, a.py, a.pz, blockIdx.x * (BLOCK * U), BLOCK, threadIdx.x, n);

  int jbeg = 0, jend = n;
  if constexpr (SPLIT) {
    jbeg = blockIdx.y * a.jchunk;
    jend = min(jbeg + a.jchunk, n);
  }
  accumulate_sources<BLOCK, TILE>(sm, T, a.px, a.py, a.pz, jbeg, jend,
                                  a.c.eps);

#pragma unroll
  for (int k = 0; k < U; ++k) {
    const int i = T.idx[k];
    if (i >= n) continue;
    float fx, fy, fz;
    T.force(k, fx, fy, fz);
    if constexpr (SPLIT) {
      const size_t s = blockIdx.y;
      a.part[(s * 3 + 0) * n + i] = fx;
      a.part[(s * 3 + 1) * n + i] = fy;
      a.part[(s * 3 + 2) * n + i] = fz;
    } else {
      integrate_ref(a.c, i, fx, fy, fz, a.px, a.py, a.pz, a.vx, a.vy, a.vz,
                    a.nx, a.ny, a.nz);
    }
  }
}

// Sums the split partial forces in chunk order and integrates.
template <bool KAHAN>
__global__ __launch_bounds__(256) void fwd_finalize(FwdArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  const size_t n = a.n;
  float f[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float s = 0.0f, comp = 0.0f;
    for (int k = 0; k < a.split; ++k) {
      const float v = a.part[(k * 3 + c) * n + i];
      if constexpr (KAHAN) {
        const float y = v - comp;
        const float t = s + y;
        comp = (t - s) - y;
        s = t;
      } else {
        s = s + v;
      }
    }
    f[c] = s;
  }
  integrate_ref(a.c, i, f[0], f[1], f[2], a.px, a.py, a.pz, a.vx, a.vy, a.vz,
                a.nx, a.ny, a.nz);
}

// ---- one launch for small systems -----------------------------------------
//
// Below a few thousand particles a step is latency: two launches, a source
// loop with few waves, a second trip through memory for the partial sums.
// Here a workgroup of 16 waves owns 4 * U targets and all their sources: each
// row of 16 lanes holds U targets, the 16 waves x 16 lanes stride through the
// sources in batches of four loads (the next batch is in flight during the
// pairs), four DPP adds sum a row, LDS brings the 16 waves' sums together, and
// the lanes that integrate have loaded their particles at the start.
// Device time at n = 1000 3.4 us, 4000 8.9 (split shapes and a second kernel:
// 23.8, 24.8); the launch and two dependent trips to L2 are about 3 of it.

template <int U, int MODE>
__global__ __launch_bounds__(kSmallBlock) void fwd_small_kernel(FwdArgs a) {
  constexpr bool KAHAN = MODE == MODE_KAHAN || MODE == MODE_KAHAN_SKIP;
  constexpr int NT = 4 * U;                  // targets per workgroup
  constexpr int WAVES = kSmallBlock / 64;
  constexpr int NV = KAHAN ? 6 : 3;
  static_assert(WAVES == kSmallLanes, "one lane of a row per wave's sum");
  __shared__ float sums[NV][NT][WAVES];
  const int n = a.n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane >> 4, sl = lane & 15;
  const int first = blockIdx.x * NT;

  // lane 0 of row r (of the workgroup) integrates target first + r
  const int fin = threadIdx.x >> 4;
  const bool owner = sl == 0 && fin < NT && first + fin < n;
  Particle own = {};
  if (owner)
    own = load_particle(first + fin, a.px, a.py, a.pz, a.vx, a.vy, a.vz);

  Targets<U, MODE> T;
  T.load(a.px, a.py, a.pz, first + row * U, 1, 0, n);

  const int s0 = wave * kSmallLanes + sl;
  constexpr int B = kSmallBatch, PASS = kSmallStride * B;
  float X[B], Y[B], Z[B];
  auto fetch = [&](int b) {
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int j = min(b + q * kSmallStride + s0, n - 1);
      X[q] = a.px[j];
      Y[q] = a.py[j];
      Z[q] = a.pz[j];
    }
  };
  fetch(0);
  for (int b = 0; b < n; b += PASS) {
    float x[B], y[B], z[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      x[q] = X[q];
      y[q] = Y[q];
      z[q] = Z[q];
    }
    if (b + PASS < n) fetch(b + PASS);
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int j = b + q * kSmallStride + s0;
      if (j < n) T.one(x[q], y[q], z[q], j, a.c.eps);
    }
  }

#pragma unroll
  for (int k = 0; k < U; ++k) {
    row_sum<KAHAN>(T.ax[k], T.cx[k]);
    row_sum<KAHAN>(T.ay[k], T.cy[k]);
    row_sum<KAHAN>(T.az[k], T.cz[k]);
    if (sl == 0) {
      sums[0][row * U + k][wave] = T.ax[k];
      sums[1][row * U + k][wave] = T.ay[k];
      sums[2][row * U + k][wave] = T.az[k];
      if constexpr (KAHAN) {
        sums[3][row * U + k][wave] = T.cx[k];
        sums[4][row * U + k][wave] = T.cy[k];
        sums[5][row * U + k][wave] = T.cz[k];
      }
    }
  }
  __syncthreads();
  if (wave >= U) return; // NT rows of 16 lanes are U waves
  float f[3], c[3] = {};
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    f[m] = sums[m][fin][sl];
    if constexpr (KAHAN) c[m] = sums[3 + m][fin][sl];
    row_sum<KAHAN>(f[m], c[m]);
    if constexpr (KAHAN) f[m] = f[m] - c[m];
  }
  if (owner)
    integrate_loaded(a.c, first + fin, own, f[0], f[1], f[2], a.vx, a.vy, a.vz,
                     a.nx, a.ny, a.nz);
}

using KernelFn = void (*)(FwdArgs);

template <int BLOCK, int U, int TILE>
KernelFn shape_kernel(int mode, bool split) {
#define NB_MODE_CASE(M)                                                        \
  case M:                                                                      \
    return split ? fwd_kernel<BLOCK, U, TILE, M, true>                         \
                 : fwd_kernel<BLOCK, U, TILE, M, false>;
  switch (mode) {
    NB_MODE_CASE(MODE_PLAIN)
    NB_MODE_CASE(MODE_PLAIN_SKIP)
    NB_MODE_CASE(MODE_KAHAN)
    NB_MODE_CASE(MODE_KAHAN_SKIP)
    NB_MODE_CASE(MODE_PREDICATED)
  default:
    return nullptr;
  }
#undef NB_MODE_CASE
}

template <int U>
KernelFn small_kernel(int mode) {
  switch (mode) {
  case MODE_PLAIN: return fwd_small_kernel<U, MODE_PLAIN>;
  case MODE_PLAIN_SKIP: return fwd_small_kernel<U, MODE_PLAIN_SKIP>;
  case MODE_KAHAN: return fwd_small_kernel<U, MODE_KAHAN>;
  case MODE_KAHAN_SKIP: return fwd_small_kernel<U, MODE_KAHAN_SKIP>;
  case MODE_PREDICATED: return fwd_small_kernel<U, MODE_PREDICATED>;
  default: return nullptr;
  }
}

struct ShapeEntry {
  int block, unroll, tile;
  KernelFn (*get)(int, bool);
};

const ShapeEntry kShapes[] = {
    {256, 1, 1024, shape_kernel<256, 1, 1024>},
    {256, 2, 1024, shape_kernel<256, 2, 1024>},
    {256, 4, 1024, shape_kernel<256, 4, 1024>},
    {128, 1, 512, shape_kernel<128, 1, 512>},
    {128, 2, 512, shape_kernel<128, 2, 512>},
    {512, 1, 2048, shape_kernel<512, 1, 2048>},
    {512, 2, 2048, shape_kernel<512, 2, 2048>},
};

// Compiled launch shapes: {block, unroll, tile, split[, scheme]}.  Index 0
// must stay the unsplit 256 x 1 shape (a valid choice for every n).  The
// symmetric shapes (nb_sym.hip) are {256, u, super-tile, super-tiles per work
// item} with super-tiles of 256 u: a wave holds rows of 512, 8 per lane, in
// workgroups of 256 threads (512 with u = 8).  Tile pairs {256, 2, 128, 1} run
// rows of 128 below 9728 particles (512 threads below 3328) and of 256, 4 per
// lane, from there, {256, 4, 256, 1} always the latter.
const FwdConfig kConfigs[] = {
    {256, 1, 1024, 1}, {256, 1, 1024, 2}, {256, 1, 1024, 4},
    {256, 1, 1024, 8}, {256, 2, 1024, 1}, {256, 2, 1024, 2},
    {256, 2, 1024, 4}, {256, 2, 1024, 8}, {256, 4, 1024, 1},
    {256, 4, 1024, 2}, {256, 4, 1024, 4}, {256, 4, 1024, 8},
    {128, 1, 512, 1},  {128, 1, 512, 2},  {128, 1, 512, 4},
    {128, 2, 512, 2},  {128, 2, 512, 4},  {512, 1, 2048, 1},
    {512, 1, 2048, 2}, {512, 2, 2048, 1}, {512, 2, 2048, 2},
    {512, 2, 2048, 4},
    {256, 8, 2048, 1, SCHEME_SYMMETRIC}, {256, 8, 2048, 2, SCHEME_SYMMETRIC},
    {256, 8, 2048, 4, SCHEME_SYMMETRIC}, {256, 4, 1024, 1, SCHEME_SYMMETRIC},
    {256, 4, 1024, 2, SCHEME_SYMMETRIC}, {256, 4, 1024, 4, SCHEME_SYMMETRIC},
    {256, 1, 1024, 16}, {256, 2, 1024, 16}, {128, 1, 512, 8},
    {128, 1, 512, 16},
    {256, 4, 256, 1, SCHEME_SYMMETRIC_TILES},
    {256, 2, 128, 1, SCHEME_SYMMETRIC_TILES},
    {256, 2, 512, 1, SCHEME_SYMMETRIC}, {256, 2, 512, 2, SCHEME_SYMMETRIC},
    {256, 2, 512, 4, SCHEME_SYMMETRIC},
    {256, 2, 128, 2, SCHEME_SYMMETRIC_TILES}, // tile pairs, rows of 128 at every n
    {kSmallBlock, 1, 1024, 1},                // one launch (fwd_small_kernel)
};
constexpr int kNumConfigs = sizeof(kConfigs) / sizeof(kConfigs[0]);

KernelFn find_kernel(const FwdConfig &c, int mode) {
  for (const ShapeEntry &s : kShapes)
    if (s.block == c.block && s.unroll == c.unroll && s.tile == c.tile)
      return s.get(mode, c.split > 1);
  return nullptr;
}

} // namespace

int forward_config_count() { return kNumConfigs; }

const FwdConfig &forward_config(int cfg) { return kConfigs[cfg]; }

int forward_default_config(size_t n, int mode) {
  // the symmetric shapes mask the self pairs where eps^3 is not a normal
  // float at the cost of the diagonal passes only: same choice
  if (mode == MODE_PLAIN_SKIP) mode = MODE_PLAIN;
  if (mode == MODE_KAHAN_SKIP) mode = MODE_KAHAN;
  // Measured on MI355X (disk ICs), us per step (device time), best others in
  // brackets.  Tile pairs: n = 4097 11.7 (target-sharded 40), 12000 35.4
  // (super-tiles of 512, 1 per item 49.0), 28000 137 (148), 32768 184 (188),
  // 36000 222 (215), 49000 397 (380).  Super-tiles win from about 34000; the
  // line is at 49152 because the allocation-free step's limits are counted for
  // the default shape: a super-tile default would have it accept sizes that it
  // refuses (26625 to 49151).  Super-tiles of 512, 1 per item: 50021 383 (tile
  // pairs 416, 1024 417), 52000 419 (448), 65536 647 (674 with 1024), 100000
  // 1471 (1468 with 2 per item, 1472 with 1024).  Of 1024: 131072 2488 (2509
  // with 512, 2605 with 2048), 200000 5849 (6001, 5895), 262144 10035 (2048:
  // 10150, with a quarter of the scratch's growth: the choice from there).  Past
  // 2^19 two super-tiles of 2048 per item need 25 % less scratch; past 2^20 four
  // per item keep the partials at 16 GB for 2^21 particles, and past 2^21 the
  // step runs in bands of source super-tiles with at most 8 GB of partials each
  // (the 4-per-lane shape with 4 per item is banded past 2^20).
  // Shapes 33 and 37 run the same kernels below 9728 particles; 37 stays the
  // name of the default below 6656.
  if (mode == MODE_PLAIN && n <= kSymBandedMaxParticles) {
    if (n > kSymMaxParticles) return 24; // 8 per lane, 4 per item (banded past 2^21)
    if (n > ((size_t)1 << 19)) return 23;  // symmetric, 8 per lane, 2 per item
    if (n >= ((size_t)1 << 18)) return 22; // symmetric, 8 per lane, 1 per item
    if (n >= ((size_t)1 << 17)) return 25; // symmetric, 4 per lane, 1 per item
    if (n >= 49152) return 34;             // symmetric, 2 per lane, 1 per item
    if (n >= 6656) return 33;              // symmetric tile pairs
    if (n >= 4096) return 37;              // the same
  }
  // Kahan, us per step: tile pairs: n = 4097 18.0 (best split target-sharded
  // 56), 5000 21.1 (one launch 33.5), 12000 64 (123), 32000 327 (575);
  // super-tiles of 512, 1 per item, and tile pairs: 32768 355 and 346, 36000
  // 416 and 418, 40960 506 and 529, 49000 724 and 750 (below 40960 the same
  // reason as above).  1 / 2 per item: 100000 2867 / 2862, 262144 19921 / 19648
  // (target-sharded 28993).  Above 2^18 four super-tiles per item run in bands
  // of source super-tiles (16 GB of (sum, compensation) partials per band).
  if (mode == MODE_KAHAN) {
    if (n > ((size_t)1 << 18) && n <= kSymBandedMaxParticles)
      return 36;               // symmetric, 2 per lane, 4 per item, banded
    if (n >= ((size_t)1 << 17) && n <= ((size_t)1 << 18))
      return 35;               // symmetric, 2 per lane, 2 per item
    if (n >= 40960 && n < ((size_t)1 << 17))
      return 34;               // symmetric, 2 per lane, 1 per item
    if (n >= 4096 && n < 40960)
      return 33;               // symmetric tile pairs
  }
  // One launch, plain / Kahan us (device time; split target-sharded plain,
  // then tile pairs plain / Kahan): n = 64 2.9 / 3.3 (10.8, 5.8 / 7.5), 1000
  // 3.3 / 4.2 (24.0, 7.4 / 9.4), 2000 4.6 / 6.7 (24.0, 7.8 / 9.9), 4000
  // 8.9 / 15.4 (24.9, 10.9 / 16.8); tile pairs from 4096.
  if (n < 4096) return 38;
  // Target-sharded, Gint/s: n = 4096: 128 x 1 split 8 629 (256 x 1 split 8
  // 480); 8192: 256 x 1 split 8 1746 (split 16 1629); 16384 .. 32768:
  // 256 x 1 split 16 2843 .. 3432 (split 8 2792 .. 3292); 65536: 256 x 4
  // split 8 3402 (256 x 1 split 8 3279).
  if (n >= (size_t)1 << 16) return 11; // 256 x 4, tile 1024, split 8
  if (n >= 12288) return 28;           // 256 x 1, tile 1024, split 16
  if (n >= 6144) return 3;             // 256 x 1, tile 1024, split 8
  return 30;                           // 128 x 1, tile 512, split 8
}

bool forward_one_launch(int cfg) { return kConfigs[cfg].block == kSmallBlock; }

// Every mode and every n below 4096, where one launch is the default: 24 us.
int forward_overlap_config() { return 30; } // 128 x 1, tile 512, split 8

int forward_launches(int cfg) {
  const FwdConfig &c = kConfigs[cfg];
  return c.scheme == SCHEME_TARGETS && c.split == 1 ? 1 : 2;
}

size_t forward_scratch_bytes(int cfg, size_t n, int mode) {
  const FwdConfig &c = kConfigs[cfg];
  if (c.scheme != SCHEME_TARGETS) // (sum, compensation) pairs for Kahan
  {
    const bool kahan = mode == MODE_KAHAN || mode == MODE_KAHAN_SKIP;
    return sym_scratch_bytes(c.unroll, c.split, n, kahan ? 6 : 3,
                             c.scheme == SCHEME_SYMMETRIC_TILES,
                             !kahan || c.unroll <= 4);
  }
  return c.split > 1 ? sizeof(float) * 3 * (size_t)c.split * n : 0;
}

size_t forward_noalloc_bytes(int cfg, size_t n, int mode) {
  const FwdConfig &c = kConfigs[cfg];
  if (c.scheme != SCHEME_SYMMETRIC_TILES || n > kSymTileMaxParticles)
    return forward_scratch_bytes(cfg, n, mode);
  const bool kahan = mode == MODE_KAHAN || mode == MODE_KAHAN_SKIP;
  const size_t P = c.tile, T = (n + P - 1) / P;
  return sizeof(float) * (kahan ? 6 : 3) * T * (T + 1) * P * c.split;
}

int launch_forward(const StepConsts &c, int mode, int cfg, const float *px,
                   const float *py, const float *pz, float *vx, float *vy,
                   float *vz, float *nx, float *ny, float *nz, int n,
                   float *scratch, hipStream_t stream) {
  if (cfg < 0 || cfg >= kNumConfigs)
    return set_error(NB_ERR_INVALID_ARG, "forward config out of range");
  if (n <= 0) return NB_OK;
  const FwdConfig &fc = kConfigs[cfg];
  if (fc.scheme != SCHEME_TARGETS) {
    // the kernels mask the self pairs themselves when eps^3 is not a normal
    // float (the SKIP modes)
    if (mode == MODE_PREDICATED)
      return set_error(NB_ERR_UNSUPPORTED,
                       "symmetric launch shapes take BRANCH only");
    const bool kahan = mode == MODE_KAHAN || mode == MODE_KAHAN_SKIP;
    if (kahan && fc.unroll > 4)
      return set_error(NB_ERR_UNSUPPORTED,
                       "symmetric Kahan shapes have 2 or 4 particles per lane");
    return launch_forward_sym(c, fc.unroll, fc.split,
                              fc.scheme == SCHEME_SYMMETRIC_TILES, kahan, px,
                              py, pz, vx, vy, vz, nx, ny, nz, n, scratch,
                              stream);
  }
  const bool small = fc.block == kSmallBlock;
  const int per_row = small ? small_targets(n) : 0;
  KernelFn fn = !small         ? find_kernel(fc, mode)
                : per_row == 1 ? small_kernel<1>(mode)
                : per_row == 2 ? small_kernel<2>(mode)
                               : small_kernel<4>(mode);
  if (!fn) return set_error(NB_ERR_UNSUPPORTED, "no kernel for this mode");
  if (fc.split > 1 && !scratch)
    return set_error(NB_ERR_INVALID_ARG, "split launch needs scratch");

  FwdArgs a;
  a.px = px;
  a.py = py;
  a.pz = pz;
  a.vx = vx;
  a.vy = vy;
  a.vz = vz;
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  a.part = scratch;
  a.n = n;
  a.split = fc.split;
  const int per_chunk = (n + fc.split - 1) / fc.split;
  a.jchunk = ((per_chunk + fc.tile - 1) / fc.tile) * fc.tile;
  a.c = c;

  const int targets = small ? 4 * per_row : fc.block * fc.unroll;
  dim3 grid((n + targets - 1) / targets, fc.split);
  dim3 block(fc.block);
  void *args[] = {&a};
  int st = hip_check(
      hipLaunchKernel(reinterpret_cast<const void *>(fn), grid, block, args,
                      0, stream),
      "forward launch");
  if (st) return st;
  if (fc.split > 1) {
    const bool kahan = (mode == MODE_KAHAN || mode == MODE_KAHAN_SKIP);
    KernelFn fin = kahan ? fwd_finalize<true> : fwd_finalize<false>;
    dim3 g2((n + 255) / 256);
    st = hip_check(hipLaunchKernel(reinterpret_cast<const void *>(fin), g2,
                                   dim3(256), args, 0, stream),
                   "forward finalize launch");
    if (st) return st;
  }
  return NB_OK;
}

} // namespace nb
