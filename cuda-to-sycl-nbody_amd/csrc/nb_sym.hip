// Symmetric all-pairs kernels for gfx950 (MI355X): each pair term is
// evaluated once and applied to both particles of the pair.
//
// Two pair rules share one decomposition:
//   ForceRule    the forward step, particle_interaction<BRANCH>
//                (src/simulator.cu:186-229):
//                  F_i = sum_{j != i} r_ij K_ij,  r_ij = x_j - x_i,
//                  K = rsqrt(d^3),  d = |r|^2 + eps  (nb_pairs.hpp arithmetic);
//   AdjointRule  the reverse-mode step of the same integrator (nb_adjoint.hip
//                derives it): A_k = sum_j K (h + t3 r),  h = g_j - g_k,
//                t3 = -3 (r . h) / d, optionally fused with the forward F.
// Both pair terms are odd under exchanging the two particles (r -> -r,
// h -> -h, d, K, t3 unchanged).  The reaction on particle j is accumulated
// negated, S' = fma(u, K, S'), which is bit for bit -fma(-u, K, S) (rounding
// is symmetric under negation), and subtracted in the finalize: particle j
// receives exactly the negative of the term added to particle i.  Only the
// order in which each particle's terms are summed differs from the
// target-sharded kernels.
//
// Particles are grouped in super-tiles of ST; a work item is one workgroup (4
// or 8 waves) and a chunk of one row of the super-tile pair triangle: super-tile
// GA against super-tiles GB in [GB0, GB1), GB >= GA.  Each item writes the
// targets' sums over its chunk as one row partial and, per pair with GB > GA,
// the (negated) reaction sums of GB's particles.  A finalize kernel sums, per
// particle, its row partials in chunk order, then subtracts the reaction
// partials of its column in GA order, and applies the rule's epilogue.  The
// order is fixed: results are deterministic.
// Inside an item a wave holds all targets of one row of GA (64 U, U = 8, 4 or
// 2 per lane) and meets GB in sets of 64 sources; a set's reaction sums rotate
// one lane down the wave after each step (meet_sources).
// The super-tile pairs of many independent systems also run on one
// persistent queue (sym_batch_kernel).
// Padding (index >= n): ForceRule puts padding particles at 1e30 in every
// coordinate, so any pair with a real particle has |r|^2 = +inf,
// rsqrt(inf) = 0 and r * 0 = 0 (exact zeros, no mask; a pair of two padding
// particles only touches padding sums).  AdjointRule masks K and t3 of pairs
// with a padding particle in the last, partial set of sources (a product
// r . h of a far padding particle could overflow).
// Self pairs: with dist_eps^3 a normal float the self term is exactly +0
// (r = 0, finite K); otherwise (eps = 0 or tiny) the passes over the
// super-tile's own sets, the only ones holding self pairs, mask them as the
// reference's `continue` skips them.
//
// Per pair term (two interactions): forward 14 VALU + v_rsq_f32 + 3/U
// reaction moves through the LDS crossbar (ds_bpermute, no VALU slot);
// adjoint 25 VALU + v_rsq_f32 (K and 1/d from rsqrt(d)) + 3/U moves; fused
// adjoint 33 VALU + v_rsq_f32 (K as the forward rule forms it, 1/d = K^2 d^2)
// + 6/U moves; Kahan sums 32 VALU + v_rsq_f32 + 6/U moves.  The
// target-sharded kernels spend 11 (forward) and 22 (adjoint) VALU per
// interaction.
//
// Build with -ffp-contract=off (explicit fmaf only).

#include "nb_pair_block.hpp"
#include "nb_pairs.hpp"
#include "nb_small.hpp"

#include <vector>

namespace nb {
namespace {

constexpr float kFar = 1.0e30f;  // coordinate of ForceRule padding particles

// Lane l receives lane (l + 1) mod 64's value: ds_bpermute_b32 through the LDS
// crossbar (no LDS memory).  It takes no VALU issue slot; a DPP move
// (wave_rol:1) costs 10-14 SIMD cycles of VALU time inside the pair loop's mix
// (measured with probe/issue_rates.hip), while the permute's latency is hidden
// (each sum is rotated as soon as it is complete and read again only in the
// next step).
__device__ __forceinline__ float lds_rol1(float v) {
  const int lane =
      (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  return __builtin_bit_cast(
      float, __builtin_amdgcn_ds_bpermute(((lane + 1) & 63) << 2,
                                          __builtin_bit_cast(int, v)));
}

// sum_{l=1..m} ceil(l / L): work items of the rows of lengths 1..m.
__host__ __device__ inline long long items_upto(int m, int L) {
  const int q = m / L, r = m - q * L; // (a 64-bit division is 150 instructions)
  return (long long)L * q * (q + 1) / 2 + (long long)r * (q + 1);
}

// First work item (= row-partial slot) of row ga.
__host__ __device__ inline long long row_first(int ga, int ts, int L) {
  if (L == 1) // no 64-bit division in the shapes of one super-tile per item
    return (long long)ga * ts - (long long)ga * (ga - 1) / 2;
  return items_upto(ts, L) - items_upto(ts - ga, L);
}

// Reaction-partial slot of super-tile pair (ga, gb), ga < gb.
__host__ __device__ inline long long pair_slot(int ga, int gb, int ts) {
  return (long long)ga * ts - (long long)ga * (ga + 1) / 2 + (gb - ga - 1);
}

__host__ __device__ inline long long tri_slot(int ga, int gb, int ts) {
  // row-major index of (ga, gb), ga <= gb, in the upper triangle with diagonal
  return (long long)ga * ts - (long long)ga * (ga - 1) / 2 + (gb - ga);
}

struct SymArgs {
  const float *px, *py, *pz;
  const float *lxn[3], *lvn[3]; // adjoint: cotangents of the step's outputs
  float *lx[3], *lv[3];         // adjoint: cotangents of its inputs
  float *vx, *vy, *vz;          // velocity in/out (forward, fused adjoint)
  float *nx, *ny, *nz;          // next positions (forward, fused adjoint)
  float *fpart;                 // [items][ACC][ST] row partials
  float *spart;                 // [ts (ts - 1) / 2][ACC][ST] reaction partials
  int n;
  int ts;    // super-tiles
  int chunk; // super-tiles per work item
  StepConsts c;
  // banded launches (sym_band_*): source super-tiles [b0, b0 + bw) of this
  // band, first band flag, running per-particle sums [3][n]
  int b0, bw, first;
  float *acc3;
};

// Finalize arithmetic of the plain rules: row partials are added, the
// negated reaction partials subtracted, in the order the caller visits them.
// fetch reads one partial ([ACC] floats, stride apart); add_v / sub_v fold it
// into the running sums.  merge / unmerge add and subtract running sums inside
// a work item, where Kahan sums keep both sides' compensation.
template <int ACC>
struct PlainPartials {
  static __device__ __forceinline__ void fetch(float (&v)[ACC], const float *p,
                                               int stride) {
#pragma unroll
    for (int e = 0; e < ACC; ++e) v[e] = p[e * stride];
  }
  static __device__ __forceinline__ void add_v(float (&f)[ACC],
                                               const float (&v)[ACC]) {
#pragma unroll
    for (int e = 0; e < ACC; ++e) f[e] = f[e] + v[e];
  }
  static __device__ __forceinline__ void sub_v(float (&f)[ACC],
                                               const float (&v)[ACC]) {
#pragma unroll
    for (int e = 0; e < ACC; ++e) f[e] = f[e] - v[e];
  }
  static __device__ __forceinline__ void merge(float (&f)[ACC],
                                               const float (&v)[ACC]) {
    add_v(f, v);
  }
  static __device__ __forceinline__ void unmerge(float (&f)[ACC],
                                                 const float (&v)[ACC]) {
    sub_v(f, v);
  }
};

struct ForceRule : PlainPartials<3> {
  static constexpr int SRC = 3; // x, y, z
  static constexpr int ACC = 3; // F
  static constexpr bool MASKED_TAIL = false;
  static constexpr bool ROWS4 = true; // has shapes with 8 per lane

  template <int U>
  static __device__ __forceinline__ void block(const float (&s)[SRC],
                                               const float (&t)[U][SRC],
                                               float (&a)[U][ACC],
                                               float (&rs)[ACC], float eps) {
    force_block<U>(s, t, a, rs, eps);
  }

  static __device__ __forceinline__ void load(const SymArgs &a, int j,
                                              float (&v)[SRC]) {
    const bool ok = j < a.n;
    v[0] = ok ? a.px[j] : kFar;
    v[1] = ok ? a.py[j] : kFar;
    v[2] = ok ? a.pz[j] : kFar;
  }

  // Source s on target t: a += r K and rs += r K: rs holds the negated
  // reaction sum of the source (the finalize subtracts it), which keeps every
  // accumulation a two-operand v_fmac_f32.  The term of a pair that is not
  // `valid` is zero (the self pair when eps^3 is not a normal float, as the
  // reference's `continue` skips it; pairs with padding where a rule needs
  // it).  block() is the same without the mask, for U targets.
  static __device__ __forceinline__ void
  pair_masked(const float (&s)[SRC], const float (&t)[SRC], float (&a)[ACC],
              float (&rs)[ACC], float eps, bool valid) {
    const float rx = s[0] - t[0];
    const float ry = s[1] - t[1];
    const float rz = s[2] - t[2];
    float d = __builtin_fmaf(rx, rx, eps);
    d = __builtin_fmaf(ry, ry, d);
    d = __builtin_fmaf(rz, rz, d);
    float K = __builtin_amdgcn_rsqf((d * d) * d);
    K = valid ? K : 0.0f;
    a[0] = __builtin_fmaf(rx, K, a[0]);
    a[1] = __builtin_fmaf(ry, K, a[1]);
    a[2] = __builtin_fmaf(rz, K, a[2]);
    rs[0] = __builtin_fmaf(rx, K, rs[0]);
    rs[1] = __builtin_fmaf(ry, K, rs[1]);
    rs[2] = __builtin_fmaf(rz, K, rs[2]);
  }

  using Own = Particle;
  static __device__ __forceinline__ Own own(const SymArgs &a, int i) {
    return load_particle(i, a.px, a.py, a.pz, a.vx, a.vy, a.vz);
  }
  static __device__ __forceinline__ void finish(const SymArgs &a, int i,
                                                const Own &p,
                                                const float (&f)[ACC]) {
    integrate_loaded(a.c, i, p, f[0], f[1], f[2], a.vx, a.vy, a.vz, a.nx, a.ny,
                     a.nz);
  }
};

// Kahan-compensated forward rule (NB_ACC_KAHAN): the target sums and the
// (negated) reaction sums each carry a running compensation c (kahan_add,
// nb_pairs.hpp: y = fma(r, K, -c), t = s + y, c = (t - s) - y, s = t; the
// sum is s - c).  A partial is (s_x, s_y, s_z, c_x, c_y, c_z); the finalize
// Kahan-adds the partials' values s - c.
struct KahanForceRule {
  static constexpr bool ROWS4 = false;
  static constexpr int SRC = 3;
  static constexpr int ACC = 6;

  template <int U>
  static __device__ __forceinline__ void block(const float (&s)[SRC],
                                               const float (&t)[U][SRC],
                                               float (&a)[U][ACC],
                                               float (&rs)[ACC], float eps) {
    kahan_block<U>(s, t, a, rs, eps);
  }

  static constexpr bool MASKED_TAIL = false;

  static __device__ __forceinline__ void load(const SymArgs &a, int j,
                                              float (&v)[SRC]) {
    ForceRule::load(a, j, v);
  }

  static __device__ __forceinline__ void
  pair_masked(const float (&s)[SRC], const float (&t)[SRC], float (&a)[ACC],
              float (&rs)[ACC], float eps, bool valid) {
    const float rx = s[0] - t[0];
    const float ry = s[1] - t[1];
    const float rz = s[2] - t[2];
    float d = __builtin_fmaf(rx, rx, eps);
    d = __builtin_fmaf(ry, ry, d);
    d = __builtin_fmaf(rz, rz, d);
    float K = __builtin_amdgcn_rsqf((d * d) * d);
    K = valid ? K : 0.0f; // as ForceRule
    kahan_add(rx, K, a[0], a[3]);
    kahan_add(ry, K, a[1], a[4]);
    kahan_add(rz, K, a[2], a[5]);
    kahan_add(rx, K, rs[0], rs[3]);
    kahan_add(ry, K, rs[1], rs[4]);
    kahan_add(rz, K, rs[2], rs[5]);
  }

  // f: running (sum, compensation) of each coordinate over the partials
  static __device__ __forceinline__ void kahan_value(float (&f)[ACC], int e,
                                                     float v) {
    const float y = v - f[3 + e];
    const float t = f[e] + y;
    f[3 + e] = (t - f[e]) - y;
    f[e] = t;
  }
  static __device__ __forceinline__ void fetch(float (&v)[ACC], const float *p,
                                               int stride) {
#pragma unroll
    for (int e = 0; e < ACC; ++e) v[e] = p[e * stride];
  }
  static __device__ __forceinline__ void add_v(float (&f)[ACC],
                                               const float (&v)[ACC]) {
#pragma unroll
    for (int e = 0; e < 3; ++e) kahan_value(f, e, v[e] - v[3 + e]);
  }
  static __device__ __forceinline__ void sub_v(float (&f)[ACC],
                                               const float (&v)[ACC]) {
#pragma unroll
    for (int e = 0; e < 3; ++e) kahan_value(f, e, v[3 + e] - v[e]);
  }
  // The waves' sums may cancel: rounding one to v - c first would leave an
  // error of the waves' size in the item's sum.
  static __device__ __forceinline__ void merge(float (&f)[ACC],
                                               const float (&v)[ACC]) {
#pragma unroll
    for (int e = 0; e < 3; ++e) meet(f[e], f[3 + e], v[e], v[3 + e]);
  }
  static __device__ __forceinline__ void unmerge(float (&f)[ACC],
                                                 const float (&v)[ACC]) {
#pragma unroll
    for (int e = 0; e < 3; ++e) meet(f[e], f[3 + e], -v[e], -v[3 + e]);
  }

  using Own = Particle;
  static __device__ __forceinline__ Own own(const SymArgs &a, int i) {
    return load_particle(i, a.px, a.py, a.pz, a.vx, a.vy, a.vz);
  }
  static __device__ __forceinline__ void finish(const SymArgs &a, int i,
                                                const Own &p,
                                                const float (&f)[ACC]) {
    integrate_loaded(a.c, i, p, f[0] - f[3], f[1] - f[4], f[2] - f[5], a.vx,
                     a.vy, a.vz, a.nx, a.ny, a.nz);
  }
};

template <bool FUSED>
struct AdjointRule : PlainPartials<FUSED ? 6 : 3> {
  static constexpr bool ROWS4 = true;
  static constexpr int SRC = 6; // x, y, z, g_x, g_y, g_z
  static constexpr int ACC = FUSED ? 6 : 3; // sum M (g_j - g_k) [, F]
  static constexpr bool MASKED_TAIL = true;

  template <int U>
  static __device__ __forceinline__ void block(const float (&s)[SRC],
                                               const float (&t)[U][SRC],
                                               float (&a)[U][ACC],
                                               float (&rs)[ACC], float eps) {
    if constexpr (FUSED) fused_block<U>(s, t, a, rs, eps);
    else adjoint_block<U>(s, t, a, rs, eps);
  }

  // g = lv' + dt lx' (the cotangent the pair sum is taken of)
  static __device__ __forceinline__ void load(const SymArgs &a, int j,
                                              float (&v)[SRC]) {
    if (j < a.n) {
      v[0] = a.px[j];
      v[1] = a.py[j];
      v[2] = a.pz[j];
#pragma unroll
      for (int c = 0; c < 3; ++c)
        v[3 + c] = __builtin_fmaf(a.c.dt, a.lxn[c][j], a.lvn[c][j]);
    } else {
#pragma unroll
      for (int c = 0; c < SRC; ++c) v[c] = 0.0f;
    }
  }

  static __device__ __forceinline__ void
  pair_masked(const float (&s)[SRC], const float (&t)[SRC], float (&a)[ACC],
              float (&rs)[ACC], float eps, bool valid) {
    const float rx = s[0] - t[0];
    const float ry = s[1] - t[1];
    const float rz = s[2] - t[2];
    float d = __builtin_fmaf(rx, rx, eps);
    d = __builtin_fmaf(ry, ry, d);
    d = __builtin_fmaf(rz, rz, d);
    float K, q;
    if constexpr (FUSED) { // K exactly as the forward kernels form it
      // 1/d = K^2 d^2: two multiplies instead of v_rcp_f32 (2 % faster at
      // N = 262144, 8 % with tile pairs at N = 16384)
      const float dd = d * d;
      K = __builtin_amdgcn_rsqf(dd * d);
      q = (K * K) * dd;
    } else { // one transcendental (8 % faster): s = d^-1/2, q = s^2, K = s^3
      const float sr = __builtin_amdgcn_rsqf(d);
      q = sr * sr;
      K = q * sr;
    }
    const float hx = s[3] - t[3];
    const float hy = s[4] - t[4];
    const float hz = s[5] - t[5];
    float rh = rx * hx;
    rh = __builtin_fmaf(ry, hy, rh);
    rh = __builtin_fmaf(rz, hz, rh);
    float t3 = (rh * q) * -3.0f;
    K = valid ? K : 0.0f;
    t3 = valid ? t3 : 0.0f;
    const float ux = __builtin_fmaf(t3, rx, hx);
    const float uy = __builtin_fmaf(t3, ry, hy);
    const float uz = __builtin_fmaf(t3, rz, hz);
    a[0] = __builtin_fmaf(K, ux, a[0]);
    a[1] = __builtin_fmaf(K, uy, a[1]);
    a[2] = __builtin_fmaf(K, uz, a[2]);
    rs[0] = __builtin_fmaf(K, ux, rs[0]); // negated, as in ForceRule
    rs[1] = __builtin_fmaf(K, uy, rs[1]);
    rs[2] = __builtin_fmaf(K, uz, rs[2]);
    if constexpr (FUSED) {
      a[3] = __builtin_fmaf(rx, K, a[3]);
      a[4] = __builtin_fmaf(ry, K, a[4]);
      a[5] = __builtin_fmaf(rz, K, a[5]);
      rs[3] = __builtin_fmaf(rx, K, rs[3]);
      rs[4] = __builtin_fmaf(ry, K, rs[4]);
      rs[5] = __builtin_fmaf(rz, K, rs[5]);
    }
  }

  // lx = lx' + dt G sum,  lv = damping g; fused: the forward step too.
  struct Own {
    float lx[3], lv[3];
    Particle p; // fused only
  };
  static __device__ __forceinline__ Own own(const SymArgs &a, int i) {
    Own o;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      o.lx[c] = a.lxn[c][i];
      o.lv[c] = a.lvn[c][i];
    }
    if constexpr (FUSED)
      o.p = load_particle(i, a.px, a.py, a.pz, a.vx, a.vy, a.vz);
    return o;
  }
  static __device__ __forceinline__ void finish(const SymArgs &a, int i,
                                                const Own &o,
                                                const float (&f)[ACC]) {
    const float cG = a.c.dt * a.c.G;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float g = __builtin_fmaf(a.c.dt, o.lx[c], o.lv[c]);
      a.lx[c][i] = __builtin_fmaf(cG, f[c], o.lx[c]);
      a.lv[c][i] = a.c.damping * g;
    }
    if constexpr (FUSED)
      integrate_loaded(a.c, i, o.p, f[3], f[4], f[5], a.vx, a.vy, a.vz, a.nx,
                       a.ny, a.nz);
  }
};

// f += partial(0), partial(1), ... in that order (SUB: f -= ...), with
// kInFlight partials loaded ahead of the running sum: the loads do not
// depend on it, so a finalize thread waits about once per kInFlight
// partials instead of once per partial.  The order, and so the result, is
// that of the plain loop.
constexpr int kInFlight = 8;

template <class R, bool SUB, class At>
__device__ __forceinline__ void sum_partials(float (&f)[R::ACC], int count,
                                             At at, int stride) {
  int k = 0;
  for (; k + kInFlight <= count; k += kInFlight) {
    float v[kInFlight][R::ACC];
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) R::fetch(v[u], at(k + u), stride);
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      if constexpr (SUB) R::sub_v(f, v[u]);
      else R::add_v(f, v[u]);
    }
  }
  if (k < count) { // the last count - k < kInFlight partials, loaded together
    float v[kInFlight][R::ACC];
#pragma unroll
    for (int u = 0; u < kInFlight; ++u)
      if (k + u < count) R::fetch(v[u], at(k + u), stride);
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      if (k + u < count) {
        if constexpr (SUB) R::sub_v(f, v[u]);
        else R::add_v(f, v[u]);
      }
    }
  }
}

// A finalize workgroup of 256 threads serves 256 / RUNS particles: with
// RUNS > 1, wave group r sums run r of each particle's partial sequence (its
// row partials, then its negated reaction partials: `rows + reacs` partials
// cut into RUNS contiguous runs), and the first group adds the runs' sums in
// run order.  The order is fixed either way, so results are deterministic.
// RUNS = 4 pays where one thread per particle leaves most CUs idle (the
// tile-pair form: 5.3 vs 10.7 us at n = 12800; 8 and 16 runs made the whole
// step 0-1 % and 3-7 % slower at n = 4096 .. 40960); with enough particles to
// fill the chip one run per particle is faster (super-tile finalize at
// n = 262144: 82 vs 91 us).
template <class R, int RUNS, class RowAt, class ReacAt>
__device__ __forceinline__ void run_sum(float (&f)[R::ACC], int rows,
                                        int reacs, int run, RowAt row_at,
                                        ReacAt reac_at, int stride) {
  const int len = rows + reacs;
  const int k0 = run * len / RUNS, k1 = (run + 1) * len / RUNS;
#pragma unroll
  for (int e = 0; e < R::ACC; ++e) f[e] = 0.0f;
  if constexpr (RUNS == 1) { // many partials: no test inside a group of loads
    if (k0 < rows)
      sum_partials<R, false>(
          f, min(k1, rows) - k0, [&](int k) { return row_at(k0 + k); }, stride);
    const int r0 = max(k0, rows) - rows, r1 = k1 - rows;
    if (r1 > r0)
      sum_partials<R, true>(
          f, r1 - r0, [&](int k) { return reac_at(r0 + k); }, stride);
  } else { // few: rows and reactions in the same groups of loads, less code
#pragma unroll 1
    for (int k = k0; k < k1; k += kInFlight) {
      float v[kInFlight][R::ACC];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u)
        if (k + u < k1)
          R::fetch(v[u], k + u < rows ? row_at(k + u) : reac_at(k + u - rows),
                   stride);
#pragma unroll
      for (int u = 0; u < kInFlight; ++u)
        if (k + u < k1) {
          if (k + u < rows) R::add_v(f, v[u]);
          else R::sub_v(f, v[u]);
        }
    }
  }
}

// First group: f (run 0's sum) plus runs 1 .. RUNS-1 in order.  A run's
// running sum has the layout and value of a row partial (Kahan: value = sum
// - compensation), so it is added as one.  Called by every thread (barrier);
// returns true in the threads that hold the total.
template <class R, int RUNS>
__device__ __forceinline__ bool combine_runs(float (&f)[R::ACC],
                                             float (*red)[256]) {
  if constexpr (RUNS == 1) {
    return true;
  } else {
    constexpr int PW = 256 / RUNS;
    const int t = threadIdx.x;
#pragma unroll
    for (int e = 0; e < R::ACC; ++e) red[e][t] = f[e];
    __syncthreads();
    if (t >= PW) return false;
#pragma unroll
    for (int q = 1; q < RUNS; ++q) {
      float v[R::ACC];
#pragma unroll
      for (int e = 0; e < R::ACC; ++e) v[e] = red[e][t + q * PW];
      R::add_v(f, v);
    }
    return true;
  }
}

// ---- pair kernels: a wave holds a whole row ---------------------------------
//
// Super-tiles of ST = 64 U M particles: M rows of 64 U, U targets per lane.
// Each wave of the workgroup holds the same row of the super-tile GA (every
// wave all its targets) and takes its share of the source super-tile GB in
// sets of 64 sources, one source per lane and step.  Per step a lane reads
// one source (SRC floats) from LDS and rotates ACC reaction sums for U pair
// terms; no barrier inside a row.
//   * U = 8 or 4: wave w meets sets w, w + W, .. of GB;  U = 2: W / 2 waves
//     share a set, each its part of the 64 steps, and add their reaction sums
//     through LDS;
//   * at the end of a row the waves' target sums are added in a fixed tree,
//     (0 + 2) + (1 + 3);
//   * M = 1: the row meets every GB of the work item before that;  M > 1: the
//     rows of GA meet one GB in turn, and the reaction sums of a set, owned by
//     one wave, wait in LDS from row to row (one reaction partial per ST x ST
//     pairs, 1 / M of M = 1's).  M = 4 runs W = 8 waves per workgroup, the
//     others 4: half as long items, a shorter last round for the same
//     partials.
// The sources lie twice in LDS (128 floats per coordinate and wave), so that
// step s reads at lane + s with no wrap, its offset in the instruction.
//
// Why: with 2 targets x 2 sources per lane a step spends 6 permutes and 3
// LDS reads on 4 pair terms (forward; 12 and 3 with Kahan sums, 6 .. 12 and 6
// for the adjoint); with 8 x 1 it is 3 and 3 for 8.  In the pair loop alone,
// sustained at 4 waves per SIMD, SIMD cycles (at 2.4 GHz) per wave pair term
// 2 x 2 -> 8 x 1: forward 56 -> 47, adjoint 85 -> 72, fused 120 -> 94, Kahan
// 102 -> 89.  8 x 8 in four-wave passes with a barrier per pass: 50 (3 waves
// per SIMD, 48 KiB of LDS).
// W: waves per workgroup.  8 with M = 4; with U = 2, 8 where one wave per
// SIMD would be all there is (see kTileWide).
template <class R, int U, int M, int W_ = (M > 2 ? 8 : 4)>
struct RowShape {
  static_assert(U == 2 || U == 4 || U == 8, "targets per lane");
  static_assert(M == 1 || U == 8, "rows per super-tile");
  static constexpr int RT = 64 * U;                  // row
  static constexpr int ST = RT * M;                  // super-tile
  static constexpr int W = W_;
  static constexpr int SETS = ST / 64;               // source sets
  static constexpr int PARTS = U >= 4 ? 1 : W / SETS; // waves per set
  static constexpr int STEPS = 64 / PARTS;           // steps of a wave per set
  // LDS: the waves' sources, and in the same place (a barrier between) the
  // two buffers of the tree; then the reaction sums that wait or meet there
  static constexpr int SRC_FLOATS = W * R::SRC * 128;
  static constexpr int SUM_FLOATS = W / 2 * R::ACC * RT;
  static constexpr int REACT = PARTS == 1 && SUM_FLOATS > SRC_FLOATS
                                   ? SUM_FLOATS
                                   : SRC_FLOATS;
  static constexpr int REACT_FLOATS = PARTS > 1 ? W * R::ACC * 64
                                      : M > 1   ? R::ACC * ST
                                                : 0;
  static constexpr int LDS_FLOATS = REACT + REACT_FLOATS > SUM_FLOATS
                                        ? REACT + REACT_FLOATS
                                        : SUM_FLOATS;
};

// Orders the wave's own LDS writes before its later reads (other lanes read
// them): the hardware runs a wave's LDS operations in order, the fences keep
// the compiler from reordering them.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Steps [s0, s0 + STEPS) of the wave's targets t against the 64 sources at
// src ([SRC][128]): target sums into a, reaction sums of source (lane + s1)
// mod 64 into rs.  masked: sources at or past index `valid` of the set and,
// in the set of the wave's own targets self (-1: another set), the self pairs
// (step 0) contribute nothing.
template <class R, int U, int STEPS>
__device__ __forceinline__ void
row_pass(const float (&t)[U][R::SRC], float (&a)[U][R::ACC],
         float (&rs)[R::ACC], const float *src, int lane, int s0, float eps,
         bool masked, int self, int valid) {
  const float *p = src + lane + s0;
  if (!masked) {
#pragma unroll 4
    for (int s = 0; s < STEPS; ++s) {
      float sv[R::SRC];
#pragma unroll
      for (int e = 0; e < R::SRC; ++e) sv[e] = p[e * 128 + s];
      R::template block<U>(sv, t, a, rs, eps);
#pragma unroll
      for (int e = 0; e < R::ACC; ++e) rs[e] = lds_rol1(rs[e]);
    }
  } else {
#pragma unroll 1
    for (int s = 0; s < STEPS; ++s) {
      float sv[R::SRC];
#pragma unroll
      for (int e = 0; e < R::SRC; ++e) sv[e] = p[e * 128 + s];
      const bool vs = ((lane + s0 + s) & 63) < valid;
#pragma unroll
      for (int k = 0; k < U; ++k)
        R::pair_masked(sv, t[k], a[k], rs, eps,
                       vs && !(k == self && s0 + s == 0));
#pragma unroll
      for (int e = 0; e < R::ACC; ++e) rs[e] = lds_rol1(rs[e]);
    }
  }
}

// Row `row` of super-tile ga (targets ga * ST + row * RT ..) against source
// super-tiles [gb0, gb1), gb0 >= ga: the wave's target sums into sum, the
// (negated) reaction sums of gb > ga after the last row to sp_at(gb)
// ([ACC][ST]).  lds: LDS_FLOATS.  Called by every thread of the workgroup.
// On the diagonal (gb == ga) a row meets its own sets without reactions (each
// of their pairs twice) and, M > 1, those of the rows after it with; their
// reaction sums wait for those rows in LDS (add_waves subtracts them).
template <class R, class S, int U, int M, class SpAt>
__device__ __forceinline__ void meet_sources(float (&sum)[U][R::ACC],
                                             const SymArgs &a, float *lds,
                                             int ga, int row, int gb0, int gb1,
                                             SpAt sp_at) {
  constexpr int ST = S::ST;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int part = w % S::PARTS, first = w / S::PARTS;
  const int s0 = part * S::STEPS;
  float t[U][R::SRC];
#pragma unroll
  for (int k = 0; k < U; ++k) {
    R::load(a, ga * ST + row * S::RT + k * 64 + lane, t[k]);
#pragma unroll
    for (int e = 0; e < R::ACC; ++e) sum[k][e] = 0.0f;
  }
  float *src = lds + w * (R::SRC * 128);
  float *react = lds + S::REACT;
  const bool self_vanishes = self_term_vanishes(a.c.eps);
  float nxt[R::SRC]; // the next set's sources, in flight during a pass
  // the diagonal's sets before the row met it there already
  int gb = gb0, q = (M > 1 && gb0 == ga ? row * U : 0) + first;
  R::load(a, gb * ST + q * 64 + lane, nxt);
  while (gb < gb1) {
    wave_lds_fence();
#pragma unroll
    for (int e = 0; e < R::SRC; ++e) {
      src[e * 128 + lane] = nxt[e];
      src[e * 128 + 64 + lane] = nxt[e];
    }
    wave_lds_fence();
    const int g = gb, set = q;
    q += S::W / S::PARTS;
    if (q >= S::SETS) {
      q = first;
      ++gb;
    }
    if (gb < gb1) R::load(a, gb * ST + q * 64 + lane, nxt);

    const int left = a.n - (g * ST + set * 64); // sources before the padding
    bool masked = g == ga && !self_vanishes;
    if constexpr (R::MASKED_TAIL) masked = masked || left < 64;
    float *held = react + set * 64 + lane; // M > 1: this wave's, row to row
    float rs[R::ACC];
#pragma unroll
    for (int e = 0; e < R::ACC; ++e) rs[e] = 0.0f;
    // (a diagonal set's first visitor is row 0, but its own row's sums are
    // not kept)
    if (M > 1 && row > 0) R::fetch(rs, held, ST);
    if (left > 0) // the same for the waves that share a set
      row_pass<R, U, S::STEPS>(t, sum, rs, src, lane, s0, a.c.eps, masked,
                               g == ga ? set - row * U : -1, left);
    if (g == ga && (M == 1 || set < (row + 1) * U)) continue;
    if constexpr (S::PARTS == 1) {
      const bool out = M == 1 || (row == M - 1 && g > ga);
      float *sp = out ? sp_at(g) + set * 64 + lane : held;
#pragma unroll
      for (int e = 0; e < R::ACC; ++e) sp[e * ST] = rs[e];
    } else {
      // lane l holds the sums of source (l + s1) mod 64
      const int m = (lane + s0 + S::STEPS) & 63;
#pragma unroll
      for (int e = 0; e < R::ACC; ++e) react[(w * R::ACC + e) * 64 + m] = rs[e];
      __syncthreads();
      if (part == 0) {
        float f[R::ACC];
        R::fetch(f, react + w * R::ACC * 64 + lane, 64);
#pragma unroll
        for (int p = 1; p < S::PARTS; ++p) {
          float v[R::ACC];
          R::fetch(v, react + (w + p) * R::ACC * 64 + lane, 64);
          R::merge(f, v);
        }
        float *sp = sp_at(g) + set * 64 + lane;
#pragma unroll
        for (int e = 0; e < R::ACC; ++e) sp[e * ST] = f[e];
      }
      __syncthreads(); // read before the next pair overwrites it
    }
  }
}

// The W waves' target sums, halves added until two are left, to fp ([ACC][RT],
// one coordinate `stride` apart), added to what it holds with ADD.  Waves 0
// and 1 each finish half of the targets and subtract the row's reaction sums
// from its own super-tile (held: [ACC][stride]; nullptr: none).  Leaves the
// LDS free for reuse.
template <class R, int U, int W, bool ADD>
__device__ __forceinline__ void add_waves(float (&sum)[U][R::ACC], float *lds,
                                          const float *held, float *fp,
                                          int stride) {
  constexpr int RT = 64 * U;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // buffer b of the tree ([ACC][RT])
  auto buf = [&](int b) { return lds + b * (R::ACC * RT) + lane; };
  // (the scheduling barriers keep one target's values in flight, not all U:
  // registers here would cost the pair loop its waves)
  auto put = [&](float *p, int k0, int k1) {
#pragma unroll
    for (int k = 0; k < U; ++k)
      if (k >= k0 && k < k1)
#pragma unroll
        for (int e = 0; e < R::ACC; ++e) p[e * RT + k * 64] = sum[k][e];
  };
  auto take = [&](const float *p, int k0, int k1) {
#pragma unroll
    for (int k = 0; k < U; ++k)
      if (k >= k0 && k < k1) {
        float v[R::ACC];
        R::fetch(v, p + k * 64, RT);
        R::merge(sum[k], v);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  __syncthreads(); // every wave is done with its sources
#pragma unroll
  for (int h = W / 2; h >= 2; h >>= 1) {
    if (w >= h && w < 2 * h) put(buf(w & (h - 1)), 0, U);
    __syncthreads();
    if (w < h) take(buf(w & (h - 1)), 0, U);
    __syncthreads();
  }
  if (w == 0) put(buf(0), U / 2, U);
  if (w == 1) put(buf(1), 0, U / 2);
  __syncthreads();
  if (w == 0) take(buf(1), 0, U / 2);
  if (w == 1) take(buf(0), U / 2, U);
#pragma unroll
  for (int k = 0; k < U; ++k)
    if (w == (k < U / 2 ? 0 : 1)) {
      float *p = fp + k * 64 + lane;
      if (held) {
        float v[R::ACC];
        R::fetch(v, held + k * 64 + lane, stride);
        R::unmerge(sum[k], v);
      }
      if constexpr (ADD) {
        float v[R::ACC];
        R::fetch(v, p, stride);
        R::merge(v, sum[k]);
#pragma unroll
        for (int e = 0; e < R::ACC; ++e) p[e * stride] = v[e];
      } else {
#pragma unroll
        for (int e = 0; e < R::ACC; ++e) p[e * stride] = sum[k][e];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  __syncthreads();
}

// Work item: super-tile ga against source super-tiles [gb0, gb1), gb0 >= ga.
// Row partial ([ACC][ST]) to fp, reaction sums to sp_at(gb) ([ACC][ST]).
template <class R, class S, int U, int M, class SpAt>
__device__ __forceinline__ void row_item(const SymArgs &a, float *lds, int ga,
                                         int gb0, int gb1, float *fp,
                                         SpAt sp_at) {
  float sum[U][R::ACC];
  if constexpr (M == 1) {
    meet_sources<R, S, U, M>(sum, a, lds, ga, 0, gb0, gb1, sp_at);
    add_waves<R, U, S::W, false>(sum, lds, nullptr, fp, S::ST);
  } else {
#pragma unroll 1
    for (int gb = gb0; gb < gb1; ++gb)
#pragma unroll 1
      for (int row = 0; row < M; ++row) {
        // rows of padding only: the last super-tile's, which has no reactions
        if (ga * S::ST + row * S::RT >= a.n) break;
        meet_sources<R, S, U, M>(sum, a, lds, ga, row, gb, gb + 1, sp_at);
        const float *held =
            gb == ga && row > 0 ? lds + S::REACT + row * S::RT : nullptr;
        float *f = fp + row * S::RT;
        if (gb == gb0) add_waves<R, U, S::W, false>(sum, lds, held, f, S::ST);
        else add_waves<R, U, S::W, true>(sum, lds, held, f, S::ST);
      }
  }
}

// Work item -> (row ga, chunk c): rows are enumerated in order, row ga
// holding ceil((ts - ga) / L) items.
__device__ __forceinline__ int item_row(long long it, int ts, int L) {
  int lo = 0, hi = ts - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (row_first(mid, ts, L) <= it) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Row of item `it` where rows hold m, m - 1, .. 1 items: counted from the end,
// the largest k with k (k + 1) / 2 <= r.  The root is off by one at most (it
// is under 2^17 and rounded to 24 bits).  item_row's search took 800
// instructions before the first load, in every workgroup at the same time.
__device__ __forceinline__ int triangle_row(unsigned it, int m) {
  const unsigned r = (unsigned)((long long)m * (m + 1) / 2) - 1 - it;
  int k = (int)((__builtin_sqrtf(8.0f * (float)r + 1.0f) - 1.0f) * 0.5f);
  if ((long long)k * (k + 1) / 2 > r) --k;
  if ((long long)(k + 1) * (k + 2) / 2 <= r) ++k;
  return __builtin_amdgcn_readfirstlane(m - 1 - k);
}

// Work item of a launch -> super-tile ga, its chunk c (row partial
// row_first(ga) + c).  With one super-tile per item the diagonal pairs, the
// shorter ones, come last: they fill the last round.
__device__ __forceinline__ void sym_item(unsigned it, int ts, int L, int &ga,
                                         int &c) {
  if (L == 1) {
    const unsigned pairs = (unsigned)((long long)ts * (ts - 1) / 2);
    if (it >= pairs) {
      ga = (int)(it - pairs);
      c = 0;
    } else { // rows of lengths ts - 1, .. 1
      ga = triangle_row(it, ts - 1);
      c = (int)(it - (unsigned)row_first(ga, ts - 1, 1)) + 1;
    }
  } else {
    ga = item_row(it, ts, L);
    c = (int)(it - row_first(ga, ts, L));
  }
}

template <class R, int U, int M, int W>
__global__ __launch_bounds__(64 * W) void sym_kernel(SymArgs a) {
  using S = RowShape<R, U, M, W>;
  constexpr int ST = S::ST;
  __shared__ float lds[S::LDS_FLOATS];
  const int ts = a.ts, L = a.chunk;
  int ga, c;
  sym_item(blockIdx.x, ts, L, ga, c);
  const int gb0 = ga + c * L;
  row_item<R, S, U, M>(
      a, lds, ga, gb0, min(gb0 + L, ts),
      a.fpart + (size_t)(row_first(ga, ts, L) + c) * (R::ACC * ST),
      [&](int gb) {
        return a.spart + (size_t)pair_slot(ga, gb, ts) * (R::ACC * ST);
      });
}

constexpr int kTileRuns = 4; // runs per particle, tile-pair finalize

// Per particle: row partials (chunk order), minus the negated reaction
// partials of its column (ga order), in RUNS runs; then the rule's epilogue.
template <class R, int ST, int RUNS>
__global__ __launch_bounds__(256) void sym_finalize(SymArgs a) {
  constexpr int PW = 256 / RUNS; // particles per workgroup
  static_assert(ST % PW == 0 && PW % 64 == 0, "one super-tile per workgroup, "
                                              "one run per wave");
  __shared__ float red[RUNS > 1 ? R::ACC : 1][256];
  // uniform: the indices of the partials are scalar arithmetic (per-lane
  // indices with 64-bit divisions were 300 instructions before the first
  // load; with that, the work items' search and the particle's own loads moved
  // here, a step takes 1 us less: n = 4097 12.9 -> 11.8, 12800 38.0 -> 37.1)
  const int base = blockIdx.x * PW, g = base / ST;
  const int run =
      RUNS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / PW) : 0;
  const int i = base + threadIdx.x % PW, o = base % ST + threadIdx.x % PW;
  const bool live = i < a.n;
  if (RUNS == 1 && !live) return;
  typename R::Own own = {}; // in flight with the partials
  if (run == 0 && live) own = R::own(a, i);
  float f[R::ACC];
  if (live) {
    const int ts = a.ts, L = a.chunk;
    const long long first = row_first(g, ts, L);
    run_sum<R, RUNS>(
        f, L == 1 ? ts - g : (ts - g + L - 1) / L, g, run,
        [&](int c) { return a.fpart + (size_t)(first + c) * (R::ACC * ST) + o; },
        [&](int ga) {
          return a.spart + (size_t)pair_slot(ga, g, ts) * (R::ACC * ST) + o;
        },
        ST);
  } else {
#pragma unroll
    for (int e = 0; e < R::ACC; ++e) f[e] = 0.0f;
  }
  if (combine_runs<R, RUNS>(f, red) && live) R::finish(a, i, own, f);
}

// ---- banded launches (n past the single-launch limit) ----------------------
//
// The super-tile pair triangle is cut by source super-tile into bands
// [B0, B0 + W): band rows GA < B0 + W, each with the sources GB in
// [max(GA, B0), B0 + W) in chunks of L.  Per band: the pair kernel writes the
// band's row partials (one per item) and reaction partials (one per pair
// with GB > GA), a fold kernel adds, per particle, its band rows minus its
// band reactions to a running sum (band order), and after the last band a
// finish kernel applies the rule's epilogue (the integrator; the adjoint's
// cotangent update).  The partials of one band stay within a fixed
// budget whatever n is; the order of every sum is fixed.

// Reaction slot of pair (ga, gb), gb > ga, gb in the band [b0, b0 + w).
__host__ __device__ inline long long band_pair_slot(int ga, int gb, int b0,
                                                    int w) {
  return ga < b0 ? (long long)ga * w + (gb - b0)
                 : (long long)b0 * w + pair_slot(ga - b0, gb - b0, w);
}

__host__ __device__ inline long long band_items(int b0, int w, int L) {
  return (long long)b0 * ((w + L - 1) / L) + items_upto(w, L);
}

__host__ __device__ inline long long band_reactions(int b0, int w) {
  return (long long)b0 * w + (long long)w * (w - 1) / 2;
}

// Work item of a band -> row ga and first source super-tile gb0.
__device__ __forceinline__ void band_item(long long it, int b0, int W, int L,
                                          int &ga, int &gb0) {
  const int c0 = (W + L - 1) / L; // items of a row above the band
  const long long head = (long long)b0 * c0;
  if (it < head) {
    ga = (int)(it / c0);
    gb0 = b0 + (int)(it % c0) * L;
  } else { // the band's own triangle, rows enumerated in order
    const long long j = it - head;
    const int lo = item_row(j, W, L);
    ga = b0 + lo;
    gb0 = ga + (int)(j - row_first(lo, W, L)) * L;
  }
}

template <class R, int U, int M, int W>
__global__ __launch_bounds__(64 * W) void sym_band_kernel(SymArgs a) {
  using S = RowShape<R, U, M, W>;
  constexpr int ST = S::ST;
  __shared__ float lds[S::LDS_FLOATS];
  const int L = a.chunk, b0 = a.b0, bw = a.bw;
  const long long it = blockIdx.x;
  int ga, gb0;
  band_item(it, b0, bw, L, ga, gb0);
  row_item<R, S, U, M>(
      a, lds, ga, gb0, min(gb0 + L, b0 + bw),
      a.fpart + (size_t)it * (R::ACC * ST), [&](int gb) {
        return a.spart + (size_t)band_pair_slot(ga, gb, b0, bw) * (R::ACC * ST);
      });
}

// Per particle: its band rows (chunk order) minus its band reactions (GA
// order), added to the running sum (band order; Kahan sums carry their
// compensation from band to band).
template <class R, int ST>
__global__ __launch_bounds__(256) void sym_band_fold(SymArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  const int g = i / ST, o = i % ST;
  const int L = a.chunk, b0 = a.b0, W = a.bw, b1 = b0 + W;
  if (g >= b1 && !a.first) return; // no band term; its sum stays
  float f[R::ACC];
#pragma unroll
  for (int e = 0; e < R::ACC; ++e) f[e] = 0.0f;
  if (g < b1) {
    const int c0 = (W + L - 1) / L;
    const long long first =
        g < b0 ? (long long)g * c0
               : (long long)b0 * c0 + row_first(g - b0, W, L);
    const int rows = g < b0 ? c0 : (b1 - g + L - 1) / L;
    run_sum<R, 1>(
        f, rows, g >= b0 ? g : 0, 0,
        [&](int c) { return a.fpart + (size_t)(first + c) * (R::ACC * ST) + o; },
        [&](int gs) {
          return a.spart +
                 (size_t)band_pair_slot(gs, g, b0, W) * (R::ACC * ST) + o;
        },
        ST);
  }
  float *acc = a.acc3 + i;
  if (!a.first) {
    float r[R::ACC];
    R::fetch(r, acc, a.n);
    R::add_v(r, f);
#pragma unroll
    for (int e = 0; e < R::ACC; ++e) f[e] = r[e];
  }
#pragma unroll
  for (int e = 0; e < R::ACC; ++e) acc[(size_t)e * a.n] = f[e];
}

template <class R>
__global__ __launch_bounds__(256) void sym_band_finish(SymArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  float f[R::ACC];
#pragma unroll
  for (int e = 0; e < R::ACC; ++e) f[e] = a.acc3[(size_t)e * a.n + i];
  R::finish(a, i, R::own(a, i), f);
}

// ---- many independent systems (batched persistent launch) ----------------
//
// Work item = (system s, super-tile pair ga <= gb of s, slot); the items of
// all systems are handed out longest first through a device counter to a
// grid sized to the GPU's resident capacity.  Slot k owns a row partial
// part[k][0] and, for ga < gb, a reaction partial part[k][1] (ACC x ST
// floats each); the slots of system s are sys_slot[s] + the row-major index
// of (ga, gb) in its upper triangle.  The finalize sums, per particle, the
// row partials of its row in gb order minus the reaction partials of its
// column in ga order: the same values in the same order as the
// single-system kernel with one super-tile per item, so a batched step
// equals the systems' single-system steps bit for bit.

struct SymBatchArgs {
  const float *px, *py, *pz; // concatenated systems
  float *vx, *vy, *vz;
  float *nx, *ny, *nz;
  const int4 *items;     // (system, ga, gb, slot)
  const int *sys_off;    // [S + 1] first particle of each system
  const int *sys_slot;   // [S + 1] first slot of each system
  const float4 *sys_par; // (eps, damping, dt, G)
  float *part;           // [slots][2][3][ST]
  int num_items;
  int num_systems;
  int total; // particles in all systems
  int *counters; // [0]: next item, [1]: workgroups finished
};

// The single-system view of system s (arrays shifted to its first particle).
__device__ __forceinline__ SymArgs system_view(const SymBatchArgs &b, int s,
                                               int ST) {
  const int off0 = b.sys_off[s];
  const float4 pr = b.sys_par[s];
  SymArgs a = {};
  a.px = b.px + off0;
  a.py = b.py + off0;
  a.pz = b.pz + off0;
  a.vx = b.vx + off0;
  a.vy = b.vy + off0;
  a.vz = b.vz + off0;
  a.nx = b.nx + off0;
  a.ny = b.ny + off0;
  a.nz = b.nz + off0;
  a.n = b.sys_off[s + 1] - off0;
  a.ts = (a.n + ST - 1) / ST;
  a.chunk = 1;
  a.c.eps = pr.x;
  a.c.damping = pr.y;
  a.c.dt = pr.z;
  a.c.G = pr.w;
  return a;
}

// The queue of a persistent grid: every thread of the workgroup gets the next
// item, or one >= num_items when the queue is drained.
__device__ __forceinline__ int next_item(const SymBatchArgs &b, int *s_item) {
  if (threadIdx.x == 0) *s_item = atomicAdd(b.counters, 1);
  __syncthreads();
  const int item = *s_item;
  __syncthreads(); // every lane has read s_item before it is rewritten
  return item;
}

// The last workgroup to leave resets the counters for the next launch.
__device__ __forceinline__ void leave_queue(const SymBatchArgs &b) {
  if (threadIdx.x == 0) {
    __threadfence(); // this workgroup's last queue access precedes the count
    const int done = atomicAdd(b.counters + 1, 1);
    if (done == (int)gridDim.x - 1) {
      atomicExch(b.counters, 0);
      atomicExch(b.counters + 1, 0);
    }
  }
}

template <int U, int M, int W>
__global__ __launch_bounds__(64 * W, 4) void sym_batch_kernel(SymBatchArgs b) {
  using R = ForceRule;
  using S = RowShape<R, U, M, W>;
  constexpr int ST = S::ST;
  __shared__ float lds[S::LDS_FLOATS];
  __shared__ int s_item;
  for (;;) {
    const int item = next_item(b, &s_item);
    if (item >= b.num_items) break;
    const int4 it = b.items[item];
    const SymArgs a = system_view(b, it.x, ST);
    float *slot = b.part + (size_t)it.w * (2 * R::ACC * ST);
    row_item<R, S, U, M>(a, lds, it.y, it.z, it.z + 1, slot,
                      [&](int) { return slot + R::ACC * ST; });
  }
  leave_queue(b);
}

template <int ST>
__global__ __launch_bounds__(256) void sym_batch_finalize(SymBatchArgs b) {
  using R = ForceRule;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= b.total) return;
  // system of particle i: the last s with sys_off[s] <= i (empty systems
  // share their offset with the next one and are skipped)
  int lo = 0, hi = b.num_systems - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (b.sys_off[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  const SymArgs a = system_view(b, lo, ST);
  const int li = i - b.sys_off[lo];
  const int g = li / ST, o = li % ST, ts = a.ts;
  const float *base = b.part + (size_t)b.sys_slot[lo] * (2 * R::ACC * ST) + o;
  float f[R::ACC];
  run_sum<R, 1>(
      f, ts - g, g, 0,
      [&](int k) {
        return base + (size_t)tri_slot(g, g + k, ts) * (2 * R::ACC * ST);
      },
      [&](int ga) {
        return base + (size_t)tri_slot(ga, g, ts) * (2 * R::ACC * ST) +
               R::ACC * ST;
      },
      ST);
  R::finish(a, li, R::own(a, li), f);
}

using KernelFn = void (*)(SymArgs);

// Kernels of one launch shape and its super-tile.  runs: finalize runs per
// particle.
struct SymShape {
  int st, threads, runs;
  KernelFn pairs, finalize;
  int even_lds; // see even_rounds (0: not for this shape)
};

// Kahan sums and the fused adjoint take 114 to 124 VGPRs with 4 targets per
// lane: four workgroups fit a CU.  Where a CU gets five, the fifth would run
// alone, one wave per SIMD with nothing to issue beside it; with LDS for three
// they run as 3 + 2.  Us per step, 4 + 1 / 3 + 2, Kahan and fused: n = 11520
// 62.9 / 62.5 and 67.2 / 66.2, 12288 65.3 / 63.8 and 69.3 / 67.8, 12800 70.3 /
// 65.0 and 74.5 / 69.5.  With four per CU (11264) 52.9 / 59.8, with six (13056)
// 72.0 / 75.2, with nine (16640) 103.7 / 105.7; the rules with more workgroups
// per CU gain nothing.
constexpr int kCUs = 256;
constexpr int kThirdOfLds = 160 * 1024 / 3 / 1280 * 1280; // bytes

bool even_rounds(long long blocks) {
  return blocks > 4 * kCUs && blocks <= 5 * kCUs;
}

template <class R, int U, int M, int RUNS, int W = (M > 2 ? 8 : 4)>
constexpr SymShape sym_shape() {
  constexpr int ST = 64 * U * M;
  constexpr bool four = U == 4 && R::ACC == 6;
  constexpr int lds = (int)sizeof(float) * RowShape<R, U, M, W>::LDS_FLOATS;
  return {ST,   64 * W, RUNS, sym_kernel<R, U, M, W>, sym_finalize<R, ST, RUNS>,
          four ? kThirdOfLds - lds : 0};
}

// Targets per lane of a tile-pair shape of `unroll` particles per lane (tiles
// of 64 * unroll).  Below kTilePairRows particles tiles of 2 per lane are taken
// one at a time (super-tiles of 128, two waves per set of sources: four times
// the workgroups); from there two at a time (4 targets per lane, half the LDS
// traffic and partials per pair term).  `items` 2 names the shape that keeps
// rows of 128 at every size.  Both sides, us per step, device time
// (forward / Kahan / adjoint / fused): n = 4097 11.8 / 17.7 / 15.1 / 19.1 vs
// 17.9 / 26.6 / 23.7 / 28.5, 9000 26.8 / 42.8 / 35.5 / 46.7 vs 25.5 / 44.2 /
// 38.5 / 49.4, 9728 29.9 / 48.6 / 39.9 / 52.8 vs 25.8 / 44.8 / 36.6 / 47.2,
// 11000 35.5 / 58.6 / 48.0 / 64.6 vs 30.9 / 52.5 / 46.4 / 60.7.
// Below kTileWide particles 8 waves share the 128 x 128 pairs, each a quarter
// of a set's steps: with fewer pairs than SIMDs the step is the latency of
// one wave (2100 8.8 / 10.3 / 10.7 / 12.0 vs 9.6 / 12.6 / 11.2 / 13.0, 3000
// 10.1 / 13.8 / 11.5 / 14.4 vs 10.2 / 13.3 / 12.4 / 14.6, 4097 12.2 / 18.2 /
// 15.1 / 19.1 vs 11.8 / 17.7 / 15.1 / 19.1).
constexpr size_t kTilePairRows = 9728;
constexpr size_t kTileWide = 3328;

int tile_targets(int unroll, int items, size_t n) {
  return unroll == 2 && items == 1 && n >= kTilePairRows ? 4 : unroll;
}

// Super-tile shapes: M = unroll / 2 rows of 512.  Tile pairs: one row per
// super-tile, of one tile or a pair of tiles.
template <class R>
const SymShape *find_shape(int unroll, bool tiles, int items, size_t n) {
  static const SymShape wide2 = sym_shape<R, 2, 1, kTileRuns, 8>(),
                        tile2 = sym_shape<R, 2, 1, kTileRuns>(),
                        tile4 = sym_shape<R, 4, 1, kTileRuns>(),
                        rows1 = sym_shape<R, 8, 1, 1>(),
                        rows2 = sym_shape<R, 8, 2, 1>();
  if (tiles) {
    if (unroll != 2 && unroll != 4) return nullptr;
    if (tile_targets(unroll, items, n) == 4) return &tile4;
    return n < kTileWide ? &wide2 : &tile2;
  }
  if (unroll == 2) return &rows1;
  if (unroll == 4) return &rows2;
  if constexpr (R::ROWS4) {
    static const SymShape rows4 = sym_shape<R, 8, 4, 1>();
    if (unroll == 8) return &rows4;
  }
  return nullptr;
}

// Banded launches: super-tile shapes with at least four super-tiles per
// item, past their single-launch limit.
bool sym_banded(int unroll, bool tiles, int chunk, int acc, size_t n) {
  return !tiles && (unroll == 2 || unroll == 4 || unroll == 8) && chunk >= 4 &&
         n > sym_max_particles(unroll, tiles, chunk, acc) &&
         n <= kSymBandedMaxParticles;
}

struct BandShape {
  int unroll, st, threads;
  KernelFn pairs, fold, finish;
};

// Band kernels of rule R: 2, 4 or 8 particles per lane (Kahan: 2 or 4).
template <class R, int M>
constexpr BandShape band_shape() {
  constexpr int W = RowShape<R, 8, M>::W;
  return {2 * M, 512 * M, 64 * W, sym_band_kernel<R, 8, M, W>,
          sym_band_fold<R, 512 * M>, sym_band_finish<R>};
}

template <class R>
const BandShape *find_band_shape(int unroll) {
  static const BandShape b2 = band_shape<R, 1>(), b4 = band_shape<R, 2>();
  if (unroll == 2) return &b2;
  if (unroll == 4) return &b4;
  if constexpr (R::ROWS4) {
    static const BandShape b8 = band_shape<R, 4>();
    if (unroll == 8) return &b8;
  }
  return nullptr;
}

// Band width (the widest whose partials fit kSymBandBytes at 3 sums per
// particle, whatever the rule's count) and the largest row-item and reaction
// slot counts over the bands.
struct BandPlan {
  int ts, w;
  long long rows, reacs;
};

BandPlan band_plan(size_t n, int unroll, int chunk) {
  const int st = 256 * unroll;
  const int ts = (int)((n + st - 1) / st);
  const size_t per_slot = sizeof(float) * 3 * st;
  for (int w = ts; w >= 1; --w) {
    long long rows = 0, reacs = 0;
    for (int b0 = 0; b0 < ts; b0 += w) {
      const int ww = std::min(w, ts - b0);
      rows = std::max(rows, band_items(b0, ww, chunk));
      reacs = std::max(reacs, band_reactions(b0, ww));
    }
    if ((size_t)(rows + reacs) * per_slot <= kSymBandBytes)
      return {ts, w, rows, reacs};
  }
  return {ts, 0, 0, 0};
}

int launch_sym_banded(const BandShape *band, SymArgs &a, int chunk, int n,
                      float *scratch, int acc, hipStream_t stream) {
  const int st = band->st;
  const BandPlan bp = band_plan((size_t)n, band->unroll, chunk);
  if (bp.w < 1)
    return set_error(NB_ERR_UNSUPPORTED, "no band plan for this size");
  a.fpart = scratch;
  a.spart = scratch + (size_t)bp.rows * acc * st;
  a.acc3 = a.spart + (size_t)bp.reacs * acc * st;
  a.ts = bp.ts;
  a.chunk = chunk;
  a.n = n;
  void *args[] = {&a};
  const dim3 block(256), part_grid((n + 255) / 256);
  for (int b0 = 0; b0 < bp.ts; b0 += bp.w) {
    a.b0 = b0;
    a.bw = std::min(bp.w, bp.ts - b0);
    a.first = b0 == 0;
    const long long items = band_items(a.b0, a.bw, chunk);
    int r = hip_check(
        hipLaunchKernel(reinterpret_cast<const void *>(band->pairs),
                        dim3((unsigned)items), dim3(band->threads), args, 0,
                        stream),
        "symmetric band launch");
    if (!r)
      r = hip_check(hipLaunchKernel(reinterpret_cast<const void *>(band->fold),
                                    part_grid, block, args, 0, stream),
                    "symmetric band fold launch");
    if (r) return r;
  }
  return hip_check(
      hipLaunchKernel(reinterpret_cast<const void *>(band->finish), part_grid,
                      block, args, 0, stream),
      "symmetric band finish launch");
}

int launch_sym(const SymShape *sh, SymArgs &a, int unroll, int chunk, int n,
               float *scratch, int acc, bool tiles, hipStream_t stream,
               const BandShape *band = nullptr) {
  if (band && sym_banded(unroll, tiles, chunk, acc, (size_t)n)) {
    if (!scratch)
      return set_error(NB_ERR_INVALID_ARG, "symmetric launch needs scratch");
    return launch_sym_banded(band, a, chunk, n, scratch, acc, stream);
  }
  const size_t cap = sym_max_particles(unroll, tiles, chunk, acc);
  if ((size_t)n > cap)
    return set_error(
        NB_ERR_UNSUPPORTED,
        tiles ? "symmetric tile-pair shapes take at most 2^17 particles"
        : chunk >= 4 && band
            ? "symmetric launch shapes take at most 2^24 particles"
        : unroll <= 2
            ? "symmetric shapes with 2 per lane take at most 2^18 particles "
              "(2^24 with 4 super-tiles per item)"
            : "symmetric launch shapes take at most 2^20 particles (2^24 with "
              "4 super-tiles per item; Kahan sums: 2 or 4 per lane)");
  if (!sh || chunk < 1)
    return set_error(NB_ERR_UNSUPPORTED, "no symmetric kernel for this shape");
  if (!scratch)
    return set_error(NB_ERR_INVALID_ARG, "symmetric launch needs scratch");
  if (tiles) {
    if (chunk > 2)
      return set_error(NB_ERR_UNSUPPORTED,
                       "tile-pair shapes take one or two items per tile pair");
    chunk = 1; // one super-tile pair per work item, whatever the shape's name
  }
  const int ts = (n + sh->st - 1) / sh->st;
  const long long blocks = items_upto(ts, chunk);
  a.fpart = scratch;
  a.spart = scratch + (size_t)blocks * acc * sh->st;
  a.ts = ts;
  a.chunk = chunk;
  a.n = n;
  void *args[] = {&a};
  int r = hip_check(hipLaunchKernel(reinterpret_cast<const void *>(sh->pairs),
                                    dim3((unsigned)blocks), dim3(sh->threads),
                                    args, even_rounds(blocks) ? sh->even_lds : 0,
                                    stream),
                    "symmetric pair launch");
  if (r) return r;
  const int per_block = 256 / sh->runs;
  return hip_check(
      hipLaunchKernel(reinterpret_cast<const void *>(sh->finalize),
                      dim3((n + per_block - 1) / per_block), dim3(256), args,
                      0, stream),
      "symmetric finalize launch");
}

} // namespace

size_t sym_scratch_bytes(int unroll, int chunk, size_t n, int acc,
                         bool tiles, bool bandable) {
  if (tiles) {
    if (n == 0 || n > sym_max_particles(unroll, tiles, chunk, acc)) return 0;
    // ts (ts + 1) / 2 row partials and ts (ts - 1) / 2 reaction partials
    const long long st = 64LL * tile_targets(unroll, chunk, n);
    const long long ts = ((long long)n + st - 1) / st;
    return sizeof(float) * acc * (size_t)(ts * ts * st);
  }
  if (bandable && sym_banded(unroll, tiles, chunk, acc, n)) {
    const BandPlan bp = band_plan(n, unroll, chunk);
    if (bp.w < 1) return 0;
    return sizeof(float) * ((size_t)(bp.rows + bp.reacs) * acc *
                                (size_t)(256 * unroll) +
                            (size_t)acc * n);
  }
  if (n == 0 || n > sym_max_particles(unroll, tiles, chunk, acc) || chunk < 1)
    return 0;
  const long long st = (long long)256 * unroll;
  const long long ts = ((long long)n + st - 1) / st;
  const long long slots = items_upto(ts, chunk) + ts * (ts - 1) / 2;
  return sizeof(float) * (size_t)slots * acc * (size_t)st;
}

int sym_batch_layout(int unroll, const int *sys_off, int num_systems,
                     std::vector<int4> &items, std::vector<int> &sys_slot,
                     size_t &part_bytes) {
  if (unroll != 2 && unroll != 4 && unroll != 8)
    return set_error(NB_ERR_UNSUPPORTED, "no symmetric batch kernel for shape");
  const int ST = 256 * unroll;
  std::vector<int4> off_diag, diag;
  sys_slot.assign(num_systems + 1, 0);
  long long slots = 0;
  for (int s = 0; s < num_systems; ++s) {
    sys_slot[s] = (int)slots;
    const int n = sys_off[s + 1] - sys_off[s];
    const int ts = (n + ST - 1) / ST;
    for (int ga = 0; ga < ts; ++ga)
      for (int gb = ga; gb < ts; ++gb) {
        const int4 it = make_int4(s, ga, gb, (int)(slots + tri_slot(ga, gb, ts)));
        (gb == ga ? diag : off_diag).push_back(it);
      }
    slots += (long long)ts * (ts + 1) / 2;
    if (slots > (1LL << 30))
      return set_error(NB_ERR_UNSUPPORTED, "too many symmetric work items");
  }
  sys_slot[num_systems] = (int)slots;
  // longest first: pairs with reactions, then the diagonal super-tiles
  items = off_diag;
  items.insert(items.end(), diag.begin(), diag.end());
  part_bytes = sizeof(float) * (size_t)slots * 2 * 3 * ST;
  return NB_OK;
}

namespace {
template <int U> const void *batch_pairs_fn() {
  return reinterpret_cast<const void *>(
      sym_batch_kernel<8, U / 2, RowShape<ForceRule, 8, U / 2>::W>);
}
template <int U> const void *batch_finalize_fn() {
  return reinterpret_cast<const void *>(sym_batch_finalize<256 * U>);
}
} // namespace

int sym_batch_threads(int unroll) {
  return 64 * (unroll == 8 ? RowShape<ForceRule, 8, 4>::W
                           : RowShape<ForceRule, 8, 1>::W);
}

const void *sym_batch_kernel_fn(int unroll) {
  switch (unroll) {
  case 2: return batch_pairs_fn<2>();
  case 4: return batch_pairs_fn<4>();
  case 8: return batch_pairs_fn<8>();
  default: return nullptr;
  }
}

int launch_sym_batch(int unroll, const SymBatchLaunch &L, hipStream_t stream) {
  const void *pairs = sym_batch_kernel_fn(unroll);
  const void *fin = unroll == 2   ? batch_finalize_fn<2>()
                    : unroll == 4 ? batch_finalize_fn<4>()
                    : unroll == 8 ? batch_finalize_fn<8>()
                                  : nullptr;
  if (!pairs || !fin)
    return set_error(NB_ERR_UNSUPPORTED, "no symmetric batch kernel for shape");
  if (L.num_items == 0) return NB_OK;
  SymBatchArgs b;
  b.px = L.pos[0];
  b.py = L.pos[1];
  b.pz = L.pos[2];
  b.vx = L.vel[0];
  b.vy = L.vel[1];
  b.vz = L.vel[2];
  b.nx = L.nxt[0];
  b.ny = L.nxt[1];
  b.nz = L.nxt[2];
  b.items = L.items;
  b.sys_off = L.sys_off;
  b.sys_slot = L.sys_slot;
  b.sys_par = L.sys_par;
  b.part = L.part;
  b.num_items = L.num_items;
  b.num_systems = L.num_systems;
  b.total = L.total;
  b.counters = L.counters;
  void *args[] = {&b};
  int r = hip_check(hipLaunchKernel(pairs, dim3(L.grid),
                                    dim3(sym_batch_threads(unroll)), args, 0,
                                    stream),
                    "symmetric batch launch");
  if (r) return r;
  return hip_check(hipLaunchKernel(fin, dim3((L.total + 255) / 256),
                                   dim3(256), args, 0, stream),
                   "symmetric batch finalize launch");
}

int launch_forward_sym(const StepConsts &c, int unroll, int chunk, bool tiles,
                       bool kahan, const float *px, const float *py,
                       const float *pz, float *vx, float *vy, float *vz,
                       float *nx, float *ny, float *nz, int n, float *scratch,
                       hipStream_t stream) {
  if (n <= 0) return NB_OK;
  SymArgs a = {};
  a.px = px;
  a.py = py;
  a.pz = pz;
  a.vx = vx;
  a.vy = vy;
  a.vz = vz;
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  a.c = c;
  if (tiles && chunk != 1 && (kahan || unroll != 2))
    return set_error(NB_ERR_UNSUPPORTED,
                     "two items per tile pair: plain sums, 2 per lane only");
  if (kahan)
    return launch_sym(
        find_shape<KahanForceRule>(unroll, tiles, chunk, (size_t)n), a, unroll, chunk, n,
        scratch, KahanForceRule::ACC, tiles, stream,
        tiles ? nullptr : find_band_shape<KahanForceRule>(unroll));
  return launch_sym(find_shape<ForceRule>(unroll, tiles, chunk, (size_t)n), a, unroll,
                    chunk, n, scratch, ForceRule::ACC, tiles, stream,
                    tiles ? nullptr : find_band_shape<ForceRule>(unroll));
}

int launch_adjoint_sym(const StepConsts &c, bool fused, int unroll, int chunk,
                       bool tiles, const float *const pos[3], const float *const lxn[3],
                       const float *const lvn[3], float *const lx[3],
                       float *const lv[3], float *const vel[3],
                       float *const nxt[3], int n, float *scratch,
                       hipStream_t stream) {
  if (n <= 0) return NB_OK;
  SymArgs a = {};
  a.c = c;
  a.px = pos[0];
  a.py = pos[1];
  a.pz = pos[2];
  for (int d = 0; d < 3; ++d) {
    a.lxn[d] = lxn[d];
    a.lvn[d] = lvn[d];
    a.lx[d] = lx[d];
    a.lv[d] = lv[d];
  }
  if (fused) {
    a.vx = vel[0];
    a.vy = vel[1];
    a.vz = vel[2];
    a.nx = nxt[0];
    a.ny = nxt[1];
    a.nz = nxt[2];
    return launch_sym(
        find_shape<AdjointRule<true>>(unroll, tiles, chunk, (size_t)n), a, unroll, chunk, n,
        scratch, AdjointRule<true>::ACC, tiles, stream,
        tiles ? nullptr : find_band_shape<AdjointRule<true>>(unroll));
  }
  return launch_sym(find_shape<AdjointRule<false>>(unroll, tiles, chunk, (size_t)n), a, unroll,
                    chunk, n, scratch, AdjointRule<false>::ACC, tiles, stream,
                    tiles ? nullptr : find_band_shape<AdjointRule<false>>(unroll));
}

} // namespace nb
