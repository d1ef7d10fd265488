// The pair terms of one source against the U targets of a lane as one block
// of gfx950 assembly: the inner loop of the symmetric kernels (nb_sym.hip),
// operation for operation the arithmetic of the rules' C++ pair() (same
// rounding, same order of every sum: the results are the same bits).
//
// Why assembly.  Two waves of a SIMD issue fp32 VALU instructions together,
// 2 cycles each, under two conditions (probe/issue_rates.hip, 2 waves):
//   * the three sources of an FMA must not all be even or all be odd VGPRs
//     (two banks, two reads each; a register read twice counts twice), and
//     none may be an SGPR: v_fmac 2.2 cycles with mixed registers, 4.2 with all
//     even, 4.2 with an SGPR.  The compiler's allocation broke this for 194 of
//     512 v_fmac and, with eps in an SGPR, for every first FMA of |r|^2 + eps;
//   * after a v_rsq_f32 the two waves stay out of step, and later instructions
//     take up to 4 cycles, until one of them issues a non-VALU instruction:
//     v_rsq + 14 FMAs take 51 cycles bare, 39 with an s_nop behind the v_rsq, 41
//     with an s_setprio on either side.
// So r and h (see AdjointRule) sit in even temporaries, d, K and t3 in odd
// ones: every FMA below mixes the two whatever registers the compiler gives
// the sums.  eps is pinned to an odd register.  Each v_rsq is bracketed by
// s_setprio 1 / 0, which also lets the wave that holds its partner up issue
// first (one s_nop instead is slower).
// The terms of two targets alternate between two sets of temporaries, so the
// sums of one are issued behind the v_rsq of the next; v_rsq results are
// read at least one instruction later (its hazard).
//
// Measured, the pair loop alone (forward, 8 sources x 8 targets per step,
// sustained; time at 2.4 GHz): 45.6 cycles per wave pair term at 3 waves per
// SIMD against 49.6 for the compiler's loop; at 4 waves 44.6 against 47.2.  The
// kernels' 1 source x 8 targets: 46.9 at 4 waves.  In the step at N = 262144 the
// counters give 40.6 clock cycles a term at 1.8 to 2.1 GHz (48.6 at 2.26 GHz
// before): the cycles are the same in every launch, the clock is what varies.
#pragma once

#include <hip/hip_runtime.h>

namespace nb {

// Temporaries: X Y Z HX HY HZ even, D E K Q R odd; one set per target parity.
#define NB_SET0 16, 18, 20, 22, 24, 26, 17, 19, 21, 23, 25
#define NB_SET1 28, 30, 32, 34, 36, 38, 29, 31, 33, 35, 37
// ForceRule needs half of them (X Y Z, D E K) and leaves the rest to the
// kernel: with 8 targets per lane its registers decide the waves per SIMD.
#define NB_FSET0 16, 18, 20, , , , 17, 19, 21, ,
#define NB_FSET1 22, 24, 26, , , , 23, 25, 27, ,
#define NB_FORCE_TEMPORARIES                                                   \
  "v16", "v17", "v18", "v19", "v20", "v21", "v22", "v23", "v24", "v25", "v26", \
      "v27"
#define NB_TEMPORARIES                                                         \
  "v16", "v17", "v18", "v19", "v20", "v21", "v22", "v23", "v24", "v25", "v26", \
      "v27", "v28", "v29", "v30", "v31", "v32", "v33", "v34", "v35", "v36",    \
      "v37", "v38"
#define NB_EPS "{v15}"

#define NB_V(r) "v" #r
#define NB_2(op, d, a, b) op " " d ", " a ", " b "\n\t"

#define NB_RSQ(d, a)                                                           \
  "s_setprio 1\n\tv_rsq_f32 " NB_V(d) ", " NB_V(a) "\n\ts_setprio 0\n\t"

// r = s - t, d = |r|^2 + eps
#define NB_TERM_D(k, X, Y, Z, D)                                               \
  NB_2("v_sub_f32", NB_V(X), "%[sx]", "%[tx" #k "]")                           \
  NB_2("v_sub_f32", NB_V(Y), "%[sy]", "%[ty" #k "]")                           \
  NB_2("v_sub_f32", NB_V(Z), "%[sz]", "%[tz" #k "]")                           \
  NB_2("v_fma_f32", NB_V(D), NB_V(X), NB_V(X) ", %[eps]")                      \
  NB_2("v_fmac_f32", NB_V(D), NB_V(Y), NB_V(Y))                                \
  NB_2("v_fmac_f32", NB_V(D), NB_V(Z), NB_V(Z))

// ---- ForceRule ----
#define NB_FORCE_TERM_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)       \
  NB_TERM_D(k, X, Y, Z, D)                                                     \
  NB_2("v_mul_f32", NB_V(E), NB_V(D), NB_V(D))                                 \
  NB_2("v_mul_f32", NB_V(E), NB_V(E), NB_V(D))                                 \
  NB_RSQ(K, E)
#define NB_FORCE_SUMS_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)                  \
  NB_2("v_fmac_f32", "%[ax" #k "]", NB_V(X), NB_V(K))                          \
  NB_2("v_fmac_f32", "%[rx]", NB_V(X), NB_V(K))                                \
  NB_2("v_fmac_f32", "%[ay" #k "]", NB_V(Y), NB_V(K))                          \
  NB_2("v_fmac_f32", "%[ry]", NB_V(Y), NB_V(K))                                \
  NB_2("v_fmac_f32", "%[az" #k "]", NB_V(Z), NB_V(K))                          \
  NB_2("v_fmac_f32", "%[rz]", NB_V(Z), NB_V(K))

// ---- AdjointRule: rh = r . h, t3 = -3 rh / d, u = h + t3 r (in place of h)
#define NB_TERM_H(k, HX, HY, HZ)                                               \
  NB_2("v_sub_f32", NB_V(HX), "%[sgx]", "%[tgx" #k "]")                        \
  NB_2("v_sub_f32", NB_V(HY), "%[sgy]", "%[tgy" #k "]")                        \
  NB_2("v_sub_f32", NB_V(HZ), "%[sgz]", "%[tgz" #k "]")
#define NB_TERM_RH(X, Y, Z, HX, HY, HZ, R)                                     \
  NB_2("v_mul_f32", NB_V(R), NB_V(X), NB_V(HX))                                \
  NB_2("v_fmac_f32", NB_V(R), NB_V(Y), NB_V(HY))                               \
  NB_2("v_fmac_f32", NB_V(R), NB_V(Z), NB_V(HZ))
#define NB_TERM_U(X, Y, Z, HX, HY, HZ, Q, R)                                   \
  NB_2("v_mul_f32", NB_V(R), NB_V(R), NB_V(Q))                                 \
  NB_2("v_mul_f32", NB_V(R), "0xc0400000", NB_V(R)) /* -3 */                   \
  NB_2("v_fmac_f32", NB_V(HX), NB_V(R), NB_V(X))                               \
  NB_2("v_fmac_f32", NB_V(HY), NB_V(R), NB_V(Y))                               \
  NB_2("v_fmac_f32", NB_V(HZ), NB_V(R), NB_V(Z))
// plain: s = rsqrt(d), q = s^2, K = s^3
#define NB_ADJOINT_TERM_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)     \
  NB_TERM_D(k, X, Y, Z, D)                                                     \
  NB_RSQ(E, D)                            \
  NB_TERM_H(k, HX, HY, HZ)                                                     \
  NB_TERM_RH(X, Y, Z, HX, HY, HZ, R)                                           \
  NB_2("v_mul_f32", NB_V(Q), NB_V(E), NB_V(E))                                 \
  NB_2("v_mul_f32", NB_V(K), NB_V(Q), NB_V(E))                                 \
  NB_TERM_U(X, Y, Z, HX, HY, HZ, Q, R)
#define NB_ADJOINT_SUMS_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)                \
  NB_2("v_fmac_f32", "%[ax" #k "]", NB_V(K), NB_V(HX))                         \
  NB_2("v_fmac_f32", "%[rx]", NB_V(K), NB_V(HX))                               \
  NB_2("v_fmac_f32", "%[ay" #k "]", NB_V(K), NB_V(HY))                         \
  NB_2("v_fmac_f32", "%[ry]", NB_V(K), NB_V(HY))                               \
  NB_2("v_fmac_f32", "%[az" #k "]", NB_V(K), NB_V(HZ))                         \
  NB_2("v_fmac_f32", "%[rz]", NB_V(K), NB_V(HZ))
// fused: K as ForceRule forms it, q = K^2 d^2
#define NB_FUSED_TERM_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)       \
  NB_TERM_D(k, X, Y, Z, D)                                                     \
  NB_2("v_mul_f32", NB_V(E), NB_V(D), NB_V(D))                                 \
  NB_2("v_mul_f32", NB_V(D), NB_V(E), NB_V(D))                                 \
  NB_RSQ(K, D)                            \
  NB_TERM_H(k, HX, HY, HZ)                                                     \
  NB_TERM_RH(X, Y, Z, HX, HY, HZ, R)                                           \
  NB_2("v_mul_f32", NB_V(Q), NB_V(K), NB_V(K))                                 \
  NB_2("v_mul_f32", NB_V(Q), NB_V(Q), NB_V(E))                                 \
  NB_TERM_U(X, Y, Z, HX, HY, HZ, Q, R)
#define NB_FUSED_SUMS_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)                  \
  NB_ADJOINT_SUMS_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)                      \
  NB_2("v_fmac_f32", "%[fx" #k "]", NB_V(X), NB_V(K))                          \
  NB_2("v_fmac_f32", "%[qx]", NB_V(X), NB_V(K))                                \
  NB_2("v_fmac_f32", "%[fy" #k "]", NB_V(Y), NB_V(K))                          \
  NB_2("v_fmac_f32", "%[qy]", NB_V(Y), NB_V(K))                                \
  NB_2("v_fmac_f32", "%[fz" #k "]", NB_V(Z), NB_V(K))                          \
  NB_2("v_fmac_f32", "%[qz]", NB_V(Z), NB_V(K))

// ---- KahanForceRule: y = fma(r, K, -c), t = s + y, c = (t - s) - y, s = t.
// The new target sums land in other registers (n..), and the reaction sums
// alternate between r.. and m.. from target to target: no moves.
#define NB_KAHAN_ADD3(X, Y, Z, K, YX, YY, YZ, SX, SY, SZ, NX, NY, NZ, CX, CY,  \
                      CZ)                                                      \
  NB_2("v_fma_f32", NB_V(YX), NB_V(X), NB_V(K) ", -" CX)                       \
  NB_2("v_fma_f32", NB_V(YY), NB_V(Y), NB_V(K) ", -" CY)                       \
  NB_2("v_fma_f32", NB_V(YZ), NB_V(Z), NB_V(K) ", -" CZ)                       \
  NB_2("v_add_f32", NX, SX, NB_V(YX))                                          \
  NB_2("v_add_f32", NY, SY, NB_V(YY))                                          \
  NB_2("v_add_f32", NZ, SZ, NB_V(YZ))                                          \
  NB_2("v_sub_f32", SX, NX, SX)                                                \
  NB_2("v_sub_f32", SY, NY, SY)                                                \
  NB_2("v_sub_f32", SZ, NZ, SZ)                                                \
  NB_2("v_sub_f32", CX, SX, NB_V(YX))                                          \
  NB_2("v_sub_f32", CY, SY, NB_V(YY))                                          \
  NB_2("v_sub_f32", CZ, SZ, NB_V(YZ))
#define NB_KAHAN_TARGET(k, X, Y, Z, K, YX, YY, YZ)                             \
  NB_KAHAN_ADD3(X, Y, Z, K, YX, YY, YZ, "%[ax" #k "]", "%[ay" #k "]",          \
                "%[az" #k "]", "%[nx" #k "]", "%[ny" #k "]", "%[nz" #k "]",    \
                "%[cx" #k "]", "%[cy" #k "]", "%[cz" #k "]")
#define NB_KAHAN_TERM_ NB_FORCE_TERM_
#define NB_KAHAN_SUMS0_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)                 \
  NB_KAHAN_TARGET(k, X, Y, Z, K, D, E, Q)                                      \
  NB_KAHAN_ADD3(X, Y, Z, K, HX, HY, HZ, "%[rx]", "%[ry]", "%[rz]", "%[mx]",    \
                "%[my]", "%[mz]", "%[qx]", "%[qy]", "%[qz]")
#define NB_KAHAN_SUMS1_(k, X, Y, Z, HX, HY, HZ, D, E, K, Q, R)                 \
  NB_KAHAN_TARGET(k, X, Y, Z, K, D, E, Q)                                      \
  NB_KAHAN_ADD3(X, Y, Z, K, HX, HY, HZ, "%[mx]", "%[my]", "%[mz]", "%[rx]",    \
                "%[ry]", "%[rz]", "%[qx]", "%[qy]", "%[qz]")

// Targets 0 .. U-1 of rule N: term, then the sums of the target before.
#define NB_X(M, ...) M(__VA_ARGS__)
#define NB_T0(N, k) NB_X(NB_##N##_TERM_, k, NB_##N##_SET0)
#define NB_T1(N, k) NB_X(NB_##N##_TERM_, k, NB_##N##_SET1)
#define NB_S0(N, k) NB_X(NB_##N##_SUMS0_, k, NB_##N##_SET0)
#define NB_S1(N, k) NB_X(NB_##N##_SUMS1_, k, NB_##N##_SET1)
#define NB_FORCE_SET0 NB_FSET0
#define NB_FORCE_SET1 NB_FSET1
#define NB_ADJOINT_SET0 NB_SET0
#define NB_ADJOINT_SET1 NB_SET1
#define NB_FUSED_SET0 NB_SET0
#define NB_FUSED_SET1 NB_SET1
#define NB_KAHAN_SET0 NB_SET0
#define NB_KAHAN_SET1 NB_SET1
#define NB_FORCE_SUMS0_ NB_FORCE_SUMS_
#define NB_FORCE_SUMS1_ NB_FORCE_SUMS_
#define NB_ADJOINT_SUMS0_ NB_ADJOINT_SUMS_
#define NB_ADJOINT_SUMS1_ NB_ADJOINT_SUMS_
#define NB_FUSED_SUMS0_ NB_FUSED_SUMS_
#define NB_FUSED_SUMS1_ NB_FUSED_SUMS_
#define NB_HEAD2(N) NB_T0(N, 0) NB_T1(N, 1) NB_S0(N, 0)
#define NB_HEAD4(N)                                                      \
  NB_HEAD2(N)                                                            \
  NB_T0(N, 2) NB_S1(N, 1) NB_T1(N, 3) NB_S0(N, 2)
#define NB_BODY2(N) NB_HEAD2(N) NB_S1(N, 1)
#define NB_BODY4(N) NB_HEAD4(N) NB_S1(N, 3)
#define NB_BODY8(N)                                                      \
  NB_HEAD4(N)                                                            \
  NB_T0(N, 4) NB_S1(N, 3) NB_T1(N, 5) NB_S0(N, 4)                  \
  NB_T0(N, 6) NB_S1(N, 5) NB_T1(N, 7) NB_S0(N, 6) NB_S1(N, 7)

// Operand lists of U targets, the first of them target o: M(0, o), ..
#define NB_LIST2(M, o) M(0, o), M(1, o)
#define NB_LIST4(M, o) NB_LIST2(M, o), M(2, o), M(3, o)
#define NB_LIST8(M, o) NB_LIST4(M, o), M(4, o), M(5, o), M(6, o), M(7, o)
#define NB_IN3(n, k, v, o)                                                     \
  [n##x##k] "v"(v[o]), [n##y##k] "v"(v[o + 1]), [n##z##k] "v"(v[o + 2])
// early-clobber: the first targets' sums are written before the last targets'
// inputs are read, so a sum must not share the register of an input whose value
// it starts from
#define NB_IO3(n, k, v, o)                                                     \
  [n##x##k] "+&v"(v[o]), [n##y##k] "+&v"(v[o + 1]), [n##z##k] "+&v"(v[o + 2])
#define NB_OUT3(n, k, v, o)                                                    \
  [n##x##k] "=&v"(v[o]), [n##y##k] "=&v"(v[o + 1]), [n##z##k] "=&v"(v[o + 2])
#define NB_T_POS(k, o) NB_IN3(t, k, t[o + k], 0)
#define NB_T_G(k, o) NB_IN3(tg, k, t[o + k], 3)
#define NB_A_0(k, o) NB_IO3(a, k, a[o + k], 0)
#define NB_A_F(k, o) NB_IO3(f, k, a[o + k], 3)
#define NB_A_C(k, o) NB_IO3(c, k, a[o + k], 3)
#define NB_A_N(k, o) NB_OUT3(n, k, n[k], 0)

// s: the source's inputs, t: the targets', a: the targets' sums, r: the
// source's (negated) reaction sums.
#define NB_BLOCK_FN(name, SRC, ACC)                                            \
  template <int U>                                                             \
  __device__ __forceinline__ void name(const float (&s)[SRC],                  \
                                       const float (&t)[U][SRC],               \
                                       float (&a)[U][ACC], float (&r)[ACC],    \
                                       float eps)
#define NB_FORCE_ASM(U)                                                        \
  asm volatile(NB_BODY##U(FORCE)                                 \
               : NB_LIST##U(NB_A_0, 0), NB_IO3(r, , r, 0)                      \
               : NB_IN3(s, , s, 0), NB_LIST##U(NB_T_POS, 0), [eps] NB_EPS(eps) \
               : NB_FORCE_TEMPORARIES)
#define NB_ADJOINT_ASM(U)                                                      \
  asm volatile(NB_BODY##U(ADJOINT)                               \
               : NB_LIST##U(NB_A_0, 0), NB_IO3(r, , r, 0)                      \
               : NB_IN3(s, , s, 0), NB_IN3(sg, , s, 3),                        \
                 NB_LIST##U(NB_T_POS, 0), NB_LIST##U(NB_T_G, 0),               \
                 [eps] NB_EPS(eps)                                             \
               : NB_TEMPORARIES)
#define NB_FUSED_ASM(U)                                                        \
  asm volatile(NB_BODY##U(FUSED)                                 \
               : NB_LIST##U(NB_A_0, 0), NB_LIST##U(NB_A_F, 0),                 \
                 NB_IO3(r, , r, 0), NB_IO3(q, , r, 3)                          \
               : NB_IN3(s, , s, 0), NB_IN3(sg, , s, 3),                        \
                 NB_LIST##U(NB_T_POS, 0), NB_LIST##U(NB_T_G, 0),               \
                 [eps] NB_EPS(eps)                                             \
               : NB_TEMPORARIES)
// targets O .. O + U - 1
#define NB_KAHAN_ASM(U, O)                                                     \
  {                                                                            \
    float n[U][3], m[3];                                                       \
    asm volatile(NB_BODY##U(KAHAN)                               \
                 : NB_LIST##U(NB_A_0, O), NB_LIST##U(NB_A_C, O),               \
                   NB_LIST##U(NB_A_N, O), NB_IO3(r, , r, 0),                   \
                   NB_IO3(q, , r, 3), NB_OUT3(m, , m, 0)                       \
                 : NB_IN3(s, , s, 0), NB_LIST##U(NB_T_POS, O),                 \
                   [eps] NB_EPS(eps)                                           \
                 : NB_TEMPORARIES);                                            \
    for (int k = 0; k < U; ++k)                                                \
      for (int c = 0; c < 3; ++c) a[O + k][c] = n[k][c];                       \
  }

NB_BLOCK_FN(force_block, 3, 3) {
  static_assert(U == 2 || U == 4 || U == 8, "targets per lane");
  if constexpr (U == 2) NB_FORCE_ASM(2);
  if constexpr (U == 4) NB_FORCE_ASM(4);
  if constexpr (U == 8) NB_FORCE_ASM(8);
}

NB_BLOCK_FN(adjoint_block, 6, 3) {
  static_assert(U == 2 || U == 4 || U == 8, "targets per lane");
  if constexpr (U == 2) NB_ADJOINT_ASM(2);
  if constexpr (U == 4) NB_ADJOINT_ASM(4);
  if constexpr (U == 8) NB_ADJOINT_ASM(8);
}

NB_BLOCK_FN(fused_block, 6, 6) {
  static_assert(U == 2 || U == 4 || U == 8, "targets per lane");
  if constexpr (U == 2) NB_FUSED_ASM(2);
  if constexpr (U == 4) NB_FUSED_ASM(4);
  if constexpr (U == 8) NB_FUSED_ASM(8);
}

NB_BLOCK_FN(kahan_block, 3, 6) {
  static_assert(U == 2 || U == 4 || U == 8, "targets per lane");
  if constexpr (U == 2) NB_KAHAN_ASM(2, 0);
  if constexpr (U >= 4) NB_KAHAN_ASM(4, 0);
  if constexpr (U == 8) NB_KAHAN_ASM(4, 4);
}

} // namespace nb
