// physics.hpp -- device point functions of the Euler, Kapila 5-equation and
// Baer-Nunziato systems.
//
// Every expression keeps the operand order of the reference function cited
// beside it, and the library is compiled without FMA contraction, so each
// value is the IEEE-FP64 result of the same operation sequence as the
// reference.  Face directions are template parameters (DIR 0: x-face, normal
// (1,0); DIR 1: y-face, normal (0,1)); products with the zero normal component
// are kept, so that a non-finite state spreads as it does there.
//
// The stage kernel is bound by the number of FP64 instructions, so where the
// reference multiplies by a power of two or by zero (an exact product) and adds,
// the two are one fused multiply-add here: it rounds once, to the same bits.
// With the constant denominators' reciprocals and the admissibility report off the
// common path, a Kapila row's faces take 860 FP64 instructions instead of 1,240.
// Halving is exact except for subnormal numbers.  Velocities and momenta do get
// there: ahead of a wave they decay by a factor per cell down to the smallest
// doubles.  So does the first phase's volume fraction where that phase vanishes,
// and its mass, momentum and energy per volume with it (the second phase's is one
// minus the first's).  S::RANGE names those components of the conservative [0] and
// the primitive [1] path; their sums keep the reference's separate operations.  So
// do the fluxes and jump terms of every component, which are products with a
// velocity.
// The other components, densities, pressures and the energies with them, are
// bounded from below by the admissibility checks, so they and their differences
// (zero or at least an ulp) are normal numbers.
#pragma once
#ifndef HYPE_KNS
#define HYPE_KNS hype  // kernel namespace; the contracted build uses its own
#endif
#include <hip/hip_runtime.h>

#include "fdiv.hpp"

namespace HYPE_KNS {

// hype.h:50-52
constexpr double PRS_FLOOR = 1.0e-12;
constexpr double RHO_FLOOR = 1.0e-14;
constexpr double SMALL_NUM = 1.0e-12;

// which numbers a component takes: normal ones and zero, any of either sign, or
// any positive one
enum Range { NORMAL, ANY, POSITIVE };

struct Eos {
  double g1, g2, p1, p2;  // GAMMA_1, GAMMA_2, PI_1, PI_2 (hype.h:42-45)
  bool bn_p2_quirk;       // baer_nunziato.c:271
  // constant denominators of the energy (S::energy_den) and their refined
  // reciprocals (recip_nr), set once per tile
  double d1, d2, y1, y2;
};

// first failing admissibility check of a flux evaluation; kinds follow the
// reference's MPI_Abort sites (see flux functions)
struct Bad {
  int kind;
  double val;
  __device__ void set(int k, double v) {
    if (kind == 0) {
      kind = k;
      val = v;
    }
  }
};

__device__ __forceinline__ double pmax(double a, double b) { return (a < b) ? b : a; }

// u nx + v ny
template <int DIR>
__device__ __forceinline__ double normal(double u, double v) {
  return DIR == 0 ? fma(v, 0.0, u) : fma(u, 0.0, v);
}
// a + n p with n the face normal's component along axis AXIS
template <int DIR, int AXIS>
__device__ __forceinline__ double add_pressure(double a, double p) {
  return DIR == AXIS ? a + p : fma(p, 0.0, a);
}

// ------------------------------------------------------------------ Euler
struct Euler {
  static constexpr int NV = 4;
  static constexpr int WAVES_PER_EU = 2;  // register budget of the stage kernel: 256 per lane
  // tile layouts the stage kernel is built for (bit HYPE_LAYOUT_*: one wave per
  // tile, split tiles, shared rows); the host picks per problem.  Two-wave tiles
  // run one wave per SIMD, one-wave tiles two: small grids gain from the shorter
  // sweeps (256^2 at order 2, us per step: split tiles 88, shared rows 80),
  // large ones from the second wave's latency hiding
  static constexpr int PAIR_MODES = 7;
  // a split tile sends its CFL maximum to memory once, from the lower wave,
  // instead of once per wave: the atomics of the last stage contend for one
  // address (Euler quadrants 256^2: 636 -> 670 Mcell-updates/s)
  static constexpr bool PAIR_CFL_COMBINE = true;
  static constexpr bool HAS_INLET = false;  // no InletBC in euler.c
  // no sound speed is shared between the admissibility check and the flux
  static constexpr bool HAS_ACACHE = false;
  static constexpr int REFX[2] = {1, -1};  // reflective x-wall negates comp 1
  static constexpr int REFY[2] = {2, -1};
  static constexpr bool HAS_NCP = false;
  // components of the face jump term D that can be nonzero
  static constexpr bool DNZ[NV] = {false, false, false, false};

  // components of the flux that are identically zero
  static constexpr bool FZERO[NV] = {false, false, false, false};
  static constexpr Range RANGE[2][NV] = {{NORMAL, ANY, ANY, NORMAL}, {NORMAL, ANY, ANY, NORMAL}};
  __device__ static __forceinline__ void energy_den(const Eos& e, double& d1, double& d2) {
    d1 = e.g1 - 1.0;
    d2 = 1.0;
  }

  // euler.c:14-23
  __device__ static __forceinline__ void cons2prim(const Eos& e, const double* Q, double* V) {
    double irho = fdiv(1.0, Q[0]);
    V[0] = Q[0];
    V[1] = irho * Q[1];
    V[2] = irho * Q[2];
    V[3] = (e.g1 - 1.0) * fma(-0.5, irho * (Q[1] * Q[1] + Q[2] * Q[2]), Q[3]);
  }
  // flux and wave speed of a conserved state (euler.c:44-84)
  template <int DIR>
  __device__ static __forceinline__ double side_cons(const Eos& e, const double* Q, double* F, bool& bad) {
    double rho = Q[0];
    double irho = fdiv(1.0, rho);
    double u = irho * Q[1];
    double v = irho * Q[2];
    double un = normal<DIR>(u, v);
    double rhoun = rho * un;
    double E = Q[3];
    double p = (e.g1 - 1.0) * fma(-0.5, rho * (u * u + v * v), E);
    bad |= (rho < RHO_FLOOR) | (p < PRS_FLOOR);
    F[0] = rhoun;
    F[1] = add_pressure<DIR, 0>(rhoun * u, p);
    F[2] = add_pressure<DIR, 1>(rhoun * v, p);
    F[3] = un * (E + p);
    return fabs(un) + sqrt_adm(e.g1 * p * irho);
  }
  // which check of the flux a state fails first (euler.c:60-70)
  __device__ static __forceinline__ void diag_cons(const Eos& e, const double* Q, Bad& b) {
    double rho = Q[0];
    double irho = fdiv(1.0, rho);
    double u = irho * Q[1];
    double v = irho * Q[2];
    double p = (e.g1 - 1.0) * fma(-0.5, rho * (u * u + v * v), Q[3]);
    if (rho < RHO_FLOOR) b.set(1, rho);
    if (p < PRS_FLOOR) b.set(2, p);
  }
  // flux, wave speed and conserved variables of a primitive state
  // (euler.c:29-38, 197-236)
  template <int DIR>
  __device__ static __forceinline__ double side_prim(const Eos& e, const double* V, double* F, double* Q, bool& bad) {
    double rho = V[0];
    double u = V[1];
    double v = V[2];
    double un = normal<DIR>(u, v);
    double rhoun = rho * un;
    double p = V[3];
    double E = fma(0.5, rho * (u * u + v * v), div_const(p, e.d1, e.y1));
    bad |= (rho < RHO_FLOOR) | (p < PRS_FLOOR);
    F[0] = rhoun;
    F[1] = add_pressure<DIR, 0>(rhoun * u, p);
    F[2] = add_pressure<DIR, 1>(rhoun * v, p);
    F[3] = un * (E + p);
    Q[0] = rho;
    Q[1] = rho * u;
    Q[2] = rho * v;
    Q[3] = E;
    return fabs(un) + sqrt_adm(fdiv(e.g1 * p, rho));
  }
  // euler.c:212-222
  __device__ static __forceinline__ void diag_prim(const Eos&, const double* V, Bad& b) {
    if (V[0] < RHO_FLOOR) b.set(1, V[0]);
    if (V[3] < PRS_FLOOR) b.set(2, V[3]);
  }
  // euler.c:169-191
  __device__ static __forceinline__ bool pad(const Eos& e, const double* Q) {
    bool ok = true;
    double rho = Q[0];
    double irho = fdiv(1.0, rho);
    double u = irho * Q[1];
    double v = irho * Q[2];
    double p = (e.g1 - 1.0) * fma(-0.5, rho * (u * u + v * v), Q[3]);
    if (rho < RHO_FLOOR) ok = false;
    if (p < PRS_FLOOR) ok = false;
    return ok;
  }
  // euler.c:292-310
  __device__ static __forceinline__ bool pad_prim(const Eos&, const double* V) {
    bool ok = true;
    if (V[0] < RHO_FLOOR) ok = false;
    if (V[3] < PRS_FLOOR) ok = false;
    return ok;
  }
  template <bool PRIM>
  __device__ static __forceinline__ void vol_ncp(const Eos&, const double*, const double*, const double*, double* B) {
    for (int c = 0; c < NV; ++c) B[c] = 0.0;
  }
  // face jump term: identically zero (euler.c:142-148, 278-286)
  template <bool PRIM, int DIR>
  __device__ static __forceinline__ void ncp_face(const Eos&, const double*, const double*, double* D) {
    for (int c = 0; c < NV; ++c) D[c] = 0.0;
  }
};

// ----------------------------------------------------------------- Kapila
struct Kapila {
  static constexpr int NV = 6;
  static constexpr int WAVES_PER_EU = 1;
  // no one-wave tiles: split ones save one reconstructed ring row per wave at the
  // same one wave per SIMD (1024 x 512 shock-bubble: 952 -> 985 Mcell-updates/s);
  // small grids share rows (512x256: 174 -> 157 us per step)
  static constexpr int PAIR_MODES = 6;
  // one atomic per split tile (Kapila 1024x512: 1087 -> 1108
  // Mcell-updates/s; the batched set, whose 64 instances already spread the
  // atomics over 64 addresses, 1320 -> 1317)
  static constexpr bool PAIR_CFL_COMBINE = true;
  // left inlet of kapila_5eqn.c:289-320, 485-513 (tabulated per row by the host)
  static constexpr bool HAS_INLET = true;
  // the admissibility check at a node computes the a_sq the primitive flux
  // at that point needs (kapila_5eqn.c:347-349 and 468-470 are the same
  // expression): the stage kernel hands it over instead of recomputing
  static constexpr bool HAS_ACACHE = true;
  static constexpr int REFX[2] = {2, -1};
  static constexpr int REFY[2] = {3, -1};
  static constexpr bool HAS_NCP = true;
  static constexpr bool DNZ[NV] = {false, false, false, false, false, true};

  static constexpr bool FZERO[NV] = {false, false, false, false, false, true};
  static constexpr Range RANGE[2][NV] = {{POSITIVE, NORMAL, ANY, ANY, NORMAL, POSITIVE},
                                         {NORMAL, NORMAL, ANY, ANY, NORMAL, POSITIVE}};
  __device__ static __forceinline__ void energy_den(const Eos& e, double& d1, double& d2) {
    d1 = (e.g1 - 1.0) * (e.g2 - 1.0);
    d2 = 1.0;
  }

  // pressure of a conserved state (kapila_5eqn.c:22-30)
  __device__ static __forceinline__ double pressure(const Eos& e, const double* Q, double rho, double u, double v,
                                                    double alpha_2) {
    double alpha_1 = Q[5];
    double en = fma(-0.5, rho * (u * u + v * v), Q[4]);
    double G1m1 = e.g1 - 1.0;
    double G2m1 = e.g2 - 1.0;
    return fdiv(en * G1m1 * G2m1 - alpha_1 * e.g1 * e.p1 * G2m1 - alpha_2 * e.g2 * e.p2 * G1m1,
                alpha_1 * G2m1 + alpha_2 * G1m1);
  }
  // the mixture's squared speed of sound (kapila_5eqn.c:89-94, 347-352)
  __device__ static __forceinline__ double sound_sq(const Eos& e, double rho_1, double rho_2, double rho, double p,
                                                    double alpha_1,
                                    double alpha_2) {
    double a1_sq = fdiv(e.g1 * (p + e.p1), rho_1);
    double a2_sq = fdiv(e.g2 * (p + e.p2), rho_2);
    return fdiv(rho_1 * a1_sq * rho_2 * a2_sq, rho * (alpha_2 * rho_1 * a1_sq + alpha_1 * rho_2 * a2_sq));
  }

  // kapila_5eqn.c:14-35
  __device__ static __forceinline__ void cons2prim(const Eos& e, const double* Q, double* V) {
    double alpha_1 = Q[5];
    double alpha_2 = 1.0 - alpha_1;
    double rho = Q[0] + Q[1];
    double u = fdiv(Q[2], rho);
    double v = fdiv(Q[3], rho);
    V[0] = fdiv(Q[0], alpha_1);
    V[1] = fdiv(Q[1], alpha_2);
    V[2] = u;
    V[3] = v;
    V[4] = pressure(e, Q, rho, u, v, alpha_2);
    V[5] = alpha_1;
  }
  // flux and wave speed of a conserved state (kapila_5eqn.c:67-113)
  template <int DIR>
  __device__ static __forceinline__ double side_cons(const Eos& e, const double* Q, double* F, bool& bad) {
    double alpha_1 = Q[5];
    double alpha_2 = 1.0 - alpha_1;
    double rho_1 = fdiv(Q[0], alpha_1);
    double rho_2 = fdiv(Q[1], alpha_2);
    double rho = Q[0] + Q[1];
    double u = fdiv(Q[2], rho);
    double v = fdiv(Q[3], rho);
    double E = Q[4];
    double p = pressure(e, Q, rho, u, v, alpha_2);
    double un = normal<DIR>(u, v);
    double a_sq = sound_sq(e, rho_1, rho_2, rho, p, alpha_1, alpha_2);
    bad |= a_sq < PRS_FLOOR;
    F[0] = alpha_1 * rho_1 * un;
    F[1] = alpha_2 * rho_2 * un;
    F[2] = add_pressure<DIR, 0>(rho * u * un, p);
    F[3] = add_pressure<DIR, 1>(rho * v * un, p);
    F[4] = (E + p) * un;
    F[5] = 0.0;
    return fabs(un) + sqrt_adm(a_sq);
  }
  __device__ static __forceinline__ double sound_sq_cons(const Eos& e, const double* Q) {
    double alpha_1 = Q[5];
    double alpha_2 = 1.0 - alpha_1;
    double rho = Q[0] + Q[1];
    double u = fdiv(Q[2], rho);
    double v = fdiv(Q[3], rho);
    return sound_sq(e, fdiv(Q[0], alpha_1), fdiv(Q[1], alpha_2), rho, pressure(e, Q, rho, u, v, alpha_2), alpha_1,
                    alpha_2);
  }
  // kapila_5eqn.c:95-99
  __device__ static __forceinline__ void diag_cons(const Eos& e, const double* Q, Bad& b) {
    const double a_sq = sound_sq_cons(e, Q);
    if (a_sq < PRS_FLOOR) b.set(3, a_sq);
  }
  // a_sq of a primitive state; the admissibility check (kapila_5eqn.c:468-470)
  // and the flux (:347-352) compute the same expression
  __device__ static __forceinline__ double sound_sq_prim(const Eos& e, const double* V) {
    double alpha_1 = V[5];
    double alpha_2 = 1.0 - alpha_1;
    double rho = alpha_1 * V[0] + alpha_2 * V[1];
    return sound_sq(e, V[0], V[1], rho, V[4], alpha_1, alpha_2);
  }
  // flux, wave speed and conserved variables of a primitive state whose a_sq
  // is given (kapila_5eqn.c:41-61, 326-371)
  template <int DIR>
  __device__ static __forceinline__ double side_prim_a(const Eos& e, const double* V, double a_sq, double* F,
                                                       double* Q, bool& bad) {
    double alpha_1 = V[5];
    double alpha_2 = 1.0 - alpha_1;
    double m1 = alpha_1 * V[0];
    double m2 = alpha_2 * V[1];
    double rho = m1 + m2;
    double u = V[2];
    double v = V[3];
    double p = V[4];
    double G1m1 = e.g1 - 1.0;
    double G2m1 = e.g2 - 1.0;
    double en = div_const(p * (alpha_1 * G2m1 + alpha_2 * G1m1) + alpha_1 * e.g1 * e.p1 * G2m1 +
                              alpha_2 * e.g2 * e.p2 * G1m1,
                          e.d1, e.y1);
    double E = fma(0.5, rho * (u * u + v * v), en);
    double un = normal<DIR>(u, v);
    double ru = rho * u;
    double rv = rho * v;
    bad |= a_sq < PRS_FLOOR;
    F[0] = m1 * un;
    F[1] = m2 * un;
    F[2] = add_pressure<DIR, 0>(ru * un, p);
    F[3] = add_pressure<DIR, 1>(rv * un, p);
    F[4] = (E + p) * un;
    F[5] = 0.0;
    Q[0] = m1;
    Q[1] = m2;
    Q[2] = ru;
    Q[3] = rv;
    Q[4] = E;
    Q[5] = alpha_1;
    return fabs(un) + sqrt_adm(a_sq);
  }
  template <int DIR>
  __device__ static __forceinline__ double side_prim(const Eos& e, const double* V, double* F, double* Q, bool& bad) {
    return side_prim_a<DIR>(e, V, sound_sq_prim(e, V), F, Q, bad);
  }
  // kapila_5eqn.c:353-357
  __device__ static __forceinline__ void diag_prim(const Eos& e, const double* V, Bad& b) {
    const double a_sq = sound_sq_prim(e, V);
    if (a_sq < PRS_FLOOR) b.set(3, a_sq);
  }
  // kapila_5eqn.c:247-283 (alpha_1 test of :278 kept)
  __device__ static __forceinline__ bool pad(const Eos& e, const double* Q) {
    const double a_sq = sound_sq_cons(e, Q);
    if (Q[0] + Q[1] < RHO_FLOOR) return false;
    if (a_sq < PRS_FLOOR) return false;
    if (Q[5] < 1.0 || Q[5] > 1.0) return false;
    return true;
  }
  // kapila_5eqn.c:450-479; also returns the a_sq it computes (for side_prim_a)
  __device__ static __forceinline__ bool pad_prim_a(const Eos& e, const double* V, double& a_out) {
    double alpha_1 = V[5];
    double alpha_2 = 1.0 - alpha_1;
    double rho = alpha_1 * V[0] + alpha_2 * V[1];
    double a_sq = sound_sq(e, V[0], V[1], rho, V[4], alpha_1, alpha_2);
    a_out = a_sq;
    if (rho < RHO_FLOOR) return false;
    if (a_sq < PRS_FLOOR) return false;
    if (alpha_1 < 0.0 || alpha_1 > 1.0) return false;
    return true;
  }
  __device__ static __forceinline__ bool pad_prim(const Eos& e, const double* V) {
    double a_sq;
    return pad_prim_a(e, V, a_sq);
  }
  // B*grad for the primitive path, comp 5 only (kapila_5eqn.c:417-444);
  // arguments: V (6 values), alpha_x, alpha_y, u_x, v_y
  __device__ static __forceinline__ double ncp5_prim(const Eos& e, const double* V, double phi_x, double phi_y,
                                     double u_x, double v_y) {
    double alpha_1 = V[5];
    double alpha_2 = 1.0 - alpha_1;
    double rho_1 = V[0];
    double rho_2 = V[1];
    double u = V[2];
    double v = V[3];
    double p = V[4];
    double a_1_sq = fdiv(e.g1 * (p + e.p1), rho_1);
    double a_2_sq = fdiv(e.g2 * (p + e.p2), rho_2);
    double K = fdiv(alpha_1 * alpha_2 * (rho_2 * a_2_sq - rho_1 * a_1_sq),
                    alpha_1 * rho_2 * a_2_sq + alpha_2 * rho_1 * a_1_sq);
    return u * phi_x + v * phi_y - K * (u_x + v_y);
  }
  // B*grad for the conservative path, comp 5 only (kapila_5eqn.c:164-198);
  // gx, gy: gradients of all components
  __device__ static __forceinline__ double ncp5_cons(const Eos& e, const double* Q, const double* gx,
                                                     const double* gy) {
    double alpha_1 = Q[5];
    double alpha_2 = 1.0 - alpha_1;
    double rho_1 = fdiv(Q[0], alpha_1);
    double rho_2 = fdiv(Q[1], alpha_2);
    double rho = Q[0] + Q[1];
    double irho = fdiv(1.0, rho);
    double u = fdiv(Q[2], rho);
    double v = fdiv(Q[3], rho);
    double p = pressure(e, Q, rho, u, v, alpha_2);
    double a1_sq = fdiv(e.g1 * (p + e.p1), rho_1);
    double a2_sq = fdiv(e.g2 * (p + e.p2), rho_2);
    double K = fdiv(alpha_1 * alpha_2 * (rho_2 * a2_sq - rho_1 * a1_sq),
                    alpha_1 * rho_2 * a2_sq + alpha_2 * rho_1 * a1_sq);
    double alpha1_x = gx[5];
    double alpha1_y = gy[5];
    double u_x = irho * irho * (gx[2] * rho - Q[2] * (gx[0] + gx[1]));
    double v_y = irho * irho * (gy[3] * rho - Q[3] * (gy[0] + gy[1]));
    return u * alpha1_x + v * alpha1_y - K * (u_x + v_y);
  }
  // volume term B(V) grad V at a quadrature point (rhs_function_prim.c:474)
  template <bool PRIM>
  __device__ static __forceinline__ void vol_ncp(const Eos& e, const double* V, const double* gx, const double* gy,
                                                 double* B) {
    for (int c = 0; c < 5; ++c) B[c] = 0.0;
    if (PRIM)
      B[5] = ncp5_prim(e, V, gx[5], gy[5], gx[2], gy[3]);
    else
      B[5] = ncp5_cons(e, V, gx, gy);
  }
  // face jump D = B(mean) (R - L) (riemann.c:95-102 / 130-137).  On the primitive
  // path the mean's factors 1/2 are kept out of the densities, where they cancel
  // exactly (rho_k a_k^2 = (2 rho_k)(a_k^2 / 2)), and out of the transverse
  // velocity, which is multiplied by zero.  Those products stay, as the zero's sign
  // does not reach a sum but a NaN does: where a transverse velocity is not finite
  // (its reconstruction overflows before any other component's does) the
  // reference's jump is NaN, also where the face's wave speed is not (PetscMax
  // keeps a left speed beside a right one that is NaN)
  template <bool PRIM, int DIR>
  __device__ static __forceinline__ void ncp_face(const Eos& e, const double* L, const double* R, double* D) {
    for (int c = 0; c < 5; ++c) D[c] = 0.0;
    if (PRIM) {
      constexpr int n = 2 + DIR, t = 3 - DIR;
      double r1 = R[0] + L[0];  // twice the means
      double r2 = R[1] + L[1];
      double un = 0.5 * (R[n] + L[n]);
      double ps = R[4] + L[4];
      double as = R[5] + L[5];
      double alpha_1 = 0.5 * as;
      double alpha_2 = fma(-0.5, as, 1.0);
      double a_1_sq = fdiv(e.g1 * fma(0.5, ps, e.p1), r1);  // half of them
      double a_2_sq = fdiv(e.g2 * fma(0.5, ps, e.p2), r2);
      double K = fdiv(alpha_1 * alpha_2 * (r2 * a_2_sq - r1 * a_1_sq), alpha_1 * r2 * a_2_sq + alpha_2 * r1 * a_1_sq);
      D[5] = fma(R[t] + L[t], 0.0, un * (R[5] - L[5])) - K * fma(R[t] - L[t], 0.0, R[n] - L[n]);
    } else {
      constexpr double nx = DIR == 0 ? 1.0 : 0.0, ny = DIR == 0 ? 0.0 : 1.0;
      double av[NV], gx[NV], gy[NV];
      for (int c = 0; c < NV; ++c) {
        av[c] = 0.5 * (R[c] + L[c]);
        gx[c] = nx * (R[c] - L[c]);
        gy[c] = ny * (R[c] - L[c]);
      }
      D[5] = ncp5_cons(e, av, gx, gy);
    }
  }
};

// ---------------------------------------------------------- Baer-Nunziato
struct BN {
  static constexpr int NV = 9;
  static constexpr int WAVES_PER_EU = 1;
  // no split tiles: two windows of nine components would halve the workgroups an
  // LDS of 160 KB holds.  Grids of few rows per wave share rows (128x128: 183 ->
  // 121 us per step), which needs one window
  static constexpr int PAIR_MODES = 5;
  static constexpr bool PAIR_CFL_COMBINE = false;  // one wave per tile
  static constexpr bool HAS_INLET = false;  // no InletBC in baer_nunziato.c
  // no sound speed is shared between the admissibility check and the flux
  static constexpr bool HAS_ACACHE = false;
  static constexpr int REFX[2] = {1, 5};
  static constexpr int REFY[2] = {2, 6};
  static constexpr bool HAS_NCP = true;
  static constexpr bool DNZ[NV] = {false, true, true, true, false, true, true, true, true};

  static constexpr bool FZERO[NV] = {false, false, false, false, false, false, false, false, true};
  static constexpr Range RANGE[2][NV] = {{POSITIVE, ANY, ANY, POSITIVE, NORMAL, ANY, ANY, NORMAL, POSITIVE},
                                         {NORMAL, ANY, ANY, NORMAL, NORMAL, ANY, ANY, NORMAL, POSITIVE}};
  __device__ static __forceinline__ void energy_den(const Eos& e, double& d1, double& d2) {
    d1 = e.g1 - 1.0;
    d2 = e.g2 - 1.0;
  }

  // pressure of a phase from its density, velocity and total energy per volume
  // (baer_nunziato.c:29-30)
  __device__ static __forceinline__ double pressure(double g, double pi, double rho, double u, double v, double E) {
    return (g - 1.0) * fma(-0.5, rho * (u * u + v * v), E) - g * pi;
  }
  // baer_nunziato.c:14-41
  __device__ static __forceinline__ void cons2prim(const Eos& e, const double* Q, double* V) {
    double phi_1 = Q[8];
    double phi_2 = 1.0 - Q[8];
    double rho_1 = fdiv(Q[0], phi_1);
    double rho_2 = fdiv(Q[4], phi_2);
    double u_1 = fdiv(Q[1], Q[0]);
    double v_1 = fdiv(Q[2], Q[0]);
    double u_2 = fdiv(Q[5], Q[4]);
    double v_2 = fdiv(Q[6], Q[4]);
    V[0] = rho_1;
    V[1] = u_1;
    V[2] = v_1;
    V[3] = pressure(e.g1, e.p1, rho_1, u_1, v_1, fdiv(Q[3], phi_1));
    V[4] = rho_2;
    V[5] = u_2;
    V[6] = v_2;
    V[7] = pressure(e.g2, e.p2, rho_2, u_2, v_2, fdiv(Q[7], phi_2));
    V[8] = phi_1;
  }
  // baer_nunziato.c:47-60
  __device__ static __forceinline__ void prim2cons(const Eos& e, const double* V, double* Q) {
    Q[0] = V[8] * V[0];
    Q[1] = Q[0] * V[1];
    Q[2] = Q[0] * V[2];
    Q[3] = Q[0] * fma(0.5, V[1] * V[1] + V[2] * V[2], fdiv(V[3] + e.g1 * e.p1, V[0] * (e.g1 - 1.0)));
    Q[4] = (1.0 - V[8]) * V[4];
    Q[5] = Q[4] * V[5];
    Q[6] = Q[4] * V[6];
    Q[7] = Q[4] * fma(0.5, V[5] * V[5] + V[6] * V[6], fdiv(V[7] + e.g2 * e.p2, V[4] * (e.g2 - 1.0)));
    Q[8] = V[8];
  }
  // the fluxes and wave speed of the two phases from their primitive variables
  // and total energies (baer_nunziato.c:115-130, 305-320)
  template <int DIR>
  __device__ static __forceinline__ double fluxes(const Eos& e, double phi_1, double rho_1, double u_1, double v_1,
                                                  double p_1,
                                  double E_1, double rho_2, double u_2, double v_2, double p_2, double E_2, double* F,
                                  bool& bad) {
    double phi_2 = 1.0 - phi_1;
    double un_1 = normal<DIR>(u_1, v_1);
    double un_2 = normal<DIR>(u_2, v_2);
    double ps_1 = p_1 + e.p1;
    double ps_2 = p_2 + e.p2;
    bad |= (rho_1 < RHO_FLOOR) | (rho_2 < RHO_FLOOR) | (ps_1 < PRS_FLOOR) | (ps_2 < PRS_FLOOR);
    F[0] = phi_1 * rho_1 * un_1;
    F[1] = phi_1 * add_pressure<DIR, 0>(rho_1 * u_1 * un_1, p_1);
    F[2] = phi_1 * add_pressure<DIR, 1>(rho_1 * v_1 * un_1, p_1);
    F[3] = phi_1 * un_1 * (E_1 + p_1);
    F[4] = phi_2 * rho_2 * un_2;
    F[5] = phi_2 * add_pressure<DIR, 0>(rho_2 * u_2 * un_2, p_2);
    F[6] = phi_2 * add_pressure<DIR, 1>(rho_2 * v_2 * un_2, p_2);
    F[7] = phi_2 * un_2 * (E_2 + p_2);
    F[8] = 0.0;
    double s_1 = fabs(un_1) + sqrt_adm(fdiv(e.g1 * ps_1, rho_1));
    double s_2 = fabs(un_2) + sqrt_adm(fdiv(e.g2 * ps_2, rho_2));
    return pmax(s_1, s_2);
  }
  // which check a state fails first (baer_nunziato.c:91-113, 281-303)
  __device__ static __forceinline__ void diag(const Eos& e, double rho_1, double p_1, double rho_2, double p_2,
                                              Bad& b) {
    if (rho_1 < RHO_FLOOR) b.set(4, rho_1);
    if (rho_2 < RHO_FLOOR) b.set(5, rho_2);
    if ((p_1 + e.p1) < PRS_FLOOR) b.set(6, p_1 + e.p1);
    if ((p_2 + e.p2) < PRS_FLOOR) b.set(7, p_2 + e.p2);
  }
  // baer_nunziato.c:66-131
  template <int DIR>
  __device__ static __forceinline__ double side_cons(const Eos& e, const double* Q, double* F, bool& bad) {
    double phi_1 = Q[8];
    double phi_2 = 1.0 - Q[8];
    double rho_1 = fdiv(Q[0], phi_1);
    double rho_2 = fdiv(Q[4], phi_2);
    double u_1 = fdiv(Q[1], Q[0]);
    double v_1 = fdiv(Q[2], Q[0]);
    double u_2 = fdiv(Q[5], Q[4]);
    double v_2 = fdiv(Q[6], Q[4]);
    double E_1 = fdiv(Q[3], phi_1);
    double E_2 = fdiv(Q[7], phi_2);
    double p_1 = pressure(e.g1, e.p1, rho_1, u_1, v_1, E_1);
    double p_2 = pressure(e.g2, e.p2, rho_2, u_2, v_2, E_2);
    return fluxes<DIR>(e, phi_1, rho_1, u_1, v_1, p_1, E_1, rho_2, u_2, v_2, p_2, E_2, F, bad);
  }
  __device__ static __forceinline__ void diag_cons(const Eos& e, const double* Q, Bad& b) {
    double V[NV];
    cons2prim(e, Q, V);
    diag(e, V[0], V[3], V[4], V[7], b);
  }
  // baer_nunziato.c:256-321
  template <int DIR>
  __device__ static __forceinline__ double side_prim(const Eos& e, const double* V, double* F, double* Q, bool& bad) {
    double p_1 = V[3];
    double p_2 = e.bn_p2_quirk ? V[8] : V[7];
    double E_1 = fma(0.5, V[0] * (V[1] * V[1] + V[2] * V[2]), div_const(p_1 + e.g1 * e.p1, e.d1, e.y1));
    double E_2 = fma(0.5, V[4] * (V[5] * V[5] + V[6] * V[6]), div_const(p_2 + e.g2 * e.p2, e.d2, e.y2));
    prim2cons(e, V, Q);
    return fluxes<DIR>(e, V[8], V[0], V[1], V[2], p_1, E_1, V[4], V[5], V[6], p_2, E_2, F, bad);
  }
  __device__ static __forceinline__ void diag_prim(const Eos& e, const double* V, Bad& b) {
    diag(e, V[0], V[3], V[4], e.bn_p2_quirk ? V[8] : V[7], b);
  }
  // baer_nunziato.c:207-250
  __device__ static __forceinline__ bool pad(const Eos& e, const double* Q) {
    double V[NV];
    cons2prim(e, Q, V);
    return pad_prim(e, V);
  }
  // baer_nunziato.c:350-385
  __device__ static __forceinline__ bool pad_prim(const Eos& e, const double* V) {
    bool ok = true;
    if (V[0] < RHO_FLOOR) ok = false;
    if (V[4] < RHO_FLOOR) ok = false;
    if ((V[3] + e.p1) < PRS_FLOOR) ok = false;
    if ((V[7] + e.p2) < PRS_FLOOR) ok = false;
    if (V[8] < 0.0 || V[8] > 1.0) ok = false;
    return ok;
  }
  // B*grad from the interface velocity u_1 and pressure p_2 (DIR: face
  // direction, whose other gradient component is a signed zero; 2: volume term)
  template <int DIR>
  __device__ static __forceinline__ void ncp(double u_I, double v_I, double p_I, double phi_x, double phi_y,
                                             double* B) {
    double adv = DIR == 0   ? fma(v_I, phi_y, u_I * phi_x)
                 : DIR == 1 ? fma(u_I, phi_x, v_I * phi_y)
                            : u_I * phi_x + v_I * phi_y;
    B[0] = 0.0;
    B[1] = -p_I * phi_x;
    B[2] = -p_I * phi_y;
    B[3] = -p_I * adv;
    B[4] = 0.0;
    B[5] = p_I * phi_x;
    B[6] = p_I * phi_y;
    B[7] = p_I * adv;
    B[8] = adv;
  }
  // primitive path (baer_nunziato.c:327-344)
  template <int DIR>
  __device__ static __forceinline__ void ncp_prim(const double* V, double phi_x, double phi_y, double* B) {
    ncp<DIR>(V[1], V[2], V[7], phi_x, phi_y, B);
  }
  // conservative path (baer_nunziato.c:137-165)
  template <int DIR>
  __device__ static __forceinline__ void ncp_cons(const Eos& e, const double* Q, double phi_x, double phi_y,
                                                  double* B) {
    double phi_2 = 1.0 - Q[8];
    double rho_2 = fdiv(Q[4], phi_2);
    double u_2 = fdiv(Q[5], Q[4]);
    double v_2 = fdiv(Q[6], Q[4]);
    double p_I = pressure(e.g2, e.p2, rho_2, u_2, v_2, fdiv(Q[7], phi_2));
    ncp<DIR>(fdiv(Q[1], Q[0]), fdiv(Q[2], Q[0]), p_I, phi_x, phi_y, B);
  }
  template <bool PRIM>
  __device__ static __forceinline__ void vol_ncp(const Eos& e, const double* V, const double* gx, const double* gy,
                                                 double* B) {
    if (PRIM)
      ncp_prim<2>(V, gx[8], gy[8], B);
    else
      ncp_cons<2>(e, V, gx[8], gy[8], B);
  }
  template <bool PRIM, int DIR>
  __device__ static __forceinline__ void ncp_face(const Eos& e, const double* L, const double* R, double* D) {
    constexpr double nx = DIR == 0 ? 1.0 : 0.0, ny = DIR == 0 ? 0.0 : 1.0;
    double av[NV];
    for (int c = 0; c < NV; ++c) av[c] = 0.5 * (R[c] + L[c]);
    double phi_x = nx * (R[8] - L[8]);
    double phi_y = ny * (R[8] - L[8]);
    if (PRIM)
      ncp_prim<DIR>(av, phi_x, phi_y, D);
    else
      ncp_cons<DIR>(e, av, phi_x, phi_y, D);
  }
};

// Twice the Rusanov flux, and the path-conservative jump (riemann.c:52-105,
// 112-140): A = F_R + F_L - s (Q_R - Q_L), whose factor 1/2 the caller folds,
// exactly, into the scaling of the assembly.  Returns s = max(s_L, s_R)
// (PetscMax); bad: a state fails its admissibility check (riemann_diag says
// which).  aL, aR: a_sq of the two states where the system shares it with the
// node check (S::HAS_ACACHE and ACACHE).
template <class S, bool PRIM, bool ACACHE, int DIR>
__device__ __forceinline__ double riemann(const Eos& e, const double* L, const double* R, double* A, double* D,
                                          bool& bad, double aL, double aR) {
  constexpr int NV = S::NV;
  double FL[NV], FR[NV], QL[NV], QR[NV];
  double sl, sr;
  bad = false;
  if constexpr (PRIM) {
    if constexpr (ACACHE) {
      sl = S::template side_prim_a<DIR>(e, L, aL, FL, QL, bad);
      sr = S::template side_prim_a<DIR>(e, R, aR, FR, QR, bad);
    } else {
      sl = S::template side_prim<DIR>(e, L, FL, QL, bad);
      sr = S::template side_prim<DIR>(e, R, FR, QR, bad);
    }
  } else {
    sl = S::template side_cons<DIR>(e, L, FL, bad);
    sr = S::template side_cons<DIR>(e, R, FR, bad);
  }
  const double s = pmax(sl, sr);
#pragma unroll
  for (int c = 0; c < NV; ++c) {
    const double dQ = PRIM ? QR[c] - QL[c] : R[c] - L[c];
    A[c] = S::FZERO[c] ? -(s * dQ) : FR[c] + FL[c] - s * dQ;
  }
  S::template ncp_face<PRIM, DIR>(e, L, R, D);
  return s;
}

// the first failing check of a face point's two states (left before right)
template <class S, bool PRIM>
__device__ __forceinline__ Bad riemann_diag(const Eos& e, const double* L, const double* R) {
  Bad b{0, 0.0};
  if constexpr (PRIM) {
    S::diag_prim(e, L, b);
    S::diag_prim(e, R, b);
  } else {
    S::diag_cons(e, L, b);
    S::diag_cons(e, R, b);
  }
  return b;
}

}  // namespace HYPE_KNS
