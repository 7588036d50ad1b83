// recon.hpp -- modal basis, quadrature tables and WENO reconstructions on the
// device (HyPE-2D/reconstruction.c, tables of hype.c:194-305).
//
// Tables are compile-time constants produced by the same basis formulas as
// the reference, so every basis value is bit-identical to the one the
// reference computes at start-up.  Sums over basis functions keep the
// reference's order k = 0..nDOF-1 starting from 0.0; terms whose basis value
// is exactly zero are skipped, which cannot change an IEEE result for finite
// coefficients (the running sum starts at +0.0 and can never become -0.0, so
// adding a signed zero is the identity).
#pragma once
#ifndef HYPE_KNS
#define HYPE_KNS hype  // kernel namespace; the contracted build uses its own
#endif
#include <hip/hip_runtime.h>

#include <utility>

#include "fdiv.hpp"
#include "physics.hpp"

namespace HYPE_KNS {

constexpr double GPT = 0.28867513459481287;  // hype.c:214-230

// reconstruction.c:11-47
constexpr double basis(double x, double y, int n) {
  return n == 0   ? 1.0
         : n == 1 ? x
         : n == 2 ? y
         : n == 3 ? x * x - 1. / 12.
         : n == 4 ? y * y - 1. / 12.
         : n == 5 ? x * y
         : n == 6 ? x * (x * x - 3. / 20.)
         : n == 7 ? y * (y * y - 3. / 20.)
         : n == 8 ? y * (x * x - 1. / 12.)
         : n == 9 ? x * (y * y - 1. / 12.)
                  : 0.0;
}
// reconstruction.c:53-100
constexpr double basis_gx(double x, double y, int n) {
  return n == 1   ? 1.0
         : n == 3 ? 2.0 * x
         : n == 5 ? y
         : n == 6 ? 3.0 * x * x - 3. / 20.
         : n == 8 ? 2.0 * x * y
         : n == 9 ? (y * y - 1. / 12.)
                  : 0.0;
}
constexpr double basis_gy(double x, double y, int n) {
  return n == 2   ? 1.0
         : n == 4 ? 2.0 * y
         : n == 5 ? x
         : n == 7 ? 3.0 * y * y - 3. / 20.
         : n == 8 ? (x * x - 1. / 12.)
         : n == 9 ? 2.0 * x * y
                  : 0.0;
}

// Quadrature for order N (hype.c:56-68, 203-230).  Face points are stored in
// the reference's node order (hype.c:207-229): right face points, left face
// points, top face points, bottom face points; the admissibility nodes are
// exactly these points.
template <int N>
struct Quad {
  static constexpr int NDOF = (N + 1) * (N + 2) / 2;
  static constexpr int NGF = N < 2 ? 1 : 2;
  static constexpr int NGV = N < 2 ? 1 : 4;
  static constexpr int NNODE = 4 * NGF;
  static constexpr double WF = N < 2 ? 1.0 : 0.5;   // wGP_Face
  static constexpr double WV = N < 2 ? 1.0 : 0.25;  // wGP_Vol
  static constexpr double xgf(int q) { return N < 2 ? 0.0 : (q == 0 ? -GPT : GPT); }
  static constexpr int R(int q) { return q; }
  static constexpr int L(int q) { return NGF + q; }
  static constexpr int T(int q) { return 2 * NGF + q; }
  static constexpr int B(int q) { return 3 * NGF + q; }
  static constexpr double nodex(int p) {
    return p < NGF ? 0.5 : p < 2 * NGF ? -0.5 : xgf(p % NGF);
  }
  static constexpr double nodey(int p) {
    return p < 2 * NGF ? xgf(p % NGF) : p < 3 * NGF ? 0.5 : -0.5;
  }
  // volume points (hype.c:217-220): (-g,-g), (-g,g), (g,-g), (g,g)
  static constexpr double volx(int q) { return N < 2 ? 0.0 : (q < 2 ? -GPT : GPT); }
  static constexpr double voly(int q) { return N < 2 ? 0.0 : ((q & 1) ? GPT : -GPT); }
  static constexpr double phin(int p, int k) { return basis(nodex(p), nodey(p), k); }
  static constexpr double phiv(int q, int k) { return basis(volx(q), voly(q), k); }
  static constexpr double gphx(int q, int k) { return basis_gx(volx(q), voly(q), k); }
  static constexpr double gphy(int q, int k) { return basis_gy(volx(q), voly(q), k); }
};

constexpr bool is_pow2(double x) {
  x = x < 0.0 ? -x : x;
  if (x == 0.0) return false;
  while (x < 1.0) x *= 2.0;
  while (x > 1.0) x *= 0.5;
  return x == 1.0;
}

// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>): a loop
// whose index is a constant expression in its body
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// sum_k s[k]*phi(k) in the reference's order, skipping exact-zero phi; T::at(k)
// is the table row.  A product with a power of two is exact, so fusing it with
// the addition rounds once, as the separate operations do, in one instruction.
// TINY: the component may hold subnormal values (S::RANGE), whose halves round
template <class T, int NDOF, bool TINY>
__device__ __forceinline__ double basis_sum(const double* s) {
  double acc = 0.0;
  static_for<NDOF>([&](auto K) {
    constexpr int k = decltype(K)::value;
    constexpr double phi = T::at(k);
    if constexpr (is_pow2(phi) && (!TINY || phi >= 1.0))
      acc = fma(s[k], phi, acc);
    else if constexpr (phi != 0.0)
      acc = acc + s[k] * phi;
  });
  return acc;
}

// rows of the tables: node P, volume point Q and its gradients
template <int N, int P>
struct RowNode { static constexpr double at(int k) { return Quad<N>::phin(P, k); } };
template <int N, int Q>
struct RowVol { static constexpr double at(int k) { return Quad<N>::phiv(Q, k); } };
template <int N, int Q>
struct RowGx { static constexpr double at(int k) { return Quad<N>::gphx(Q, k); } };
template <int N, int Q>
struct RowGy { static constexpr double at(int k) { return Quad<N>::gphy(Q, k); } };

// reconstruction.c:106-117
__device__ __forceinline__ double minmod(double a, double b) {
  if (a * b < 0.0) return 0.0;
  if (fabs(a) < fabs(b)) return a;
  return b;
}

__device__ __forceinline__ double pow4(double a) {  // reconstruction.c:123-127
  double a2 = a * a;
  return a2 * a2;
}

// One direction of weno3 (reconstruction.c:155-187): the three candidates'
// slopes and curvatures and their nonlinear combination.  The candidates are
// kept doubled (S_i = 2 u_x,i, s_i = 2 u_xx,i): scaling by a power of two is
// exact, so every sum and product is the reference's times a power of two, and
// its products with 2 and 1/2 become the exact operand of a fused
// multiply-add: 11 operations for the six candidate values instead of 20.  The
// smoothness terms are then 4 times, their fourth powers 256 times the
// reference's, which cancels in the weights; dividing by twice the weights' sum
// undoes the doubling.
// TINY: the component may hold subnormal values, whose products with
// 1/2 round; the candidates then keep the reference's halves (17 operations).
// The smoothness terms may still use the doubled curvatures: below 1e-28 they
// vanish beside the 1e-12 they are added to.
// h0 = 3/2 u_0 (TINY), else 3 u_0.  top: running maximum of the high words of
// the divisors.
template <bool TINY>
__device__ __forceinline__ void weno3_dir(double m2, double m1, double u0, double p1, double p2, double h0,
                                          double& slope, double& curv, unsigned& top) {
  const double r13_3 = 13. / 3.;
  const double s0 = fma(-2.0, m1, m2) + u0;
  const double s1 = fma(-2.0, u0, m1) + p1;
  const double s2 = fma(-2.0, p1, u0) + p2;
  const double S0 = TINY ? fma(-2.0, m1, 0.5 * m2) + h0 : fma(-4.0, m1, m2) + h0;
  const double S1 = TINY ? 0.5 * (p1 - m1) : p1 - m1;
  const double S2 = TINY ? fma(2.0, p1, -h0) - 0.5 * p2 : fma(4.0, p1, -h0) - p2;
  // TINY: S^2 + (r s) s / 4 + eps, else 4 times that
  const double is0 = r13_3 * s0 * s0, is1 = r13_3 * s1 * s1, is2 = r13_3 * s2 * s2;
  const double eps = TINY ? SMALL_NUM : 4.0 * SMALL_NUM;
  const double d0 = pow4((TINY ? fma(0.25, is0, S0 * S0) : S0 * S0 + is0) + eps);
  const double d1 = pow4((TINY ? fma(0.25, is1, S1 * S1) : S1 * S1 + is1) + eps);
  const double d2 = pow4((TINY ? fma(0.25, is2, S2 * S2) : S2 * S2 + is2) + eps);
  top = max(top, max(max(hi_word(d0), hi_word(d1)), hi_word(d2)));
  double w0 = inv_y(d0, recip_nr(d0));
  double w1 = div_y(100.0, d1, recip_nr(d1));  // the central cell's linear weight
  double w2 = inv_y(d2, recip_nr(d2));
  const double total = w0 + w1 + w2;
  const double sum = TINY ? total : total + total;
  const double yt = recip_nr(sum);
  w0 = div_y(w0, sum, yt);
  w1 = div_y(w1, sum, yt);
  w2 = div_y(w2, sum, yt);
  slope = w0 * S0 + w1 * S1 + w2 * S2;
  if constexpr (TINY)
    curv = w0 * (0.5 * s0) + w1 * (0.5 * s1) + w2 * (0.5 * s2);
  else
    curv = w0 * s0 + w1 * s1 + w2 * s2;
}

// weno3 with every division done by fdiv.hpp's shared-reciprocal sequence.
// Same expressions and operation order as the reference weno3
// (reconstruction.c:144-221) up to exact scalings by powers of two, so the
// coefficients are bitwise those of the IEEE-division version whenever all
// divisors are in range; returns false otherwise (the caller then recomputes
// with plain division).  The divisors are the pow4 terms, >= 1e-48, and the
// weight sums; all are in range when every pow4 term is below 2^388.  The
// terms are positive (or NaN, whose high word is larger still), so their high
// words compare as they do.
//
// The stage kernel is bound by FP64 issue and this is half of a row's
// instructions: 248 per component, 258 where it may be subnormal (288 with the
// unscaled candidates, two Newton steps per reciprocal and FP64 range checks).  Measured over an SSP-RK
// solve: Kapila 1024x512 4802 -> 4503 us per 10 steps, Baer-Nunziato 2048x1024
// 9191 -> 8647 us per 3, Euler 256x256 2007 -> 1934 us per 20.
//
// A positive component (RANGE POSITIVE) is subnormal only where a phase vanishes.
// Its doubled candidates are exact wherever the cell's own value is far above the
// subnormal numbers: every candidate but the central slope contains that value, in
// whose sum a subnormal neighbour's rounded half is lost, and the central slope's
// is lost in the sum of the three.  Elsewhere (below 2^-800, or not positive, or
// beyond 2^610) the cell is left to the plain form too: two integer operations
// instead of weno3_dir<TINY>'s ten FP64 ones (Kapila 1024x512, 10 steps: 4136 and
// 4043 us; 48 Kapila grids 14955 and 14637).
constexpr unsigned POSITIVE_LOW_WORD = (1023u - 800u) << 20;  // high word of 2^-800

template <Range RANGE>
__device__ __forceinline__ bool weno3_fast(const double* U_x, const double* U_y, const double* U_xy,
                                           double* coeffs) {
  constexpr bool TINY = RANGE == ANY;
  const double u_0 = U_xy[0];
  const double h0 = (TINY ? 1.5 : 3.0) * u_0;
  // wraps below 2^-800 to more than FDIV_TOP_WORD
  unsigned top = RANGE == POSITIVE ? hi_word(u_0) - POSITIVE_LOW_WORD : 0;
  double c1, c2, c3, c4;
  weno3_dir<TINY>(U_x[0], U_x[1], u_0, U_x[3], U_x[4], h0, c1, c3, top);
  weno3_dir<TINY>(U_y[0], U_y[1], u_0, U_y[3], U_y[4], h0, c2, c4, top);
  coeffs[0] = u_0;
  coeffs[1] = c1;
  coeffs[2] = c2;
  coeffs[3] = c3;
  coeffs[4] = c4;

  // U_xy: u_0, u_ip1jp1, u_ip1jm1, u_im1jp1, u_im1jm1
  const double uxy0 = U_xy[1] - u_0 - c1 - c2 - c3 - c4;
  const double uxy1 = -U_xy[2] + u_0 + c1 - c2 + c3 + c4;
  const double uxy2 = -U_xy[3] + u_0 - c1 + c2 + c3 + c4;
  const double uxy3 = U_xy[4] - u_0 + c1 + c2 - c3 - c4;
  const double t = c3 * c3 + c4 * c4;
  const double d0 = pow4(fma(4.0, t, uxy0 * uxy0) + SMALL_NUM);
  const double d1 = pow4(fma(4.0, t, uxy1 * uxy1) + SMALL_NUM);
  const double d2 = pow4(fma(4.0, t, uxy2 * uxy2) + SMALL_NUM);
  const double d3 = pow4(fma(4.0, t, uxy3 * uxy3) + SMALL_NUM);
  top = max(top, max(max(hi_word(d0), hi_word(d1)), hi_word(d2)));
  top = max(top, hi_word(d3));
  double w0 = inv_y(d0, recip_nr(d0));
  double w1 = inv_y(d1, recip_nr(d1));
  double w2 = inv_y(d2, recip_nr(d2));
  double w3 = inv_y(d3, recip_nr(d3));
  const double total = w0 + w1 + w2 + w3;
  const double yt = recip_nr(total);
  w0 = div_y(w0, total, yt);
  w1 = div_y(w1, total, yt);
  w2 = div_y(w2, total, yt);
  w3 = div_y(w3, total, yt);
  coeffs[5] = w0 * uxy0 + w1 * uxy1 + w2 * uxy2 + w3 * uxy3;
  return top < FDIV_TOP_WORD;
}

// reconstruction.c:223-357: CWENO with one fourth-degree central candidate
// and five third-degree candidates (gamma_hi = gamma_lo = 0.85).  FAST divides
// with shared reciprocals, as weno3_fast does, and returns false where a divisor
// is out of their range; the other form divides plainly.  The 13 divisions were
// 182 of a component's issue slots and are 88; halving joins the additions where
// the component is never subnormal (TINY as in weno3_dir).  Kapila 256x256, 3
// RK104 steps: 1238 -> 1143 us; Baer-Nunziato 1024x1024, one step: 7642 -> 4319 us (its
// registers no longer spill as far).
template <bool FAST, bool TINY>
__device__ __forceinline__ bool weno4(const double* U_x, const double* U_y, const double* U_xy, double* coeffs) {
  // a + x / 2
  auto add_half = [](double a, double x) { return TINY ? a + 0.5 * x : fma(0.5, x, a); };
  constexpr double r1_6 = 1. / 6., r13_3 = 13. / 3., r7_6 = 7. / 6., r11_120 = 11. / 120., r1_12 = 1. / 12.,
                   r41_60 = 41. / 60.;
  const double gammaHi = 0.85, gammaLo = 0.85;
  double u_0 = U_xy[0];
  double u_ip1 = U_x[3], u_jp1 = U_y[3], u_ip1jp1 = U_xy[1];
  double u_im1 = U_x[1], u_jm1 = U_y[1], u_ip1jm1 = U_xy[2];
  double u_ip2 = U_x[4], u_jp2 = U_y[4], u_im1jp1 = U_xy[3];
  double u_im2 = U_x[0], u_jm2 = U_y[0], u_im1jm1 = U_xy[4];
  double gR3[5], xR3[5], yR3[5], xxR3[5], yyR3[5], xyR3[5], wR3[5];
  const double gR4 = gammaHi;
  gR3[0] = (1.0 - gammaHi) * gammaLo;
#pragma unroll
  for (int i = 1; i < 5; ++i) gR3[i] = 0.25 * (1 - gammaHi) * (1 - gammaLo);

  const double xR4 = r41_60 * (-u_im1 + u_ip1) + r11_120 * (u_im2 - u_ip2);
  const double yR4 = r41_60 * (-u_jm1 + u_jp1) + r11_120 * (u_jm2 - u_jp2);
  const double xxR4 = add_half(-u_0, u_im1 + u_ip1);
  const double yyR4 = add_half(-u_0, u_jm1 + u_jp1);
  const double xyR4 = 0.25 * (u_im1jm1 - u_im1jp1 - u_ip1jm1 + u_ip1jp1);
  const double xxxR4 = r1_6 * (u_im1 - u_ip1) + r1_12 * (u_ip2 - u_im2);
  const double yyyR4 = r1_6 * (u_jm1 - u_jp1) + r1_12 * (u_jp2 - u_jm2);
  const double xxyR4 = add_half(0.25 * (-u_im1jm1 + u_im1jp1 - u_ip1jm1 + u_ip1jp1), u_jm1 - u_jp1);
  const double xyyR4 = add_half(0.25 * (u_ip1jp1 - u_im1jm1 - u_im1jp1 + u_ip1jm1), u_im1 - u_ip1);
  const double IS_R4 = (xR4 + 0.1 * xxxR4) * (xR4 + 0.1 * xxxR4) + r13_3 * (xxR4 * xxR4 + yyR4 * yyR4) +
                       (yR4 + 0.1 * yyyR4) * (yR4 + 0.1 * yyyR4) + 39.05 * (xxxR4 * xxxR4 + yyyR4 * yyyR4) +
                       r7_6 * xyR4 * xyR4 + 4.7 * (xxyR4 * xxyR4 + xyyR4 * xyyR4);
  unsigned top = 0;
  auto weight = [&](double g, double IS) {
    const double d = pow4(IS + SMALL_NUM);
    top = max(top, hi_word(d));
    return FAST ? div_y(g, d, recip_nr(d)) : g / d;
  };
  double wR4 = weight(gR4, IS_R4);
  double sum = wR4;

  xR3[0] = 0.5 * (-u_im1 + u_ip1);
  yR3[0] = 0.5 * (-u_jm1 + u_jp1);
  xxR3[0] = xxR4;
  yyR3[0] = yyR4;
  xyR3[0] = xyR4;

  xR3[1] = add_half(fma(-2.0, u_im1, 1.5 * u_0), u_im2);
  yR3[1] = 0.5 * (-u_jm1 + u_jp1);
  xxR3[1] = add_half(add_half(-u_im1, u_0), u_im2);
  yyR3[1] = add_half(add_half(-u_0, u_jm1), u_jp1);
  xyR3[1] = 0.5 * (u_im1jm1 - u_im1jp1 - u_jm1 + u_jp1);

  xR3[2] = add_half(fma(2.0, u_ip1, -1.5 * u_0), -u_ip2);
  yR3[2] = 0.5 * (-u_jm1 + u_jp1);
  xxR3[2] = add_half(add_half(-u_ip1, u_0), u_ip2);
  yyR3[2] = yyR3[1];
  xyR3[2] = 0.5 * (-u_ip1jm1 + u_ip1jp1 + u_jm1 - u_jp1);

  xR3[3] = 0.5 * (-u_im1 + u_ip1);
  yR3[3] = add_half(fma(-2.0, u_jm1, 1.5 * u_0), u_jm2);
  xxR3[3] = add_half(add_half(-u_0, u_im1), u_ip1);
  yyR3[3] = add_half(add_half(-u_jm1, u_0), u_jm2);
  xyR3[3] = 0.5 * (-u_im1 + u_im1jm1 + u_ip1 - u_ip1jm1);

  xR3[4] = 0.5 * (-u_im1 + u_ip1);
  yR3[4] = add_half(fma(2.0, u_jp1, -1.5 * u_0), -u_jp2);
  xxR3[4] = xxR3[3];
  yyR3[4] = add_half(add_half(-u_jp1, u_0), u_jp2);
  xyR3[4] = 0.5 * (u_im1 - u_im1jp1 - u_ip1 + u_ip1jp1);

#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const double IS = xR3[i] * xR3[i] + yR3[i] * yR3[i] + r13_3 * (xxR3[i] * xxR3[i] + yyR3[i] * yyR3[i]) +
                      r7_6 * xyR3[i] * xyR3[i];
    wR3[i] = weight(gR3[i], IS);
    sum = sum + wR3[i];
  }
  const double ys = recip_nr(sum);
  wR4 = FAST ? div_y(wR4, sum, ys) : wR4 / sum;
#pragma unroll
  for (int i = 0; i < 5; ++i) wR3[i] = FAST ? div_y(wR3[i], sum, ys) : wR3[i] / sum;
  constexpr double yg = 1.0 / 0.85;  // rounded, as div_y needs it
  const double wt_ratio = FAST ? div_y(wR4, gR4, yg) : wR4 / gR4;

  auto coef = [&](double R4, const double* R3) {
    return wt_ratio * (R4 - gR3[0] * R3[0] - gR3[1] * R3[1] - gR3[2] * R3[2] - gR3[3] * R3[3] - gR3[4] * R3[4]) +
           wR3[0] * R3[0] + wR3[1] * R3[1] + wR3[2] * R3[2] + wR3[3] * R3[3] + wR3[4] * R3[4];
  };
  coeffs[0] = u_0;
  coeffs[1] = coef(xR4, xR3);
  coeffs[2] = coef(yR4, yR3);
  coeffs[3] = coef(xxR4, xxR3);
  coeffs[4] = coef(yyR4, yyR3);
  coeffs[5] = coef(xyR4, xyR3);
  coeffs[6] = wt_ratio * xxxR4;
  coeffs[7] = wt_ratio * yyyR4;
  coeffs[8] = wt_ratio * xxyR4;
  coeffs[9] = wt_ratio * xyyR4;
  return top < FDIV_TOP_WORD;
}

// Stencil of one component: x[0..4] = u(i-2..i+2, j), y[0..4] = u(i, j-2..j+2),
// d[0..4] = u(i,j), u(i+1,j+1), u(i+1,j-1), u(i-1,j+1), u(i-1,j-1)
// (rhs_function_prim.c:332-348).
template <int N, Range RANGE>
__device__ __forceinline__ void reconstruct(const double* U_x, const double* U_y, const double* U_xy,
                                            double* coeffs) {
  if constexpr (N == 0) {
    coeffs[0] = U_xy[0];
  } else if constexpr (N == 1) {
    // reconstruction.c:129-142
    double u_0 = U_xy[0];
    coeffs[0] = u_0;
    coeffs[1] = minmod(U_x[3] - u_0, u_0 - U_x[1]);
    coeffs[2] = minmod(U_y[3] - u_0, u_0 - U_y[1]);
  } else if constexpr (N == 3) {
    constexpr bool TINY = RANGE != NORMAL;
    if (!__builtin_expect((weno4<true, TINY>(U_x, U_y, U_xy, coeffs)), 1)) weno4<false, TINY>(U_x, U_y, U_xy, coeffs);
  } else {
    if (__builtin_expect(weno3_fast<RANGE>(U_x, U_y, U_xy, coeffs), 1)) return;
    // reconstruction.c:144-221
    const double central_cell_wt = 100.0;
    const double r13_3 = 13. / 3.;
    double u_0 = U_xy[0];
    double u_ip1 = U_x[3], u_jp1 = U_y[3], u_ip1jp1 = U_xy[1];
    double u_im1 = U_x[1], u_jm1 = U_y[1], u_ip1jm1 = U_xy[2];
    double u_ip2 = U_x[4], u_jp2 = U_y[4], u_im1jp1 = U_xy[3];
    double u_im2 = U_x[0], u_jm2 = U_y[0], u_im1jm1 = U_xy[4];
    double ux0, ux1, ux2, uxx0, uxx1, uxx2, w0, w1, w2, w3, total, temp;

    ux0 = -2.0 * u_im1 + 0.5 * u_im2 + 1.5 * u_0;
    uxx0 = 0.5 * (u_im2 - 2.0 * u_im1 + u_0);
    ux1 = 0.5 * (u_ip1 - u_im1);
    uxx1 = 0.5 * (u_im1 - 2.0 * u_0 + u_ip1);
    ux2 = -1.5 * u_0 + 2.0 * u_ip1 - 0.5 * u_ip2;
    uxx2 = 0.5 * (u_0 - 2.0 * u_ip1 + u_ip2);
    w0 = 1.0 / (pow4(ux0 * ux0 + r13_3 * uxx0 * uxx0 + SMALL_NUM));
    w1 = central_cell_wt / (pow4(ux1 * ux1 + r13_3 * uxx1 * uxx1 + SMALL_NUM));
    w2 = 1.0 / (pow4(ux2 * ux2 + r13_3 * uxx2 * uxx2 + SMALL_NUM));
    total = w0 + w1 + w2;
    w0 = w0 / total;
    w1 = w1 / total;
    w2 = w2 / total;
    coeffs[0] = u_0;
    coeffs[1] = w0 * ux0 + w1 * ux1 + w2 * ux2;
    coeffs[3] = w0 * uxx0 + w1 * uxx1 + w2 * uxx2;

    ux0 = -2.0 * u_jm1 + 0.5 * u_jm2 + 1.5 * u_0;
    uxx0 = 0.5 * (u_jm2 - 2.0 * u_jm1 + u_0);
    ux1 = 0.5 * (u_jp1 - u_jm1);
    uxx1 = 0.5 * (u_jm1 - 2.0 * u_0 + u_jp1);
    ux2 = -1.5 * u_0 + 2.0 * u_jp1 - 0.5 * u_jp2;
    uxx2 = 0.5 * (u_0 - 2.0 * u_jp1 + u_jp2);
    w0 = 1.0 / (pow4(ux0 * ux0 + r13_3 * uxx0 * uxx0 + SMALL_NUM));
    w1 = central_cell_wt / (pow4(ux1 * ux1 + r13_3 * uxx1 * uxx1 + SMALL_NUM));
    w2 = 1.0 / (pow4(ux2 * ux2 + r13_3 * uxx2 * uxx2 + SMALL_NUM));
    total = w0 + w1 + w2;
    w0 = w0 / total;
    w1 = w1 / total;
    w2 = w2 / total;
    coeffs[2] = w0 * ux0 + w1 * ux1 + w2 * ux2;
    coeffs[4] = w0 * uxx0 + w1 * uxx1 + w2 * uxx2;

    double c1 = coeffs[1], c2 = coeffs[2], c3 = coeffs[3], c4 = coeffs[4];
    double uxy0 = u_ip1jp1 - u_0 - c1 - c2 - c3 - c4;
    double uxy1 = -u_ip1jm1 + u_0 + c1 - c2 + c3 + c4;
    double uxy2 = -u_im1jp1 + u_0 - c1 + c2 + c3 + c4;
    double uxy3 = u_im1jm1 - u_0 + c1 + c2 - c3 - c4;
    temp = 4.0 * (c3 * c3 + c4 * c4);
    w0 = 1.0 / (pow4(temp + uxy0 * uxy0 + SMALL_NUM));
    w1 = 1.0 / (pow4(temp + uxy1 * uxy1 + SMALL_NUM));
    w2 = 1.0 / (pow4(temp + uxy2 * uxy2 + SMALL_NUM));
    w3 = 1.0 / (pow4(temp + uxy3 * uxy3 + SMALL_NUM));
    total = w0 + w1 + w2 + w3;
    w0 = w0 / total;
    w1 = w1 / total;
    w2 = w2 / total;
    w3 = w3 / total;
    coeffs[5] = w0 * uxy0 + w1 * uxy1 + w2 * uxy2 + w3 * uxy3;
  }
}

}  // namespace HYPE_KNS
