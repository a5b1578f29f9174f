// FP64 sine and cosine for the particle maps.
//
// The maps count their phases in turns (phx_turns_n below).  Arguments in
// radians (the wake functions; a few hundred at most):  For |x| < 2^20 the argument is reduced by Cody and
// Waite's method with pi/2 split into P1 + P2 + P3: P1 and P2 carry 33
// significant bits, so k*P1 and k*P2 are exact for |k| < 2^20 and x - k*P1
// is exact (both are multiples of ulp(x) there); the remainder
// r = x - k*pi/2, |r| <~ pi/4, is then within ~1 ulp.  sin(r) and cos(r)
// are their Taylor series to r^17 and r^16 (truncation below 1e-19 at
// pi/4), evaluated by Horner's rule in r^2, and the quadrant k mod 4 picks
// and signs them.  Larger arguments go to the device library through calls
// kept out of line that return by value (an output pointer would put the
// results, and the callers' every launch, on scratch memory).
//
// The constants: P1, P2 are pi/2 truncated to 33 and the next 33 bits, P3
// the rest rounded to double (pi from Machin's formula to 80 digits);
// 2/pi rounded to double; the coefficients are (-1)^k/(2k+1)! and
// (-1)^k/(2k)! rounded to double.
#pragma once

#include <hip/hip_runtime.h>

namespace phx_math {

constexpr double TWO_OVER_PI = 0x1.45f306dc9c883p-1;
constexpr double PIO2_1 = 0x1.921fb54400000p+0;
constexpr double PIO2_2 = 0x1.0b4611a600000p-34;
constexpr double PIO2_3 = 0x1.3198a2e037073p-69;
constexpr double REDUCE_MAX = 0x1p20;

// sin: r + r^3 * (S1 + r^2 (S2 + ...)),  S_k = (-1)^k / (2k+1)!
constexpr double S1 = -1.0 / 6.0;
constexpr double S2 = 1.0 / 120.0;
constexpr double S3 = -1.0 / 5040.0;
constexpr double S4 = 1.0 / 362880.0;
constexpr double S5 = -1.0 / 39916800.0;
constexpr double S6 = 1.0 / 6227020800.0;
constexpr double S7 = -1.0 / 1307674368000.0;
constexpr double S8 = 1.0 / 355687428096000.0;
// cos: 1 + r^2 * (C1 + r^2 (C2 + ...)),  C_k = (-1)^k / (2k)!
constexpr double C1 = -0.5;
constexpr double C2 = 1.0 / 24.0;
constexpr double C3 = -1.0 / 720.0;
constexpr double C4 = 1.0 / 40320.0;
constexpr double C5 = -1.0 / 3628800.0;
constexpr double C6 = 1.0 / 479001600.0;
constexpr double C7 = -1.0 / 87178291200.0;
constexpr double C8 = 1.0 / 20922789888000.0;

// sin and cos of r + r_lo, |r| <= ~pi/4, with r_lo the tail of the reduced
// argument: sin(r + r_lo) ~ sin(r) + r_lo cos(r), cos(r + r_lo) ~
// cos(r) - r_lo sin(r), both folded in before the last rounding.
__host__ __device__ __forceinline__ void kernel_sincos(double r, double r_lo, double &s,
                                                       double &c) {
  const double z = r * r;
  double ps = S8;
  ps = fma(ps, z, S7);
  ps = fma(ps, z, S6);
  ps = fma(ps, z, S5);
  ps = fma(ps, z, S4);
  ps = fma(ps, z, S3);
  ps = fma(ps, z, S2);
  ps = fma(ps, z, S1);
  double pc = C8;
  pc = fma(pc, z, C7);
  pc = fma(pc, z, C6);
  pc = fma(pc, z, C5);
  pc = fma(pc, z, C4);
  pc = fma(pc, z, C3);
  pc = fma(pc, z, C2);
  pc = fma(pc, z, C1);
  // 1 + z*pc - r*r_lo: the tail enters through the low part of z*pc
  const double zpc = z * pc;
  const double zpc_lo = fma(z, pc, -zpc) - r * r_lo;
  c = 1.0 + (zpc + zpc_lo);
  s = r + fma(r * z, ps, r_lo * (1.0 + zpc));
}

// Argument reduction: x - k*pi/2 = r + r_lo and the quadrant k mod 4.
// x - k*P1 is exact; the subtraction of k*P2 (exact product) is done as an
// exact two-sum, k*P3 is a correction far below ulp(r).
__host__ __device__ __forceinline__ double reduce(double x, double &r_lo, int &quadrant) {
  const double k = rint(x * TWO_OVER_PI);
  const double a = fma(-k, PIO2_1, x);
  const double b = k * PIO2_2;
  const double w = k * PIO2_3;
  const double hi = a - b;
  const double bv = a - hi;  // two-sum of a and -b
  const double lo = (a - (hi + bv)) + (bv - b);
  const double r = hi - w;
  r_lo = ((hi - r) - w) + lo;
  quadrant = ((int)k) & 3;
  return r;
}

// sin(2 pi r) = r T(r^2) and cos(2 pi r) = 1 + r^2 U(r^2) for |r| <= 1/8:
// the polynomials that interpolate sin(2 pi sqrt(z))/sqrt(z) and
// (cos(2 pi sqrt(z)) - 1)/z at the Chebyshev nodes of [0, 1/64] (degree 6,
// formed in 70-digit arithmetic and rounded to double; within 3.5e-18
// relative and 1.3e-19 absolute of the functions).
constexpr double T0 = 0x1.921fb54442d18p+2;
constexpr double T1 = -0x1.4abbce625be41p+5;
constexpr double T2 = 0x1.466bc677587f8p+6;
constexpr double T3 = -0x1.32d2cce2e5b18p+6;
constexpr double T4 = 0x1.50782fda12c1ep+5;
constexpr double T5 = -0x1.e30071afacecep+3;
constexpr double T6 = 0x1.e3f38390face5p+1;
constexpr double U1 = -0x1.3bd3cc9be45dep+4;
constexpr double U2 = 0x1.03c1f081b5ac0p+6;
constexpr double U3 = -0x1.55d3c7e3cb241p+6;
constexpr double U4 = 0x1.e1f5068688d5ap+5;
constexpr double U5 = -0x1.a6d1eef479ab9p+4;
constexpr double U6 = 0x1.f9ce245c9b912p+2;
constexpr double U7 = -0x1.b2f3eafeb9c45p+0;
constexpr double TURNS_MAX = 0x1p40;
constexpr double TWO_PI = 0x1.921fb54442d18p+2;
constexpr double INV_TWO_PI = 1.0 / TWO_PI;
constexpr double TWO_PI_REL = -0x1.678afae35cdd1p-55;  // TWO_PI / (2 pi) - 1

__device__ __noinline__ double cos_library(double x) { return ::cos(x); }

__device__ __noinline__ double sin_library(double x) { return ::sin(x); }

}  // namespace phx_math

// -v where bit 1 of quadrant is set.
__device__ __forceinline__ double phx_flip(double v, int quadrant) {
  return __longlong_as_double(__double_as_longlong(v) ^
                              ((long long)((unsigned)(quadrant & 2) << 30) << 32));
}

// sin(x_k) and cos(x_k) of M arguments; within ~1 ulp for |x| < 2^20, the
// device library's values beyond (and for NaN / infinity).  The M reductions
// and polynomials run in lockstep (2 M independent chains of dependent FP64
// operations, which the compiler interleaves), with one branch for arguments
// out of range after all of them: a branch per argument keeps each chain in a
// basic block of its own, and a wave then waits for one chain at a time.
template <int M>
__device__ __forceinline__ void phx_sincos_n(const double (&x)[M], double (&sp)[M],
                                             double (&cp)[M]) {
  bool far = false;
#pragma unroll
  for (int k = 0; k < M; ++k) {
    int q;
    double r_lo, s, c;
    const double r = phx_math::reduce(x[k], r_lo, q);
    phx_math::kernel_sincos(r, r_lo, s, c);
    // quadrant q: (sin, cos) = (s, c), (c, -s), (-s, -c), (-c, s)
    sp[k] = phx_flip((q & 1) ? c : s, q);
    cp[k] = phx_flip((q & 1) ? s : c, q + 1);
    far |= !(fabs(x[k]) < phx_math::REDUCE_MAX);
  }
  if (__builtin_expect(far, 0)) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
      if (fabs(x[k]) < phx_math::REDUCE_MAX) continue;
      sp[k] = phx_math::sin_library(x[k]);
      cp[k] = phx_math::cos_library(x[k]);
    }
  }
}

// Sine and cosine of the maps' phases, counted in turns: u minus its nearest
// quarter is exact, so no multiple of pi has to be subtracted in parts and the
// reduced argument has no tail.  The quarter is rounded off by adding
// 1.5 * 2^52, whose sum's low bits are the quadrant.  |u| >= 2^40 (and NaN,
// infinity) go to the library.
// COS (the betatron phases): sin(t) and cos(t) of t = u * (2.*np.pi) as the
// reference rounds it; its distance from 2 pi u (up to 7e-15 rad by the
// product's rounding and 5e-15 by the constant's at a tune of 20, ten times
// what the rest of a segment map rounds) is put back after the reduction,
// with three operations.  33 operations a pair against 45 with the reduction
// in radians.  Otherwise (RF phases) sin(2 pi u) alone.
template <int M, bool COS>
__device__ __forceinline__ void phx_turns_n(const double (&u)[M], double (&sp)[M],
                                            double (&cp)[M]) {
  using namespace phx_math;
  bool far = false;
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const double t = fma(u[k], 4.0, 0x1.8p52);
    const int q = (int)__double_as_longlong(t);
    double r = fma(t - 0x1.8p52, -0.25, u[k]);
    if constexpr (COS) {
      const double th = u[k] * TWO_PI;
      r = fma(u[k], TWO_PI_REL, r);
      r = fma(fma(u[k], TWO_PI, -th), -INV_TWO_PI, r);
    }
    const double z = r * r;
    double ps = fma(T6, z, T5);
    ps = fma(ps, z, T4);
    ps = fma(ps, z, T3);
    ps = fma(ps, z, T2);
    ps = fma(ps, z, T1);
    ps = fma(ps, z, T0);
    double pc = fma(U7, z, U6);
    pc = fma(pc, z, U5);
    pc = fma(pc, z, U4);
    pc = fma(pc, z, U3);
    pc = fma(pc, z, U2);
    pc = fma(pc, z, U1);
    const double s = r * ps, c = fma(pc, z, 1.0);
    sp[k] = phx_flip((q & 1) ? c : s, q);
    if constexpr (COS) cp[k] = phx_flip((q & 1) ? s : c, q + 1);
    far |= !(fabs(u[k]) < TURNS_MAX);
  }
  if (__builtin_expect(far, 0)) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
      if (fabs(u[k]) < TURNS_MAX) continue;
      sp[k] = sin_library(u[k] * TWO_PI);
      if constexpr (COS) cp[k] = cos_library(u[k] * TWO_PI);
    }
  }
}

template <int M>
__device__ __forceinline__ void phx_sincos_turns_n(const double (&u)[M], double (&sp)[M],
                                                   double (&cp)[M]) {
  phx_turns_n<M, true>(u, sp, cp);
}

template <int M>
__device__ __forceinline__ void phx_sin_turns_n(const double (&u)[M], double (&sp)[M]) {
  phx_turns_n<M, false>(u, sp, sp);
}

__device__ __forceinline__ void phx_sincos(double x, double *sp, double *cp) {
  const double a[1] = {x};
  double s[1], c[1];
  phx_sincos_n<1>(a, s, c);
  *sp = s[0];
  *cp = c[0];
}

__device__ __forceinline__ double phx_sin(double x) {
  double s, c;
  phx_sincos(x, &s, &c);
  return s;
}
