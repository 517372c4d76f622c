// FP64 functions of the pair terms, written for gfx950's FP64 pipe: sine and
// cosine of a phase difference, the square root of a squared separation and a
// division by a launch constant.  The pair walks evaluate them per partner, so
// their instruction counts set the FP64 forms' rate: an FP64 instruction issues
// in 4 cycles per wavefront, as an FP32 one, and the general library functions
// take 60-70 (sin), 17 (sqrt) and 12 (division) of them for the whole range of
// doubles.  Compiled with -ffp-contract=off: every fused operation is written
// out.
#pragma once

#include <hip/hip_runtime.h>

namespace spc2 {

// pi = kPiHi + kPiLo to 107 bits (the nearest double and the nearest double to
// the rest); kRound: adding it rounds a double below 2^51 in magnitude to the
// nearest whole number, whose parity is then bit 0 of the sum.
constexpr double kPiHi = 0x1.921fb54442d18p+1, kPiLo = 0x1.1a62633145c07p-53, kInvPi = 0x1.45f306dc9c883p-2;
constexpr double kRound = 0x1.8p+52;
constexpr double kTrigMax = 0x1p+45;  // larger arguments, infinities and NaN take the library functions

// a * b + c, c a constant in scalar registers.  The compiler forms an accumulating
// v_fmac for these and copies each coefficient into its destination first, 7 more
// instructions per sine; in vector registers the coefficients, hoisted out of the
// walks, took 14 of them (a wavefront per SIMD less in the chimera cell walks: 143
// against 134 us in pass 1 at N = 262,144, 168 against 160 in pass 2).
__device__ __forceinline__ double fma3(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}

// sin(r) for |r| <= pi / 2 (and a hair beyond): r + r^3 p(r^2), p the degree-7
// minimax polynomial of (sin(r) / r - 1) / r^2 in relative error of sin, found
// by a Remez exchange in 60-digit arithmetic; the fit's error is 2^-61.6.
__device__ __forceinline__ double sin_half_turn(double r) {
  const double z = r * r;
  double p = fma3(0x1.882935a9c68d3p-49, z, -0x1.ae43199df130ap-41);
  p = fma3(p, z, 0x1.6123cb1a05428p-33);
  p = fma3(p, z, -0x1.ae6454cb1cd5fp-26);
  p = fma3(p, z, 0x1.71de3a52874a4p-19);
  p = fma3(p, z, -0x1.a01a01a0148abp-13);
  p = fma3(p, z, 0x1.11111111110c1p-7);
  p = fma3(p, z, -0x1.5555555555555p-3);
  return __builtin_fma(r * z, p, r);
}

// The library's functions, for arguments outside the fast reduction: called, not
// inlined, so that their registers do not count against the pair walks'.
static __device__ __attribute__((noinline, cold)) double sin_any(double x) { return sin(x); }
static __device__ __attribute__((noinline, cold)) double cos_any(double x) { return cos(x); }

__device__ __forceinline__ double flip_sign(double s, int odd) {
  return __hiloint2double(__double2hiint(s) ^ (odd << 31), __double2loint(s));
}

// sin(x) for |x| <= kTrigMax: x = k pi + r, k the nearest whole number.  k pi_hi
// is a multiple of 2^-51, so x - k pi_hi is exact in one fma, and the part of
// k pi beyond pi_hi + pi_lo stays below 2^-62.  18 FP64-rate instructions; at
// most 1.64 ulp off and 3.8e-17 rms over |x| <= 2000 (a correctly rounded sine:
// 2.7e-17), far below the rounding of the sums of 30 to 150 such terms.
__device__ __forceinline__ double sin_fast(double x) {
  const double kr = __builtin_fma(x, kInvPi, kRound), k = kr - kRound;
  const double r = __builtin_fma(-k, kPiLo, __builtin_fma(-k, kPiHi, x));
  return flip_sign(sin_half_turn(r), __double2loint(kr));
}

// cos(x) for |x| <= kTrigMax: x = (k + 1/2) pi + r, cos(x) = -(-1)^k sin(r).
__device__ __forceinline__ double cos_fast(double x) {
  const double kr = __builtin_fma(x, kInvPi, -0.5) + kRound, k = (kr - kRound) + 0.5;
  const double r = __builtin_fma(-k, kPiLo, __builtin_fma(-k, kPiHi, x));
  return flip_sign(sin_half_turn(r), ~__double2loint(kr));
}

// The same for any x.  FAST: the caller has checked the phases (phase_fits).
template <bool FAST = false>
__device__ __forceinline__ double sin_term(double x) {
  if (!FAST && __builtin_expect(!(__builtin_fabs(x) <= kTrigMax), 0)) return sin_any(x);
  return sin_fast(x);
}
template <bool FAST = false>
__device__ __forceinline__ double cos_term(double x) {
  if (!FAST && __builtin_expect(!(__builtin_fabs(x) <= kTrigMax), 0)) return cos_any(x);
  return cos_fast(x);
}

// Whether differences of such phases stay within kTrigMax.
__device__ __forceinline__ bool phase_fits(double p) { return __builtin_fabs(p) <= kTrigMax / 4; }

// sqrt(a) of a squared separation: the hardware estimate of 1 / sqrt(a) and two
// Goldschmidt steps with a residual correction, the correctly rounded root for
// normal a without the library's scaling of denormals; 0 for a == 0 and NaN for
// NaN (a separation that is not finite fails every test of the root, as with the
// library's).  For 0 <= a < 1e300 and NaN only.
__device__ __forceinline__ double sqrt_sep(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  e = __builtin_fma(-g, g, a);
  g = __builtin_fma(e, h, g);
  e = __builtin_fma(-g, g, a);
  g = __builtin_fma(e, h, g);
  return a > 0.0 ? g : a;
}

// a / c for a launch constant c with rc = 1 / c rounded: the product and one
// residual correction (Markstein), the correctly rounded quotient for normal
// values; 3 instructions.
__device__ __forceinline__ double div_by(double a, double c, double rc) {
  const double q = a * rc;
  return __builtin_fma(__builtin_fma(-q, c, a), rc, q);
}

}  // namespace spc2
