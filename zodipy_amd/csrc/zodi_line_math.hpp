// Elementary functions of the line kernels (gfx950), and the tables that they read.
//
//  * PowTable: x^p for an exponent p that is fixed for the launch (the temperature law,
//    the cloud's two powers). x = 2^e m, inv_j close to 1/m and short enough that
//    r = m inv_j - 1 is exact before its one rounding, x^p = 2^(p e) inv_j^-p (1 + r)^p:
//    two table entries and a binomial series of five terms, 12 operations where
//    exp(p log x) takes 32. The tables are built in LDS by each block from
//    the device model block (about 5 entries per thread).
//  * exp_neg_node: exp with its argument reduced in units of ln2/256 by two FMAs, 13
//    operations where exp_fast takes 15.
//
// Host builds (tests/test_line_math_accuracy.py, with g++) run the same steps on the same
// tables.
#pragma once

#include "zodi_math.hpp"
#include "zodi_trig.hpp"

#ifdef __HIPCC__
#include "zodi_device.hpp"
#endif

#ifndef __HIPCC__
struct double2 {
  double x, y;
};
#endif

namespace zodi {

// ---------------------------------------------------------------- host and device
#ifdef __HIPCC__
// 2^(j/256) in LDS (stage_line_tables).
__shared__ __attribute__((aligned(2048))) double g_exp2[256];

__constant__ double kLineInv[256] = {ZODI_LINE_INV_TABLE};  // inv_j of PowTable
__constant__ double kLineLog[256] = {ZODI_LINE_LOG_TABLE};  // -log inv_j
__constant__ double kLineAngle[258] = {ZODI_LINE_ANGLE_TABLE};
__constant__ double kExp2Lo[256] = {ZODI_EXP2_LO_TABLE};        // 2^(j/256) - g_exp2[j]
__constant__ double kLineLog2[512] = {ZODI_LINE_LOG2_TABLE};    // -log2 inv_j, two words

// Every thread of the block must call this before exp_neg_node.
__device__ __forceinline__ void stage_line_tables() {
  for (int i = threadIdx.x; i < 256; i += blockDim.x) g_exp2[i] = kMathTablesConst[i];
  __syncthreads();
}
#else
inline constexpr double kLineInv[256] = {ZODI_LINE_INV_TABLE};
inline constexpr double kLineLog[256] = {ZODI_LINE_LOG_TABLE};
inline constexpr double kLineAngle[258] = {ZODI_LINE_ANGLE_TABLE};
inline constexpr double kExp2Lo[256] = {ZODI_EXP2_LO_TABLE};
inline constexpr double kLineLog2[512] = {ZODI_LINE_LOG2_TABLE};
#endif

#if defined(__HIP_DEVICE_COMPILE__)
#define ZODI_LINE_EXP2 g_exp2
#else
#define ZODI_LINE_EXP2 kHostExp2
#endif

// Entry of a table in bytes from its start.
template <class T>
ZODI_MATH_FN T table_at(const T* tab, uint32_t bytes) {
  return *(const T*)((const char*)tab + bytes);
}

// Mantissa in [1/2, 1) and exponent of a positive normal number (NaN keeps its mantissa).
ZODI_MATH_FN double frexp_mant(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_frexp_mant(x);
#else
  int e;
  return std::frexp(x, &e);
#endif
}

ZODI_MATH_FN int frexp_exponent(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_frexp_exp(x);
#else
  int e;
  std::frexp(x, &e);
  return e;
#endif
}

// Conversions to 32-bit integers that saturate (NaN: 0), as the hardware's do; a C++ cast of a
// value out of range is undefined. The sources here are results of plain arithmetic, never of
// the reciprocal or root instructions, after which a reader needs a wait state that the
// compiler does not add before an asm.
ZODI_MATH_FN uint32_t saturate_u32(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t r;
  asm("v_cvt_u32_f64 %0, %1" : "=v"(r) : "v"(x));
  return r;
#else
  return x > 0.0 ? (x < 4294967296.0 ? (uint32_t)x : 0xffffffffu) : 0u;
#endif
}

ZODI_MATH_FN uint32_t saturate_u32(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t r;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
#else
  return saturate_u32((double)x);
#endif
}

ZODI_MATH_FN int saturate_i32(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  int r;
  asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(x));
  return r;
#else
  if (x != x) return 0;
  return x < -2147483648.0 ? INT32_MIN : (x > 2147483647.0 ? INT32_MAX : (int)x);
#endif
}

// ---------------------------------------------------------------- exp
// exp_neg_node: exp(-x) for |x| < 5.8e6 (NaN passes), within 1.2 ulp. With
// |x 256/ln2| < 2^31 the integer k = rint(x 256/ln2) is the low word of
// x 256/ln2 + 1.5 2^52 (x negated); f = x 256/ln2 - k by two FMAs, the second with what
// 256/ln2 leaves out of a double (one alone has an error of 1.4e-17 x, 1e-14 at x = 700; the
// second costs 1.8 % of the large forward batches, DIRBE 50.7 M rays 24.1 -> 24.5 ms, and 0.7
// to 0.9 % of the maps and gradients); exp(x) = 2^(k/256) (1 + q(f)), q the Taylor series of
// 2^(f/256) - 1 to f^4 (first term left out 3.8e-17).
//
// An FP64 instruction takes one scalar-register operand and no 64-bit literal, so a
// step with two constants needs one of them in a vector register. ExpConst holds them all
// for the whole kernel: rebuilt per use they would cost two moves each, and as vector
// operands the compiler copies them first to use the two-address FMA.
struct ExpConst {
  double shift, c3;                 // vector registers
  double inv_l, inv_lo, c1, c2, c4;  // scalar registers
};

ZODI_MATH_FN ExpConst exp_const() {
  ExpConst e = {0x1.8p52,                // rounds to an integer in the low word
                0x1.c6b08d704a0c0p-29,   // (ln2/256)^3/6
                kExpInvL,                // 256/ln2
                0x1.777d0ffda0d24p-48,   // 256/ln2 - kExpInvL
                0x1.62e42fefa39efp-9,    // ln2/256
                0x1.ebfbdff82c58fp-19,   // (ln2/256)^2/2
                0x1.3b2ab6fba4e77p-39};  // (ln2/256)^4/24
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(e.shift), "+v"(e.c3));
  asm volatile("" : "+s"(e.inv_l), "+s"(e.inv_lo), "+s"(e.c1), "+s"(e.c2), "+s"(e.c4));
#endif
  return e;
}

ZODI_MATH_FN double exp_node_tail(const ExpConst& e, double f, int k) {
  double q = fma(f, e.c4, e.c3);
  q = fma(q, f, e.c2);
  q = fma(q, f, e.c1);
  q = q * f;
  const double t = table_at(ZODI_LINE_EXP2, (uint32_t)k << 3 & 0x7f8u);
  return math_ldexp(fma(t, q, t), k >> 8);
}

// exp(-x)
ZODI_MATH_FN double exp_neg_node(const ExpConst& e, double x) {
  const double sh = fma(-x, e.inv_l, e.shift);
  const double kd = sh - e.shift;
  double f = fma(-x, e.inv_l, -kd);
  f = fma(-x, e.inv_lo, f);
  return exp_node_tail(e, f, (int)(uint32_t)__builtin_bit_cast(uint64_t, sh));
}

// exp(-x), |x| < 5.8e6, for 1 - exp(-x) and x exp(-x) (a band's radial cut-off): the one-word
// reduction adds at most 1.4e-17 x exp(-x) < 6e-18 and 1.4e-17 x^2 exp(-x) < 8e-18 to them.
ZODI_MATH_FN double exp_neg_cut(const ExpConst& e, double x) {
  const double sh = fma(-x, e.inv_l, e.shift);
  const double f = fma(-x, e.inv_l, -(sh - e.shift));
  return exp_node_tail(e, f, (int)(uint32_t)__builtin_bit_cast(uint64_t, sh));
}

// exp(-x) for any x above -5.8e6 up to 1e90 (the result underflows to 0 above 745 by
// itself: the integer conversion saturates, which still gives 0).
ZODI_MATH_FN double exp_neg_any(const ExpConst& e, double x) {
  const double kd = __builtin_rint(-x * e.inv_l);
  double f = fma(-x, e.inv_l, -kd);
  f = fma(-x, e.inv_lo, f);
  return exp_node_tail(e, f, saturate_i32(kd));
}

// ---------------------------------------------------------------- x^p, p fixed
// In LDS: entry j is (inv_j, inv_j^-p) for mantissas in [1/2 + j/512, 1/2 + (j+1)/512);
// scale[i] = factor 2^(p e) for the exponents e whose biased value is i modulo 256 and
// that lie in [e_first, e_first + 256). An argument outside [2^(e_first - 1),
// 2^(e_first + 255)) is the caller's to exclude (NaN passes).
struct PowTable {
  double2 c[256];
  double scale[256];
};

// Binomial coefficients of (1 + r)^p, r^1..r^5, in scalar registers but the fourth:
// |r| < 2^-8.9, the first term left out is below 8.4e-17 |binom(p, 6)|, for -1 <= p <= 6 at
// most 8.4e-17 (p = -1 and 6), 5e-18 for the temperature law of the registry.
struct PowPoly {
  double b1, b2, b3, b4, b5;
};

// A value that all lanes hold, moved to scalar registers. (With the builtin the compiler,
// which sees that the value is uniform, leaves it in vector registers.)
ZODI_MATH_FN double to_scalar(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint64_t v = __builtin_bit_cast(uint64_t, x);
  uint32_t lo, hi;
  // s_nop: a lane read needs a wait state after the vector write it reads, and a vector
  // or scalar read of the result further ones (the compiler adds none around an asm)
  asm volatile("s_nop 4\n\tv_readfirstlane_b32 %0, %2\n\tv_readfirstlane_b32 %1, %3\n\ts_nop 4"
               : "=&s"(lo), "=&s"(hi)
               : "v"((uint32_t)v), "v"((uint32_t)(v >> 32)));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
#else
  return x;
#endif
}

ZODI_MATH_FN PowPoly pow_poly(double p) {
  PowPoly q;
  q.b1 = p;
  q.b2 = q.b1 * (p - 1.0) * 0.5;
  q.b3 = q.b2 * (p - 2.0) * (1.0 / 3.0);
  q.b4 = q.b3 * (p - 3.0) * 0.25;
  q.b5 = q.b4 * (p - 4.0) * 0.2;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(q.b4));
#endif
  return {to_scalar(q.b1), to_scalar(q.b2), to_scalar(q.b3), q.b4, to_scalar(q.b5)};
}

// inv_j (kLineInv): 2/(1 + (j + 1/2)/256) rounded to a multiple of 2^-12 (13 significant
// bits), so its product with a 53-bit mantissa fits the FMA exactly and only r is rounded.

// factor 2^(zh + zl), |zl| tiny, rounded once: 2^(j/256) in two words, the series of
// 2^(f/256) - 1 to f^5 (first term left out 9e-21), and the product with `factor` exact.
ZODI_MATH_FN double exp2_scaled(const ExpConst& ec, double zh, double zl, double factor) {
  const double kd = __builtin_rint(zh * 256.0);
  const double f = fma(zh, 256.0, -kd) + zl * 256.0;
  double q = fma(f, 0x1.5d87fe78a6731p-50, ec.c4);  // (ln2/256)^5/120
  q = fma(q, f, ec.c3);
  q = fma(q, f, ec.c2);
  q = fma(q, f, ec.c1);
  const int k = saturate_i32(kd), j = k & 255;
  const double t = ZODI_LINE_EXP2[j];
  const double low = fma(t, q * f, kExp2Lo[j]);
  const double p = factor * t;
  return math_ldexp(p + fma(factor, low, fma(factor, t, -p)), k >> 8);
}

// Entries i, i + stride, ... of the table of x^p, the whole multiplied by `factor`;
// exponents from e_first on. Every entry is the exact value rounded once. Mean relative
// errors of x^p, 1e-16, with entries of exp's accuracy -> these, and of exp(p log x):
// temperature law (p = -0.233) 0.94 -> 0.81 and 0.64, cloud's radius (-0.67) 0.93 -> 0.77 and
// 1.1, its g (0.942) 0.91 -> 0.81 and 1.7; of T/dT on the table's axis (pow_table_less, where
// the last product is not rounded) the mean is 6.1e-15 and the largest 3.5e-14, where
// exp(p log x) gives 5.7e-15 and 6.3e-14. stage_line_tables() must have run.
ZODI_MATH_FN void build_pow_table(PowTable& t, const ExpConst& ec, double p, double factor,
                                  int e_first, int i, int stride) {
  for (int j = i; j < 256; j += stride) {
    const double lh = kLineLog2[2 * j], zh = p * lh;
    const double zl = fma(p, lh, -zh) + p * kLineLog2[2 * j + 1];
    t.c[j] = double2{kLineInv[j], exp2_scaled(ec, zh, zl, 1.0)};
  }
  for (int j = i; j < 256; j += stride) {
    const int e = e_first + j;
    const double zh = p * (double)e;
    const double zl = fma(p, (double)e, -zh);
    // frexp's exponent e: x = 2^e m, m in [1/2, 1); its biased exponent is e + 1022
    t.scale[(e + 1022) & 255] = exp2_scaled(ec, zh, zl, factor);
  }
}

// inv_j^-p and factor 2^(p e) (1 + r)^p, whose product is factor x^p, for x in the table's
// range (NaN passes).
ZODI_MATH_FN double2 pow_factors(const PowTable& t, const PowPoly& q, double x) {
  const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, x) >> 32);
  const double m = frexp_mant(x);
  // byte offsets: 16 (hi >> 12 & 255) and 8 (hi >> 20 & 255), a shift right and an and
  // each (2 cycles apiece; a shift left takes 4)
  const double2 c = table_at(t.c, hi >> 8 & 0xff0u);
  const double s = table_at(t.scale, hi >> 17 & 0x7f8u);
  const double r = fma(m, c.x, -1.0);
  double y = fma(r, q.b5, q.b4);
  y = fma(y, r, q.b3);
  y = fma(y, r, q.b2);
  y = fma(y, r, q.b1);
  y = y * r;
  return double2{c.y, fma(s, y, s)};
}

// factor x^p
ZODI_MATH_FN double pow_table(const PowTable& t, const PowPoly& q, double x) {
  const double2 w = pow_factors(t, q, x);
  return w.x * w.y;
}

// factor x^p - u, the product unrounded (the temperature on the Planck table's axis)
ZODI_MATH_FN double pow_table_less(const PowTable& t, const PowPoly& q, double x, double u) {
  const double2 w = pow_factors(t, q, x);
  return fma(w.x, w.y, -u);
}

// ---------------------------------------------------------------- log
// log x for positive normal x from a table of (inv_j, -log inv_j) (kLineInv) and the
// Taylor series of log(1 + r) to r^5, |r| < 2^-8.9 (first term left out 1.4e-17); e ln2 with
// both words of ln2 (with one the error is 2.3e-17 |e| more).
struct LogConst {
  double c4;                   // vector register: -1/4
  double c5, c3, ln2, ln2_lo;  // scalar registers
};

ZODI_MATH_FN LogConst log_const() {
  LogConst l = {-0.25, 0.2, 1.0 / 3.0, 0x1.62e42fefa39efp-1, 0x1.abc9e3b39803fp-56};
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(l.c4));
  asm volatile("" : "+s"(l.c5), "+s"(l.c3), "+s"(l.ln2), "+s"(l.ln2_lo));
#endif
  return l;
}

ZODI_MATH_FN double log_node(const double2* tab, const LogConst& l, double x) {
  const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, x) >> 32);
  const double m = frexp_mant(x);
  const double de = (double)frexp_exponent(x);
  const double2 c = table_at(tab, hi >> 8 & 0xff0u);
  const double r = fma(m, c.x, -1.0);
  double p = fma(r, l.c5, l.c4);
  p = fma(p, r, l.c3);
  p = fma(p, r, -0.5);
  const double l1p = fma(p * r, r, r);
  return fma(de, l.ln2, c.y + fma(de, l.ln2_lo, l1p));
}

// ---------------------------------------------------------------- angles
// Angle of the unit vector (c, s), s >= 0, from the x axis: turned by the nearest of 129
// tabulated directions j C, C the double nearest pi/128, found from the arc cosine in single
// precision (within 4e-4, Abramowitz and Stegun 4.4.45), its sine is below 0.0127 and the arc
// sine's series ends at the seventh power (next term 1e-18): 11 FP64 operations and no
// quotient where axis_angle takes some 37. The table holds the directions of the exact
// products j C, so that the last FMA is the angle's only rounding. An error that c and s
// share (of 1/|X|) only scales the small turn. Near 0 the direction is (1, 0), so the angle
// keeps the digits of s.
struct AngleTable {
  double2 e[129];
};

// Entries i, i + stride, ...
ZODI_MATH_FN void load_angles(AngleTable& t, int i, int stride) {
  for (; i < 129; i += stride) t.e[i] = double2{kLineAngle[2 * i], kLineAngle[2 * i + 1]};
}

ZODI_MATH_FN double unit_angle(const AngleTable& t, double c, double s) {
  constexpr float kPerRad = 40.743665f;  // 128 / pi
  const float x = (float)c, a = fminf(fabsf(x), 1.0f);
  float q = fmaf(a, -0.0187293f * kPerRad, 0.0742610f * kPerRad);
  q = fmaf(q, a, -0.2121144f * kPerRad);
  q = fmaf(q, a, 1.5707288f * kPerRad);
#if defined(__HIP_DEVICE_COMPILE__)
  q *= __builtin_amdgcn_sqrtf(1.0f - a);
#else
  q *= sqrtf(1.0f - a);
#endif
  q = x < 0.0f ? 128.0f - q : q;
  const uint32_t j = saturate_u32(rintf(q)) & 0xffu;
  const uint32_t jc = j < 128u ? j : 128u;  // NaN converts to 0
  const double2 e = t.e[jc];
  const double d = fma(s, e.x, -(c * e.y)), z = d * d;
  double w = fma(z, 15.0 / 336.0, 3.0 / 40.0);
  w = fma(w, z, 1.0 / 6.0);
  return fma((double)jc, 0x1.921fb54442d18p-6, fma(d * z, w, d));
}

// Angle of (x, y) from the x axis, in [0, pi]; the octant, half-angle and quadrant steps of
// atan2_fast as multiplications by 0, 1 and -1 instead of selections: the angle is
// +-atan(t) + k pi/4 for an integer k, with both words of pi/4.
ZODI_MATH_FN double axis_angle(double x, double y) {
  constexpr double kP[] = {ZODI_ATAN_POLY};
  const double m = fmax(fabs(x), fabs(y)), n = fmin(fabs(x), fabs(y));
  const double up = n > zodi_trig::kTanPi8 * m ? 1.0 : 0.0;
  const double t = zodi_trig::quotient(fma(-up, m, n), fma(up, n, m));
  const double s = t * t;
  const double a = fma(t * s, zodi_trig::horner(kP, s), t);
  const double sw = fabs(y) > fabs(x) ? -1.0 : 1.0;
  const double sx = __builtin_copysign(1.0, x);
  // sx (sw (a + up pi/4) + (1 - sw) pi/4) + (1 - sx) pi/2
  const double k = fma(sx, fma(sw, up - 1.0, -1.0), 2.0);
  const double r = fma(k, zodi_trig::kPiQuarterHi, (sx * sw) * a);
  return fma(k, zodi_trig::kPiQuarterLo, r);
}

// asin(s) for 0 <= s <= 1 (the reduction of acos_fast). The half above 1/2 costs a
// square root and is entered only by the waves that have such a point.
ZODI_MATH_FN double asin_unit(double s) {
  constexpr double kQ[] = {ZODI_ASIN_POLY};
  double w = s, z = s * s, up = 0.0;
  if (s > 0.5) {
    z = fma(-0.5, s, 0.5);
#if defined(__HIP_DEVICE_COMPILE__)
    double inv;
    norm_and_inverse(z, w, inv);
    w = z == 0.0 ? 0.0 : w;
#else
    w = sqrt(z);
#endif
    up = 1.0;
  }
  const double v = fma(w * z, zodi_trig::horner(kQ, z), w);
  // pi/2 - 2 asin(sqrt((1 - s)/2)) above 1/2
  const double r = fma(up, zodi_trig::kPiHalfHi, fma(-3.0 * up, v, v));
  return fma(up, zodi_trig::kPiHalfLo, r);
}

}  // namespace zodi
