// The line-of-sight node arithmetic of the Kelsall registry kernels (gfx950).
//
// What bounds these kernels is the issue of FP64 vector instructions: measured on
// MI355X, an FP64 operation, a three-operand integer operation or a shift left
// takes a SIMD 4 cycles, a plain 32-bit and/add/shift right 2, v_rsq_f64 and
// v_rcp_f64 16. (FP64 MFMA shares the vector unit: 8 FMAs and one 16x16x4 MFMA
// take the sum of their times.) So everything here takes work out of the node loop:
//
//  * Line: a ray is parametrised by its signed distance t from the point P closest to
//    the Sun, X = P + t V with V a unit vector normal to P. Then |X|^2 = t^2 + |P|^2,
//    the distance from a component's symmetry plane is A + t B and the squared
//    distance from its centre (t - t_c)^2 + d_c^2, with A, B, t_c, d_c formed once per
//    ray: a node's geometry takes one operation for t and one for |X|^2 instead of
//    seven, a plane distance one instead of three, an offset centre two instead of
//    six. Both squares are sums of non-negative terms, so nothing cancels: the error
//    of |X| is that of the position itself.
//  * PowTable: x^p for an exponent p that is fixed for the launch (the temperature law,
//    the cloud's two powers). x = 2^e m, inv_j close to 1/m and short enough that
//    r = m inv_j - 1 is exact before its one rounding, x^p = 2^(p e) inv_j^-p (1 + r)^p:
//    two table entries and a binomial series of five terms, 12 operations where
//    exp(p log x) takes 32. The tables are built in LDS by each block from
//    the device model block (about 5 entries per thread).
//  * exp_neg_node: exp with its argument reduced in units of ln2/256 (the product with
//    256/ln2, whose rounded value is within 1.5e-17 relative of the exact one, inside
//    one FMA), 12 operations instead of 15.
#pragma once

#include "zodi_device.hpp"
#include "zodi_line_domain.hpp"

namespace zodi {

// ---------------------------------------------------------------- the ray's line
// X(t) = P + t V; t = n s + t0 for the distance s along the pointing (n its length,
// 1 up to rounding; a zero vector gives n = 0 and V = 0, so that X stays the
// observer, as s u + o does).
struct Line {
  double px, py, pz, vx, vy, vz;
  double n, t0, d2;
};

__device__ __forceinline__ Line make_line(double ux, double uy, double uz, double ox, double oy,
                                          double oz) {
  Line l;
  const double uu = fma(ux, ux, fma(uy, uy, uz * uz));
  double inv;
  norm_and_inverse(uu, l.n, inv);
  if (uu == 0.0) {
    l.n = 0.0;
    inv = 0.0;
  }
  l.vx = ux * inv;
  l.vy = uy * inv;
  l.vz = uz * inv;
  l.t0 = fma(l.vx, ox, fma(l.vy, oy, l.vz * oz));
  l.px = fma(-l.t0, l.vx, ox);
  l.py = fma(-l.t0, l.vy, oy);
  l.pz = fma(-l.t0, l.vz, oz);
  l.d2 = fma(l.px, l.px, fma(l.py, l.py, l.pz * l.pz));
  return l;
}

// a + b t along the line.
struct Linear {
  double a, b;
  __device__ __forceinline__ double at(double t) const { return fma(b, t, a); }
};

// The linear form c . (X - (x0, y0, z0)).
__device__ __forceinline__ Linear line_form(const Line& l, double cx, double cy, double cz,
                                            double x0, double y0, double z0) {
  return {fma(cx, l.px - x0, fma(cy, l.py - y0, cz * (l.pz - z0))),
          fma(cx, l.vx, fma(cy, l.vy, cz * l.vz))};
}

__device__ __forceinline__ Linear line_form(const Line& l, double cx, double cy, double cz) {
  return {fma(cx, l.px, fma(cy, l.py, cz * l.pz)), fma(cx, l.vx, fma(cy, l.vy, cz * l.vz))};
}

// |X - X0|^2 = (t - tc)^2 + d2 along the line.
struct OffsetLine {
  double tc, d2;
  __device__ __forceinline__ double r2(double t) const {
    const double d = t - tc;
    return fma(d, d, d2);
  }
};

__device__ __forceinline__ OffsetLine offset_line(const Line& l, double x0, double y0, double z0) {
  const double qx = l.px - x0, qy = l.py - y0, qz = l.pz - z0;
  OffsetLine o;
  o.tc = -fma(qx, l.vx, fma(qy, l.vy, qz * l.vz));
  const double wx = fma(o.tc, l.vx, qx), wy = fma(o.tc, l.vy, qy), wz = fma(o.tc, l.vz, qz);
  o.d2 = fma(wx, wx, fma(wy, wy, wz * wz));
  return o;
}

// ---------------------------------------------------------------- exp
// exp_neg_node: exp(-x) for |x| < 5.8e6 (NaN passes), within 1 ulp + 1.5e-17 |x| relative. With
// |x 256/ln2| < 2^31 the integer k = rint(x 256/ln2) is the low word of
// x 256/ln2 + 1.5 2^52 (x negated); f = x 256/ln2 - k in one FMA; exp(x) = 2^(k/256) (1 + q(f)),
// q the Taylor series of 2^(f/256) - 1 to f^4 (first term left out 3.8e-17).
//
// An FP64 instruction takes one scalar-register operand and no 64-bit literal, so a
// step with two constants needs one of them in a vector register. ExpConst holds them all
// for the whole kernel: rebuilt per use they would cost two moves each, and as vector
// operands the compiler copies them first to use the two-address FMA.
struct ExpConst {
  double shift, c3;          // vector registers
  double inv_l, c1, c2, c4;  // scalar registers
};

__device__ __forceinline__ ExpConst exp_const() {
  ExpConst e = {0x1.8p52,              // rounds to an integer in the low word
                0x1.c6b08d704a0c0p-29,  // (ln2/256)^3/6
                kExpInvL,               // 256/ln2
                0x1.62e42fefa39efp-9,   // ln2/256
                0x1.ebfbdff82c58fp-19,  // (ln2/256)^2/2
                0x1.3b2ab6fba4e77p-39};  // (ln2/256)^4/24
  asm volatile("" : "+v"(e.shift), "+v"(e.c3));
  asm volatile("" : "+s"(e.inv_l), "+s"(e.c1), "+s"(e.c2), "+s"(e.c4));
  return e;
}

// 2^(j/256) in LDS (stage_line_tables).
__shared__ __attribute__((aligned(2048))) double g_exp2[256];

__constant__ double kLineInv[256] = {ZODI_LINE_INV_TABLE};  // inv_j of PowTable
__constant__ double kLineLog[256] = {ZODI_LINE_LOG_TABLE};  // -log inv_j

// Every thread of the block must call this before exp_neg_node.
__device__ __forceinline__ void stage_line_tables() {
  for (int i = threadIdx.x; i < 256; i += blockDim.x) g_exp2[i] = kMathTablesConst[i];
  __syncthreads();
}

__device__ __forceinline__ double exp_node_tail(const ExpConst& e, double f, int k) {
  double q = fma(f, e.c4, e.c3);
  q = fma(q, f, e.c2);
  q = fma(q, f, e.c1);
  q = q * f;
  const double t = *(const double*)((const char*)g_exp2 + ((uint32_t)(k << 3) & 0x7f8u));
  return __builtin_amdgcn_ldexp(fma(t, q, t), k >> 8);
}

// exp(-x)
__device__ __forceinline__ double exp_neg_node(const ExpConst& e, double x) {
  const double sh = fma(-x, e.inv_l, e.shift);
  const double kd = sh - e.shift;
  const double f = fma(-x, e.inv_l, -kd);
  return exp_node_tail(e, f, (int)(uint32_t)__builtin_bit_cast(uint64_t, sh));
}

// exp(-x) for any x above -5.8e6 up to 9e15 (the result underflows to 0 above 745 by
// itself: the integer conversion saturates, which still gives 0).
__device__ __forceinline__ double exp_neg_any(const ExpConst& e, double x) {
  const double kd = __builtin_rint(-x * e.inv_l);
  const double f = fma(-x, e.inv_l, -kd);
  return exp_node_tail(e, f, (int)kd);
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

// Binomial coefficients of (1 + r)^p, r^1..r^5, in scalar registers but the fourth: |r| < 2^-8.9, the
// first term left out is below 2^-53.4 |binom(p, 6)| < 5e-17 for -1 <= p <= 6.
struct PowPoly {
  double b1, b2, b3, b4, b5;
};

// A value that all lanes hold, moved to scalar registers. (With the builtin the compiler,
// which sees that the value is uniform, leaves it in vector registers.)
__device__ __forceinline__ double to_scalar(double x) {
  const uint64_t v = __builtin_bit_cast(uint64_t, x);
  uint32_t lo, hi;
  // s_nop: a lane read needs a wait state after the vector write it reads, and a vector
  // or scalar read of the result further ones (the compiler adds none around an asm)
  asm volatile("s_nop 4\n\tv_readfirstlane_b32 %0, %2\n\tv_readfirstlane_b32 %1, %3\n\ts_nop 4"
               : "=&s"(lo), "=&s"(hi)
               : "v"((uint32_t)v), "v"((uint32_t)(v >> 32)));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ PowPoly pow_poly(double p) {
  PowPoly q;
  q.b1 = p;
  q.b2 = q.b1 * (p - 1.0) * 0.5;
  q.b3 = q.b2 * (p - 2.0) * (1.0 / 3.0);
  q.b4 = q.b3 * (p - 3.0) * 0.25;
  q.b5 = q.b4 * (p - 4.0) * 0.2;
  asm volatile("" : "+v"(q.b4));
  return {to_scalar(q.b1), to_scalar(q.b2), to_scalar(q.b3), q.b4, to_scalar(q.b5)};
}

// inv_j (kLineInv): 2/(1 + (j + 1/2)/256) rounded to a multiple of 2^-12 (13 significant
// bits), so its product with a 53-bit mantissa fits the FMA exactly and only r is rounded.

// 2^z for the exact z = zh + zl, |zl| tiny.
__device__ __forceinline__ double exp2_table(const ExpConst& ec, double zh, double zl) {
  const double k = __builtin_rint(zh);
  const double f = (zh - k) + zl;
  constexpr double kLn2Hi = 0x1.62e42fefa39efp-1, kLn2Lo = 0x1.abc9e3b39803fp-56;
  const double y = f * kLn2Hi;
  const double yl = fma(f, kLn2Hi, -y) + f * kLn2Lo;
  const double e = exp_neg_any(ec, -y);
  return __builtin_amdgcn_ldexp(fma(e, yl, e), (int)k);
}

// Entries i, i + stride, ... of the table of x^p, the whole multiplied by `factor`;
// exponents from e_first on. stage_line_tables() must have run.
__device__ __forceinline__ void build_pow_table(PowTable& t, const ExpConst& ec, double p,
                                                double factor, int e_first, int i, int stride) {
  for (int j = i; j < 256; j += stride) {
    // inv^-p; -p log(inv) is below |p| 0.7, so its rounding stays below an ulp
    t.c[j] = double2{kLineInv[j], exp_neg_any(ec, -(p * kLineLog[j]))};
  }
  for (int j = i; j < 256; j += stride) {
    const int e = e_first + j;
    const double zh = p * (double)e;
    const double zl = fma(p, (double)e, -zh);
    // frexp's exponent e: x = 2^e m, m in [1/2, 1); its biased exponent is e + 1022
    t.scale[(e + 1022) & 255] = factor * exp2_table(ec, zh, zl);
  }
}

// factor x^p from the table, for x in the table's range (NaN passes).
__device__ __forceinline__ double pow_table(const PowTable& t, const PowPoly& q, double x) {
  const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, x) >> 32);
  const double m = __builtin_amdgcn_frexp_mant(x);
  // byte offsets: 16 (hi >> 12 & 255) and 8 (hi >> 20 & 255), a shift right and an and
  // each (2 cycles apiece; a shift left takes 4)
  const double2 c = *(const double2*)((const char*)t.c + ((hi >> 8) & 0xff0u));
  const double s = *(const double*)((const char*)t.scale + ((hi >> 17) & 0x7f8u));
  const double r = fma(m, c.x, -1.0);
  double y = fma(r, q.b5, q.b4);
  y = fma(y, r, q.b3);
  y = fma(y, r, q.b2);
  y = fma(y, r, q.b1);
  y = y * r;
  const double w = c.y * s;
  return fma(w, y, w);
}

// Exponent ranges: squared radii from 2^-101 (below which a position's own rounding,
// 1e-16 AU, leaves nothing of it) to 2^155, and the cloud's g from 2^-254 to 2^2; the host
// sends blocks that can leave them to the general kernel (zodi_line_domain.hpp).
constexpr int kPowRadiusFirst = -100;
constexpr int kPowUnitFirst = -253;

// ---------------------------------------------------------------- Planck table
// In LDS, shifted by one entry: entry 0 is (B_0, 0), entry i (T_{i-1}'s interval) is
// (B_{i-1}, B_i - B_{i-1}), and from the last temperature on (B_last, 0). With
// u' = (T - T_first)/dT + 1 the unsigned conversion of u' takes everything below the
// table to entry 0 and one integer minimum everything above it to the last entry, whose
// zero differences give the end values of np.interp: five operations without a clamp of u'.
// NaN passes (fract keeps it).
__device__ __forceinline__ void load_planck(ModelPtr M, double2* tab, int i, int stride) {
  const int n = M->n_temps;
  for (; i <= ZODI_N_TEMPS; i += stride) {
    const int k = i - 1;
    const bool in = i >= 1 && k < n - 1;
    const int kc = k < 0 ? 0 : (k > n - 1 ? n - 1 : k);
    const double b = M->tab_B[kc];
    tab[i] = double2{b, in ? M->tab_B[kc + 1] - b : 0.0};
  }
}

__device__ __forceinline__ double planck_shifted(double u1, const double2* tab) {
  uint32_t j = (uint32_t)u1;  // saturating: 0 below 0 and for NaN
  j = j < (uint32_t)ZODI_N_TEMPS ? j : (uint32_t)ZODI_N_TEMPS;
  const double2 e = tab[j];
  return fma(__builtin_amdgcn_fract(u1), e.y, e.x);
}

// ---------------------------------------------------------------- angles
// Angle of the unit vector (c, s), s >= 0, from the x axis: turned by the nearest of 129
// tabulated directions j pi/128, found from the arc cosine in single precision (within
// 4e-4, Abramowitz and Stegun 4.4.45), its sine is below 0.0127 and the arc sine's series
// ends at the seventh power (next term 1e-18): 11 FP64 operations and no quotient where
// axis_angle takes some 35. An error that c and s share (of 1/|X|) only scales the small
// turn. Near 0 the direction is (1, 0), so the angle keeps the digits of s.
struct AngleTable {
  double2 e[129];
};

__constant__ double kLineAngle[258] = {ZODI_LINE_ANGLE_TABLE};

__device__ __forceinline__ void load_angles(AngleTable& t) {
  for (int i = threadIdx.x; i < 129; i += blockDim.x)
    t.e[i] = double2{kLineAngle[2 * i], kLineAngle[2 * i + 1]};
}

__device__ __forceinline__ double unit_angle(const AngleTable& t, double c, double s) {
  constexpr float kPerRad = 40.743665f;  // 128 / pi
  const float x = (float)c, a = fminf(fabsf(x), 1.0f);
  float q = fmaf(a, -0.0187293f * kPerRad, 0.0742610f * kPerRad);
  q = fmaf(q, a, -0.2121144f * kPerRad);
  q = fmaf(q, a, 1.5707288f * kPerRad);
  q *= __builtin_amdgcn_sqrtf(1.0f - a);
  q = x < 0.0f ? 128.0f - q : q;
  const uint32_t j = (uint32_t)rintf(q) & 0xffu;
  const uint32_t jc = j < 128u ? j : 128u;  // NaN converts to 0
  const double2 e = t.e[jc];
  const double d = fma(s, e.x, -(c * e.y)), z = d * d;
  double w = fma(z, 15.0 / 336.0, 3.0 / 40.0);
  w = fma(w, z, 1.0 / 6.0);
  return fma((double)jc, 0x1.921fb54442d18p-6, fma(d * z, w, d));
}

// ---------------------------------------------------------------- per-launch tables
struct LineTables {
  PowTable temperature;  // T0/dT (|X|^2)^(-delta/2)
  PowTable radial;       // the cloud's n_0 (r^2)^(-alpha/2)
  PowTable vertical;     // the cloud's g^gamma
  double2 planck[ZODI_N_TEMPS + 1];
  AngleTable angles;
};

// Everything the node loops read besides the model block.
struct LineCtx {
  ModelPtr M;
  const LineTables* tab;
  PowPoly pt, pr, pv;
  double uo1;  // T_first/dT - 1
  ExpConst ec;
  int K, sub;
};

// Builds the block's tables (every thread of the block must call it).
__device__ __forceinline__ LineCtx line_ctx(ModelPtr M, LineTables& tab, int sub) {
  stage_line_tables();
  const ExpConst ec = exp_const();
  const int i = threadIdx.x, n = blockDim.x;
  const ParamPtr P = M->comp[0];  // the cloud (the layouts' first component)
  const double pt = -0.5 * M->group_delta[0], pr = -0.5 * P[7], pv = P[9];
  build_pow_table(tab.temperature, ec, pt, M->group_T0[0] * M->tab_inv_step, kPowRadiusFirst, i, n);
  build_pow_table(tab.radial, ec, pr, P[6], kPowRadiusFirst, i, n);
  build_pow_table(tab.vertical, ec, pv, 1.0, kPowUnitFirst, i, n);
  load_planck(M, tab.planck, i, n);
  load_angles(tab.angles);
  __syncthreads();
  LineCtx cx;
  cx.M = M;
  cx.tab = &tab;
  cx.pt = pow_poly(pt);
  cx.pr = pow_poly(pr);
  cx.pv = pow_poly(pv);
  cx.uo1 = to_scalar(M->tab_T[0] * M->tab_inv_step - 1.0);
  cx.ec = ec;
  cx.K = M->n_nodes;
  cx.sub = sub;
  return cx;
}

// ---------------------------------------------------------------- densities
// The reference's densities (see zodi_device.hpp for each expression's source) on the
// line's linear forms; LineComp<KIND> holds a component's constants for one ray.
template <int KIND>
struct LineComp;

template <>
struct LineComp<ZODI_CLOUD> {
  OffsetLine o;
  Linear z;
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : o(offset_line(l, P[ZODI_P_X0], P[ZODI_P_Y0], P[ZODI_P_Z0])),
        z(line_form(l, P[ZODI_P_NX], -P[ZODI_P_NY], P[ZODI_P_NZ], P[ZODI_P_X0], P[ZODI_P_Y0],
                    P[ZODI_P_Z0])) {}
};

template <>
struct LineComp<ZODI_BAND> {  // the plane normal over delta_zeta
  Linear z;
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : z(line_form(l, P[ZODI_P_D0 + 3], -P[ZODI_P_D0 + 4], P[ZODI_P_D0 + 5])) {}
};

template <>
struct LineComp<ZODI_RING> {
  Linear z;
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : z(line_form(l, P[ZODI_P_NX], -P[ZODI_P_NY], P[ZODI_P_NZ])) {}
};

template <>
struct LineComp<ZODI_FEATURE> {  // x, y: the point rotated by the centre line's longitude
  Linear z, x, y;
  FeatureDir d;
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double ex, double ey)
      : z(line_form(l, P[ZODI_P_NX], -P[ZODI_P_NY], P[ZODI_P_NZ])),
        d(feature_dir(P, ex, ey)) {
    x = line_form(l, d.c, d.s, 0.0);
    y = line_form(l, -d.s, d.c, 0.0);
  }
};

struct LineNode {
  double t, R2, R, inv_R;
};

__device__ __forceinline__ double line_cloud(ParamPtr P, const LineComp<ZODI_CLOUD>& c,
                                             const LineCtx& cx, const LineNode& nd) {
  const double mu = P[10], inv_2mu = P[13];
  const double r2 = c.o.r2(nd.t);
  double r, inv_r;
  norm_and_inverse_node(r2, r, inv_r);
  const double zeta = fabs(c.z.at(nd.t)) * inv_r;
  // m^2/(2 mu) + (zeta - m) with m = min(zeta, mu): the reference's two cases without a
  // selection (two vcc-masked moves in a row stall the SIMD for about 20 cycles)
  const double m = fmin(zeta, mu);
  const double g = fma(m * m, inv_2mu, zeta - m);
  // the floor changes nothing: with gamma >= 1/2 both powers are below 2^-126
  const double gg = pow_table(cx.tab->vertical, cx.pv, fmax(g, 0x1p-253));
  return pow_table(cx.tab->radial, cx.pr, r2) * exp_neg_node(cx.ec, P[8] * gg);
}

// What a band of the line kernels does with its cut-off term: forms it for itself, forms
// it for the bands of its group that share it too, or takes the published one.
enum BandCut { kCutOwn = 0, kCutPublish = 1, kCutReuse = 2 };

// exp(-zeta_d^6) is 0 from 746 on: those nodes add nothing and are left out for the waves
// whose lanes all lie there (a map's rings at higher latitudes). NaN takes the branch.
template <int CUT>
__device__ __forceinline__ double line_band(ParamPtr P, const LineComp<ZODI_BAND>& c,
                                            const LineCtx& cx, const LineNode& nd, double& cut) {
  double term4;
  if constexpr (CUT == kCutReuse) {
    term4 = cut;
  } else {
    const double y = nd.R2 * P[ZODI_P_D0 + 6];
    const double y2 = y * y;
    const double y4 = y2 * y2;
    const double x = (y4 * y4) * y2;
    double ex = 0.0;
    if (x < 38.0) ex = exp_neg_node(cx.ec, x);
    term4 = 1.0 - ex;
    if constexpr (CUT == kCutPublish) cut = term4;
  }
  const double zd = fabs(c.z.at(nd.t)) * nd.inv_R;
  const double zd2 = zd * zd;
  const double zd4 = zd2 * zd2;
  const double zd6 = zd4 * zd2;
  double n = 0.0;
  if (!(zd6 >= 746.0)) {
    const double term3 = fma(zd4, P[14], 1.0);
    n = (P[6] * nd.inv_R) * exp_neg_node(cx.ec, zd6) * term3 * term4;
  }
  return n;
}

__device__ __forceinline__ double line_ring(ParamPtr P, const LineComp<ZODI_RING>& c,
                                            const LineCtx& cx, const LineNode& nd) {
  const double d = nd.R - P[7];
  return P[6] * exp_neg_any(cx.ec, fma(d * d, P[13], fabs(c.z.at(nd.t)) * P[14]));
}

// Angle of (x, y) from the x axis, in [0, pi]; the octant, half-angle and quadrant steps of
// atan2_fast as multiplications by 0, 1 and -1 instead of selections.
__device__ __forceinline__ double axis_angle(double x, double y) {
  constexpr double kP[] = {ZODI_ATAN_POLY};
  const double m = fmax(fabs(x), fabs(y)), n = fmin(fabs(x), fabs(y));
  const double up = n > zodi_trig::kTanPi8 * m ? 1.0 : 0.0;
  const double t = zodi_trig::quotient(fma(-up, m, n), fma(up, n, m));
  const double s = t * t;
  double a = fma(t * s, zodi_trig::horner(kP, s), t);
  a = fma(up, zodi_trig::kPiQuarterHi, a);
  const double sw = fabs(y) > fabs(x) ? -1.0 : 1.0;
  a = fma(sw, a, fma(-sw, zodi_trig::kPiQuarterHi, zodi_trig::kPiQuarterHi));
  const double sx = __builtin_copysign(1.0, x);
  return fma(sx, a, fma(-sx, zodi_trig::kPiHalfHi, zodi_trig::kPiHalfHi));
}

// What the scattering angle needs of a ray: d = |P| and, for a pointing whose length is not
// 1, k = 1 - n^2 (0 below 1e-12, where the length is 1 up to rounding).
struct LinePhase {
  double d, k;
};

__device__ __forceinline__ LinePhase line_phase(const Line& l) {
  const double k = fma(-l.n, l.n, 1.0);
  return {sqrt(l.d2), fabs(k) < 1e-12 ? 0.0 : k};
}

// Phase function at the node (phase_function): the scattering angle is
// arccos(-u . X / |X|), whose cosine is -n t / |X|. As the angle of (-n t, sqrt(|X|^2 -
// n^2 t^2)) it needs no quotient by |X| and keeps its digits near 0 and pi, where the
// arc cosine loses half of them; for a unit pointing the second is the ray's d.
__device__ __forceinline__ double scattering_angle(const LinePhase& p, const Line& l, double t) {
  double y = p.d;
  if (p.k != 0.0) y = sqrt(fmax(fma(t * t, p.k, l.d2), 0.0));  // clipped like the cosine
  return axis_angle(-l.n * t, y);
}

__device__ __forceinline__ double scattering_angle(const LinePhase& p, const Line& l, double t,
                                                   const AngleTable& tab, double inv_R) {
  if (p.k != 0.0) return scattering_angle(p, l, t);
  return unit_angle(tab, (-l.n * t) * inv_R, p.d * inv_R);
}

__device__ __forceinline__ double line_phase_function(const LinePhase& p, const Line& l,
                                                      const AngleTable& tab, const ExpConst& e,
                                                      double t, double inv_R, ParamPtr S) {
  const double theta = scattering_angle(p, l, t, tab, inv_R);
  return S[ZODI_S_PHASE_NORM] *
         (S[ZODI_S_C1] + S[ZODI_S_C2] * theta + exp_neg_any(e, -(S[ZODI_S_C3] * theta)));
}

// |theta| of the feature at the node: the angle of the rotated point from the centre line,
// by the table, with its y, rho^2 and 1/rho (of a point scaled up where rho^2 would leave
// the normal range).
__device__ __forceinline__ double feature_angle(const LineComp<ZODI_FEATURE>& c, const Line& l,
                                                const AngleTable& tab, double t, double& y,
                                                double& rho2, double& inv_rho) {
  double x = c.x.at(t);
  y = c.y.at(t);
  rho2 = fma(x, x, y * y);
  double r2 = rho2, rho;
  if (r2 < 0x1p-900) {
    if (x == 0.0 && y == 0.0) {  // on the axis: see feature_dtheta
      const double sg = __builtin_signbit(fma(l.vx, t, l.px)) ? -1.0 : 1.0;
      x = sg * c.d.c;
      y = -sg * c.d.s;
    } else {
      x *= 0x1p600;
      y *= 0x1p600;
    }
    r2 = fma(x, x, y * y);
  }
  norm_and_inverse_node(r2, rho, inv_rho);
  return unit_angle(tab, x * inv_rho, fabs(y) * inv_rho);
}

__device__ __forceinline__ double line_feature(ParamPtr P, const LineComp<ZODI_FEATURE>& c,
                                               const LineCtx& cx, const Line& l,
                                               const LineNode& nd) {
  const double d = nd.R - P[7];
  double e = (d * d) * P[13];
  e = fma(fabs(c.z.at(nd.t)), P[14], e);
  double y, rho2, inv_rho;
  const double theta = feature_angle(c, l, cx.tab->angles, nd.t, y, rho2, inv_rho);
  e = fma(theta * theta, P[15], e);
  return P[6] * exp_neg_any(cx.ec, e);
}

}  // namespace zodi
