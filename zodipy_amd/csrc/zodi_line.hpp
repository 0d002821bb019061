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
//  * Powers, exponentials, logarithms and angles from tables in LDS (zodi_line_math.hpp).
#pragma once

#include "zodi_device.hpp"
#include "zodi_line_domain.hpp"
#include "zodi_line_math.hpp"

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

// ---------------------------------------------------------------- power tables
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
  uint32_t j = saturate_u32(u1);  // saturating: 0 below 0 and for NaN
  j = j < (uint32_t)ZODI_N_TEMPS ? j : (uint32_t)ZODI_N_TEMPS;
  const double2 e = tab[j];
  return fma(__builtin_amdgcn_fract(u1), e.y, e.x);
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
  load_angles(tab.angles, i, n);
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

// The same with powers as exp(p log x), for the passes that need the logarithms anyway (the
// gradients, RRM) and for exponents that the power tables do not hold (line_match).
struct LineLogTables {
  double2 log_tab[256];
  double2 planck[ZODI_N_TEMPS + 1];
};

struct LineLogCtx {
  ModelPtr M;
  const LineLogTables* tab;
  ExpConst ec;
  LogConst lc;
  int K, sub, split;
  bool share;  // gradients: band 3 takes band 1's cut-off (props_match with kShareCut)
  const AngleTable* angles;
  static constexpr bool kAngles = false;
};

// Builds the block's tables, `angles` too if given (every thread of the block must call it).
__device__ __forceinline__ LineLogCtx line_log_ctx(ModelPtr M, LineLogTables& tab,
                                                   AngleTable* angles = nullptr) {
  stage_line_tables();
  for (int j = threadIdx.x; j < 256; j += blockDim.x)
    tab.log_tab[j] = double2{kLineInv[j], kLineLog[j]};
  load_planck(M, tab.planck, threadIdx.x, blockDim.x);
  if (angles != nullptr) load_angles(*angles, threadIdx.x, blockDim.x);
  __syncthreads();
  LineLogCtx cx;
  cx.M = M;
  cx.tab = &tab;
  cx.ec = exp_const();
  cx.lc = log_const();
  cx.K = M->n_nodes;
  cx.sub = 0;
  cx.split = 1;
  cx.share = false;
  cx.angles = angles;
  return cx;
}

// A group's temperature law as the node loop takes it: T/dT - T_first/dT + 1.
struct LineLaw {
  double half_delta, us, uo1;
};

__device__ __forceinline__ LineLaw line_law(const LineCtx& cx, int) { return {0.0, 0.0, cx.uo1}; }

__device__ __forceinline__ LineLaw line_law(const LineLogCtx& cx, int g) {
  const ModelPtr M = cx.M;
  return {to_scalar(0.5 * M->group_delta[g]), to_scalar(M->group_T0[g] * M->tab_inv_step),
          to_scalar(M->tab_T[0] * M->tab_inv_step - 1.0)};
}

__device__ __forceinline__ double line_axis(const LineCtx& cx, const LineLaw& law, double R2) {
  return pow_table_less(cx.tab->temperature, cx.pt, R2, law.uo1);
}

__device__ __forceinline__ double line_axis(const LineLogCtx& cx, const LineLaw& law, double R2) {
  const double Rd = exp_neg_any(cx.ec, law.half_delta * log_node(cx.tab->log_tab, cx.lc, R2));
  return fma(Rd, law.us, -law.uo1);
}

// The cloud's density from r^2 and g. The floor under g changes nothing: with gamma >= 1/2
// both powers are below 2^-126.
__device__ __forceinline__ double cloud_profile(ParamPtr P, const LineCtx& cx, double r2,
                                                double g) {
  const double gg = pow_table(cx.tab->vertical, cx.pv, fmax(g, 0x1p-253));
  return pow_table(cx.tab->radial, cx.pr, r2) * exp_neg_node(cx.ec, P[8] * gg);
}

__device__ __forceinline__ double cloud_profile(ParamPtr P, const LineLogCtx& cx, double r2,
                                                double g) {
  const double lg = log_node(cx.tab->log_tab, cx.lc, fmax(g, 0x1p-253));
  const double gg = exp_neg_any(cx.ec, -(P[9] * lg));
  const double lr = log_node(cx.tab->log_tab, cx.lc, r2);
  return P[6] * exp_neg_any(cx.ec, fma(0.5 * P[7], lr, P[8] * gg));
}

__device__ __forceinline__ const AngleTable& line_angles(const LineCtx& cx) {
  return cx.tab->angles;
}
__device__ __forceinline__ const AngleTable& line_angles(const LineLogCtx& cx) {
  return *cx.angles;
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

template <class CTX>
__device__ __forceinline__ double line_cloud(ParamPtr P, const LineComp<ZODI_CLOUD>& c,
                                             const CTX& cx, const LineNode& nd) {
  const double mu = P[10], inv_2mu = P[13];
  const double r2 = c.o.r2(nd.t);
  double r, inv_r;
  norm_and_inverse_node(r2, r, inv_r);
  const double zeta = fabs(c.z.at(nd.t)) * inv_r;
  // m^2/(2 mu) + (zeta - m) with m = min(zeta, mu): the reference's two cases without a
  // selection (two vcc-masked moves in a row stall the SIMD for about 20 cycles)
  const double m = fmin(zeta, mu);
  const double g = fma(m * m, inv_2mu, zeta - m);
  return cloud_profile(P, cx, r2, g);
}

// What a band of the line kernels does with its cut-off term: forms it for itself, forms
// it for the bands of its group that share it too, or takes the published one.
enum BandCut { kCutOwn = 0, kCutPublish = 1, kCutReuse = 2 };

// exp(-zeta_d^6) is 0 from 746 on: those nodes add nothing and are left out for the waves
// whose lanes all lie there (a map's rings at higher latitudes). NaN takes the branch.
template <int CUT, class CTX>
__device__ __forceinline__ double line_band(ParamPtr P, const LineComp<ZODI_BAND>& c,
                                            const CTX& cx, const LineNode& nd, double& cut) {
  double term4;
  if constexpr (CUT == kCutReuse) {
    term4 = cut;
  } else {
    const double y = nd.R2 * P[ZODI_P_D0 + 6];
    const double y2 = y * y;
    const double y4 = y2 * y2;
    const double x = (y4 * y4) * y2;
    double ex = 0.0;
    if (x < 38.0) ex = exp_neg_cut(cx.ec, x);
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

template <class CTX>
__device__ __forceinline__ double line_ring(ParamPtr P, const LineComp<ZODI_RING>& c,
                                            const CTX& cx, const LineNode& nd) {
  const double d = nd.R - P[7];
  return P[6] * exp_neg_any(cx.ec, fma(d * d, P[13], fabs(c.z.at(nd.t)) * P[14]));
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

template <class CTX>
__device__ __forceinline__ double line_feature(ParamPtr P, const LineComp<ZODI_FEATURE>& c,
                                               const CTX& cx, const Line& l,
                                               const LineNode& nd) {
  const double d = nd.R - P[7];
  double e = (d * d) * P[13];
  e = fma(fabs(c.z.at(nd.t)), P[14], e);
  double y, rho2, inv_rho;
  const double theta = feature_angle(c, l, line_angles(cx), nd.t, y, rho2, inv_rho);
  e = fma(theta * theta, P[15], e);
  return P[6] * exp_neg_any(cx.ec, e);
}

}  // namespace zodi
