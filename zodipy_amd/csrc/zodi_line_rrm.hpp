// The Rowan-Robinson & May components on the ray's line (gfx950): densities for the forward
// kernel and their partials for the adjoint and Jacobian passes.
//
// Bound by FP64 vector issue. Beside the line's geometry (zodi_line.hpp):
//
//  * One logarithm of |X|^2 per node serves the temperature law and every radial power;
//    a component's powers and exponentials multiply as one exponential of a sum.
//  * The fan's and comet's latitude term sin(|beta|^eps) is |sin(beta)| = |Z|/R wherever
//    |Z| >= Z_0 (eps = 1): the arc sine, the power and the sine run only for the waves that
//    have a point closer to the plane, cos(beta)^Q is exp(Q/2 log(1 - sin^2 beta)).
//  * Bands whose mask or latitude limit leaves no lane of a wave are skipped.
//
// zodipy/number_density.py:184-404, zodipy/brightness.py:59-83.
#pragma once

#include "zodi_line_adjoint.hpp"

namespace zodi {

// sin(beta) of a point, its size capped at 1 (1/R carries an error of 5e-15).
__device__ __forceinline__ double line_sin_beta(const Linear& z, const GradNode& nd, double& zc) {
  zc = z.at(nd.t);
  return fmin(fabs(zc) * nd.inv_R, 1.0);
}

// The fan's and comet's sin(|beta|^eps): zc, the size of sin(beta) and log |beta| terms are
// needed by the partials.
struct LatSine {
  double su;                      // sin(u), u = |beta|^eps
  double cu, du_db, u_logb, beta;  // cos(u), |du/dbeta|, u log|beta|, |beta|
  bool inner;
};

template <bool GRAD>
__device__ __forceinline__ LatSine lat_sine(const LineLogCtx& cx, ParamPtr P, double Z0,
                                            double inv_Z0, double za, double s, double cb) {
  LatSine o;
  o.su = s;
  o.cu = cb;
  o.du_db = 1.0;
  o.u_logb = 0.0;
  o.beta = 0.0;
  o.inner = za < Z0;
  if (o.inner) {
    const double eps = fma(-za, inv_Z0, 2.0);
    const double b = asin_unit(s);
    const double bb = fmax(b, 0x1p-500);  // |beta| = 0: u = 0 to 2^-500
    const double lb = log_node(cx.tab->log_tab, cx.lc, bb);
    const double u = exp_neg_any(cx.ec, -(eps * lb));
    double sn, cn;
    zodi_trig::sincos_moderate(u, &sn, &cn);
    o.su = b > 0.0 ? sn : 0.0;
    if constexpr (GRAD) {
      o.cu = cn;
      o.du_db = b > 0.0 ? eps * u * rcp_fast(bb) : 0.0;
      o.u_logb = b > 0.0 ? u * lb : 0.0;
      o.beta = b;
    }
  }
  return o;
}

// The RRM kinds' constants for one ray: a plane, and what their exponents need in scalar
// registers (halved, since lR2 is log |X|^2).
struct PlaneComp {
  Linear z;
  double hg;  // gamma/2
  __device__ __forceinline__ PlaneComp(ParamPtr P, const Line& l, double gamma)
      : z(line_form(l, P[ZODI_P_NX], -P[ZODI_P_NY], P[ZODI_P_NZ])), hg(to_scalar(0.5 * gamma)) {}
};

template <>
struct LineComp<ZODI_FAN> : PlaneComp {
  double hq;  // Q/2
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : PlaneComp(P, l, P[8]), hq(to_scalar(0.5 * P[6])) {}
};
template <>
struct LineComp<ZODI_COMET> : PlaneComp {
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : PlaneComp(P, l, P[6]) {}
};
template <>
struct LineComp<ZODI_NARROW_BAND> : PlaneComp {
  double lo2;  // log R_outer^2
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : PlaneComp(P, l, P[8]), lo2(to_scalar(2.0 * log(P[11]))) {}
};
template <>
struct LineComp<ZODI_BROAD_BAND> : PlaneComp {
  double lo2;
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : PlaneComp(P, l, P[8]), lo2(to_scalar(2.0 * log(P[11]))) {}
};
template <>
struct LineComp<ZODI_RING_RRM> : LineComp<ZODI_RING> {
  using LineComp<ZODI_RING>::LineComp;
};
template <>
struct LineComp<ZODI_FEATURE_RRM> : LineComp<ZODI_FEATURE> {
  using LineComp<ZODI_FEATURE>::LineComp;
};
template <>
struct LineComp<ZODI_INTERSTELLAR> {
  __device__ __forceinline__ LineComp(ParamPtr, const Line&, double, double) {}
};

// Density of an RRM component at a node; lR2 = log |X|^2.
template <int KIND>
__device__ __forceinline__ double rrm_density(ParamPtr P, const LineComp<KIND>& c,
                                              const LineLogCtx& cx, const Line& l,
                                              const GradNode& nd, double lR2) {
  if constexpr (KIND == ZODI_INTERSTELLAR) {
    return P[6];
  } else if constexpr (KIND == ZODI_FAN) {
    double n = 0.0;
    if (nd.R <= P[10]) {
      double zc;
      const double s = line_sin_beta(c.z, nd, zc);
      const double lc2 = log_node(cx.tab->log_tab, cx.lc, fmax(fma(-s, s, 1.0), 0x1p-900));
      const LatSine t = lat_sine<false>(cx, P, P[9], P[13], fabs(zc), s, 0.0);
      n = exp_neg_any(cx.ec, fma(P[7], t.su, fma(c.hg, lR2, -(c.hq * lc2))));
    }
    return n;
  } else if constexpr (KIND == ZODI_COMET) {
    double n = 0.0;
    if (nd.R >= P[10] && nd.R <= P[11]) {
      double zc;
      const double s = line_sin_beta(c.z, nd, zc);
      const LatSine t = lat_sine<false>(cx, P, P[7], P[13], fabs(zc), s, 0.0);
      n = P[9] * exp_neg_any(cx.ec, fma(P[8], t.su, c.hg * lR2));
    }
    return n;
  } else if constexpr (KIND == ZODI_NARROW_BAND) {
    double n = 0.0;
    if (nd.R >= P[10] && nd.R <= P[11]) {
      double zc;
      const double s = line_sin_beta(c.z, nd, zc);
      const double b = asin_unit(s) * kRad2Deg;
      if (b < P[6]) {
        n = P[9] * exp_neg_any(cx.ec, fma(P[7], P[6] - b, c.hg * (lR2 - c.lo2)));
      }
    }
    return n;
  } else if constexpr (KIND == ZODI_BROAD_BAND) {
    double n = 0.0;
    if (nd.R >= P[10] && nd.R <= P[11]) {
      double zc;
      const double s = line_sin_beta(c.z, nd, zc);
      const double b = asin_unit(s) * kRad2Deg;  // the density is even in beta
      const double a = (b - P[6]) * P[13], d = (b + P[6]) * P[13];
      const double r = c.hg * (lR2 - c.lo2);
      n = P[9] * (exp_neg_any(cx.ec, fma(0.5 * a, a, r)) + exp_neg_any(cx.ec, fma(0.5 * d, d, r)));
    }
    return n;
  } else if constexpr (KIND == ZODI_RING_RRM) {
    const double d = nd.R - P[7];
    return (P[10] * P[6]) *
           exp_neg_any(cx.ec, fma(d * d, P[13], fabs(c.z.at(nd.t)) * P[14]));
  } else {
    static_assert(KIND == ZODI_FEATURE_RRM, "an RRM component");
    double y, rho2, inv_rho;
    const double th = feature_angle(c, l, *cx.angles, nd.t, y, rho2, inv_rho);
    const double d = nd.R - P[7];
    double e = (d * d) * P[13];
    e = fma(fabs(c.z.at(nd.t)), P[14], e);
    e = fma(th * th, P[15], e);
    return (P[12] * P[6]) * exp_neg_any(cx.ec, e);
  }
}

// The node's geometry, log |X|^2, R^-delta and Planck lookup of a group.
struct RrmNode {
  GradNode nd;
  double lR2, Rd, B, dB;
};

__device__ __forceinline__ RrmNode rrm_node(const LineLogCtx& cx, const Line& l, double t,
                                            double half_delta, double us, double uo1) {
  RrmNode o;
  o.nd.t = t;
  o.nd.R2 = fma(t, t, l.d2);
  norm_and_inverse_node(o.nd.R2, o.nd.R, o.nd.inv_R);
  o.nd.iR2 = o.nd.inv_R * o.nd.inv_R;
  o.lR2 = log_node(cx.tab->log_tab, cx.lc, o.nd.R2);
  // |X| = 0 exactly: the reference's quotient 0/0 makes the node NaN
  if (o.nd.R2 == 0.0) o.lR2 = __builtin_nan("");
  o.Rd = exp_neg_any(cx.ec, half_delta * o.lR2);
  const double u1 = fma(o.Rd, us, -uo1);
  uint32_t j = saturate_u32(u1);
  j = j < (uint32_t)ZODI_N_TEMPS ? j : (uint32_t)ZODI_N_TEMPS;
  const double2 pl = cx.tab->planck[j];
  o.B = fma(__builtin_amdgcn_fract(u1), pl.y, pl.x);
  o.dB = pl.y;
  return o;
}

// ---------------------------------------------------------------- forward
template <int SPLIT, int... Ks, int... J>
__device__ __forceinline__ void rrm_group(Grp<Ks...>, std::integer_sequence<int, J...>,
                                          const LineLogCtx& cx, const FwdArgs& a, const Ray& y,
                                          const Line& l, int g, int first, double2* terms,
                                          double& total) {
  constexpr int C = sizeof...(Ks);
  constexpr int kinds[C] = {Ks...};
  const ModelPtr M = cx.M;
  double h, mid;
  group_range(M, g, y, h, mid);
  const double th = l.n * h, tm = fma(l.n, mid, l.t0);
  const double half_delta = to_scalar(0.5 * M->group_delta[g]);
  const double us = to_scalar(M->group_T0[g] * M->tab_inv_step);
  const double uo1 = to_scalar(M->tab_T[0] * M->tab_inv_step - 1.0);
  const std::tuple<LineComp<Ks>...> lc{LineComp<Ks>(M->comp[first + J], l, y.ex, y.ey)...};
  const int lanes = SPLIT == 8 ? a.lanes : SPLIT;
  LaneSums<SPLIT, C> acc;
  for (int k0 = 0; k0 < cx.K; k0 += lanes) {
    const int k = SPLIT == 1 ? k0 : (k0 + cx.sub < cx.K ? k0 + cx.sub : cx.K - 1);
    const ModelPtr Mk = opaque(M);
    const double wk = Mk->gl_w[k];
    const RrmNode o = rrm_node(cx, l, fma(th, Mk->gl_x[k], tm), half_delta, us, uo1);
    const double wB = wk * o.B;
    const NodeTerm t[C] = {NodeTerm{
        wB, rrm_density<kinds[J]>(Mk->comp[first + J], std::get<J>(lc), cx, l, o.nd, o.lR2)}...};
    acc.add(t, terms, lanes, cx.sub, cx.K - k0);
  }
  const double cal = M->shared[ZODI_S_CALIBRATION];
  acc.finish(a, y, first, lanes, cx.sub, total, [&](int c, double sum) {
    return finish<ZODI_INTEGRAND_RRM>(M->comp[c], M->comp_flags[c], sum, h, cal);
  });
}

template <int SPLIT, class... Gs, int... G>
__device__ __forceinline__ void rrm_groups(Layout<ZODI_INTEGRAND_RRM, Gs...>,
                                           std::integer_sequence<int, G...>,
                                           const LineLogCtx& cx, const FwdArgs& a, const Ray& y,
                                           const Line& l, double2* terms, double& total) {
  (rrm_group<SPLIT>(Gs{}, std::make_integer_sequence<int, Gs::size>{}, cx, a, y, l, G,
                    group_first<Gs...>(G), terms, total),
   ...);
}

template <int SPLIT, class... Gs>
__device__ __forceinline__ void run_rrm(Layout<ZODI_INTEGRAND_RRM, Gs...> lay,
                                        const LineLogCtx& cx, const FwdArgs& a, const Ray& y,
                                        double2* terms, double& total) {
  const Line l = make_line(y.ux, y.uy, y.uz, y.ox, y.oy, y.oz);
  rrm_groups<SPLIT>(lay, std::make_integer_sequence<int, sizeof...(Gs)>{}, cx, a, y, l, terms,
                    total);
}

// ---------------------------------------------------------------- partials
// Sums of an RRM component, as LineGrad's: add() takes the node's weight u = w B and
// lR2 and returns nu; partials() the geometry sums m and the kind's partials at unit
// weight from the sums and b = sum u nu (the amplitude multiplies what it must).
struct RrmSums {
  __device__ __forceinline__ static double sign(double zc) {
    return zc == 0.0 ? 0.0 : __builtin_copysign(1.0, zc);
  }
};

// Adds the geometry terms: dl the derivative of the density with respect to |beta|, dz one
// with respect to |Z| besides, both times the weight; q the weighted density, gamma its
// radial power.
__device__ __forceinline__ void rrm_geometry(double* s, const GradNode& nd, double sb,
                                             double inv_cb, double sgn, double q, double gamma,
                                             double dl, double dz) {
  const double tan_b = sb * inv_cb;
  const double mr = -fma(gamma, q, dl * tan_b) * nd.iR2;
  s[0] += mr;
  s[1] = fma(mr, nd.t, s[1]);
  const double mz = sgn * fma(dl, nd.inv_R * inv_cb, dz);
  s[2] += mz;
  s[3] = fma(mz, nd.t, s[3]);
}

template <>
struct LineGrad<ZODI_FAN> : RrmSums {
  static constexpr int kSlots = 8;
  LineComp<ZODI_FAN> c;
  double s[kSlots];
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{} {}
  __device__ __forceinline__ static double amplitude(ParamPtr) { return 1.0; }
  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line&,
                                        const GradNode& nd, double lR2, double u) {
    double nu = 0.0;
    if (nd.R <= P[10]) {
      double zc;
      const double sb = line_sin_beta(c.z, nd, zc);
      const double cb2 = fmax(fma(-sb, sb, 1.0), 0x1p-900);
      double cb, inv_cb;
      norm_and_inverse_node(cb2, cb, inv_cb);
      const double lc2 = log_node(cx.tab->log_tab, cx.lc, cb2);
      const LatSine t = lat_sine<true>(cx, P, P[9], P[13], fabs(zc), sb, cb);
      nu = exp_neg_any(cx.ec, fma(P[7], t.su, fma(c.hg, lR2, -(c.hq * lc2))));
      const double q = u * nu;
      const double pq = (P[7] * t.cu) * q;
      const double de = pq * t.u_logb;  // - dn/deps
      const double dl = -fma(P[6] * (sb * inv_cb), q, pq * t.du_db);
      rrm_geometry(s, nd, sb, inv_cb, sign(zc), q, P[8], dl, de * P[13]);
      s[4] = fma(q, lR2, s[4]);
      s[5] = fma(-de, fabs(zc), s[5]);
      s[6] = fma(q, lc2, s[6]);
      s[7] = fma(q, t.su, s[7]);
    }
    return nu;
  }
  __device__ __forceinline__ void partials(ParamPtr P, double, double m[4], double* dp) const {
    for (int k = 0; k < 4; ++k) m[k] = s[k];
    dp[0] = -0.5 * s[4];
    dp[1] = (P[13] * P[13]) * s[5];
    dp[2] = 0.5 * s[6];
    dp[3] = -s[7];
    dp[4] = 0.0;
  }
};

template <>
struct LineGrad<ZODI_COMET> : RrmSums {
  static constexpr int kSlots = 7;
  LineComp<ZODI_COMET> c;
  double s[kSlots];
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{} {}
  __device__ __forceinline__ static double amplitude(ParamPtr P) { return P[9]; }
  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line&,
                                        const GradNode& nd, double lR2, double u) {
    double nu = 0.0;
    if (nd.R >= P[10] && nd.R <= P[11]) {
      double zc;
      const double sb = line_sin_beta(c.z, nd, zc);
      double cb, inv_cb;
      norm_and_inverse_node(fmax(fma(-sb, sb, 1.0), 0x1p-900), cb, inv_cb);
      const LatSine t = lat_sine<true>(cx, P, P[7], P[13], fabs(zc), sb, cb);
      nu = exp_neg_any(cx.ec, fma(P[8], t.su, c.hg * lR2));
      const double q = u * nu;
      const double pq = (P[8] * t.cu) * q;
      const double de = pq * t.u_logb;
      rrm_geometry(s, nd, sb, inv_cb, sign(zc), q, P[6], -(pq * t.du_db), de * P[13]);
      s[4] = fma(q, lR2, s[4]);
      s[5] = fma(-de, fabs(zc), s[5]);
      s[6] = fma(q, t.su, s[6]);
    }
    return nu;
  }
  __device__ __forceinline__ void partials(ParamPtr P, double b, double m[4], double* dp) const {
    const double amp = P[9];
    for (int k = 0; k < 4; ++k) m[k] = amp * s[k];
    dp[0] = -0.5 * amp * s[4];
    dp[1] = amp * (P[13] * P[13]) * s[5];
    dp[2] = -amp * s[6];
    dp[3] = b;
    dp[4] = 0.0;
    dp[5] = 0.0;
  }
};

template <>
struct LineGrad<ZODI_NARROW_BAND> : RrmSums {
  static constexpr int kSlots = 6;
  LineComp<ZODI_NARROW_BAND> c;
  double s[kSlots];
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{} {}
  __device__ __forceinline__ static double amplitude(ParamPtr P) { return P[9]; }
  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line&,
                                        const GradNode& nd, double lR2, double u) {
    double nu = 0.0;
    if (nd.R >= P[10] && nd.R <= P[11]) {
      double zc;
      const double sb = line_sin_beta(c.z, nd, zc);
      const double b = asin_unit(sb) * kRad2Deg;
      if (b < P[6]) {
        double cb, inv_cb;
        norm_and_inverse_node(fmax(fma(-sb, sb, 1.0), 0x1p-900), cb, inv_cb);
        const double lr = lR2 - c.lo2;
        nu = exp_neg_any(cx.ec, fma(P[7], P[6] - b, c.hg * lr));
        const double q = u * nu;
        rrm_geometry(s, nd, sb, inv_cb, sign(zc), q, P[8], q * (P[7] * kRad2Deg), 0.0);
        s[4] = fma(q, lr, s[4]);
        s[5] = fma(q, b - P[6], s[5]);
      }
    }
    return nu;
  }
  __device__ __forceinline__ void partials(ParamPtr P, double b, double m[4], double* dp) const {
    const double A = P[9];
    for (int k = 0; k < 4; ++k) m[k] = A * s[k];
    dp[0] = -0.5 * A * s[4];
    dp[1] = b;
    dp[2] = A * s[5];
    dp[3] = 0.0;
    dp[4] = A * b * P[8] * P[13];
    dp[5] = -P[7] * (A * b);
  }
};

template <>
struct LineGrad<ZODI_BROAD_BAND> : RrmSums {
  static constexpr int kSlots = 7;
  LineComp<ZODI_BROAD_BAND> c;
  double s[kSlots];
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{} {}
  __device__ __forceinline__ static double amplitude(ParamPtr P) { return P[9]; }
  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line&,
                                        const GradNode& nd, double lR2, double u) {
    double nu = 0.0;
    if (nd.R >= P[10] && nd.R <= P[11]) {
      double zc;
      const double sb = line_sin_beta(c.z, nd, zc);
      const double b = asin_unit(sb) * kRad2Deg;
      double cb, inv_cb;
      norm_and_inverse_node(fmax(fma(-sb, sb, 1.0), 0x1p-900), cb, inv_cb);
      const double a = (b - P[6]) * P[13], d = (b + P[6]) * P[13];
      const double lr = lR2 - c.lo2, r = c.hg * lr;
      const double ea = exp_neg_any(cx.ec, fma(0.5 * a, a, r));
      const double ed = exp_neg_any(cx.ec, fma(0.5 * d, d, r));
      nu = ea + ed;
      const double q = u * nu, wa = (u * ea) * a, wd = (u * ed) * d;
      rrm_geometry(s, nd, sb, inv_cb, sign(zc), q, P[8], -(wa + wd) * (P[13] * kRad2Deg), 0.0);
      s[4] = fma(q, lr, s[4]);
      s[5] += wa - wd;
      s[6] += fma(wa, a, wd * d);
    }
    return nu;
  }
  __device__ __forceinline__ void partials(ParamPtr P, double b, double m[4], double* dp) const {
    const double A = P[9];
    for (int k = 0; k < 4; ++k) m[k] = A * s[k];
    dp[0] = -0.5 * A * s[4];
    dp[1] = b;
    dp[2] = 0.0;
    dp[3] = A * b * P[8] * P[14];
    dp[4] = A * P[13] * s[5];
    dp[5] = A * P[13] * s[6];
  }
};

template <>
struct LineGrad<ZODI_INTERSTELLAR> : RrmSums {
  static constexpr int kSlots = 1;
  double s[kSlots];
  __device__ __forceinline__ LineGrad(ParamPtr, const Line&, double, double) : s{} {}
  __device__ __forceinline__ static double amplitude(ParamPtr P) { return P[6]; }
  __device__ __forceinline__ double add(ParamPtr, const LineLogCtx&, const Line&, const GradNode&,
                                        double, double) {
    return 1.0;
  }
  __device__ __forceinline__ void partials(ParamPtr, double b, double m[4], double* dp) const {
    for (int k = 0; k < 4; ++k) m[k] = 0.0;
    dp[0] = b;
  }
};

// The ring and the feature: the Kelsall ones with a second amplitude A.
template <>
struct LineGrad<ZODI_RING_RRM> : LineGrad<ZODI_RING> {
  using LineGrad<ZODI_RING>::LineGrad;
  __device__ __forceinline__ static double amplitude(ParamPtr P) { return P[10] * P[6]; }
  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line& l,
                                        const GradNode& nd, double, double u) {
    return LineGrad<ZODI_RING>::add(P, cx, l, nd, u);
  }
  __device__ __forceinline__ void partials(ParamPtr P, double b, double m[4], double* dp) const {
    LineGrad<ZODI_RING>::partials(P, m, dp);
    const double amp = amplitude(P);
    for (int k = 0; k < 4; ++k) m[k] *= amp;
    for (int k = 1; k < 4; ++k) dp[k] *= amp;
    dp[0] = P[10] * b;
    dp[4] = P[6] * b;
  }
};

template <>
struct LineGrad<ZODI_FEATURE_RRM> : LineGrad<ZODI_FEATURE> {
  using LineGrad<ZODI_FEATURE>::LineGrad;
  __device__ __forceinline__ static double amplitude(ParamPtr P) { return P[12] * P[6]; }
  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line& l,
                                        const GradNode& nd, double, double u) {
    return LineGrad<ZODI_FEATURE>::add(P, cx, l, nd, u);
  }
  __device__ __forceinline__ void partials(ParamPtr P, double b, double m[7], double* dp) const {
    LineGrad<ZODI_FEATURE>::partials(P, m, dp);
    const double amp = amplitude(P);
    for (int k = 0; k < 7; ++k) m[k] *= amp;
    for (int k = 1; k < 6; ++k) dp[k] *= amp;
    dp[0] = P[12] * b;
    dp[6] = P[6] * b;
  }
};

// Group g of one ray: line_adj_group for the RRM integrand, f = calibration B(T_c) n. Every
// component has a temperature law of its own in the parameter vector.
template <bool JAC, int... Ks, int... J>
__device__ __forceinline__ void rrm_adj_group(Grp<Ks...>, std::integer_sequence<int, J...>,
                                              const LineLogCtx& cx, const AdjArgs& a, Ray& y,
                                              int g, int first, double gscale, double* row,
                                              int lane, double (&sh)[6], double& total) {
  constexpr int C = sizeof...(Ks);
  constexpr int kinds[C] = {Ks...};
  const ModelPtr M = cx.M;
  double h, mid;
  group_range(M, g, y, h, mid);
  const Line l = make_line(y.ux, y.uy, y.uz, y.ox, y.oy, y.oz);
  const double tscale = l.n * h, tmid = fma(l.n, mid, l.t0);
  const double T0 = M->group_T0[g];
  const double half_delta = to_scalar(0.5 * M->group_delta[g]);
  const double us = to_scalar(T0 * M->tab_inv_step);
  const double uo1 = to_scalar(M->tab_T[0] * M->tab_inv_step - 1.0);
  std::tuple<LineGrad<Ks>...> lg{LineGrad<Ks>(M->comp[first + J], l, y.ex, y.ey)...};
  double s0[C] = {}, st[C] = {}, sd[C] = {};
  const int K = y.active ? cx.K : 0;
  double xnext = M->gl_x[cx.sub], wnext = M->gl_w[cx.sub];
  for (int k = cx.sub; k < K; k += cx.split) {
    const ModelPtr Mk = opaque(M);
    const double wk = wnext;
    const RrmNode o = rrm_node(cx, l, fma(tscale, xnext, tmid), half_delta, us, uo1);
    {
      const int kn = k + cx.split < ZODI_MAX_NODES ? k + cx.split : 0;
      xnext = M->gl_x[kn];
      wnext = M->gl_w[kn];
    }
    const double wB = wk * o.B, wT = (wk * o.dB) * o.Rd;
    (
        [&] {
          const double nu =
              std::get<J>(lg).add(Mk->comp[first + J], cx, l, o.nd, o.lR2, wB);
          s0[J] = fma(wB, nu, s0[J]);
          const double x = wT * nu;
          st[J] += x;
          sd[J] = fma(x, o.lR2, sd[J]);
        }(),
        ...);
  }

  if (!y.active) h = 0.0;
  const auto sum = [&](double v) { return JAC ? split_sum(v, cx.split) : v; };
  const double cal = M->shared[ZODI_S_CALIBRATION];
  (
      [&] {
        constexpr int KIND = kinds[J];
        constexpr bool FEATURE = is_feature(KIND);
        constexpr int NP = kind_nparams<KIND>();
        auto& A = std::get<J>(lg);
        const int c = first + J;
        const ParamPtr P = M->comp[c];
#pragma unroll
        for (int q = 0; q < A.kSlots; ++q) A.s[q] = sum(A.s[q]);
        const double b = sum(s0[J]);
        const double amp = A.amplitude(P);
        double wr = h;
        if (!JAC) {
          wr = a.mode == ZODI_ADJ_VJP_COMPS
                   ? (y.active ? h * a.weights[(int64_t)c * a.f.n_rays + y.r] : 0.0)
                   : h * gscale;
        }
        const double W = wr * cal;
        double m[7], dp[NP], geo[5];
        A.partials(P, b, m, dp);
        line_geo<FEATURE>(P, l, m, FEATURE ? earth_term(P, y.ex, y.ey) : EarthTerm{0.0, 0.0},
                          geo);
#pragma unroll
        for (int q = 0; q < 5; ++q) geo[q] *= W;
#pragma unroll
        for (int q = 0; q < NP; ++q) dp[q] *= W;
        const double wt = W * amp * M->tab_inv_step;
        const double dT = wt * sum(st[J]);
        const double dd = (-0.5 * T0) * wt * sum(sd[J]);
        sh[0] += wr * (amp * b);  // calibration
        if constexpr (JAC) {
          total = __dadd_rn(total, h * (cal * (amp * b)));
          if (y.active && cx.sub == 0) {
            double* col = a.jac + y.r;
            const int64_t ld = a.ld_jac;
            const int off = M->grad_comp[c];
#pragma unroll
            for (int q = 0; q < 5; ++q) col[(off + q) * ld] = geo[q];
#pragma unroll
            for (int q = 0; q < NP; ++q) col[(off + 5 + q) * ld] = dp[q];
            col[M->grad_spec_a[c] * ld] = dT;
            col[M->grad_spec_b[c] * ld] = dd;
          }
        } else {
          double v[5 + NP + 2];
#pragma unroll
          for (int q = 0; q < 5; ++q) v[q] = geo[q];
#pragma unroll
          for (int q = 0; q < NP; ++q) v[5 + q] = dp[q];
          v[5 + NP] = dT;
          v[6 + NP] = dd;
          add_folded(v, row, lane, M->grad_comp[c], M->grad_spec_a[c], M->grad_spec_b[c]);
        }
      }(),
      ...);
}

template <bool JAC, class... Gs, int... G>
__device__ __forceinline__ void rrm_adj_groups(Layout<ZODI_INTEGRAND_RRM, Gs...>,
                                               std::integer_sequence<int, G...>,
                                               const LineLogCtx& cx, const AdjArgs& a, Ray& y,
                                               double gscale, double* row, int lane,
                                               double (&sh)[6], double& total) {
  (rrm_adj_group<JAC>(Gs{}, std::make_integer_sequence<int, Gs::size>{}, cx, a, y, G,
                      group_first<Gs...>(G), gscale, row, lane, sh, total),
   ...);
}

template <int SCAT, int PASS, class... Gs>
__device__ __forceinline__ void line_adj_layout(Layout<ZODI_INTEGRAND_RRM, Gs...> lay,
                                                const LineLogCtx& cx, const AdjArgs& a, Ray& y,
                                                double gscale, double* row, int lane,
                                                double (&sh)[6], double& total, double&,
                                                double*) {
  rrm_adj_groups<PASS == kPassJac>(lay, std::make_integer_sequence<int, sizeof...(Gs)>{}, cx, a, y, gscale,
                      row, lane, sh, total);
}

template <class LAYOUT, bool JAC>
__global__ __launch_bounds__(kAdjBlock)
__attribute__((amdgpu_waves_per_eu(kRrmAdjWaves, kRrmAdjWaves))) void
rrm_adjoint(AdjArgs a) {
  line_adj_body<LAYOUT, 0, JAC ? kPassJac : kPassVjp>(a);
}

}  // namespace zodi
