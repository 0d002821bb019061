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

// asin(s) for 0 <= s <= 1 (the reduction of acos_fast). The half above 1/2 costs a
// square root and is entered only by the waves that have such a point.
__device__ __forceinline__ double asin_unit(double s) {
  constexpr double kQ[] = {ZODI_ASIN_POLY};
  double w = s, z = s * s, up = 0.0;
  if (s > 0.5) {
    z = fma(-0.5, s, 0.5);
    double inv;
    norm_and_inverse(z, w, inv);
    w = z == 0.0 ? 0.0 : w;
    up = 1.0;
  }
  const double v = fma(w * z, zodi_trig::horner(kQ, z), w);
  // pi/2 - 2 asin(sqrt((1 - s)/2)) above 1/2
  return fma(up, zodi_trig::kPiHalfHi, fma(up, -3.0 * v, v));
}

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
__device__ __forceinline__ LatSine lat_sine(const LineAdjCtx& cx, ParamPtr P, double Z0,
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
      : PlaneComp(P, l, P[8]), lo2(to_scalar(2.0 * log_pos(P[11]))) {}
};
template <>
struct LineComp<ZODI_BROAD_BAND> : PlaneComp {
  double lo2;
  __device__ __forceinline__ LineComp(ParamPtr P, const Line& l, double, double)
      : PlaneComp(P, l, P[8]), lo2(to_scalar(2.0 * log_pos(P[11]))) {}
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
                                              const LineAdjCtx& cx, const Line& l,
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
    double x = c.x.at(nd.t), y = c.y.at(nd.t);
    if (x == 0.0 && y == 0.0) {
      const double sg = __builtin_signbit(fma(l.vx, nd.t, l.px)) ? -1.0 : 1.0;
      x = sg * c.d.c;
      y = -sg * c.d.s;
    }
    const double th = axis_angle(x, y);
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

__device__ __forceinline__ RrmNode rrm_node(const LineAdjCtx& cx, const Line& l, double t,
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
  uint32_t j = (uint32_t)u1;
  j = j < (uint32_t)ZODI_N_TEMPS ? j : (uint32_t)ZODI_N_TEMPS;
  const double2 pl = cx.tab->planck[j];
  o.B = fma(__builtin_amdgcn_fract(u1), pl.y, pl.x);
  o.dB = pl.y;
  return o;
}

// ---------------------------------------------------------------- forward
template <int L, int... Ks, int... J>
__device__ __forceinline__ void rrm_group(Grp<Ks...>, std::integer_sequence<int, J...>,
                                          const LineAdjCtx& cx, const FwdArgs& a, const Ray& y,
                                          const Line& l, int g, int first, double& total) {
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
  double acc[C] = {};
  for (int k0 = 0; k0 < cx.K; k0 += L) {
    const int k = L == 1 ? k0 : (k0 + cx.sub < cx.K ? k0 + cx.sub : cx.K - 1);
    const ModelPtr Mk = opaque(M);
    const double wk = Mk->gl_w[k];
    const RrmNode o = rrm_node(cx, l, fma(th, Mk->gl_x[k], tm), half_delta, us, uo1);
    const double wB = wk * o.B;
    const NodeTerm t[C] = {NodeTerm{
        wB, rrm_density<kinds[J]>(Mk->comp[first + J], std::get<J>(lc), cx, l, o.nd, o.lR2)}...};
    if constexpr (L == 1) {
      ((acc[J] = node_add(acc[J], t[J])), ...);
    } else {
      add_in_node_order<L>(acc, t, cx.K - k0);
    }
  }
  const double cal = M->shared[ZODI_S_CALIBRATION];
  const bool write = y.active && cx.sub == 0;
  (
      [&] {
        const double e = finish<ZODI_INTEGRAND_RRM>(M->comp[first + J], M->comp_flags[first + J],
                                                    acc[J], h, cal);
        if (a.out_mode == ZODI_OUT_COMPS) {
          if (write) a.out[(int64_t)(first + J) * a.n_rays + y.r] = e;
        } else {
          total = __dadd_rn(total, e);
        }
      }(),
      ...);
}

template <int L, class... Gs, int... G>
__device__ __forceinline__ void rrm_groups(Layout<ZODI_INTEGRAND_RRM, Gs...>,
                                           std::integer_sequence<int, G...>,
                                           const LineAdjCtx& cx, const FwdArgs& a, const Ray& y,
                                           const Line& l, double& total) {
  (rrm_group<L>(Gs{}, std::make_integer_sequence<int, Gs::size>{}, cx, a, y, l, G,
                group_first<Gs...>(G), total),
   ...);
}

template <int L, class... Gs>
__device__ __forceinline__ void run_rrm(Layout<ZODI_INTEGRAND_RRM, Gs...> lay,
                                        const LineAdjCtx& cx, const FwdArgs& a, const Ray& y,
                                        double& total) {
  const Line l = make_line(y.ux, y.uy, y.uz, y.ox, y.oy, y.oz);
  rrm_groups<L>(lay, std::make_integer_sequence<int, sizeof...(Gs)>{}, cx, a, y, l, total);
}

}  // namespace zodi
