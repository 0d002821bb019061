// The Kelsall registry layouts' adjoint and Jacobian passes on the ray's line (gfx950).
//
// Bound by FP64 vector issue, like the forward (zodi_line.hpp), at the occupancy that the
// accumulators leave. Besides the line's cheaper geometry:
//
//  * The partials with respect to a component's offset and tilts are linear in dn/dR' and
//    dn/dZ with the point's coordinates as coefficients, and the point is P + t V: four
//    sums a component (of dn/dR'/R', t dn/dR'/R', dn/dZ, t dn/dZ) stand for the seven
//    of the coordinate form, and line_geo combines them with P and V once per ray
//    (seven instead of ten for the feature).
//  * Every sum is of the density at unit amplitude; the amplitude, the emissivity and
//    the other constants of a component multiply the finished sums. The amplitude's own
//    partial is then the emissivity's sum, not a sum of its own.
//  * The weights of a vector-Jacobian product multiply the finished sums too, so both
//    passes share the node loop.
//  * A power is exp(p log x) here, since the partials need the logarithm anyway;
//    g^(gamma - 1) = exp((gamma - 1) log g) takes the place of g^gamma / g.
//
// SCAT: 0 no component scatters and there is no solar irradiance (block_noscat); 1 no
// component scatters, but d/d(albedo) needs the scattered light; 2 some component scatters.
#pragma once

#include "zodi_adjoint.hpp"

namespace zodi {

// ---------------------------------------------------------------- angles
// For the passes that take angles from the table: with scattering (SCAT 2), chi^2 of 196 608
// rays of DIRBE at 1.25 um takes 296 us for 314, of 400 000 672 for 741. The passes without,
// whose only angle is the feature's, spill more registers for it than it saves (VJP of
// 150 000 rays 210 us for 205, RRM chi^2 of 49 152 168 for 165) and keep axis_angle.
struct LineLogCtxAngles : LineLogCtx {
  static constexpr bool kAngles = true;
};

template <int SCAT>
using AdjCtx = std::conditional_t<SCAT == 2, LineLogCtxAngles, LineLogCtx>;

// One node as the components see it.
struct GradNode {
  double t, R2, R, inv_R, iR2;
};

// ---------------------------------------------------------------- components
// Sums of one component over the nodes, of the density nu at unit amplitude with weight u
// (w_k B, or with a scattering component w_k e): slots 0-3 the geometry sums u dnu/dR'/R'
// and u dnu/dZ, each times 1 and t (up to the constants in partials()), then the kind's.
// add() returns nu; partials() gives the geometry sums m and the partials with respect
// to the kind's parameters after its amplitude.
template <int KIND>
struct LineGrad;

template <>
struct LineGrad<ZODI_CLOUD> {
  static constexpr int kSlots = 8;
  LineComp<ZODI_CLOUD> c;
  double s[kSlots];
  double kz, ha, og;  // beta gamma / mu, alpha/2, 1 - gamma
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{}, kz(to_scalar(P[8] * P[9] * (2.0 * P[13]))),
        ha(to_scalar(0.5 * P[7])), og(to_scalar(1.0 - P[9])) {}

  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line&,
                                        const GradNode& nd, double u) {
    const double alpha = P[7], beta = P[8], mu = P[10], inv_2mu = P[13];
    const double r2 = c.o.r2(nd.t);
    double r, inv_r;
    norm_and_inverse_node(r2, r, inv_r);
    const double zc = c.z.at(nd.t);
    const double zeta = fabs(zc) * inv_r;
    const double m = fmin(zeta, mu);  // see line_cloud
    const double g = fmax(fma(m * m, inv_2mu, zeta - m), 0x1p-127);
    const double lg = log_node(cx.tab->log_tab, cx.lc, g);
    const double H = exp_neg_node(cx.ec, og * lg);
    const double G = H * g;
    const double lr = log_node(cx.tab->log_tab, cx.lc, r2);
    const double nu = exp_neg_node(cx.ec, fma(ha, lr, beta * G));
    const double q = u * nu;
    const double a = (q * H) * m;
    const double mr = fma(kz, a * zeta, -(alpha * q)) * (inv_r * inv_r);
    s[0] += mr;
    s[1] = fma(mr, nd.t, s[1]);
    const double mz = a * __builtin_copysign(inv_r, zc);
    s[2] += mz;
    s[3] = fma(mz, nd.t, s[3]);
    const double qG = q * G;
    s[4] = fma(q, lr, s[4]);
    s[5] += qG;
    s[6] = fma(qG, lg, s[6]);
    s[7] = fma(a, m, s[7]);
    return nu;
  }

  __device__ __forceinline__ void partials(ParamPtr P, double m[4], double* dp) const {
    const double bg = P[8] * P[9];
    m[0] = s[0];
    m[1] = s[1];
    m[2] = -kz * s[2];
    m[3] = -kz * s[3];
    dp[1] = -0.5 * s[4];
    dp[2] = -s[5];
    dp[3] = -P[8] * s[6];
    dp[4] = 2.0 * (P[13] * P[13]) * bg * s[7];
  }
};

// A band's radial cut-off argument x = (R/delta_r)^20 and exp(-x) (0 where
// 1 - exp(-x) rounds to 1), shared within a node by bands with the same cut-off.
struct CutShare {
  double x, ex;
};

template <>
struct LineGrad<ZODI_BAND> {
  static constexpr int kSlots = 8;
  LineComp<ZODI_BAND> c;
  double s[kSlots];
  double k23;  // 2/(3 v)
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{}, k23(to_scalar(P[14] * (2.0 / 3.0))) {}

  // cs: the radial cut-off's x and exp(-x), formed here unless `have`. Past zeta_d^6 =
  // 746 the density and every partial are exact zeros (line_band).
  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const GradNode& nd,
                                        CutShare& cs, bool have, double u) {
    if (!have) {
      const double y = nd.R2 * P[ZODI_P_D0 + 6];
      const double y2 = y * y;
      const double y4 = y2 * y2;
      cs.x = (y4 * y4) * y2;
      cs.ex = 0.0;
      if (cs.x < 38.0) cs.ex = exp_neg_cut(cx.ec, cs.x);
    }
    const double zq = c.z.at(nd.t) * nd.inv_R;  // signed
    const double zd2 = zq * zq;
    const double zd4 = zd2 * zd2;
    const double zd6 = zd4 * zd2;
    double nu = 0.0;
    if (!(zd6 >= 746.0)) {
      const double lz = log_node(cx.tab->log_tab, cx.lc, zd2);
      const double t3 = fma(zd4, P[14], 1.0);
      const double t12 = nd.inv_R * exp_neg_node(cx.ec, zd6);
      const double t124 = t12 * (1.0 - cs.ex);
      nu = t124 * t3;
      const double q = u * nu;
      const double w124 = u * t124;
      const double zv = w124 * zd4;
      // zeta_d dn/dzeta_d = -6 p with p = zeta_d^2 b, b = t124 zeta_d^2 (zeta_d^2 t3 - 2/(3 v))
      const double b = (w124 * zd2) * fma(zd2, t3, -k23);
      const double p = b * zd2;
      const double rx = (u * (t12 * t3)) * (cs.x * cs.ex);
      const double mr = fma(6.0, p, fma(20.0, rx, -q)) * nd.iR2;
      s[0] += mr;
      s[1] = fma(mr, nd.t, s[1]);
      const double mz = b * (zq * nd.inv_R);
      s[2] += mz;
      s[3] = fma(mz, nd.t, s[3]);
      s[4] += p;
      s[5] += zv;
      s[6] = fma(zv, lz, s[6]);
      s[7] += rx;
    }
    return nu;
  }

  __device__ __forceinline__ void partials(ParamPtr P, double m[4], double* dp) const {
    const double inv_dzeta = P[13], inv_v = P[14], inv_dr = P[15];
    m[0] = s[0];
    m[1] = s[1];
    m[2] = -6.0 * inv_dzeta * s[2];
    m[3] = -6.0 * inv_dzeta * s[3];
    dp[1] = 6.0 * (inv_dzeta * kDegToRad) * s[4];
    dp[2] = -(inv_v * inv_v) * s[5];
    dp[3] = 0.5 * inv_v * s[6];
    dp[4] = -20.0 * inv_dr * s[7];
  }
};

template <>
struct LineGrad<ZODI_RING> {
  static constexpr int kSlots = 7;
  LineComp<ZODI_RING> c;
  double s[kSlots];
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{} {}

  __device__ __forceinline__ double add(ParamPtr P, const LineLogCtx& cx, const Line&,
                                        const GradNode& nd, double u) {
    const double d = nd.R - P[7];
    const double zc = c.z.at(nd.t);
    const double nu = exp_neg_any(cx.ec, fma(d * d, P[13], fabs(zc) * P[14]));
    const double q = u * nu;
    const double qd = q * d;
    const double mr = qd * nd.inv_R;
    s[0] += mr;
    s[1] = fma(mr, nd.t, s[1]);
    const double mz = q * (zc == 0.0 ? 0.0 : __builtin_copysign(1.0, zc));
    s[2] += mz;
    s[3] = fma(mz, nd.t, s[3]);
    s[4] += qd;
    s[5] = fma(qd, d, s[5]);
    s[6] = fma(q, fabs(zc), s[6]);
    return nu;
  }

  __device__ __forceinline__ void partials(ParamPtr P, double m[4], double* dp) const {
    const double inv_sr2 = P[13], inv_sz = P[14], inv_sr = P[15];
    m[0] = -2.0 * inv_sr2 * s[0];
    m[1] = -2.0 * inv_sr2 * s[1];
    m[2] = -inv_sz * s[2];
    m[3] = -inv_sz * s[3];
    dp[1] = 2.0 * inv_sr2 * s[4];
    dp[2] = 2.0 * inv_sr2 * inv_sr * s[5];
    dp[3] = (inv_sz * inv_sz) * s[6];
  }
};

template <>
struct LineGrad<ZODI_FEATURE> {
  static constexpr int kSlots = 11;
  LineComp<ZODI_FEATURE> c;
  double s[kSlots];
  __device__ __forceinline__ LineGrad(ParamPtr P, const Line& l, double ex, double ey)
      : c(P, l, ex, ey), s{} {}

  template <class CTX>
  __device__ __forceinline__ double add(ParamPtr P, const CTX& cx, const Line& l,
                                        const GradNode& nd, double u) {
    double y, inv_rho2, angle;
    if constexpr (CTX::kAngles) {
      double rho2, inv_rho;
      angle = feature_angle(c, l, *cx.angles, nd.t, y, rho2, inv_rho);
      inv_rho2 = inv_rho * inv_rho;
      inv_rho2 = fma(inv_rho2, fma(-rho2, inv_rho2, 1.0), inv_rho2);
      if (rho2 < 0x1p-900) inv_rho2 = rcp_fast(rho2);  // inv_rho is that of a scaled point
    } else {
      double x = c.x.at(nd.t);
      y = c.y.at(nd.t);
      inv_rho2 = rcp_fast(fma(x, x, y * y));
      if (x == 0.0 && y == 0.0) {  // on the axis: see feature_dtheta
        const double sg = __builtin_signbit(fma(l.vx, nd.t, l.px)) ? -1.0 : 1.0;
        x = sg * c.d.c;
        y = -sg * c.d.s;
      }
      angle = axis_angle(x, y);
    }
    const double th = __builtin_copysign(angle, y);
    const double d = nd.R - P[7];
    const double zc = c.z.at(nd.t);
    double e = (d * d) * P[13];
    e = fma(fabs(zc), P[14], e);
    e = fma(th * th, P[15], e);
    const double nu = exp_neg_any(cx.ec, e);
    const double q = u * nu;
    const double qd = q * d;
    const double mr = qd * nd.inv_R;
    s[0] += mr;
    s[1] = fma(mr, nd.t, s[1]);
    const double mz = q * (zc == 0.0 ? 0.0 : __builtin_copysign(1.0, zc));
    s[2] += mz;
    s[3] = fma(mz, nd.t, s[3]);
    s[4] += qd;
    s[5] = fma(qd, d, s[5]);
    s[6] = fma(q, fabs(zc), s[6]);
    const double qt = q * th;
    s[7] += qt;
    s[8] = fma(qt, th, s[8]);
    const double qr = qt * inv_rho2;
    s[9] += qr;
    s[10] = fma(qr, nd.t, s[10]);
    return nu;
  }

  __device__ __forceinline__ void partials(ParamPtr P, double m[7], double* dp) const {
    const double inv_sr2 = P[13], inv_sz = P[14], inv_sth2 = P[15], inv_sr = P[16],
                 inv_sth = P[17];
    m[0] = -2.0 * inv_sr2 * s[0];
    m[1] = -2.0 * inv_sr2 * s[1];
    m[2] = -inv_sz * s[2];
    m[3] = -inv_sz * s[3];
    m[4] = -2.0 * inv_sth2 * s[9];   // dth / rho^2
    m[5] = -2.0 * inv_sth2 * s[10];  // and times t
    m[6] = -2.0 * inv_sth2 * s[7];   // dth
    dp[1] = 2.0 * inv_sr2 * s[4];
    dp[2] = 2.0 * inv_sr2 * inv_sr * s[5];
    dp[3] = (inv_sz * inv_sz) * s[6];
    dp[4] = 2.0 * inv_sth2 * kDegToRad * s[7];
    dp[5] = 2.0 * inv_sth2 * inv_sth * kDegToRad * s[8];
  }
};

// Partials with respect to x_0, y_0, z_0, i, Omega from the geometry sums of a component
// with centre X0: geo_finish on the coordinate moments that they stand for.
template <bool FEATURE>
__device__ __forceinline__ void line_geo(ParamPtr P, const Line& l, const double* m,
                                         const EarthTerm& et, double out[5]) {
  const double px = l.px - P[ZODI_P_X0], py = l.py - P[ZODI_P_Y0], pz = l.pz - P[ZODI_P_Z0];
  double A[10];
  A[0] = fma(px, m[0], l.vx * m[1]);
  A[1] = fma(py, m[0], l.vy * m[1]);
  A[2] = fma(pz, m[0], l.vz * m[1]);
  A[3] = fma(px, m[2], l.vx * m[3]);
  A[4] = fma(py, m[2], l.vy * m[3]);
  A[5] = fma(pz, m[2], l.vz * m[3]);
  A[6] = m[2];
  if constexpr (FEATURE) {
    A[7] = fma(py, m[4], l.vy * m[5]);
    A[8] = fma(px, m[4], l.vx * m[5]);
    A[9] = m[6];
  }
  geo_finish<FEATURE>(P, A, et, out);
}

// ---------------------------------------------------------------- one group
// Kelsall phase function at the node with its partials (phase_grad) on the line.
__device__ __forceinline__ PhaseGrad line_phase_grad(double theta, const ExpConst& e,
                                                     ParamPtr S) {
  const double C1 = S[ZODI_S_C1], C2 = S[ZODI_S_C2], C3 = S[ZODI_S_C3];
  const double N = S[ZODI_S_PHASE_NORM];
  const double e3 = exp_neg_any(e, -(C3 * theta));
  const double inv_D = kTwoPi * N;
  PhaseGrad o;
  o.phi = N * (C1 + C2 * theta + e3);
  o.d1 = N - o.phi * 2.0 * inv_D;
  o.d2 = N * theta - o.phi * kPi * inv_D;
  o.d3 = N * theta * e3 - o.phi * S[ZODI_S_DD_DC3] * inv_D;
  return o;
}

// Sum over the `split` lanes that share a ray (every lane gets it).
__device__ __forceinline__ double split_sum(double v, int split) {
  for (int off = split >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// The chi^2 pass: a ray's gradient is g = 2 (I - d) / sigma^2 times its derivatives, and I
// is whole only after the last group. So the groups after the first go before it and leave
// their derivatives at unit weight in LDS (kHoldRow doubles a component and thread), and
// group 0, whose sums are still in registers then, forms I and g. Against the Jacobian
// pass and J^T g (78 columns written and read), in us of both: 196 608 rays of DIRBE 250
// -> 212, 400 000 rays of planck13 533 -> 481; the VJP pass with I known takes 209 and 479.
constexpr int kHoldRow = 13;  // most of a later component: the feature's 5 + 6 + 2
template <int NC, int C0>
struct Chi2Ray {
  // first double of component c (not of group 0) in a thread's held derivatives
  static __device__ __forceinline__ int held(int c) { return (c - C0) * kHoldRow * kAdjBlock; }
  double e[NC];  // the components' emission
  double g, chi;
};

// Group g of one ray. sh: the ray's sums for the shared parameters (T0, delta, F, C1..C3),
// weighted in kPassVjp, else at unit weight.
template <int SCAT, int PASS, uint32_t PROPS, int NC, int C0, int... Ks, int... J>
__device__ __forceinline__ void line_adj_group(Grp<Ks...>, std::integer_sequence<int, J...>,
                                               const LineLogCtx& cx, const AdjArgs& a, Ray& y,
                                               int g, int first, double gscale, double* row,
                                               int lane, double (&sh)[6], double& total,
                                               Chi2Ray<NC, C0>& cr, double* hold) {
  constexpr bool JAC = PASS == kPassJac, CHI2 = PASS == kPassChi2;
  constexpr int C = sizeof...(Ks);
  constexpr int kinds[C] = {Ks...};
  const ModelPtr M = cx.M;
  double h, mid;
  group_range(M, g, y, h, mid);
  const double T0 = M->group_T0[g];
  const double half_delta = to_scalar(0.5 * M->group_delta[g]);
  const double us = to_scalar(T0 * M->tab_inv_step);
  const double uo1 = to_scalar(M->tab_T[0] * M->tab_inv_step - 1.0);
  const double solar = M->shared[ZODI_S_SOLAR];
  double st = 0.0, sd = 0.0;  // T0 and delta sums
  double sf[4] = {0.0, 0.0, 0.0, 0.0};
  double s0[C] = {}, s1[C] = {};  // sum w B nu, sum w F Phi / R^2 nu
  // What multiplies nu in the shared sums: amplitude times (1 - a) eps, and times a; with
  // weights per component, the ray's weight too.
  double cn[C], ca[C];
  (
      [&] {
        const ParamPtr P = M->comp[first + J];
        cn[J] = to_scalar(P[ZODI_P_K0] * P[ZODI_P_SCALE]);
        ca[J] = SCAT == 2 ? to_scalar(P[ZODI_P_K0] * P[ZODI_P_ALBEDO]) : 0.0;
        if (PASS == kPassVjp && a.mode == ZODI_ADJ_VJP_COMPS) {
          const double gc = y.active ? a.weights[(int64_t)(first + J) * a.f.n_rays + y.r] : 0.0;
          cn[J] *= gc;
          ca[J] *= gc;
        }
      }(),
      ...);
  std::tuple<LineGrad<Ks>...> lg = [&] {
    const Line l = make_line(y.ux, y.uy, y.uz, y.ox, y.oy, y.oz);
    return std::tuple<LineGrad<Ks>...>{LineGrad<Ks>(M->comp[first + J], l, y.ex, y.ey)...};
  }();
  {
    const Line l = make_line(y.ux, y.uy, y.uz, y.ox, y.oy, y.oz);
    const double tscale = l.n * h, tmid = fma(l.n, mid, l.t0);
    // Phi: see adjoint_group (with every albedo 0 and C2 = C3 = 0 it is a constant)
    const bool need_angle = SCAT == 2 || (SCAT == 1 && (M->shared[ZODI_S_C2] != 0.0 ||
                                                        M->shared[ZODI_S_C3] != 0.0));
    const double phi_const = M->shared[ZODI_S_PHASE_NORM] * (M->shared[ZODI_S_C1] + 1.0);
    LinePhase lp = {0.0, 0.0};
    if (SCAT != 0 && need_angle) lp = line_phase(l);
    const int K = y.active ? cx.K : 0;
    // The next node's abscissa and weight are loaded a node ahead, and the parameters stay
    // in scalar registers: two waves do not cover a load in the loop (2 % on 4.5 M rays).
    double xnext = M->gl_x[cx.sub], wnext = M->gl_w[cx.sub];
    for (int k = cx.sub; k < K; k += cx.split) {
      const double wk = wnext;
      GradNode nd;
      nd.t = fma(tscale, xnext, tmid);
      {
        const int kn = k + cx.split < ZODI_MAX_NODES ? k + cx.split : 0;
        xnext = M->gl_x[kn];
        wnext = M->gl_w[kn];
      }
      nd.R2 = fma(nd.t, nd.t, l.d2);
      norm_and_inverse_node(nd.R2, nd.R, nd.inv_R);
      nd.iR2 = nd.inv_R * nd.inv_R;
      const double lR2 = log_node(cx.tab->log_tab, cx.lc, nd.R2);
      const double Rd = exp_neg_node(cx.ec, half_delta * lR2);  // R^-delta = dT/dT0
      // B and its step over the table interval (0 outside the table): planck_shifted
      const double u1 = fma(Rd, us, -uo1);
      uint32_t j = saturate_u32(u1);
      j = j < (uint32_t)ZODI_N_TEMPS ? j : (uint32_t)ZODI_N_TEMPS;
      const double2 pl = cx.tab->planck[j];
      const double B = fma(__builtin_amdgcn_fract(u1), pl.y, pl.x);
      const double wB = wk * B;
      PhaseGrad pg = {phi_const, 0.0, 0.0, 0.0};
      double ws = 0.0;  // w F Phi / R^2
      if constexpr (SCAT != 0) {
        if (need_angle) {
          double theta;
          if constexpr (SCAT == 2)
            theta = scattering_angle(lp, l, nd.t, *cx.angles, nd.inv_R);
          else
            theta = scattering_angle(lp, l, nd.t);
          pg = line_phase_grad(theta, cx.ec, M->shared);
        }
        ws = wk * ((solar * nd.iR2) * pg.phi);
      }
      double sn = 0.0;  // sum of (1 - a) eps n over the components
      double sa = 0.0;  // sum of a n
      CutShare cs = {0.0, 0.0};  // the published cut-off
      (
          [&] {
            const ParamPtr P = M->comp[first + J];
            auto& A = std::get<J>(lg);
            double u = wB;
            if constexpr (SCAT == 2) u = fma(P[ZODI_P_ALBEDO], ws, P[ZODI_P_SCALE] * wB);
            double nu;
            if constexpr (kinds[J] == ZODI_BAND) {
              constexpr int CUT = cut_mode<PROPS, J, Ks...>();
              CutShare own = {0.0, 0.0};
              nu = A.add(P, cx, nd, CUT == kCutOwn ? own : cs, CUT == kCutReuse && cx.share, u);
            } else {
              nu = A.add(P, static_cast<const AdjCtx<SCAT>&>(cx), l, nd, u);
            }
            s0[J] = fma(wB, nu, s0[J]);
            if constexpr (SCAT != 0) s1[J] = fma(ws, nu, s1[J]);
            sn = fma(cn[J], nu, sn);
            if constexpr (SCAT == 2) sa = fma(ca[J], nu, sa);
          }(),
          ...);
      const double x = (wk * pl.y) * (sn * Rd);
      st += x;
      sd = fma(x, lR2, sd);
      if constexpr (SCAT == 2) {
        const double wa = wk * (sa * nd.iR2);
        sf[0] = fma(wa, pg.phi, sf[0]);
        sf[1] = fma(wa, pg.d1, sf[1]);
        sf[2] = fma(wa, pg.d2, sf[2]);
        sf[3] = fma(wa, pg.d3, sf[3]);
      }
    }
  }

  // The ray's own values again (nothing of them lived across the node loop).
  FwdArgs again = a.f;
  asm volatile("" : "+s"(again.u), "+s"(again.obs), "+s"(again.earth));
  read_ray(again, y);
  const Line l = make_line(y.ux, y.uy, y.uz, y.ox, y.oy, y.oz);
  if (!y.active) h = 0.0;
  const auto sum = [&](double v) { return JAC ? split_sum(v, cx.split) : v; };
  const double wsh = PASS != kPassVjp || a.mode == ZODI_ADJ_VJP_COMPS ? h : h * gscale;
  // Component J's emission over h amp: e = (1 - a) eps B + a F Phi/R^2 (with SCAT 2 already
  // in the sums of the derivatives)
  const auto value = [&](ParamPtr P, double b, double f) {
    return SCAT == 2 ? fma(P[ZODI_P_ALBEDO], f, P[ZODI_P_SCALE] * b) : P[ZODI_P_SCALE] * b;
  };
  if constexpr (CHI2) {
    (
        [&] {
          const ParamPtr P = M->comp[first + J];
          const double b = split_sum(s0[J], cx.split);
          const double f = SCAT == 2 ? split_sum(s1[J], cx.split) : 0.0;
          cr.e[first + J] = h * (P[ZODI_P_K0] * value(P, b, f));
        }(),
        ...);
    if (g == 0) {
#pragma unroll
      for (int c = 0; c < NC; ++c) total = __dadd_rn(total, cr.e[c]);
      cr.g = 0.0;
      cr.chi = 0.0;
      if (y.active) {
        const double iv = a.inv_var != nullptr ? a.inv_var[y.r] : a.inv_var_scalar;
        const double res = total - a.target[y.r];
        if (cx.sub == 0) {
          cr.chi = res * res * iv;
          if (a.model_vals_out != nullptr) a.model_vals_out[y.r] = total;
        }
        cr.g = 2.0 * res * iv;
      }
    }
  }
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
        const double b = sum(s0[J]), f = sum(s1[J]);
        const double amp = P[ZODI_P_K0];
        const double scale = P[ZODI_P_SCALE];
        double W = CHI2 && g == 0 ? h * cr.g : h;
        if (PASS == kPassVjp) {
          W = a.mode == ZODI_ADJ_VJP_COMPS
                  ? (y.active ? h * a.weights[(int64_t)c * a.f.n_rays + y.r] : 0.0)
                  : h * gscale;
        }
        const double We = SCAT == 2 ? W * amp : W * amp * scale;
        double m[7], dp[NP], geo[5];
        A.partials(P, m, dp);
        line_geo<FEATURE>(P, l, m, FEATURE ? earth_term(P, y.ex, y.ey) : EarthTerm{0.0, 0.0},
                          geo);
        const double e0 = value(P, b, f);
        dp[0] = (KIND == ZODI_BAND ? 3.0 : 1.0) * (W * e0);
#pragma unroll
        for (int q = 0; q < 5; ++q) geo[q] *= We;
#pragma unroll
        for (int q = 1; q < NP; ++q) dp[q] *= We;
        const double hb = (W * amp) * b;
        const double de = P[ZODI_P_ONE_MINUS_ALBEDO] * hb;
        const double da = (W * amp) * f - P[ZODI_P_EMISSIVITY] * hb;
        if constexpr (JAC) {
          total = __dadd_rn(total, h * (amp * e0));
          if (y.active && cx.sub == 0) {
            double* col = a.jac + y.r;
            const int64_t ld = a.ld_jac;
            const int off = M->grad_comp[c];
#pragma unroll
            for (int q = 0; q < 5; ++q) col[(off + q) * ld] = geo[q];
#pragma unroll
            for (int q = 0; q < NP; ++q) col[(off + 5 + q) * ld] = dp[q];
            col[M->grad_spec_a[c] * ld] = de;
            col[M->grad_spec_b[c] * ld] = da;
          }
        } else {
          double v[5 + NP + 2];
#pragma unroll
          for (int q = 0; q < 5; ++q) v[q] = geo[q];
#pragma unroll
          for (int q = 0; q < NP; ++q) v[5 + q] = dp[q];
          v[5 + NP] = de;
          v[6 + NP] = da;
          if (CHI2 && g != 0) {
            static_assert(KIND == ZODI_CLOUD || 5 + NP + 2 <= kHoldRow);
#pragma unroll
            for (int q = 0; q < 5 + NP + 2; ++q) hold[cr.held(c) + q * kAdjBlock] = v[q];
            return;
          }
          add_folded(v, row, lane, M->grad_comp[c], M->grad_spec_a[c], M->grad_spec_b[c]);
        }
      }(),
      ...);
  const double inv_step = M->tab_inv_step;
  sh[0] += wsh * (inv_step * sum(st));
  sh[1] += wsh * ((-0.5 * T0 * inv_step) * sum(sd));  // -T0 R^-delta log R
  if constexpr (SCAT == 2) {
    sh[2] += wsh * sum(sf[0]);
#pragma unroll
    for (int q = 1; q < 4; ++q) sh[2 + q] += wsh * (solar * sum(sf[q]));
  }
}

// The held derivatives of a later group's components, weighted onto the wave's row.
template <int NC, int C0, int... Ks, int... J>
__device__ __forceinline__ void add_held(Grp<Ks...>, std::integer_sequence<int, J...>,
                                         ModelPtr M, int first, const Chi2Ray<NC, C0>& cr,
                                         double* row, int lane, const double* hold) {
  constexpr int kinds[sizeof...(Ks)] = {Ks...};
  (
      [&] {
        const int c = first + J;
        double v[5 + kind_nparams<kinds[J]>() + 2];
#pragma unroll
        for (int q = 0; q < 5 + kind_nparams<kinds[J]>() + 2; ++q)
          v[q] = cr.g * hold[cr.held(c) + q * kAdjBlock];
        add_folded(v, row, lane, M->grad_comp[c], M->grad_spec_a[c], M->grad_spec_b[c]);
      }(),
      ...);
}

// Components of a Kelsall layout, and of its group 0.
template <class... Gs>
constexpr int layout_comps(Layout<ZODI_INTEGRAND_KELSALL, Gs...>) {
  return (Gs::size + ...);
}
template <class G0, class... Gs>
constexpr int layout_group0(Layout<ZODI_INTEGRAND_KELSALL, G0, Gs...>) {
  return G0::size;
}

template <int SCAT, int PASS, uint32_t PROPS, class... Gs, int... G>
__device__ __forceinline__ void line_adj_groups(Layout<ZODI_INTEGRAND_KELSALL, Gs...>,
                                                std::integer_sequence<int, G...>,
                                                const LineLogCtx& cx, const AdjArgs& a, Ray& y,
                                                double gscale, double* row, int lane,
                                                double (&sh)[6], double& total, double& chi,
                                                double* hold) {
  using L = Layout<ZODI_INTEGRAND_KELSALL, Gs...>;
  Chi2Ray<layout_comps(L{}), layout_group0(L{})> cr;
  const auto run = [&](auto grp, auto index) {
    constexpr int g = decltype(index)::value, first = group_first<Gs...>(g);
    line_adj_group<SCAT, PASS, props_shift(PROPS, first)>(
        grp, std::make_integer_sequence<int, decltype(grp)::size>{}, cx, a, y, g, first, gscale,
        row, lane, sh, total, cr, hold);
  };
  if constexpr (PASS == kPassChi2) {
    ((G != 0 ? run(Gs{}, std::integral_constant<int, G>{}) : void()), ...);
    ((G == 0 ? run(Gs{}, std::integral_constant<int, G>{}) : void()), ...);
    ((G != 0 ? add_held(Gs{}, std::make_integer_sequence<int, Gs::size>{}, cx.M,
                        group_first<Gs...>(G), cr, row, lane, hold)
             : void()),
     ...);
#pragma unroll
    for (int q = 0; q < 6; ++q) sh[q] *= cr.g;
    chi = cr.chi;
  } else {
    (run(Gs{}, std::integral_constant<int, G>{}), ...);
  }
}

template <int SCAT, int PASS, class... Gs>
__device__ __forceinline__ void line_adj_layout(Layout<ZODI_INTEGRAND_KELSALL, Gs...> lay,
                                                const LineLogCtx& cx, const AdjArgs& a, Ray& y,
                                                double gscale, double* row, int lane,
                                                double (&sh)[6], double& total, double& chi,
                                                double* hold) {
  line_adj_groups<SCAT, PASS, RegistryProps<Layout<ZODI_INTEGRAND_KELSALL, Gs...>>::value>(
      lay, std::make_integer_sequence<int, sizeof...(Gs)>{}, cx, a, y, gscale, row, lane, sh,
      total, chi, hold);
}

// The passes that leave a row: one wave per tile of 64 / a.split rays, whose lanes are
// adjacent; see adjoint_body, whose rows and order of additions these are. Every thread of
// the block must call it, after the tables are built.
template <class RAY>
__device__ __forceinline__ void rows_body(const AdjArgs& a, RAY ray) {
  extern __shared__ double sRows[];  // kAdjWaves rows of n_params + 1
  const int tid = threadIdx.x;
  const int wave = tid / kWave, lane = tid % kWave;
  const int np1 = a.n_params + 1;
  for (int i = tid; i < np1 * kAdjWaves; i += kAdjBlock) sRows[i] = 0.0;
  __syncthreads();
  const int rays = kWave / a.split;
  double* row = sRows + wave * np1;
  const int64_t stride = (int64_t)gridDim.x * kAdjWaves;
  for (int64_t tile = (int64_t)blockIdx.x * kAdjWaves + wave; tile < a.f.n_tiles;
       tile += stride) {
    Ray y = find_ray(a.f, tile * rays, lane / a.split);
    read_ray(a.f, y);
    ray(y, row, lane);
  }
  __syncthreads();
  for (int p = tid; p < np1; p += kAdjBlock) {
    double s = sRows[p];
#pragma unroll
    for (int w = 1; w < kAdjWaves; ++w) s += sRows[w * np1 + p];
    a.partials[(int64_t)blockIdx.x * np1 + p] = s;
  }
}

// The weighted passes, with the weights of a.mode (chi^2: from the stored I).
template <class RAY>
__device__ __forceinline__ void weighted_body(const AdjArgs& a, RAY ray) {
  rows_body(a, [&](Ray& y, double* row, int lane) {
    double gscale = 0.0;
    if (a.mode == ZODI_ADJ_CHI2) {
      double chi = 0.0;
      if (y.active) {
        const double I = a.model_vals[y.r];
        const double iv = a.inv_var != nullptr ? a.inv_var[y.r] : a.inv_var_scalar;
        const double res = I - a.target[y.r];
        chi = (lane & (a.split - 1)) == 0 ? res * res * iv : 0.0;
        gscale = 2.0 * res * iv;
      }
      chi = wave_sum(chi);
      if (lane == 0) row[a.n_params] += chi;
    } else if (a.mode == ZODI_ADJ_VJP_SUM) {
      gscale = y.active ? a.weights[y.r] : 0.0;
    }
    ray(y, gscale, row, lane);
  });
}

// A layout's Jacobian pass (each ray's column and I_r), weighted pass or chi^2 pass.
template <class LAYOUT, int SCAT, int PASS>
__device__ __forceinline__ void line_adj_body(const AdjArgs& a) {
  constexpr int NSH = layout_integrand<LAYOUT>() == ZODI_INTEGRAND_KELSALL ? 6 : 1;
  __shared__ LineLogTables tables;
  const ModelPtr M = as_const(a.f.m);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  __shared__ AngleTable angles;
  AdjCtx<SCAT> cx{line_log_ctx(M, tables, SCAT == 2 ? &angles : nullptr)};
  cx.split = a.split;
  cx.sub = lane & (a.split - 1);
  cx.share = a.share != 0;
  double chi = 0.0;
  if constexpr (PASS == kPassJac) {
    const int rays = kWave / a.split;
    const int64_t stride = (int64_t)gridDim.x * kAdjWaves;
    for (int64_t tile = (int64_t)blockIdx.x * kAdjWaves + wave; tile < a.f.n_tiles;
         tile += stride) {
      Ray y = find_ray(a.f, tile * rays, lane / a.split);
      read_ray(a.f, y);
      double sh[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      double total = 0.0;
      line_adj_layout<SCAT, PASS>(LAYOUT{}, cx, a, y, 1.0, nullptr, lane, sh, total, chi,
                                  nullptr);
      if (y.active && cx.sub == 0) {
        a.model_vals_out[y.r] = total;
#pragma unroll
        for (int q = 0; q < NSH; ++q) a.jac[M->grad_shared[q] * a.ld_jac + y.r] = sh[q];
      }
    }
  } else if constexpr (PASS == kPassChi2) {
    constexpr int kHeld = (layout_comps(LAYOUT{}) - layout_group0(LAYOUT{})) * kHoldRow;
    __shared__ double held[kHeld > 0 ? kHeld * kAdjBlock : 1];
    static_assert(sizeof(g_exp2) + sizeof(tables) + sizeof(angles) + sizeof(held) +
                      (kOnePassParams + 1) * kAdjWaves * sizeof(double) <=
                  kLineAdjLds);
    double* hold = held + (kHeld > 0 ? threadIdx.x : 0);
    rows_body(a, [&](Ray& y, double* row, int ln) {
      double v[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      double sh[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      double total = 0.0;
      line_adj_layout<SCAT, PASS>(LAYOUT{}, cx, a, y, 0.0, row, ln, sh, total, chi, hold);
#pragma unroll
      for (int q = 0; q < 6; ++q) v[q] = sh[q];
      v[6] = chi;
      const double s = wave_fold<32>(v);
      const int i = fold_index(ln);
      if ((ln & 3) == 0 && i < 7) lds_add(row + (i < 6 ? M->grad_shared[i] : a.n_params), s);
    });
  } else {
    weighted_body(a, [&](Ray& y, double gscale, double* row, int ln) {
      double sh[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      double total = 0.0;
      line_adj_layout<SCAT, PASS>(LAYOUT{}, cx, a, y, gscale, row, ln, sh, total, chi, nullptr);
      double v[NSH];
#pragma unroll
      for (int q = 0; q < NSH; ++q) v[q] = sh[q];
      const double s = wave_fold<32>(v);
      const int i = fold_index(ln);
      if ((ln & 3) == 0 && i < NSH) lds_add(row + M->grad_shared[i], s);
    });
  }
}

template <class LAYOUT, int SCAT, int PASS>
__global__ __launch_bounds__(kAdjBlock)
__attribute__((amdgpu_waves_per_eu(kLineAdjWaves, kLineAdjWaves))) void
line_adjoint(AdjArgs a) {
  line_adj_body<LAYOUT, SCAT, PASS>(a);
}

template <class LAYOUT, int SCAT>
AdjKernel pick_line_pass(int pass) {
  return pass == kPassVjp   ? line_adjoint<LAYOUT, SCAT, kPassVjp>
         : pass == kPassJac ? line_adjoint<LAYOUT, SCAT, kPassJac>
                            : line_adjoint<LAYOUT, SCAT, kPassChi2>;
}

template <class LAYOUT>
AdjKernel pick_line_adjoint(int scat, int pass) {
  return scat == 0   ? pick_line_pass<LAYOUT, 0>(pass)
         : scat == 1 ? pick_line_pass<LAYOUT, 1>(pass)
                     : pick_line_pass<LAYOUT, 2>(pass);
}

}  // namespace zodi
