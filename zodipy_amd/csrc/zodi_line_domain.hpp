// Which model blocks the line kernels may take, beside the frames and forms that props_match
// tests: the ranges inside which their tables and exponentials hold. Plain C++, so that a
// host test builds it alone.
#pragma once

#include <cmath>

#include "zodi_hip.h"

namespace zodi {

// false for NaN
inline bool within(double v, double lo, double hi) { return v >= lo && v <= hi; }

// The forward's power tables (PowTable) hold the exponents of a squared radius from 2^-101
// up to 2^155 and of the cloud's g from 2^-254 to 2^2. Offsets and cut-off radii up to 2^60
// AU leave r^2 below 2^124, and a pointing that is not of unit length multiplies the
// distance along it by its length, up to 2^16 then. g is at most 1, or 1 + |mu|/2 for mu < 0.
constexpr double kLineMaxRadius = 0x1p60;
constexpr double kLineMinMu = -4.0;
constexpr double kLineMaxExponent = 5e6;  // beta g^gamma (exp_neg_node)

// Largest size of a parameter or derived constant (of offsets, kLineMaxRadius). NaN and
// infinities do not pass through the line kernels as through the general ones: a NaN tilt
// leaves fmin(|sin beta|, 1) = 1 and fmax(g, floor) finite, a node past a band's edge is not
// multiplied by a NaN amplitude, an infinite R_outer gives log |X| - inf. And an exponent
// takes the square of a distance over a width, which exp_neg_any holds to 1e93. It bounds
// 1/(2 mu) too: g is formed as m^2/(2 mu) + (zeta - m), m = min(zeta, mu), which is NaN where
// 1/(2 mu) is infinite (mu = 0), and the partial with respect to mu squares it.
constexpr double kLineMaxParameter = 1e15;

// Exponent of the temperature law, up to which R^-delta stays finite down to R = 2^-80.
// A NaN temperature law passes (a NaN T makes B NaN).
constexpr double kLineMaxDelta = 12.0;

inline bool line_bounded(const zodi_model* m) {
  for (int c = 0; c < m->n_comps; ++c)
    for (int q = 0; q < ZODI_COMP_SLOTS; ++q) {
      const double most = q <= ZODI_P_Z0 ? kLineMaxRadius : kLineMaxParameter;
      if (!within(m->comp[c][q], -most, most)) return false;
    }
  for (int g = 0; g < m->n_groups; ++g)
    if (std::fabs(m->group_T0[g]) > kLineMaxParameter ||
        std::fabs(m->group_delta[g]) > kLineMaxDelta)
      return false;
  return !(std::fabs(m->shared[ZODI_S_C3]) > kLineMaxParameter);
}

// The cloud's fall-off (component 0 of the Kelsall layouts).
inline bool line_cloud_match(const zodi_model* m) {
  const double* P = m->comp[0];
  const double beta = P[8], gamma = P[9], mu = P[10];
  return mu >= kLineMinMu && within(beta, -1e6, 1e6) &&
         (mu > 0.0 || std::fabs(beta) * std::pow(1.0 - 0.5 * mu, gamma) <= kLineMaxExponent);
}

// Whether a block that meets a layout's registry properties (props_match) may take the line
// kernels that form powers as exp(p log x): the gradients, and the forward and table kernels
// where line_match fails.
inline bool line_log_match(const zodi_model* m) {
  if (!line_bounded(m)) return false;
  if (m->integrand == ZODI_INTEGRAND_RRM) return true;
  const double* P = m->comp[0];
  return line_cloud_match(m) && within(P[7], -1e3, 1e3) && within(P[9], -1e3, 1e3);
}

// Whether the Kelsall forward and table kernels may take their powers from tables: one
// temperature law for all groups, the three exponents inside the ranges in which the
// tables' series holds (PowPoly), the radii inside those of the exponents.
inline bool line_match(const zodi_model* m) {
  if (!line_log_match(m)) return false;
  if (m->integrand == ZODI_INTEGRAND_RRM) return true;
  const auto same = [](double a, double b) { return a == b || (a != a && b != b); };
  const double delta = m->group_delta[0];
  for (int g = 0; g < m->n_groups; ++g) {
    if (!same(m->group_T0[g], m->group_T0[0]) || !same(m->group_delta[g], delta)) return false;
    if (!within(m->group_r_in[g], 0.0, kLineMaxRadius) ||
        !within(m->group_r_out[g], 0.0, kLineMaxRadius))
      return false;
  }
  const double* P = m->comp[0];
  return !(delta > 2.0) && within(P[7], -12.0, 2.0) && within(P[9], 0.5, 6.0);
}

}  // namespace zodi
