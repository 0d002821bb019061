// Which model blocks the line kernels may take, beside the frames and forms that props_match
// tests: the ranges inside which their tables and exponentials hold. Plain C++, so that a
// host test builds it alone. NaN fails every test here.
#pragma once

#include <cmath>

#include "zodi_hip.h"

namespace zodi {

inline bool within(double v, double lo, double hi) { return v >= lo && v <= hi; }

// The forward's power tables (PowTable) hold the exponents of a squared radius from 2^-101
// up to 2^155 and of the cloud's g from 2^-254 to 2^2. Offsets and cut-off radii up to 2^60
// AU leave r^2 below 2^124, and a pointing that is not of unit length multiplies the
// distance along it by its length, up to 2^16 then. g is at most 1, or 1 + |mu|/2 for mu < 0.
constexpr double kLineMaxRadius = 0x1p60;
constexpr double kLineMinMu = -4.0;
constexpr double kLineMaxExponent = 5e6;  // beta g^gamma (exp_neg_node)

// Of 1/(2 mu): g is formed as m^2/(2 mu) + (zeta - m), m = min(zeta, mu), which is NaN where
// 1/(2 mu) is infinite (mu = 0), and the partial with respect to mu squares it.
constexpr double kLineMaxInverse = 1e15;

// The cloud's centre and fall-off (component 0 of the Kelsall layouts).
inline bool line_cloud_match(const zodi_model* m) {
  const double* P = m->comp[0];
  for (int q = ZODI_P_X0; q <= ZODI_P_Z0; ++q)
    if (!within(P[q], -kLineMaxRadius, kLineMaxRadius)) return false;
  const double beta = P[8], gamma = P[9], mu = P[10];
  return mu >= kLineMinMu && within(P[13], -kLineMaxInverse, kLineMaxInverse) &&
         within(beta, -1e6, 1e6) &&
         (mu > 0.0 || std::fabs(beta) * std::pow(1.0 - 0.5 * mu, gamma) <= kLineMaxExponent);
}

// Whether a block that meets a Kelsall layout's registry properties (props_match) may take
// the line kernels: one temperature law for all groups, the three exponents and the radii
// inside the power tables' ranges.
inline bool line_match(const zodi_model* m) {
  for (int g = 0; g < m->n_groups; ++g) {
    if (m->group_T0[g] != m->group_T0[0] || m->group_delta[g] != m->group_delta[0]) return false;
    if (!within(m->group_r_in[g], 0.0, kLineMaxRadius) ||
        !within(m->group_r_out[g], 0.0, kLineMaxRadius))
      return false;
  }
  const double* P = m->comp[0];
  return line_cloud_match(m) && within(m->group_delta[0], -12.0, 2.0) &&
         within(P[7], -12.0, 2.0) && within(P[9], 0.5, 6.0);
}

// The same for the adjoint and Jacobian kernels, which take logarithms instead of tables.
inline bool line_adjoint_match(const zodi_model* m) {
  if (m->integrand == ZODI_INTEGRAND_RRM) return true;
  for (int g = 0; g < m->n_groups; ++g)
    if (!within(m->group_delta[g], -1e3, 1e3)) return false;
  const double* P = m->comp[0];
  return line_cloud_match(m) && within(P[7], -1e3, 1e3) && within(P[9], -1e3, 1e3);
}

}  // namespace zodi
