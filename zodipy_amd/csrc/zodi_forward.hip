// Fused FP64 line-of-sight kernels for MI355X (gfx950) and their C ABI.
//
// One ray per lane (or per group of adjacent lanes, which then split the
// Gauss-Legendre nodes and add their terms in node order). For each ray the
// per-ray sphere-intersection setup runs once; then, per group of components
// sharing a line-of-sight range and temperature law, the node loop evaluates
// position, 1/R, temperature and the Planck lookup once and every component
// density of the group on top, accumulating in registers. The model block is
// read through the constant address space with wave-uniform addresses (scalar
// loads into SGPRs); the Planck table is staged in LDS.
//
// Two kernel families:
//  * forward_layout<Layout, BLOCK, L>: the component kinds of every group are
//    template parameters, so each slot carries only its own density code
//    (registry layouts: DIRBE/planck13, planck15/18/odegard, RRM), with forward_line and
//    forward_rrm for blocks that have the registry models' properties;
//  * forward_generic<BLOCK, L>: any layout the model block can describe; one
//    density switch per slot, per-slot accumulators in LDS.
//
// Reference: zodipy/model.py:253-277 and the functions it calls (see zodi_hip.h).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <utility>

#include "zodi_common.hpp"
#include "zodi_line_rrm.hpp"

namespace zodi {

namespace {
thread_local std::string g_last_error;
}  // namespace




zodi_status fail(zodi_status code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

zodi_status check_hip(hipError_t e, const char* what) {
  if (e != hipSuccess) {
    return fail(ZODI_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  }
  return ZODI_OK;
}

int cu_count() {
  static int counts[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (counts[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0) {
      n = 256;
    }
    counts[dev] = n;
  }
  return counts[dev];
}

zodi_status validate_model(const zodi_model* m) {
  if (m == nullptr) return fail(ZODI_ERR_ARG, "model_host is null");
  if (m->abi_version != ZODI_ABI_VERSION)
    return fail(ZODI_ERR_MODEL, "model abi_version %d, library %d", m->abi_version,
                ZODI_ABI_VERSION);
  if (m->integrand != ZODI_INTEGRAND_KELSALL && m->integrand != ZODI_INTEGRAND_RRM)
    return fail(ZODI_ERR_MODEL, "unknown integrand %d", m->integrand);
  if (m->n_comps < 1 || m->n_comps > ZODI_MAX_COMPS)
    return fail(ZODI_ERR_MODEL, "n_comps %d outside [1, %d]", m->n_comps, ZODI_MAX_COMPS);
  if (m->n_groups < 1 || m->n_groups > ZODI_MAX_GROUPS)
    return fail(ZODI_ERR_MODEL, "n_groups %d outside [1, %d]", m->n_groups, ZODI_MAX_GROUPS);
  if (m->n_nodes < 1 || m->n_nodes > ZODI_MAX_NODES)
    return fail(ZODI_ERR_MODEL, "n_nodes %d outside [1, %d]", m->n_nodes, ZODI_MAX_NODES);
  if (m->n_temps < 2 || m->n_temps > ZODI_N_TEMPS)
    return fail(ZODI_ERR_MODEL, "n_temps %d outside [2, %d]", m->n_temps, ZODI_N_TEMPS);
  int next = 0;
  for (int g = 0; g < m->n_groups; ++g) {
    if (m->group_first[g] != next)
      return fail(ZODI_ERR_MODEL, "group %d starts at %d, expected %d", g, m->group_first[g],
                  next);
    if (m->group_count[g] < 1 || m->group_count[g] > kMaxSlots)
      return fail(ZODI_ERR_MODEL, "group %d has %d components (1..%d)", g, m->group_count[g],
                  kMaxSlots);
    next += m->group_count[g];
  }
  if (next != m->n_comps)
    return fail(ZODI_ERR_MODEL, "groups cover %d components, model has %d", next, m->n_comps);
  for (int c = 0; c < m->n_comps; ++c) {
    if (m->comp_kind[c] < ZODI_CLOUD || m->comp_kind[c] > ZODI_FEATURE_RRM)
      return fail(ZODI_ERR_MODEL, "component %d has unknown kind %d", c, m->comp_kind[c]);
  }
  return ZODI_OK;
}


// Minimum waves per SIMD the register allocator must leave room for, per layout
// (1 = no constraint): the Kelsall layouts at 5 (96 VGPRs; at 4, without the 6-component
// kernel's 10 spilled registers, the batches take the same time within 0.5 %: DIRBE 24.62 and
// 24.55 ms, planck18 6.19 and 6.22), RRM at 4 (110 VGPRs, no spill; at 5 it is 1 % slower).
// The kind switch (forward_generic) runs at 3. The split-lane variants (L > 1) run only where
// the launch is small, so they ask for 2 and keep their registers.
template <class LAYOUT>
struct ForwardOccupancy {
  static constexpr int value = 1;
};
template <>
struct ForwardOccupancy<LayoutDirbe> {
  static constexpr int value = 5;
};
template <>
struct ForwardOccupancy<LayoutRRM> {
  static constexpr int value = 4;
};
template <>
struct ForwardOccupancy<LayoutRRMSplit> {
  static constexpr int value = 4;
};
template <>
struct ForwardOccupancy<LayoutKelsall4> {
  static constexpr int value = 5;
};

// A layout whose components' frames are tested per node: blocks that the line kernels do
// not take (an offset component, a band with p other than 4).
template <class LAYOUT, int BLOCK, int L>
__global__ __launch_bounds__(BLOCK)
__attribute__((amdgpu_waves_per_eu(L == 1 ? ForwardOccupancy<LAYOUT>::value : 2))) void
forward_layout(FwdArgs a) {
  __shared__ double sTab[4 * ZODI_N_TEMPS];
  const ModelPtr M = as_const(a.m);
  stage_math_tables();
  load_table(M, sTab);
  const Ctx cx = make_ctx(M, sTab, threadIdx.x % L);
  constexpr int RAYS = BLOCK / L;
  const int local = threadIdx.x / L;
  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    const Ray y = load_ray<RAYS>(a, tile, local);
    double total = 0.0;
    run_layout<L>(LAYOUT{}, cx, a, y, total);
    if (a.out_mode == ZODI_OUT_SUM && y.active && cx.sub == 0) a.out[y.r] = total;
  }
}

// The context of a forward line kernel and its tables in LDS (every thread must call it).
template <bool LOGS>
__device__ __forceinline__ auto line_tables(ModelPtr M, int sub) {
  if constexpr (LOGS) {
    __shared__ LineLogTables tables;
    __shared__ AngleTable angles;
    LineLogCtx cx = line_log_ctx(M, tables, &angles);
    cx.sub = sub;
    return cx;
  } else {
    __shared__ LineTables tables;
    return line_ctx(M, tables, sub);
  }
}

// The Kelsall layouts' registry blocks (props_match without the shared cut-off, and
// line_log_match) on the ray's line (zodi_line.hpp): bound by FP64 vector issue, 339 vector
// instructions a ray and node of the DIRBE layout where forming every node's position and
// its powers by exp(p log x) took 487. Measured: DIRBE 12 um, 50.7 M rays, 35.0 -> 24.8 ms
// (7.2e10 -> 1.02e11 ray-nodes/s); planck18 857 GHz, 22.5 M rays, 8.38 -> 6.22 ms; DIRBE
// 1.25 um with scattering, 196 608 rays, 0.321 -> 0.223 ms (compiled for 4 waves a SIMD,
// without spills: 214 -> 200 us of kernel against 5). SHARE: the bands that share a radial
// cut-off reuse it (kShareCut), for blocks whose delta_r values allow it (the registry
// parameters; a fit that moves them runs without). NOSCAT (with SHARE): no component
// scatters, so no scattering code is compiled in. LOGS (without NOSCAT): powers by
// logarithms, for exponents that the tables do not hold (line_match): 1 M rays at alpha =
// 2.5 623 us, with tables at 1.34 510.
template <class LAYOUT, int BLOCK, bool SHARE, bool NOSCAT, bool LOGS = false>
__global__ __launch_bounds__(BLOCK)
__attribute__((amdgpu_waves_per_eu(NOSCAT ? ForwardOccupancy<LAYOUT>::value : 4))) void
forward_line(FwdArgs a) {
  const auto cx = line_tables<LOGS>(as_const(a.m), 0);
  constexpr uint32_t kProps = SHARE ? RegistryProps<LAYOUT>::value
                                    : props_without_share(RegistryProps<LAYOUT>::value);
  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    Ray y = load_ray<BLOCK>(a, tile, threadIdx.x);
    double total = 0.0;
    run_line<1, kProps, NOSCAT>(LAYOUT{}, cx, a, y, nullptr, total);
    if (a.out_mode == ZODI_OUT_SUM && y.active) a.out[y.r] = total;
  }
}

// The same for small launches, a.lanes lanes per ray (2 to 32).
template <class LAYOUT, int SPLIT, bool SHARE, bool NOSCAT, bool LOGS = false>
__global__ __launch_bounds__(kSplitBlock) __attribute__((amdgpu_waves_per_eu(2))) void
forward_line_split(FwdArgs a) {
  __shared__ double2 terms[SPLIT == 8 ? kMaxSlots * kSplitStride : 1];
  const int lanes = SPLIT == 8 ? a.lanes : SPLIT;
  const auto cx = line_tables<LOGS>(as_const(a.m), threadIdx.x & (lanes - 1));
  constexpr uint32_t kProps = SHARE ? RegistryProps<LAYOUT>::value
                                    : props_without_share(RegistryProps<LAYOUT>::value);
  const int rays = blockDim.x / lanes;
  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    Ray y = find_ray(a, tile * rays, threadIdx.x / lanes);
    read_ray(a, y);
    double total = 0.0;
    run_line<SPLIT, kProps, NOSCAT>(LAYOUT{}, cx, a, y, terms, total);
    if (a.out_mode == ZODI_OUT_SUM && y.active && cx.sub == 0) a.out[y.r] = total;
  }
}

// The RRM layouts' registry blocks (every component centred) on the ray's line: 3580 issue
// cycles per wave and node over the six groups where the arc sines, sines, cosines and
// powers of every node took 6750 (and less where a wave skips a branch). Measured: RRM 25
// um, 196 608 rays with the pixel vectors, 0.532 -> 0.309 ms (two lanes a ray).
template <class LAYOUT, int BLOCK>
__global__ __launch_bounds__(BLOCK)
__attribute__((amdgpu_waves_per_eu(ForwardOccupancy<LAYOUT>::value))) void
forward_rrm(FwdArgs a) {
  __shared__ LineLogTables tables;
  __shared__ AngleTable angles;
  const LineLogCtx cx = line_log_ctx(as_const(a.m), tables, &angles);
  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    const Ray y = load_ray<BLOCK>(a, tile, threadIdx.x);
    double total = 0.0;
    run_rrm<1>(LAYOUT{}, cx, a, y, nullptr, total);
    if (a.out_mode == ZODI_OUT_SUM && y.active) a.out[y.r] = total;
  }
}

template <class LAYOUT, int SPLIT>
__global__ __launch_bounds__(kSplitBlock) __attribute__((amdgpu_waves_per_eu(2))) void
forward_rrm_split(FwdArgs a) {
  __shared__ LineLogTables tables;
  __shared__ double2 terms[SPLIT == 8 ? kMaxSlots * kSplitStride : 1];
  __shared__ AngleTable angles;
  LineLogCtx cx = line_log_ctx(as_const(a.m), tables, &angles);
  const int lanes = SPLIT == 8 ? a.lanes : SPLIT;
  cx.sub = threadIdx.x & (lanes - 1);
  const int rays = blockDim.x / lanes;
  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    Ray y = find_ray(a, tile * rays, threadIdx.x / lanes);
    read_ray(a, y);
    double total = 0.0;
    run_rrm<SPLIT>(LAYOUT{}, cx, a, y, terms, total);
    if (a.out_mode == ZODI_OUT_SUM && y.active && cx.sub == 0) a.out[y.r] = total;
  }
}

// ------------------------------------------------------------ generic kernel
template <int INTEGRAND, int BLOCK>
__device__ __forceinline__ void generic_groups(const Ctx& cx, const FwdArgs& a, const Ray& y,
                                               double (*sAcc)[BLOCK], int tid, int L,
                                               double& total) {
  const ModelPtr M = cx.M;
  const int n_groups = M->n_groups;
  for (int g = 0; g < n_groups; ++g) {
    const int first = M->group_first[g];
    const int cnt = M->group_count[g];
    double h, mid;
    group_range(M, g, y, h, mid);
    const double T0 = M->group_T0[g];
    const double mdelta = -M->group_delta[g];
    const double us = T0 * cx.tb.inv_step;
    const double uo = cx.tb.T_first * cx.tb.inv_step;
    bool scatter = false;
    for (int j = 0; j < cnt; ++j) {
      sAcc[j][tid] = 0.0;
      scatter = scatter || (M->comp_flags[first + j] & ZODI_CF_SCATTER);
    }
    // L lanes evaluate L consecutive nodes; each lane adds the L terms in node
    // order (as forward_layout does), past the last node repeating it unadded.
    for (int k0 = 0; k0 < cx.K; k0 += L) {
      const int k = k0 + cx.sub < cx.K ? k0 + cx.sub : cx.K - 1;
      const int left = cx.K - k0;
      const double xk = M->gl_x[k];
      const double wk = M->gl_w[k];
      Node nd = node_geometry(y, h, mid, xk, us, uo, mdelta, cx.tb);
      if (INTEGRAND == ZODI_INTEGRAND_KELSALL && scatter) {
        nd.phi = phase_function(h * xk + mid, y.ux, y.uy, y.uz, nd.X0, nd.X1, nd.X2, nd.R,
                                M->shared);
      }
      const double wB = wk * nd.B;
#pragma unroll 1
      for (int j = 0; j < cnt; ++j) {
        const int c = first + j;
        const ParamPtr P = M->comp[c];
        const uint32_t flags = M->comp_flags[c];
        const int kind = M->comp_kind[c];
        const FeatureDir fd = is_feature(kind) ? feature_dir(P, y.ex, y.ey) : FeatureDir{1.0, 0.0};
        const double dens =
            density(kind, P, flags, nd.X0, nd.X1, nd.X2, nd.R, nd.inv_R, nd.R2, fd);
        const NodeTerm t = node_term<INTEGRAND>(P, flags, nd, wk, wB, dens, cx.solar);
        double acc = sAcc[j][tid];
        if (L == 1) {
          acc = node_add(acc, t);
        } else {
          for (int s = 0; s < L && s < left; ++s)
            acc = node_add(acc, NodeTerm{__shfl(t.a, s, L), __shfl(t.b, s, L)});
        }
        sAcc[j][tid] = acc;
      }
    }
    for (int j = 0; j < cnt; ++j) {
      const double acc = sAcc[j][tid];
      const double e = finish<INTEGRAND>(M->comp[first + j], M->comp_flags[first + j], acc, h,
                                         cx.calibration);
      if (a.out_mode == ZODI_OUT_COMPS) {
        if (y.active && cx.sub == 0) a.out[(int64_t)(first + j) * a.n_rays + y.r] = e;
      } else {
        total = __dadd_rn(total, e);
      }
    }
  }
}

// Three waves per SIMD (167-168 VGPRs, up to a 16-byte spill with split lanes):
// 22-30 % faster than the unconstrained 169-175 VGPRs at two (DIRBE through the
// kind switch on 196 608 to 3.1 M rays; the same on 49 152).
template <int BLOCK, int L>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(3))) void
forward_generic(FwdArgs a) {
  __shared__ double sTab[4 * ZODI_N_TEMPS];
  __shared__ double sAcc[kMaxSlots][BLOCK];  // one node sum per lane and component slot
  const ModelPtr M = as_const(a.m);
  stage_math_tables();
  load_table(M, sTab);
  const int tid = threadIdx.x;
  const Ctx cx = make_ctx(M, sTab, tid % L);
  constexpr int RAYS = BLOCK / L;
  const int local = tid / L;
  const bool kelsall = M->integrand == ZODI_INTEGRAND_KELSALL;
  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    const Ray y = load_ray<RAYS>(a, tile, local);
    double total = 0.0;
    if (kelsall) {
      generic_groups<ZODI_INTEGRAND_KELSALL>(cx, a, y, sAcc, tid, L, total);
    } else {
      generic_groups<ZODI_INTEGRAND_RRM>(cx, a, y, sAcc, tid, L, total);
    }
    if (a.out_mode == ZODI_OUT_SUM && y.active && cx.sub == 0) a.out[y.r] = total;
  }
}

// Per-group start/stop distances (zodipy/line_of_sight.py:88-105).
__global__ __launch_bounds__(256) void line_of_sight_kernel(FwdArgs a, double* __restrict__ start,
                                                            double* __restrict__ stop) {
  const ModelPtr M = as_const(a.m);
  const int64_t n = a.n_rays;
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  int64_t s = a.obs_mode == ZODI_OBS_PER_RAY ? r : find_segment(a.seg, a.n_seg, r);
  const uint32_t bits = a.beyond[a.obs_mode == ZODI_OBS_PER_RAY ? 0 : s];
  const int64_t os = a.obs_stride;
  const RayGeom G = ray_geometry(a.u[r], a.u[n + r], a.u[2 * n + r], a.obs[s], a.obs[os + s],
                                 a.obs[2 * os + s]);
  for (int g = 0; g < M->n_groups; ++g) {
    start[(int64_t)g * n + r] =
        ((bits >> (2 * g)) & 1u) ? kEps : sphere_distance(G, M->group_r_in[g]);
    stop[(int64_t)g * n + r] =
        ((bits >> (2 * g + 1)) & 1u) ? kEps : sphere_distance(G, M->group_r_out[g]);
  }
}

// Component densities at heliocentric points (zodipy/number_density.py:47-420).
__global__ __launch_bounds__(256) void number_density_kernel(const zodi_model* model,
                                                             const double* __restrict__ X,
                                                             int64_t n, const double* earth,
                                                             double* __restrict__ out) {
  const ModelPtr M = as_const(model);
  stage_math_tables();
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double x0 = X[i], x1 = X[n + i], x2 = X[2 * n + i];
  const double R2 = x0 * x0 + x1 * x1 + x2 * x2;
  double R, inv_R;
  norm_and_inverse(R2, R, inv_R);
  if (R2 == 0.0) {  // the Sun's centre (a grid may hold it): R = 0 as sqrt gives it
    R = 0.0;
    inv_R = __builtin_inf();
  }
  const double ex = earth[0], ey = earth[1];
  for (int c = 0; c < M->n_comps; ++c) {
    const ParamPtr P = M->comp[c];
    const int kind = M->comp_kind[c];
    const FeatureDir fd = is_feature(kind) ? feature_dir(P, ex, ey) : FeatureDir{1.0, 0.0};
    out[(int64_t)c * n + i] = density(kind, P, M->comp_flags[c], x0, x1, x2, R, inv_R, R2, fd);
  }
}

namespace {

using FwdKernel = void (*)(FwdArgs);

template <class LAYOUT, int BLOCK>
FwdKernel pick_layout_lanes(int L) {
  switch (L) {
    case 1:
      return forward_layout<LAYOUT, BLOCK, 1>;
    case 2:
      return forward_layout<LAYOUT, BLOCK, 2>;
    case 4:
      return forward_layout<LAYOUT, BLOCK, 4>;
    case 8:
      return forward_layout<LAYOUT, BLOCK, 8>;
    default:
      return nullptr;
  }
}

template <class LAYOUT>
FwdKernel pick_layout_block(int block, int L) {
  switch (block) {
    case 64:
      return pick_layout_lanes<LAYOUT, 64>(L);
    case 128:
      return pick_layout_lanes<LAYOUT, 128>(L);
    case 256:
      return pick_layout_lanes<LAYOUT, 256>(L);
    case 512:
      return pick_layout_lanes<LAYOUT, 512>(L);
    default:
      return nullptr;
  }
}

template <class LAYOUT>
FwdKernel pick_rrm(int block, int L) {
  if (block != 256 && block != 512) return nullptr;
  if (L == 2) return forward_rrm_split<LAYOUT, 2>;
  if (L == 4) return forward_rrm_split<LAYOUT, 4>;
  if (L > 4) return forward_rrm_split<LAYOUT, 8>;
  return block == 256 ? forward_rrm<LAYOUT, 256> : forward_rrm<LAYOUT, 512>;
}

// Whether no component of the block has its scattering term (ZODI_CF_SCATTER).
inline bool no_scattering(const zodi_model* m) {
  for (int c = 0; c < m->n_comps; ++c)
    if (m->comp_flags[c] & ZODI_CF_SCATTER) return false;
  return true;
}

template <class LAYOUT, bool SHARE, bool NOSCAT, bool LOGS = false>
FwdKernel pick_line_block(int block, int L) {
  if (block != 256 && block != 512) return nullptr;
  if (L == 2) return forward_line_split<LAYOUT, 2, SHARE, NOSCAT, LOGS>;
  if (L == 4) return forward_line_split<LAYOUT, 4, SHARE, NOSCAT, LOGS>;
  if (L > 4) return forward_line_split<LAYOUT, 8, SHARE, NOSCAT, LOGS>;
  return block == 256 ? forward_line<LAYOUT, 256, SHARE, NOSCAT, LOGS>
                      : forward_line<LAYOUT, 512, SHARE, NOSCAT, LOGS>;
}

template <class LAYOUT>
FwdKernel pick_line(const zodi_model* m, int block, int L) {
  const bool share = props_match(m, RegistryProps<LAYOUT>::value);
  if (!line_match(m))
    return share ? pick_line_block<LAYOUT, true, false, true>(block, L)
                 : pick_line_block<LAYOUT, false, false, true>(block, L);
  if (!share) return pick_line_block<LAYOUT, false, false>(block, L);
  return no_scattering(m) ? pick_line_block<LAYOUT, true, true>(block, L)
                          : pick_line_block<LAYOUT, true, false>(block, L);
}

// The line kernels when the block has the layout's registry properties (the Kelsall
// layouts: with the shared cut-offs where the delta_r values allow it, and then without
// scattering code when no component scatters), else the one that tests each component's
// flags.
template <class LAYOUT>
bool line_eligible(const zodi_model* m) {
  return props_match(m, props_without_share(RegistryProps<LAYOUT>::value)) && line_log_match(m);
}

bool takes_line(const zodi_model* m, LayoutId id) {
  switch (id) {
    case kLayoutDirbe:
      return line_eligible<LayoutDirbe>(m);
    case kLayoutKelsall4:
      return line_eligible<LayoutKelsall4>(m);
    case kLayoutRRM:
      return line_eligible<LayoutRRM>(m);
    case kLayoutRRMSplit:
      return line_eligible<LayoutRRMSplit>(m);
    default:
      return false;
  }
}

template <class LAYOUT>
FwdKernel pick_layout(const zodi_model* m, int block, int L) {
  if (line_eligible<LAYOUT>(m)) {
    if constexpr (layout_integrand<LAYOUT>() == ZODI_INTEGRAND_KELSALL) {
      return pick_line<LAYOUT>(m, block, L);
    } else {
      return pick_rrm<LAYOUT>(block, L);
    }
  }
  return pick_layout_block<LAYOUT>(block, L);
}

template <int BLOCK>
FwdKernel pick_generic_lanes(int L) {
  switch (L) {
    case 1:
      return forward_generic<BLOCK, 1>;
    case 2:
      return forward_generic<BLOCK, 2>;
    case 4:
      return forward_generic<BLOCK, 4>;
    case 8:
      return forward_generic<BLOCK, 8>;
    default:
      return nullptr;
  }
}

FwdKernel pick_generic(int block, int L) {
  switch (block) {
    case 64:
      return pick_generic_lanes<64>(L);
    case 128:
      return pick_generic_lanes<128>(L);
    case 256:
      return pick_generic_lanes<256>(L);
    case 512:
      return pick_generic_lanes<512>(L);
    default:
      return nullptr;
  }
}

constexpr int kGenericWaves = 3;

// Resident waves per SIMD of the kernel pick_forward chooses.
int forward_waves(const zodi_model* m, int variant) {
  switch (variant == 0 ? kLayoutGeneric : match_layout(m)) {
    case kLayoutDirbe:
      return ForwardOccupancy<LayoutDirbe>::value;
    case kLayoutKelsall4:
      return ForwardOccupancy<LayoutKelsall4>::value;
    case kLayoutRRM:
      return ForwardOccupancy<LayoutRRM>::value;
    case kLayoutRRMSplit:
      return ForwardOccupancy<LayoutRRMSplit>::value;
    default:
      return kGenericWaves;
  }
}

// Lanes per ray when the caller leaves it open: the node terms are added in node order
// whatever the split, so it only sets the speed.
//
// The line kernels: with r waves of L lanes a ray on a SIMD and K nodes a ray, a launch
// takes (r + 1) (ceil(K / L) + 4) units within some 10 % (4: a wave's work beside its
// nodes; 1: the latency of its chains, which r waves share; below two waves it shows in
// full), and the cheapest L is taken. Measured with 50 nodes (us, up to 8 lanes with the
// sums fetched by ds_bpermute -> this rule; DIRBE, then RRM): 3072 rays 33 -> 14 and
// 48 -> 21, 12 288 rays 43 -> 22 and 57 -> 38, 49 152 rays 67 -> 43 and 101 -> 92,
// 150 000 rays 141 -> 108 and 297 -> 244. Past 5 waves a SIMD the Kelsall kernels of one
// lane a ray, which keep 5, are as fast or faster (196 608 rays: 123 at 1, 126 at 2); the
// RRM kernels, which keep 4, up to 8 (196 608 rays: 298 at 1, 282 at 2).
//
// The general kernel: up to 8 lanes while the waves still fit the resident slots.
int default_lanes(const zodi_model* m, int variant, int64_t n_rays) {
  const LayoutId id = variant == 0 ? kLayoutGeneric : match_layout(m);
  const int64_t simds = (int64_t)4 * cu_count();
  if (takes_line(m, id)) {
    const int most = id == kLayoutDirbe || id == kLayoutKelsall4 ? 5 : 8;
    int best = 1;
    int64_t least = INT64_MAX;
    for (int L : {1, 2, 4, 8, 16, 32}) {
      const int64_t waves = (n_rays * L + 63) / 64, r = (waves + simds - 1) / simds;
      if (L > 1 && r > most) break;
      const int64_t cost = (std::max<int64_t>(r, 2) + 1) * ((m->n_nodes + L - 1) / L + 4);
      if (cost <= least) {
        least = cost;
        best = L;
      }
    }
    return best;
  }
  const int64_t slots = forward_waves(m, variant) * simds;
  for (int L : {8, 4, 2})
    if ((n_rays * L + 63) / 64 <= slots) return L;
  return 1;
}

// The line kernels' tables take 10 KB of LDS a block (logarithms, RRM) or 24 KB (power tables),
// the terms of 8 lanes a ray and more 33 KB besides, so that blocks of 64 and 128 threads would
// leave a CU with few waves: smaller requests run as 256.
constexpr int kLineMinBlock = 256;

FwdKernel pick_forward(const zodi_model* m, int& block, int L, int variant) {
  const LayoutId id = variant == 0 ? kLayoutGeneric : match_layout(m);
  if (takes_line(m, id) && (block == 64 || block == 128)) block = kLineMinBlock;
  switch (id) {
    case kLayoutDirbe:
      return pick_layout<LayoutDirbe>(m, block, L);
    case kLayoutKelsall4:
      return pick_layout<LayoutKelsall4>(m, block, L);
    case kLayoutRRM:
      return pick_layout<LayoutRRM>(m, block, L);
    case kLayoutRRMSplit:
      return pick_layout<LayoutRRMSplit>(m, block, L);
    default:
      return pick_generic(block, L);
  }
}

// See zodi_forward_route.
int forward_route(const zodi_model* m, int variant) {
  const LayoutId id = variant == 0 ? kLayoutGeneric : match_layout(m);
  if (id == kLayoutGeneric) return ZODI_ROUTE_GENERIC;
  if (!takes_line(m, id)) return ZODI_ROUTE_LAYOUT;
  int route = line_match(m) ? ZODI_ROUTE_LINE : ZODI_ROUTE_LINE_LOGS;
  if (no_scattering(m)) route |= ZODI_ROUTE_NO_SCATTERING;
  const bool share =
      (id == kLayoutDirbe && props_match(m, RegistryProps<LayoutDirbe>::value)) ||
      (id == kLayoutKelsall4 && props_match(m, RegistryProps<LayoutKelsall4>::value));
  return share ? route | ZODI_ROUTE_SHARED_CUT : route;
}

zodi_status fill_args(FwdArgs& a, const zodi_model* model_host, const zodi_model* model_dev,
                      const double* u, int64_t n_rays, const int64_t* seg_offsets, int32_t n_seg,
                      const double* obs, const double* earth, int32_t obs_mode,
                      const uint32_t* beyond) {
  zodi_status st = validate_model(model_host);
  if (st != ZODI_OK) return st;
  if (model_dev == nullptr) return fail(ZODI_ERR_ARG, "model_dev is null");
  if (n_rays < 0) return fail(ZODI_ERR_ARG, "n_rays %lld < 0", (long long)n_rays);
  if (u == nullptr || obs == nullptr || earth == nullptr || beyond == nullptr)
    return fail(ZODI_ERR_ARG, "null input pointer");
  if (obs_mode == ZODI_OBS_PER_SEGMENT) {
    if (seg_offsets == nullptr || n_seg < 1)
      return fail(ZODI_ERR_ARG, "per-segment mode needs seg_offsets and n_seg >= 1");
  } else if (obs_mode != ZODI_OBS_PER_RAY) {
    return fail(ZODI_ERR_ARG, "unknown obs_mode %d", obs_mode);
  }
  a.m = model_dev;
  a.u = u;
  a.n_rays = n_rays;
  a.seg = seg_offsets;
  a.n_seg = n_seg;
  a.obs_mode = obs_mode;
  a.obs = obs;
  a.earth = earth;
  a.obs_stride = obs_mode == ZODI_OBS_PER_RAY ? n_rays : n_seg;
  a.beyond = beyond;
  a.out = nullptr;
  a.out_mode = 0;
  a.lanes = 1;
  a.n_tiles = 0;
  return ZODI_OK;
}

}  // namespace
}  // namespace zodi

using namespace zodi;

extern "C" {

int32_t zodi_abi_version(void) { return ZODI_ABI_VERSION; }

int64_t zodi_model_size(void) { return (int64_t)sizeof(zodi_model); }

const char* zodi_last_error(void) { return g_last_error.c_str(); }

int32_t zodi_forward_route(const zodi_model* model_host, int32_t variant) {
  if (model_host == nullptr || validate_model(model_host) != ZODI_OK) return -1;
  return forward_route(model_host, variant);
}

zodi_status zodi_forward(const zodi_model* model_host, const zodi_model* model_dev,
                         const double* u, int64_t n_rays, const int64_t* seg_offsets,
                         int32_t n_seg, const double* obs, const double* earth, int32_t obs_mode,
                         const uint32_t* beyond, double* out, int32_t out_mode,
                         const zodi_launch* launch, void* stream) {
  FwdArgs a;
  zodi_status st = fill_args(a, model_host, model_dev, u, n_rays, seg_offsets, n_seg, obs, earth,
                             obs_mode, beyond);
  if (st != ZODI_OK) return st;
  if (out == nullptr) return fail(ZODI_ERR_ARG, "out is null");
  if (out_mode != ZODI_OUT_COMPS && out_mode != ZODI_OUT_SUM)
    return fail(ZODI_ERR_ARG, "unknown out_mode %d", out_mode);
  if (n_rays == 0) return ZODI_OK;

  int block = 256, L = 0, per_cu = 0, variant = 1;
  if (launch != nullptr) {
    if (launch->block) block = launch->block;
    L = launch->lanes_per_ray;
    per_cu = launch->blocks_per_cu;
    variant = launch->variant;
  }
  if (variant < 0 || variant > 1) return fail(ZODI_ERR_ARG, "unknown variant %d", variant);
  if (L < 0) return fail(ZODI_ERR_ARG, "lanes_per_ray %d < 0", L);
  if (L > block) return fail(ZODI_ERR_ARG, "lanes_per_ray %d > block %d", L, block);
  const bool lanes_ok = L <= 8 && (L & (L - 1)) == 0;  // 16 and 32 are the default's own
  if (L == 0) L = std::min(default_lanes(model_host, variant, n_rays), block);
  FwdKernel k = lanes_ok ? pick_forward(model_host, block, L, variant) : nullptr;
  if (k == nullptr)
    return fail(ZODI_ERR_ARG, "unsupported launch: block %d, lanes_per_ray %d", block, L);
  if (per_cu < 0 || per_cu > 64)
    return fail(ZODI_ERR_ARG, "blocks_per_cu %d outside [0, 64]", per_cu);

  const int64_t rays_per_block = block / L;
  const int64_t n_tiles = (n_rays + rays_per_block - 1) / rays_per_block;
  int64_t grid = n_tiles;
  if (per_cu > 0) grid = std::min<int64_t>(grid, (int64_t)per_cu * cu_count());
  if (grid > 0x7fffffff) return fail(ZODI_ERR_TOO_LARGE, "grid of %lld blocks", (long long)grid);
  a.out = out;
  a.out_mode = out_mode;
  a.lanes = L;
  a.n_tiles = n_tiles;
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(block), 0, (hipStream_t)stream, a);
  return check_hip(hipGetLastError(), "forward launch");
}

zodi_status zodi_host_device_pointer(const void* host, void** device) {
  if (host == nullptr || device == nullptr) return fail(ZODI_ERR_ARG, "null pointer");
  *device = nullptr;
  hipPointerAttribute_t attr;
  hipError_t e = hipPointerGetAttributes(&attr, host);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return fail(ZODI_ERR_ARG, "%p is not memory known to HIP (%s)", host, hipGetErrorString(e));
  }
  if (attr.type != hipMemoryTypeHost)
    return fail(ZODI_ERR_ARG, "%p is not page-locked host memory (memory type %d)", host,
                (int)attr.type);
  void* d = nullptr;
  e = hipHostGetDevicePointer(&d, const_cast<void*>(host), 0);
  if (e != hipSuccess || d == nullptr) {
    (void)hipGetLastError();
    return fail(ZODI_ERR_ARG, "no device mapping for host memory %p (%s)", host,
                hipGetErrorString(e));
  }
  *device = d;
  return ZODI_OK;
}

zodi_status zodi_line_of_sight(const zodi_model* model_host, const zodi_model* model_dev,
                               const double* u, int64_t n_rays, const int64_t* seg_offsets,
                               int32_t n_seg, const double* obs, int32_t obs_mode,
                               const uint32_t* beyond, double* start, double* stop,
                               void* stream) {
  FwdArgs a;
  zodi_status st = fill_args(a, model_host, model_dev, u, n_rays, seg_offsets, n_seg, obs, obs,
                             obs_mode, beyond);
  if (st != ZODI_OK) return st;
  if (start == nullptr || stop == nullptr) return fail(ZODI_ERR_ARG, "null output pointer");
  if (n_rays == 0) return ZODI_OK;
  const int64_t grid = (n_rays + 255) / 256;
  if (grid > 0x7fffffff) return fail(ZODI_ERR_TOO_LARGE, "too many rays");
  hipLaunchKernelGGL(line_of_sight_kernel, dim3((unsigned)grid), dim3(256), 0,
                     (hipStream_t)stream, a, start, stop);
  return check_hip(hipGetLastError(), "line_of_sight launch");
}

zodi_status zodi_number_density(const zodi_model* model_host, const zodi_model* model_dev,
                                const double* X, int64_t n_points, const double* earth,
                                double* out, void* stream) {
  zodi_status st = validate_model(model_host);
  if (st != ZODI_OK) return st;
  if (model_dev == nullptr || X == nullptr || earth == nullptr || out == nullptr)
    return fail(ZODI_ERR_ARG, "null pointer");
  if (n_points < 0) return fail(ZODI_ERR_ARG, "n_points < 0");
  if (n_points == 0) return ZODI_OK;
  const int64_t grid = (n_points + 255) / 256;
  if (grid > 0x7fffffff) return fail(ZODI_ERR_TOO_LARGE, "too many points");
  hipLaunchKernelGGL(number_density_kernel, dim3((unsigned)grid), dim3(256), 0,
                     (hipStream_t)stream, model_dev, X, n_points, earth, out);
  return check_hip(hipGetLastError(), "number_density launch");
}

}  // extern "C"

