// Point kernels of libtbx for one Chebyshev degree.  This file is compiled
// once per degree with -DTBX_Q=<q>; each build defines the launchers
// launch_{eval,traj,step}_q<q> declared in tbx_internal.h.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "tbx_device.h"
#include "tbx_mfma.h"
#include "tbx_rows.h"

#ifndef TBX_Q
#error "compile with -DTBX_Q=<degree>"
#endif

namespace tbx {
namespace {

constexpr int D = TBX_Q + 1;

// Waves per SIMD asked of the row kernels: the basis in registers, 2 D
// values, leaves FP64 four up to degree 9 and three above, FP32 five and
// four.  Nothing is spilled but in the step through four velocity trees (2 to
// 12 vector registers, by degree and mode).
constexpr int rows_waves(int mode) {
  return mode == kFma64 ? (TBX_Q <= 9 ? 4 : 3) : (TBX_Q <= 9 ? 5 : 4);
}

// EvalTree at caller points (tree_functor.h:397-791) in the reference's
// arithmetic: wrap, locate, contract.  out[i][l] point-major.
__global__ __launch_bounds__(kBlock) void k_eval_exact(TreeView t, double *__restrict__ pts,
                                                       int64_t n, int bc, int write_back,
                                                       double *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double x = pts[3 * i + 0], y = pts[3 * i + 1], z = pts[3 * i + 2];
  if (bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
    if (write_back) {
      pts[3 * i + 0] = x;
      pts[3 * i + 1] = y;
      pts[3 * i + 2] = z;
    }
  }
  const int dof = t.dof;
  double *o = out + i * dof;
  eval_dof<D, kExact64>(t, x, y, z, [&](int l, double v) { o[l] = v; });
}

// A velocity functor (FieldExtrapFunctor / FieldSetFunctor / a scaled tree)
// at caller points at time t, as k_eval_exact; the extrapolating kind
// evaluates its extrapolation (the second-stage functor).
template <int KIND>
__global__ __launch_bounds__(kBlock) void k_veval_exact(VelSource vel, double *__restrict__ pts,
                                                        int64_t n, int bc, int write_back,
                                                        double t, int scaled, double g,
                                                        double *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double x = pts[3 * i + 0], y = pts[3 * i + 1], z = pts[3 * i + 2];
  if (bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
  }
  double v0, v1, v2;
  eval_velocity<D, kExact64, KIND>(vel, 2, t, scaled, g, bc, x, y, z, v0, v1, v2);
  if (bc == TBX_BC_PERIODIC && write_back) {  // wrapped once per tree
    pts[3 * i + 0] = x;
    pts[3 * i + 1] = y;
    pts[3 * i + 2] = z;
  }
  out[3 * i + 0] = v0;
  out[3 * i + 1] = v1;
  out[3 * i + 2] = v2;
}

// IntegrateRK2 substeps for caller points (x0 may be xs), as k_eval_exact.
template <int KIND>
__global__ __launch_bounds__(kBlock) void k_traj_exact(VelSource vel, const double *x0,
                                                       double *xs, int64_t n, SubArgs a) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double x = x0[3 * i + 0], y = x0[3 * i + 1], z = x0[3 * i + 2];
#pragma unroll 1
  for (int s = 0; s < a.nsub; ++s)
    rk2_substep<D, kExact64, KIND>(vel, a.bc, a.htau, a.tau, a.scaled, a.g[2 * s],
                                   a.g[2 * s + 1], a.ts[2 * s], a.ts[2 * s + 1], x, y, z);
  xs[3 * i + 0] = x;
  xs[3 * i + 1] = y;
  xs[3 * i + 2] = z;
}

// The same three in the other modes: a workgroup's points ordered by leaf
// and contracted row by row (tbx_rows.h).  Threads past the last point hold
// a copy of it and take no part.  BLOCK: with_rows_block.
//
// RUNS: the call's points were looked at (perm), and may come in runs of a
// leaf.  In place only up to three components (200,000 points of degree 4, 16
// components: 51 us in order, 69 in place), and not for points taken through
// perm, whose components are stored together (4 M of degree 4, three: 360 us,
// in place 406).  A kernel of its own: with the branch in it, scattered points
// that are not looked at took 3 % longer (846,243 on eight leaves of degree 12
// 41.6 us, 43.2).
template <int MODE, int BLOCK, bool RUNS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(rows_waves(MODE)))) void k_eval(
    TreeView t, double *__restrict__ pts, int64_t n, int bc, int write_back,
    double *__restrict__ out, PointPerm perm) {
  __shared__ RowsLds<BLOCK> sh;
  const int64_t i0 = (int64_t)blockIdx.x * BLOCK;
  const bool live = i0 + (int)threadIdx.x < n;
  int64_t i = live ? i0 + (int)threadIdx.x : n - 1;
  bool ordered = true;
  if constexpr (RUNS) {
    ordered = *perm.use;
    if (ordered) i = perm.perm[i];
  }
  double x = pts[3 * i + 0], y = pts[3 * i + 1], z = pts[3 * i + 2];
  if (bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
    if (write_back && live) {
      pts[3 * i + 0] = x;
      pts[3 * i + 1] = y;
      pts[3 * i + 2] = z;
    }
  }
  const int lf = locate(t, x, y, z);
  double *o = out + i * t.dof;
  bool rest = live;
  if constexpr (RUNS) {
    if (!ordered && t.dof <= 3 && rows_in_place(lf)) {
      in_place_dof<D, MODE>(t, lf, x, y, z, [&](int l, double v) {
        if (live) o[l] = v;
      });
      rest = false;
    }
  }
  const int count = order_by_leaf(sh, rest, lf);
  if (RUNS && count == 0) return;  // uniform over the workgroup
  rows_dof<D, MODE>(sh, t, count, lf, x, y, z, [&](int l, double v) {
    if (rest) o[l] = v;
  });
}

template <int MODE, int KIND, int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(rows_waves(MODE)))) void k_veval(
    VelSource vel, double *__restrict__ pts, int64_t n, int bc, int write_back, double t,
    int scaled, double g, double *__restrict__ out) {
  __shared__ RowsLds<BLOCK> sh;
  const int64_t i0 = (int64_t)blockIdx.x * BLOCK;
  const bool live = i0 + (int)threadIdx.x < n;
  const int64_t i = live ? i0 + (int)threadIdx.x : n - 1;
  double x = pts[3 * i + 0], y = pts[3 * i + 1], z = pts[3 * i + 2];
  if (bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
  }
  const int lf = locate(vel.t[0], x, y, z);
  const int count = order_by_leaf(sh, live, lf);
  double v[3];
  rows_velocity<D, MODE, KIND>(sh, vel, 2, t, scaled, g, bc, count, lf, x, y, z, v);
  if (!live) return;
  if (bc == TBX_BC_PERIODIC && write_back) {  // wrapped once per tree
    pts[3 * i + 0] = x;
    pts[3 * i + 1] = y;
    pts[3 * i + 2] = z;
  }
  out[3 * i + 0] = v[0];
  out[3 * i + 1] = v[1];
  out[3 * i + 2] = v[2];
}

template <int MODE, int KIND, int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(rows_waves(MODE)))) void k_traj(
    VelSource vel, const double *x0, double *xs, int64_t n, SubArgs a,
    PointPerm perm) {
  __shared__ RowsLds<BLOCK> sh;
  const int64_t i0 = (int64_t)blockIdx.x * BLOCK;
  const bool live = i0 + (int)threadIdx.x < n;
  int64_t i = live ? i0 + (int)threadIdx.x : n - 1;
  if (perm.perm && *perm.use) i = perm.perm[i];
  double x = x0[3 * i + 0], y = x0[3 * i + 1], z = x0[3 * i + 2];
#pragma unroll 1
  for (int s = 0; s < a.nsub; ++s)
    rows_substep<D, MODE, KIND>(sh, vel, a.bc, a.htau, a.tau, a.scaled, a.g[2 * s],
                                a.g[2 * s + 1], a.ts[2 * s], a.ts[2 * s + 1], live, x, y, z);
  if (!live) return;
  xs[3 * i + 0] = x;
  xs[3 * i + 1] = y;
  xs[3 * i + 2] = z;
}

// SolveSemilagInSitu fused (tree_semilag.h:92-135), TBX_EXACT's: arrival point of
// (leaf, node) -> num_rk_step RK2 substeps through vel -> conc at the
// departure point -> vals[leaf][l][node] for the refit.  Workgroups are
// remapped so that each XCD runs a contiguous range of arrival points and a
// leaf's coefficients are fetched into one XCD's L2.  BLOCK and WPE (the
// minimum waves per SIMD the register budget must allow) select the launch
// shape: wide workgroups keep the waves resident on a CU inside one or two
// leaves, so their scalar coefficient loads hit the same cache lines.
template <int KIND, int BLOCK, int WPE>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WPE))) void k_step(
    VelSource vel, TreeView conc, StepArgs a, double *__restrict__ vals,
    double *__restrict__ dep) {
  const uint32_t b = blockIdx.x;
  const int64_t lb = (int64_t)(b & 7u) * a.per_xcd + (int64_t)(b >> 3);
  if (lb >= a.nblocks) return;
  const int64_t i = lb * BLOCK + threadIdx.x;
  if (i >= a.npts) return;
  const int64_t leaf = i / a.P;
  const int m = (int)(i - leaf * a.P);
  // arrival point: corner + 2^-depth * node (tree_utils.h:480-491)
  const uint4 inf = conc.info[leaf];
  const double len = 1.0 / (double)(1u << inf.w);
  double x = (double)inf.x * len + len * a.node[m % D];
  double y = (double)inf.y * len + len * a.node[(m / D) % D];
  double z = (double)inf.z * len + len * a.node[m / (D * D)];
  // ComputeTrajRK2 (traj.inc:48-68), tinit -> tfinal = tinit - dt
  for (int s = 0; s < a.nsub; ++s)
    rk2_substep<D, kExact64, KIND>(vel, a.bc, a.htau, a.tau, a.scaled, a.g[2 * s],
                                   a.g[2 * s + 1], a.ts[2 * s], a.ts[2 * s + 1], x, y, z);
  // con_evaluator(departure points) wraps them in place (semilag.inc:43)
  if (a.bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
  }
  if (dep) {
    dep[3 * i + 0] = x;
    dep[3 * i + 1] = y;
    dep[3 * i + 2] = z;
  }
  const int dof = conc.dof;
  double *o = vals + leaf * dof * a.P + m;
  eval_dof<D, kExact64>(conc, x, y, z,
                        [&](int l, double v) { o[(int64_t)l * a.P] = v; });
}

// The start point of this thread's RK2 substep, read back from its row of
// the regroup buffer after a velocity evaluation instead of being held in
// registers through it (the row is this thread's until the next regroup,
// whose first barrier every thread reaches after its evaluation).  The
// empty asm with a memory clobber makes the compiler load it again rather
// than keep the value it loaded at the regroup.
template <int BLOCK, int NF>
__device__ __forceinline__ void reload_start(RegroupLds<BLOCK, NF> &sh, double (&st)[6]) {
  asm volatile("" ::: "memory");
  st[0] = sh.f[0][threadIdx.x];
  st[1] = sh.f[1][threadIdx.x];
  st[2] = sh.f[2][threadIdx.x];
}

// The same step with the workgroup's points regrouped by leaf before each
// of the 2 num_rk_step + 1 evaluations (regroup_pos in tbx_device.h).  The
// thread that holds a point after a regroup carries it on: the RK2 state
// (start point, wrapped midpoint) travels with the point through LDS, and
// the leaf found for the regroup is the one the evaluation uses.  Lanes
// past the last arrival point carry a copy of it and store nothing.
template <int KIND, int BLOCK, int WPE>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WPE))) void k_step_rg(
    VelSource vel, TreeView conc, StepArgs a, double *__restrict__ vals,
    double *__restrict__ dep) {
  __shared__ RegroupLds<BLOCK, 6> sh;
  const uint32_t b = blockIdx.x;
  const int64_t lb = (int64_t)(b & 7u) * a.per_xcd + (int64_t)(b >> 3);
  if (lb >= a.nblocks) return;  // uniform over the workgroup
  const int64_t i0 = lb * BLOCK;
  int orig = (int)threadIdx.x;
  {
    const int64_t i = i0 + orig < a.npts ? i0 + orig : a.npts - 1;
    const int64_t leaf = i / a.P;
    const int m = (int)(i - leaf * a.P);
    const uint4 inf = conc.info[leaf];
    const double len = 1.0 / (double)(1u << inf.w);
    double st[6];
    st[0] = (double)inf.x * len + len * a.node[m % D];
    st[1] = (double)inf.y * len + len * a.node[(m / D) % D];
    st[2] = (double)inf.z * len + len * a.node[m / (D * D)];
    int lf = 0;
    for (int s = 0; s < a.nsub; ++s) {
      // stage 1 at the (wrapped in place) start point (traj.inc:33)
      if (a.bc == TBX_BC_PERIODIC) {
        st[0] = wrap1(st[0]);
        st[1] = wrap1(st[1]);
        st[2] = wrap1(st[2]);
      }
      lf = locate(vel.t[0], st[0], st[1], st[2]);
      double v0, v1, v2;
      {
        double p3[3] = {st[0], st[1], st[2]};
        regroup(sh, orig, lf, p3);
        st[0] = p3[0];
        st[1] = p3[1];
        st[2] = p3[2];
      }
      eval_velocity<D, kExact64, KIND>(vel, 1, a.ts[2 * s], a.scaled, a.g[2 * s], a.bc, st[0],
                                       st[1], st[2], v0, v1, v2, lf);
      reload_start(sh, st);
      // midpoint xtmp = xinit + (0.5 * dt) * vtmp (traj.inc:36), wrapped
      // for its evaluation only
      st[3] = st[0] + a.htau * v0;
      st[4] = st[1] + a.htau * v1;
      st[5] = st[2] + a.htau * v2;
      if (a.bc == TBX_BC_PERIODIC) {
        st[3] = wrap1(st[3]);
        st[4] = wrap1(st[4]);
        st[5] = wrap1(st[5]);
      }
      lf = locate(vel.t[0], st[3], st[4], st[5]);
      regroup(sh, orig, lf, st);
      eval_velocity<D, kExact64, KIND>(vel, 2, a.ts[2 * s + 1], a.scaled, a.g[2 * s + 1], a.bc,
                                       st[3], st[4], st[5], v0, v1, v2, lf);
      reload_start(sh, st);
      // xsol = xinit + dt * vtmp (traj.inc:41-42)
      st[0] = st[0] + a.tau * v0;
      st[1] = st[1] + a.tau * v1;
      st[2] = st[2] + a.tau * v2;
    }
    // con_evaluator(departure points) wraps them in place (semilag.inc:43)
    if (a.bc == TBX_BC_PERIODIC) {
      st[0] = wrap1(st[0]);
      st[1] = wrap1(st[1]);
      st[2] = wrap1(st[2]);
    }
    lf = locate(conc, st[0], st[1], st[2]);
    double p3[3] = {st[0], st[1], st[2]};
    regroup(sh, orig, lf, p3);
    const int64_t gi = i0 + orig;
    const bool live = gi < a.npts;
    if (live && dep) {
      dep[3 * gi + 0] = p3[0];
      dep[3 * gi + 1] = p3[1];
      dep[3 * gi + 2] = p3[2];
    }
    const int64_t al = gi / a.P;
    const int am = (int)(gi - al * a.P);
    double *o = vals + al * conc.dof * a.P + am;
    eval_dof<D, kExact64>(
        conc, p3[0], p3[1], p3[2],
        [&](int l, double v) {
          if (live) o[(int64_t)l * a.P] = v;
        },
        lf);
  }
}

// The step in every mode but TBX_EXACT (tbx_rows.h).  A thread keeps its
// arrival point; before each velocity evaluation the workgroup's points are
// ordered by leaf and its wavefronts take 64 places at a time from that
// order.  The first substep's first stage takes the nodal values, and only
// points without one are ordered and contracted.  MF: many components (a
// multiple of 16) through eval_dof_mfma.
template <int MODE, int KIND, int BLOCK, bool MF>
__device__ __forceinline__ void k_step_rows_body(const VelSource &vel, const TreeView &conc,
                                                 const StepArgs &a, double *__restrict__ vals,
                                                 double *__restrict__ dep) {
  constexpr int P = D * D * D;
  __shared__ RowsLds<BLOCK> sh;
  const uint32_t b = blockIdx.x;
  const int64_t lb = (int64_t)(b & 7u) * a.per_xcd + (int64_t)(b >> 3);
  if (lb >= a.nblocks) return;  // uniform over the workgroup
  // leaf l0 + r / P, node r % P of the workgroup's arrival point t: the
  // 64-bit division is the workgroup's, lanes divide 32-bit by a constant
  const int64_t i0 = lb * BLOCK, l0 = i0 / P;
  const uint32_t r0 = (uint32_t)(i0 - l0 * P);
  const int np = a.npts - i0 < BLOCK ? (int)(a.npts - i0) : BLOCK;
  const bool live = (int)threadIdx.x < np;
  const uint32_t r = r0 + (live ? threadIdx.x : (uint32_t)np - 1u);
  const int64_t leaf = l0 + r / (uint32_t)P;
  const int m = (int)(r % (uint32_t)P);
  double x, y, z;
  {
    const uint4 inf = conc.info[leaf];
    const double len = leaf_edge(inf.w);
    x = (double)inf.x * len + len * a.node[m % D];
    y = (double)inf.y * len + len * a.node[(m / D) % D];
    z = (double)inf.z * len + len * a.node[m / (D * D)];
  }
  int count = 0;
#pragma unroll 1
  for (int s = 0; s < a.nsub; ++s) {
    // stage 1 at the (wrapped in place) start point (traj.inc:33)
    if (a.bc == TBX_BC_PERIODIC) {
      x = wrap1(x);
      y = wrap1(y);
      z = wrap1(z);
    }
    int lf = locate(vel.t[0], x, y, z);
    double v[3] = {0.0, 0.0, 0.0};
    bool need = live;
    if constexpr (KIND == kVelTree || KIND == kVelExtrap) {
      if (s == 0 && a.vnode)
        need = live && !nodal_velocity<D>((const NodalT<MODE> *)a.vnode, vel.t[0],
                                          conc.info[leaf], m, lf, P, a.scaled, a.g[0], v[0],
                                          v[1], v[2]);
    }
    if (__syncthreads_or(need)) {
      double u[3];
      count = order_by_leaf(sh, need, lf);
      rows_velocity<D, MODE, KIND>(sh, vel, 1, a.ts[2 * s], a.scaled, a.g[2 * s], a.bc, count,
                                   lf, x, y, z, u);
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = need ? u[c] : v[c];
    }
    count = rows_midpoint<D, MODE, KIND>(sh, vel, a.bc, a.htau, a.tau, a.scaled, a.g[2 * s + 1],
                                         a.ts[2 * s + 1], live, v, x, y, z);
  }
  // con_evaluator(departure points) wraps them in place (semilag.inc:43)
  if (a.bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
  }
  if (live && dep) {
    dep[3 * (i0 + threadIdx.x) + 0] = x;
    dep[3 * (i0 + threadIdx.x) + 1] = y;
    dep[3 * (i0 + threadIdx.x) + 2] = z;
  }
  const int lf = locate(conc, x, y, z);
  if constexpr (MF) {
    // a wavefront takes 64 places of the order by leaf at a time (a padding
    // place stores its point's values a second time)
    using T = typename ModeType<MODE>::T;
    sh.e[0][threadIdx.x] = x;
    sh.e[1][threadIdx.x] = y;
    sh.e[2][threadIdx.x] = z;
    sh.leaf[threadIdx.x] = lf;
    count = order_by_leaf(sh, live, lf);
    __syncthreads();
#pragma unroll 1
    for (int p0 = (int)(threadIdx.x & ~63u); p0 < count; p0 += BLOCK) {
      const int pos = p0 + (int)(threadIdx.x & 63u);
      const int src = sh.order[pos < count ? pos : count - 1] & kPlaceMask;
      const uint32_t q = r0 + (uint32_t)src;
      eval_dof_mfma<D, T>(conc, sh.leaf[src], sh.e[0][src], sh.e[1][src], sh.e[2][src], vals,
                          (l0 + q / (uint32_t)P) * conc.dof * P + (int64_t)(q % (uint32_t)P), P,
                          pos < count);
    }
  } else {
    // a departure point lies mostly in its midpoint's leaf: the midpoints'
    // order serves the concentration too
    double *o = vals + leaf * conc.dof * P + m;
    rows_dof<D, MODE>(sh, conc, count, lf, x, y, z, [&](int l, double v) {
      if (live) o[(int64_t)l * P] = v;
    });
  }
}

template <int MODE, int KIND, int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(rows_waves(MODE)))) void k_step_rows(
    VelSource vel, TreeView conc, StepArgs a, double *__restrict__ vals,
    double *__restrict__ dep) {
  k_step_rows_body<MODE, KIND, BLOCK, false>(vel, conc, a, vals, dep);
}

// The same step with the concentration's components contracted on the
// matrix cores (conc.dof a multiple of 16; FP64 or FP32 arithmetic).
template <int MODE, int KIND, int BLOCK, int WPE>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WPE))) void k_step_rows_mfma(
    VelSource vel, TreeView conc, StepArgs a, double *__restrict__ vals,
    double *__restrict__ dep) {
  k_step_rows_body<MODE, KIND, BLOCK, true>(vel, conc, a, vals, dep);
}

inline unsigned grid_for(int64_t n) {
  return (unsigned)((n + kBlock - 1) / kBlock);
}

// Calls f with the workgroup size of the point kernels for n points and the
// grid: 64 threads while 256 would leave some of the 256 compute units
// without a workgroup, 256 above (the larger group finds fewer runs of a
// leaf to pad).
template <typename F>
void with_rows_block(int64_t n, F f) {
  if (n <= 256 * 256)
    f(std::integral_constant<int, 64>{}, (unsigned)((n + 63) / 64));
  else
    f(std::integral_constant<int, 256>{}, (unsigned)((n + 255) / 256));
}

// Calls f with the arithmetic mode as a compile-time constant.
template <typename F>
hipError_t with_mode(int mode, F f) {
  switch (mode) {
    case kFma64:
      return f(std::integral_constant<int, kFma64>{});
    case kExact64:
      return f(std::integral_constant<int, kExact64>{});
    case kFp32:
      return f(std::integral_constant<int, kFp32>{});
    case kFp32h:
      return f(std::integral_constant<int, kFp32h>{});
    default:
      return hipErrorInvalidValue;
  }
}

// The leaf contraction alone, without the step around it: point i sits in
// leaf (w / waves_per_leaf) mod L, w = i / 64 its wavefront, at a position in
// the leaf's box from a hash of i; every component of the leaf is
// contracted there one after another (as in a velocity evaluation) and
// out[i] = ((0 + u_0) + u_1) + ... .  pts (optional) receives the points.
// It measures the rate of the contraction with scalar operands (TBX_EXACT's
// form, in each mode's arithmetic).
__device__ __forceinline__ double unit_hash(uint64_t v) {
  v += 0x9E3779B97F4A7C15ull;  // SplitMix64 finaliser
  v = (v ^ (v >> 30)) * 0xBF58476D1CE4E5B9ull;
  v = (v ^ (v >> 27)) * 0x94D049BB133111EBull;
  v ^= v >> 31;
  return (double)(v >> 11) * (1.0 / 9007199254740992.0);  // [0, 1)
}

template <int MODE>
__global__ __launch_bounds__(kBlock) void k_contract_only(TreeView t, int64_t n,
                                                          int waves_per_leaf,
                                                          double *__restrict__ out,
                                                          double *__restrict__ pts) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t w = __builtin_amdgcn_readfirstlane((int)((i >> 6) / waves_per_leaf % t.L));
  const int lf = (int)w;
  const uint4 inf = t.info[lf];
  const double len = 1.0 / (double)(1u << inf.w);
  const double x = (double)inf.x * len + len * unit_hash(3 * (uint64_t)i);
  const double y = (double)inf.y * len + len * unit_hash(3 * (uint64_t)i + 1);
  const double z = (double)inf.z * len + len * unit_hash(3 * (uint64_t)i + 2);
  PointBasis<D, MODE> b;
  b.build(t, x, y, z, lf);
  double acc = 0.0;
#pragma unroll 1
  for (int c = 0; c < t.dof; ++c) acc += leaf_value<D, MODE>(t, lf, c, b);
  if (i < n) {
    out[i] = acc;
    if (pts) {
      pts[3 * i + 0] = x;
      pts[3 * i + 1] = y;
      pts[3 * i + 2] = z;
    }
  }
}

// Calls f with the velocity kind as a compile-time constant.
template <typename F>
hipError_t with_kind(int kind, F f) {
  switch (kind) {
    case kVelTree:
      return f(std::integral_constant<int, kVelTree>{});
    case kVelExtrap:
      return f(std::integral_constant<int, kVelExtrap>{});
    case kVelSet:
      return f(std::integral_constant<int, kVelSet>{});
    default:
      return hipErrorInvalidValue;
  }
}

template <int KIND, int BLOCK, int WPE>
hipError_t launch_step_shape(const VelSource &vel, const TreeView &conc, const StepArgs &a,
                             double *vals, double *dep, hipStream_t s) {
  hipLaunchKernelGGL((k_step<KIND, BLOCK, WPE>), dim3((unsigned)(8 * a.per_xcd)),
                     dim3(BLOCK), 0, s, vel, conc, a, vals, dep);
  return hipGetLastError();
}

template <int KIND, int BLOCK, int WPE>
hipError_t launch_step_rg_shape(const VelSource &vel, const TreeView &conc, const StepArgs &a,
                                double *vals, double *dep, hipStream_t s) {
  hipLaunchKernelGGL((k_step_rg<KIND, BLOCK, WPE>), dim3((unsigned)(8 * a.per_xcd)),
                     dim3(BLOCK), 0, s, vel, conc, a, vals, dep);
  return hipGetLastError();
}

template <int MODE>
hipError_t launch_step_mode(const VelSource &vel, const TreeView &conc, const StepArgs &a,
                            double *vals, double *dep, hipStream_t s) {
  // many components on the matrix cores: workgroups of mfma_step_block
  // threads (the tile operands and accumulators need the registers)
  if (a.mfma) {
    if constexpr (MODE == kFma64 || MODE == kFp32) {
      if (vel.kind != kVelTree || a.shape != kMfmaStepShape) return hipErrorInvalidValue;
      constexpr int B = mfma_step_block(MODE), W = mfma_step_waves(MODE);
      hipLaunchKernelGGL((k_step_rows_mfma<MODE, kVelTree, B, W>), dim3((unsigned)(8 * a.per_xcd)),
                         dim3(B), 0, s, vel, conc, a, vals, dep);
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
  if constexpr (MODE != kExact64) {
    constexpr int kB = rows_step_block(MODE);
    return with_kind(vel.kind, [&](auto k) {
      hipLaunchKernelGGL((k_step_rows<MODE, decltype(k)::value, kB>),
                         dim3((unsigned)(8 * a.per_xcd)), dim3(kB), 0, s, vel, conc, a,
                         vals, dep);
      return hipGetLastError();
    });
  } else {
  // the composite velocity kinds run the default shape only (the host
  // sizes the grid for the shape it asks for: kDefaultStepShape then)
  if (vel.kind == kVelExtrap)
    return launch_step_rg_shape<kVelExtrap, 1024, 4>(vel, conc, a, vals, dep, s);
  if (vel.kind == kVelSet)
    return launch_step_rg_shape<kVelSet, 1024, 4>(vel, conc, a, vals, dep, s);
  // launch shapes of kStepShapes (tbx_internal.h); the extra shapes are
  // built for the degrees of the benchmark workloads only
  constexpr int T = kVelTree;
  switch (a.shape) {
    case 0:
      return launch_step_shape<T, 256, 1>(vel, conc, a, vals, dep, s);
#if TBX_Q == 8 || TBX_Q == 14
    case 4:
      return launch_step_rg_shape<T, 256, 2>(vel, conc, a, vals, dep, s);
    case 1:
      return launch_step_shape<T, 256, 4>(vel, conc, a, vals, dep, s);
    case 2:
      return launch_step_shape<T, 1024, 4>(vel, conc, a, vals, dep, s);
    case 3:
      return launch_step_shape<T, 512, 4>(vel, conc, a, vals, dep, s);
    case 5:
      return launch_step_rg_shape<T, 512, 2>(vel, conc, a, vals, dep, s);
    case 7:
      return launch_step_rg_shape<T, 512, 4>(vel, conc, a, vals, dep, s);
    case 8:
      return launch_step_rg_shape<T, 1024, 8>(vel, conc, a, vals, dep, s);
    case 9:
      return launch_step_rg_shape<T, 512, 6>(vel, conc, a, vals, dep, s);
    case 10:
      return launch_step_rg_shape<T, 768, 6>(vel, conc, a, vals, dep, s);
#endif
    default:  // shape 6, and the shapes not built for this degree
      return launch_step_rg_shape<T, 1024, 4>(vel, conc, a, vals, dep, s);
  }
  }
}

}  // namespace

#define TBX_CAT2(a, b) a##b
#define TBX_CAT(a, b) TBX_CAT2(a, b)

hipError_t TBX_CAT(launch_eval_q, TBX_Q)(int mode, const TreeView &t,
                                         double *pts, int64_t n, int bc,
                                         int write_back, double *out,
                                         PointPerm perm, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  return with_mode(mode, [&](auto m) {
    constexpr int M = decltype(m)::value;
    if constexpr (M == kExact64) {
      hipLaunchKernelGGL(k_eval_exact, dim3(grid_for(n)), dim3(kBlock), 0, s, t, pts, n, bc,
                         write_back, out);
    } else {
      with_rows_block(n, [&](auto b, unsigned grid) {
        constexpr int B = decltype(b)::value;
        if (perm.perm)
          hipLaunchKernelGGL((k_eval<M, B, true>), dim3(grid), dim3(B), 0, s, t, pts, n, bc,
                             write_back, out, perm);
        else
          hipLaunchKernelGGL((k_eval<M, B, false>), dim3(grid), dim3(B), 0, s, t, pts, n, bc,
                             write_back, out, perm);
      });
    }
    return hipGetLastError();
  });
}

hipError_t TBX_CAT(launch_contract_q, TBX_Q)(int mode, const TreeView &t, int64_t n,
                                             int waves_per_leaf, double *out, double *pts,
                                             hipStream_t s) {
  if (n <= 0) return hipSuccess;
  return with_mode(mode, [&](auto m) {
    hipLaunchKernelGGL(k_contract_only<decltype(m)::value>, dim3(grid_for(n)), dim3(kBlock), 0, s,
                       t, n, waves_per_leaf, out, pts);
    return hipGetLastError();
  });
}

hipError_t TBX_CAT(launch_veval_q, TBX_Q)(int mode, const VelSource &vel,
                                          double *pts, int64_t n, int bc,
                                          int write_back, double t, int scaled,
                                          double g, double *out,
                                          hipStream_t s) {
  if (n <= 0) return hipSuccess;
  return with_mode(mode, [&](auto m) {
    return with_kind(vel.kind, [&](auto k) {
      constexpr int M = decltype(m)::value, K = decltype(k)::value;
      if constexpr (M == kExact64) {
        hipLaunchKernelGGL(k_veval_exact<K>, dim3(grid_for(n)), dim3(kBlock), 0, s, vel, pts, n,
                           bc, write_back, t, scaled, g, out);
      } else {
        with_rows_block(n, [&](auto b, unsigned grid) {
          hipLaunchKernelGGL((k_veval<M, K, decltype(b)::value>), dim3(grid),
                             dim3(decltype(b)::value), 0, s, vel, pts, n, bc, write_back, t,
                             scaled, g, out);
        });
      }
      return hipGetLastError();
    });
  });
}

hipError_t TBX_CAT(launch_traj_q, TBX_Q)(int mode, const VelSource &vel,
                                         const double *x0, double *x,
                                         int64_t n, const SubArgs &a,
                                         PointPerm perm, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  return with_mode(mode, [&](auto m) {
    return with_kind(vel.kind, [&](auto k) {
      constexpr int M = decltype(m)::value, K = decltype(k)::value;
      if constexpr (M == kExact64) {
        hipLaunchKernelGGL(k_traj_exact<K>, dim3(grid_for(n)), dim3(kBlock), 0, s, vel, x0, x, n,
                           a);
      } else {
        with_rows_block(n, [&](auto b, unsigned grid) {
          hipLaunchKernelGGL((k_traj<M, K, decltype(b)::value>), dim3(grid),
                             dim3(decltype(b)::value), 0, s, vel, x0, x, n, a, perm);
        });
      }
      return hipGetLastError();
    });
  });
}

hipError_t TBX_CAT(launch_step_q, TBX_Q)(int mode, const VelSource &vel,
                                         const TreeView &conc,
                                         const StepArgs &a, double *vals,
                                         double *dep, hipStream_t s) {
  if (a.npts <= 0) return hipSuccess;
  return with_mode(mode, [&](auto m) {
    return launch_step_mode<decltype(m)::value>(vel, conc, a, vals, dep, s);
  });
}

}  // namespace tbx
