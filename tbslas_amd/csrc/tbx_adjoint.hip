// Adjoint of one SolveSemilagInSitu step for one Chebyshev degree
// (compiled once per degree with -DTBX_Q=<q>, like tbx_kernels.hip).
//
// The forward step is c' = R E_D(V) c: E_D interpolates c at the departure
// points D(V) of the grid points (RK2 through the velocity tree V), R is the
// per-leaf refit.  For a cotangent lam' of c':
//   dc = E_D^T R^T lam'          transposed interpolation: every departure
//                                point adds u_p B_m(D_p) into the
//                                coefficients of its leaf (u = R^T lam')
//   dV = sum_p a_p . dD_p/dV     a_p = sum_c u_{p,c} grad c_c(D_p), chained
//                                through the midpoint RK2 substep
// R^T lam' is a GEMM on the host side.  The reference has no adjoint; these
// kernels differentiate exactly what the forward kernels compute (the same
// trajectory arithmetic, the same leaf assignment), for one RK2 substep and
// a single velocity tree.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "tbx_rows.h"

#ifndef TBX_Q
#error "compile with -DTBX_Q=<degree>"
#endif

namespace tbx {
namespace {

constexpr int D = TBX_Q + 1;
constexpr int NC = D * (D + 1) * (D + 2) / 6;

// T_0..T_{D-1} and dT/dxi by differentiating the three-term recurrence,
// dT_{k+1} = 2 T_k + 2 xi dT_k - dT_{k-1}, at x inside [-1, 1].
__device__ __forceinline__ void cheb_poly_d(double x, double (&p)[D], double (&dp)[D]) {
  const double x2 = 2.0 * x;
  p[0] = 1.0;
  dp[0] = 0.0;
  if constexpr (D > 1) {
    p[1] = x;
    dp[1] = 1.0;
  }
#pragma unroll
  for (int k = 2; k < D; ++k) {
    p[k] = __builtin_fma(x2, p[k - 1], -p[k - 2]);
    dp[k] = __builtin_fma(2.0, p[k - 1], __builtin_fma(x2, dp[k - 1], -dp[k - 2]));
  }
}

// Gradient (d/dxi_x, d/dxi_y, d/dxi_z) of one component at the lane's
// point, the lane's DPP row sharing the leaf (row_contract in tbx_rows.h):
// one pass over the packed triangle, every coefficient feeding the value
// and the x-derivative sums along k; the (i, j) sums are then combined with
// the y and z bases and derivatives.
__device__ __forceinline__ void row_grad(const double *__restrict__ c, const double (&px)[D],
                                         const double (&dx)[D], const double (&py)[D],
                                         const double (&dy)[D], double z, double &gx,
                                         double &gy, double &gz) {
  constexpr int NB = (NC + 15) / 16, kRing = 4;
  double r[kRing];
  static_for<(kRing - 1 < NB ? kRing - 1 : NB)>([&](auto bc) {
    constexpr int b = decltype(bc)::value;
    r[b] = c[16 * b];
  });
  gx = gy = gz = 0.0;
  const double z2 = 2.0 * z;
  double zm = 0.0, zc = 1.0, dm = 0.0, dc = 0.0;  // T_{i-1}, T_i and derivatives
  static_for<D>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    double vx = 0.0, vy = 0.0, v = 0.0;
    static_for<D - i>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      constexpr int first = tri_start(D, i, j), len = D - i - j;
      double w = 0.0, wx = 0.0;
      static_for<2>([&](auto hc) {  // the row's coefficients, cut at multiples of 16
        constexpr int h = decltype(hc)::value;
        constexpr int b = first / 16 + h;
        constexpr int lo = h == 0 ? first : 16 * b;
        constexpr int hi = first + len < 16 * (b + 1) ? first + len : 16 * (b + 1);
        if constexpr (lo < hi) {
          if constexpr (lo % 16 == 0 && b + kRing - 1 < NB) {
            asm volatile("" ::: "memory");  // loads stay kRing - 1 blocks ahead
            r[(b + kRing - 1) % kRing] = c[16 * (b + kRing - 1)];
            __builtin_amdgcn_sched_barrier(0);
          }
          const double cb = r[b % kRing];
          if constexpr (lo == first) {
            row_start<lo % 16, hi - lo>(w, cb, px + 1);
            if constexpr (hi - lo > 1) row_add<lo % 16 + 1, hi - lo - 1>(wx, cb, dx + 1);
          } else {
            row_add<0, hi - lo>(w, cb, px + (lo - first));
            row_add<0, hi - lo>(wx, cb, dx + (lo - first));
          }
        }
      });
      if constexpr (j == 0) {
        v = w;
        vx = wx;
      } else {
        fmac_here(v, py[j], w);
        fmac_here(vx, py[j], wx);
        fmac_here(vy, dy[j], w);
      }
    });
    if constexpr (i == 0) {
      gx = vx;
      gy = vy;
    } else {
      if constexpr (i == 1) {
        zm = 1.0;
        zc = z;
        dc = 1.0;
      } else {
        const double zn = __builtin_fma(z2, zc, -zm);
        const double dn = __builtin_fma(2.0, zc, __builtin_fma(z2, dc, -dm));
        zm = zc;
        zc = zn;
        dm = dc;
        dc = dn;
      }
      fmac_here(gx, zc, vx);
      fmac_here(gy, zc, vy);
      fmac_here(gz, dc, v);
    }
  });
}

// Rows (i, j) of the transposed interpolation's tiles, sorted by n = i + j.
struct ScatterRows {
  static constexpr int R = D * (D + 1) / 2;
  static constexpr int NT = (R + 15) / 16;
  int8_t i[16 * NT], j[16 * NT];  // i = -1: padding
  int len[NT];                    // values of k of the tile's longest row
  constexpr ScatterRows() : i(), j(), len() {
    int r = 0;
    for (int n = 0; n < D; ++n)
      for (int a = 0; a <= n; ++a) {
        i[r] = (int8_t)a;
        j[r] = (int8_t)(n - a);
        ++r;
      }
    for (; r < 16 * NT; ++r) {
      i[r] = -1;
      j[r] = 0;
    }
    for (int t = 0; t < NT; ++t) len[t] = D - i[16 * t] - j[16 * t];
  }
};
constexpr ScatterRows kRows{};
__device__ const ScatterRows kDevRows{};

// Tiles of 16 (k, component) columns an M tile needs, and the first tile's
// index among all.
constexpr int scatter_cols(int t, int ncomp) { return (kRows.len[t] * ncomp + 15) / 16; }
constexpr int scatter_first(int t, int ncomp) {
  int n = 0;
  for (int a = 0; a < t; ++a) n += scatter_cols(a, ncomp);
  return n;
}

// A workgroup's adjoint points: RowsLds holds their leaf coordinates, w the
// weights per component, g the gradients; scratch per wavefront.
template <int BLOCK>
struct AdjLds {
  RowsLds<BLOCK> r;
  double w[3][BLOCK];
  double g[3][BLOCK];
  double t[BLOCK / 64][3][D][16];  // T_k of a group's 16 points per axis
  double sw[BLOCK / 64][3][16];    // their weights
  int rows[16 * ScatterRows::NT];  // per tile row: start | values of k << 10 | i << 15 | j << 20
};

// The tile rows' table, read through LDS (from global memory its loads'
// latency stood before every sum that left the registers: 4,096 leaves of
// degree 8, the concentration kernel 820 us, now 511; the velocity kernel
// 1,185, now 1,097).  The caller synchronises before its use.
template <int BLOCK>
__device__ __forceinline__ void scatter_table(AdjLds<BLOCK> &s) {
  for (int r = (int)threadIdx.x; r < 16 * ScatterRows::NT; r += BLOCK) {
    const int i = kDevRows.i[r], j = kDevRows.j[r];
    s.rows[r] = i < 0 ? 0 : tri_start(D, i, j) | ((D - i - j) << 10) | (i << 15) | (j << 20);
  }
}

// s.g = sum over c < nc of w[c] grad_xi(component c of t) at the points in
// order[0, count) (zero outside the leaf's box, as the basis).  The caller
// synchronises before and after.
template <int BLOCK>
__device__ __forceinline__ void rows_gradient(AdjLds<BLOCK> &s, const TreeView &t, int c0, int nc,
                                              int count) {
  const int lane = (int)(threadIdx.x & 63u);
#pragma unroll 1
  for (int p0 = (int)(threadIdx.x & ~63u); p0 < count; p0 += BLOCK) {
    const int src = s.r.order[p0 + lane < count ? p0 + lane : count - 1] & kPlaceMask;
    const int leaf = s.r.leaf[src];
    const double ex = s.r.e[0][src], ey = s.r.e[1][src], ez = s.r.e[2][src];
    const bool in = fabs(ex) <= 1.0 && fabs(ey) <= 1.0 && fabs(ez) <= 1.0;
    double px[D], dx[D], py[D], dy[D];
    cheb_poly_d(in ? ex : 0.0, px, dx);
    cheb_poly_d(in ? ey : 0.0, py, dy);
    const double z = in ? ez : 0.0;
    double jx = 0.0, jy = 0.0, jz = 0.0;
    uint64_t pending = __builtin_amdgcn_ballot_w64(true);
#pragma unroll 1
    while (pending) {
      const int lf = row_leaf(pending, leaf);
      const bool mine = leaf == lf;
      pending &= ~__builtin_amdgcn_ballot_w64(mine);
      const double *cb = t.coeff + ((size_t)lf * t.dof + c0) * NC + (lane & 15);
      // summed from zero in each pass: a row that is done goes through its
      // first lane's leaf again while another row has leaves left
      double kx = 0.0, ky = 0.0, kz = 0.0;
#pragma unroll 1
      for (int c = 0; c < nc; ++c) {
        double gx, gy, gz;
        row_grad(cb, px, dx, py, dy, z, gx, gy, gz);
        const double a = s.w[c][src];
        kx = __builtin_fma(a, gx, kx);
        ky = __builtin_fma(a, gy, ky);
        kz = __builtin_fma(a, gz, kz);
        cb += NC;
      }
      jx = mine ? kx : jx;
      jy = mine ? ky : jy;
      jz = mine ? kz : jz;
    }
    s.g[0][src] = in_box(in, jx);
    s.g[1][src] = in_box(in, jy);
    s.g[2][src] = in_box(in, jz);
  }
}

// Transposed interpolation: G[leaf][c0 + c][ijk] += sum over the points in
// order[0, count) of scale w[c] T_i(z) T_j(y) T_k(x), c < NCOMP.  Per leaf it
// is a product [rows (i, j)] x [points] . [points] x [columns (k, c)]:
// 16 x 16 x 4 FP64 MFMAs over groups of 16 places, the sums of a leaf kept in
// registers until the wavefront's next group is another leaf's, then added
// to memory.  Columns are ordered k first, so that shorter rows need fewer
// column tiles: at degree 8 and three components 16 MFMAs per 16 points.
// (Reducing every product over the wavefront took 5 to 8 vector
// instructions per coefficient and component: 2.2 of the velocity
// kernel's 3.1 ms on 3.0 M points.)  The caller synchronises before and
// after.
template <int NCOMP, int BLOCK>
__device__ __forceinline__ void rows_scatter(AdjLds<BLOCK> &s, double *__restrict__ G, int dof,
                                             int c0, double scale, int count) {
  typedef MfmaAcc<double>::V V;
  constexpr int NT = ScatterRows::NT, NCT = scatter_cols(0, NCOMP);
  constexpr int NACC = scatter_first(NT, NCOMP);
  const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
  const int g = lane >> 4, p = lane & 15;
  double(*T)[D][16] = s.t[wave];
  double(*sw)[16] = s.sw[wave];
  V acc[NACC];
  auto clear = [&]() {
#pragma unroll
    for (int a = 0; a < NACC; ++a) acc[a] = V{0, 0, 0, 0};
  };
  auto flush = [&](int leaf) {
    static_for<NT>([&](auto tc) {
      constexpr int t = decltype(tc)::value;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = s.rows[16 * t + g + 4 * r];
#pragma unroll
        for (int n = 0; n < scatter_cols(t, NCOMP); ++n) {
          const int q = 16 * n + p, k = q / NCOMP, c = q % NCOMP;
          if (k < ((row >> 10) & 31))
            atomicAdd(G + ((size_t)leaf * dof + c0 + c) * NC + (row & 1023) + k,
                      acc[scatter_first(t, NCOMP) + n][r]);
        }
      }
    });
  };
  // the lane's row per M tile (the A operand's address)
  int zi[NT], yj[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    zi[t] = (s.rows[16 * t + p] >> 15) & 31;
    yj[t] = s.rows[16 * t + p] >> 20;
  }
  const int ng = count / 16, per = (ng + BLOCK / 64 - 1) / (BLOCK / 64);
  const int g1 = (wave + 1) * per < ng ? (wave + 1) * per : ng;
  int cur = -1;
  clear();
#pragma unroll 1
  for (int grp = wave * per; grp < g1; ++grp) {
    const int o = s.r.order[16 * grp + p], src = o & kPlaceMask;
    const int leaf = s.r.leaf[src];
    {
      double v[D];
      row_cheb<D>(s.r.e[g < 3 ? g : 2][src], v);
      if (g < 3) {
#pragma unroll
        for (int k = 0; k < D; ++k) T[g][k][p] = v[k];
      }
    }
    // copies that pad a leaf's places carry no weight
    const double w = o == src && g < NCOMP ? scale * s.w[g < NCOMP ? g : 0][src] : 0.0;
    uint64_t pending = __builtin_amdgcn_ballot_w64(true);
#pragma unroll 1
    while (pending) {  // one pass; per leaf in the overflow run
      const int lf = __builtin_amdgcn_readlane(leaf, __builtin_ctzll(pending));
      const bool mine = leaf == lf;
      pending &= ~__builtin_amdgcn_ballot_w64(mine);
      if (lf != cur) {
        if (cur >= 0) {
          flush(cur);
          clear();
        }
        cur = lf;
      }
      if (g < NCOMP) sw[g][p] = mine ? w : 0.0;
      wave_lds_order();
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int pt = 4 * st + g;  // the lane's point of this K step
        double b[NCT];
#pragma unroll
        for (int n = 0; n < NCT; ++n) {
          const int q = 16 * n + p, k = q / NCOMP;
          b[n] = sw[q % NCOMP][pt] * T[0][k < D ? k : 0][pt];
        }
        static_for<NT>([&](auto tc) {
          constexpr int t = decltype(tc)::value;
          const double a = T[2][zi[t]][pt] * T[1][yj[t]][pt];
#pragma unroll
          for (int n = 0; n < scatter_cols(t, NCOMP); ++n)
            acc[scatter_first(t, NCOMP) + n] =
                MfmaAcc<double>::mma(a, b[n], acc[scatter_first(t, NCOMP) + n]);
        });
      }
      wave_lds_order();  // the scratch is written again
    }
  }
  if (cur >= 0) flush(cur);
}

// Arrival point of global grid index gi (tree_utils.h:480-491).
__device__ __forceinline__ void arrival_point(const TreeView &conc, const StepArgs &a,
                                              int64_t gi, double &x, double &y, double &z) {
  const int64_t leaf = gi / a.P;
  const int m = (int)(gi - leaf * a.P);
  const uint4 inf = conc.info[leaf];
  const double len = 1.0 / (double)(1u << inf.w);
  x = (double)inf.x * len + len * a.node[m % D];
  y = (double)inf.y * len + len * a.node[(m / D) % D];
  z = (double)inf.z * len + len * a.node[m / (D * D)];
}

// The first-stage velocity at arrival point i (its wrapped position x, y,
// z) as the forward step takes it from the velocity's nodal values
// (a.vnode, FP64; nodal_velocity); false where the forward evaluates it.
__device__ __forceinline__ bool adj_nodal_stage1(const VelSource &vel, const TreeView &conc,
                                                 const StepArgs &a, int64_t i, double x,
                                                 double y, double z, double &v0, double &v1,
                                                 double &v2) {
  if (!a.vnode) return false;
  const int64_t jl = i / a.P;
  const int lf = locate(vel.t[0], x, y, z);
  return nodal_velocity<D>((const double *)a.vnode, vel.t[0], conc.info[jl],
                           (int)(i - jl * a.P), lf, a.P, a.scaled, a.g[0], v0, v1, v2);
}

__device__ __forceinline__ void wrap3(const StepArgs &a, double &x, double &y, double &z) {
  if (a.bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
  }
}

// Velocity of stage `stage` of substep s at the needing threads' points.
template <int MODE, int BLOCK>
__device__ __forceinline__ void adj_velocity(RowsLds<BLOCK> &sh, const VelSource &vel,
                                             const StepArgs &a, int stage, int s, bool need,
                                             double &x, double &y, double &z, double (&v)[3]) {
  const int k = 2 * s + stage - 1;
  if constexpr (MODE == kExact64) {
    eval_velocity<D, MODE, kVelTree>(vel, stage, a.ts[k], a.scaled, a.g[k], a.bc, x, y, z, v[0],
                                     v[1], v[2]);
  } else {
    const int lf = locate(vel.t[0], x, y, z);
    const int count = order_by_leaf(sh, need, lf);
    rows_velocity<D, MODE, kVelTree>(sh, vel, stage, a.ts[k], a.scaled, a.g[k], a.bc, count, lf,
                                     x, y, z, v);
  }
}

// The first stage of substep s at (x, y, z) as the forward step takes it:
// the nodal value of arrival point i where it has one (a.vnode).
template <int MODE, int BLOCK>
__device__ __forceinline__ void adj_stage1(RowsLds<BLOCK> &sh, const VelSource &vel,
                                           const TreeView &conc, const StepArgs &a, int64_t i,
                                           bool live, int s, double &x, double &y, double &z,
                                           double (&v)[3]) {
  bool need = live;
  v[0] = v[1] = v[2] = 0.0;
  if (s == 0 && a.vnode)
    need = live && !adj_nodal_stage1(vel, conc, a, i, x, y, z, v[0], v[1], v[2]);
  if (__syncthreads_or(need)) {
    double u[3];
    adj_velocity<MODE>(sh, vel, a, 1, s, need, x, y, z, u);
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = need ? u[c] : v[c];
  }
}

// Substep s of the forward step for a workgroup's points, in place.
template <int MODE, int BLOCK>
__device__ __forceinline__ void adj_substep(RowsLds<BLOCK> &sh, const VelSource &vel,
                                            const TreeView &conc, const StepArgs &a, int64_t i,
                                            bool live, int s, double &x, double &y, double &z) {
  wrap3(a, x, y, z);
  double v[3];
  adj_stage1<MODE>(sh, vel, conc, a, i, live, s, x, y, z, v);
  double hx = x + a.htau * v[0], hy = y + a.htau * v[1], hz = z + a.htau * v[2];
  wrap3(a, hx, hy, hz);
  adj_velocity<MODE>(sh, vel, a, 2, s, live, hx, hy, hz, v);
  x = x + a.tau * v[0];
  y = y + a.tau * v[1];
  z = z + a.tau * v[2];
}

// Cotangent of c and, when A is given, the per-point velocity cotangent
// factor a_p += sum_c u_{p,c} grad c_c(D_p).  ua[al][c][am] = (R^T lam')
// at arrival point (al, am).  MODE is the forward's trajectory arithmetic;
// with STORED the departure points are read from dep[3 gi] (the forward
// step's own output, wrapped as the concentration saw them) instead of
// being integrated again.
template <int MODE, int BLOCK, bool STORED>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void k_adj_conc(
    VelSource vel, TreeView conc, StepArgs a, const double *__restrict__ dep,
    const double *__restrict__ ua, double *__restrict__ lam, double *__restrict__ A) {
  __shared__ AdjLds<BLOCK> sh;
  const uint32_t b = blockIdx.x;
  const int64_t lb = (int64_t)(b & 7u) * a.per_xcd + (int64_t)(b >> 3);
  if (lb >= a.nblocks) return;  // uniform over the workgroup
  scatter_table(sh);
  const int tid = (int)threadIdx.x;
  const int64_t i0 = lb * BLOCK;
  const bool live = i0 + tid < a.npts;
  const int64_t i = live ? i0 + tid : a.npts - 1;
  double x, y, z;
  if constexpr (STORED) {
    x = dep[3 * i + 0];
    y = dep[3 * i + 1];
    z = dep[3 * i + 2];
  } else {
    arrival_point(conc, a, i, x, y, z);
#pragma unroll 1
    for (int s = 0; s < a.nsub; ++s)
      adj_substep<MODE>(sh.r, vel, conc, a, i, live, s, x, y, z);
    wrap3(a, x, y, z);
  }
  const int lf = locate(conc, x, y, z);
  const int count = order_by_leaf(sh.r, live, lf);
  put_point(sh.r, conc, lf, x, y, z);
  const int64_t al = i / a.P;
  const int am = (int)(i - al * a.P);
  const int dof = conc.dof;
  double ax = 0.0, ay = 0.0, az = 0.0;
#pragma unroll 1
  for (int c = 0; c < dof; ++c) {
    sh.w[0][tid] = ua[(al * dof + c) * a.P + am];
    __syncthreads();
    if (A) rows_gradient(sh, conc, c, 1, count);
    rows_scatter<1>(sh, lam, dof, c, 1.0, count);
    __syncthreads();
    if (A) {
      ax += sh.g[0][tid];
      ay += sh.g[1][tid];
      az += sh.g[2][tid];
    }
  }
  if (A && live) {
    const double s2 = 2.0 * (double)(1u << conc.info[lf].w);  // d xi / dx
    A[3 * i + 0] += s2 * ax;
    A[3 * i + 1] += s2 * ay;
    A[3 * i + 2] += s2 * az;
  }
}

// Velocity cotangent through the num_rk_step substeps.  Substep s maps x_s
// to x_{s+1} = x_s + tau g2_s V(h_s), h_s = x_s + (tau/2) g1_s V(x_s)
// (traj.inc:20-46; the periodic wraps are translations), so with a_{s+1}
// the cotangent of x_{s+1} (a_S = A, the departure point's):
//   a . dx_{s+1} gives   tau g2_s a_{s+1} . dV(h_s)
//                      + w_s . dV(x_s),  w_s = tau g2_s (tau/2) g1_s J_V(h_s)^T a_{s+1}
//   a_s = a_{s+1} + tau g2_s J_V(h_s)^T a_{s+1} + J_V(x_s)^T w_s,
// each dV scattered into G[leaf][k][m] at its point (in its leaf).  The
// substeps run backwards; x_s is integrated again from the arrival point
// (s substeps) for each one.  A thread keeps its arrival point; the work at
// h_s and at x_s goes through the workgroup's order by leaf.
template <int MODE>
__global__ __launch_bounds__(kAdjBlock) __attribute__((amdgpu_waves_per_eu(2))) void k_adj_vel(
    VelSource vel, TreeView conc, StepArgs a, const double *__restrict__ A,
    double *__restrict__ G) {
  __shared__ AdjLds<kAdjBlock> sh;
  const uint32_t b = blockIdx.x;
  const int64_t lb = (int64_t)(b & 7u) * a.per_xcd + (int64_t)(b >> 3);
  if (lb >= a.nblocks) return;  // uniform over the workgroup
  scatter_table(sh);
  const TreeView &V = vel.t[0];
  const int tid = (int)threadIdx.x;
  const int64_t i0 = lb * kAdjBlock;
  const bool live = i0 + tid < a.npts;
  const int64_t i = live ? i0 + tid : a.npts - 1;
  double ax = A[3 * i + 0], ay = A[3 * i + 1], az = A[3 * i + 2];
#pragma unroll 1
  for (int s = a.nsub - 1; s >= 0; --s) {
    double x, y, z;
    arrival_point(conc, a, i, x, y, z);
#pragma unroll 1
    for (int r = 0; r < s; ++r) adj_substep<MODE>(sh.r, vel, conc, a, i, live, r, x, y, z);
    wrap3(a, x, y, z);
    // the forward's midpoint of substep s (rk2_substep, stage 1)
    double v[3];
    adj_stage1<MODE>(sh.r, vel, conc, a, i, live, s, x, y, z, v);
    double hx = x + a.htau * v[0], hy = y + a.htau * v[1], hz = z + a.htau * v[2];
    wrap3(a, hx, hy, hz);
    const double g1 = a.scaled ? a.g[2 * s] : 1.0, g2 = a.scaled ? a.g[2 * s + 1] : 1.0;
    const double fh = a.tau * g2, fx = a.tau * g2 * a.htau * g1;
    // work at h: J^T a, (J^T a)_k = sum_c a_c dV_c/dy_k, and fh a scattered
    const int lh = locate(V, hx, hy, hz);
    int count = order_by_leaf(sh.r, live, lh);
    put_point(sh.r, V, lh, hx, hy, hz);
    sh.w[0][tid] = ax;
    sh.w[1][tid] = ay;
    sh.w[2][tid] = az;
    __syncthreads();
    rows_gradient(sh, V, 0, 3, count);
    rows_scatter<3>(sh, G, 3, 0, fh, count);
    __syncthreads();
    const double sh2 = 2.0 * (double)(1u << V.info[lh].w);  // d xi / dx
    const double jx = sh2 * sh.g[0][tid], jy = sh2 * sh.g[1][tid], jz = sh2 * sh.g[2][tid];
    const double wx = fx * jx, wy = fx * jy, wz = fx * jz;
    // work at x
    const int lx = locate(V, x, y, z);
    bool rest = live;
    if (s == 0 && a.wnode) {
      // x is the point's arrival node: where that is a grid node of its
      // velocity leaf, its weights go to the node's slot (the slots are then
      // projected, G += B^T slots, in one pass per leaf); only the others
      // scatter, and only workgroups holding one
      const int64_t jl = i / a.P;
      const int mm = live ? node_of(conc.info[jl], V.info[lx], (int)(i - jl * a.P), D) : -1;
      if (mm >= 0) {
        double *wn = a.wnode + (int64_t)lx * 3 * a.P + mm;
        atomicAdd(wn, wx);
        atomicAdd(wn + a.P, wy);
        atomicAdd(wn + 2 * a.P, wz);
        rest = false;
      }
      if (!__syncthreads_or(rest)) continue;  // s == 0: the last substep
    }
    count = order_by_leaf(sh.r, rest, lx);
    put_point(sh.r, V, lx, x, y, z);
    sh.w[0][tid] = wx;
    sh.w[1][tid] = wy;
    sh.w[2][tid] = wz;
    __syncthreads();
    if (s > 0) rows_gradient(sh, V, 0, 3, count);
    rows_scatter<3>(sh, G, 3, 0, 1.0, count);
    __syncthreads();
    if (s > 0) {
      // a_s = a_{s+1} + tau g2 J(h)^T a_{s+1} + J(x)^T w
      const double sx2 = 2.0 * (double)(1u << V.info[lx].w);
      ax = ax + fh * jx + sx2 * sh.g[0][tid];
      ay = ay + fh * jy + sx2 * sh.g[1][tid];
      az = az + fh * jz + sx2 * sh.g[2][tid];
    }
  }
}

}  // namespace

#define TBX_CAT2(a, b) a##b
#define TBX_CAT(a, b) TBX_CAT2(a, b)

hipError_t TBX_CAT(launch_adj_conc_q, TBX_Q)(int mode, const VelSource &vel,
                                             const TreeView &conc, const StepArgs &a,
                                             const double *dep, const double *ua, double *lam,
                                             double *A, hipStream_t s) {
  if (a.npts <= 0) return hipSuccess;
  const dim3 g((unsigned)(8 * a.per_xcd)), blk(kAdjBlock);
  if (dep)  // the stored trajectories carry the forward's arithmetic
    hipLaunchKernelGGL((k_adj_conc<kFma64, kAdjBlock, true>), g, blk, 0, s, vel, conc, a, dep,
                       ua, lam, A);
  else if (mode == kFma64)
    hipLaunchKernelGGL((k_adj_conc<kFma64, kAdjBlock, false>), g, blk, 0, s, vel, conc, a, dep,
                       ua, lam, A);
  else if (mode == kExact64)
    hipLaunchKernelGGL((k_adj_conc<kExact64, kAdjBlock, false>), g, blk, 0, s, vel, conc, a,
                       dep, ua, lam, A);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t TBX_CAT(launch_adj_vel_q, TBX_Q)(int mode, const VelSource &vel,
                                            const TreeView &conc, const StepArgs &a,
                                            const double *A, double *G, hipStream_t s) {
  if (a.npts <= 0) return hipSuccess;
  const dim3 g((unsigned)(8 * a.per_xcd)), blk(kAdjBlock);
  if (mode == kFma64)
    hipLaunchKernelGGL((k_adj_vel<kFma64>), g, blk, 0, s, vel, conc, a, A, G);
  else if (mode == kExact64)
    hipLaunchKernelGGL((k_adj_vel<kExact64>), g, blk, 0, s, vel, conc, a, A, G);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace tbx
