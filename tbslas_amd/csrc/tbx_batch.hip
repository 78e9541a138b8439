// Many small problems in one persistent launch: every problem is one
// velocity tree and one single-component concentration tree (its own
// leaves, degree and time step), all advanced by one in-situ step in FP32
// in a single kernel.
//
// Work items are (problem, run of LPI leaves), numbered problem by problem;
// persistent workgroups claim them from a global counter until none are
// left.  An item computes the departure points of its leaves' grid points
// (one RK2 substep through the problem's velocity tree, FP32 contraction,
// points ordered by leaf in LDS as in the fused step), the concentration
// there (FP32), keeps the values in LDS and refits them at once (the
// per-leaf product of SetTreeGridValues, tree_utils.h:534-546, factored as
// in the tree's refit and summed in FP64), so no value buffer exists.  Coefficients
// are FP32 and ping-pong between two buffers; the step of parity k reads
// buffer k and writes buffer 1 - k.  With vnode (the stationary velocity's
// values at its own grid nodes, expanded once when the batch is made) the
// first RK2 stage at the arrival nodes reads them, as the single-tree step
// does.
//
// Bound by the FP32 contractions' issue rate and the refit's reads of H from
// L2.  24 problems of 4,096 leaves, degrees 6, 8 and 10, one step: 7.5 ms
// with scalar-operand contractions and the refit as one dense P x Nc product
// (3 MB of operator per item at degree 10), 4.1 ms with the rows and the
// factored refit (0.65 MB), both with 512 threads and four leaves an item.
#include <hip/hip_runtime.h>

#include "tbx_rows.h"

namespace tbx {
namespace {

__device__ __forceinline__ int find_problem(const BatchProblem *pb, int nprob, int64_t item) {
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {  // last problem whose first item is <= item
    const int mid = (lo + hi + 1) >> 1;
    if (pb[mid].item0 <= item)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// A workgroup's LDS: the points' buffers while the values are made, then the
// refit's intermediate [LPI][D][D][D]; the values, then the refit's
// projection [LPI][Nc].
template <int BLOCK, int LPI>
struct BatchLds {
  union {
    RowsLds<BLOCK> rows;
    double a[LPI * 11 * 11 * 11];
  };
  union {
    float vals[LPI * 11 * 11 * 11];
    double w[LPI * 11 * 12 * 13 / 6];
  };
  long long item;
};

// Refit of an item's leaves from their values: c' = H (B^T v), B^T by the
// three one-axis contractions x, y, z (a line of D values a thread, in place
// in s.a), summed in FP64 throughout.  The one-axis table sits in registers,
// column a across the 16 lanes of each DPP row (row_outer).  H: one thread
// per coefficient (and group of leaves, where the workgroup has threads for
// several), each entry streamed from L2 once per group.
template <int D, int BLOCK, int LPI>
__device__ __forceinline__ void batch_refit(const BatchProblem &pb, float *__restrict__ out,
                                            int64_t leaf0, int nleaf, BatchLds<BLOCK, LPI> &s) {
  constexpr int P = D * D * D;
  constexpr int NC = D * (D + 1) * (D + 2) / 6;
  const int tid = (int)threadIdx.x, lane = tid & 15;
  double tr[D];  // T_lane at node a
#pragma unroll
  for (int a = 0; a < D; ++a) tr[a] = pb.T[(lane < D ? lane : 0) * D + a];
  const int nl = nleaf * D * D;  // lines per axis
  auto line = [&](const double (&x)[D], double (&o)[D]) {
#pragma unroll
    for (int k = 0; k < D; ++k) o[k] = 0.0;
#pragma unroll
    for (int a = 0; a < D; ++a) row_outer<0, D>(o, tr[a], x[a]);
  };
  // every lane computes a line (its table entries are read by its
  // neighbours); those past the last repeat it and are dropped
#pragma unroll 1
  for (int t0 = 0; t0 < nl; t0 += BLOCK) {
    const int t = t0 + tid < nl ? t0 + tid : nl - 1;  // (leaf, c, b)
    double x[D], o[D];
#pragma unroll
    for (int a = 0; a < D; ++a) x[a] = (double)s.vals[t * D + a];
    line(x, o);
    if (t0 + tid < nl) {
#pragma unroll
      for (int k = 0; k < D; ++k) s.a[t * D + k] = o[k];
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int t0 = 0; t0 < nl; t0 += BLOCK) {
    const int t = t0 + tid < nl ? t0 + tid : nl - 1;  // (leaf, c), k
    double *p = s.a + t / D * (D * D) + t % D;
    double x[D], o[D];
#pragma unroll
    for (int b = 0; b < D; ++b) x[b] = p[b * D];
    line(x, o);
    if (t0 + tid < nl) {
#pragma unroll
      for (int j = 0; j < D; ++j) p[j * D] = o[j];
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int t0 = 0; t0 < nl; t0 += BLOCK) {
    const int t = t0 + tid < nl ? t0 + tid : nl - 1;  // leaf, (j, k)
    const int leaf = t / (D * D), jk = t % (D * D), j = jk / D, k = jk % D;
    const double *p = s.a + leaf * P + jk;
    double x[D], o[D];
#pragma unroll
    for (int c = 0; c < D; ++c) x[c] = p[c * (D * D)];
    line(x, o);
    if (t0 + tid < nl) {
      double *w = s.w + leaf * NC + k;
#pragma unroll
      for (int i = 0; i < D; ++i)
        if (i + j + k < D) w[tri_start(D, i, j)] = o[i];
    }
  }
  __syncthreads();
  // the sums of the item's missing leaves (b >= nleaf) run on whatever the
  // LDS holds there and are not stored
  constexpr int W = (NC + 63) / 64 * 64;
  constexpr int fit = BLOCK / W > 1 ? BLOCK / W : 1;
  constexpr int G = fit >= 4 && LPI >= 4 ? 4 : fit >= 2 && LPI >= 2 ? 2 : 1;
  constexpr int LB = LPI / G;
  const int g = G > 1 ? tid / W : 0;
  if (g < G) {
    const double *w = s.w + g * LB * NC;
    for (int m = G > 1 ? tid - g * W : tid; m < NC; m += G > 1 ? W : BLOCK) {
      double acc[LB];
#pragma unroll
      for (int b = 0; b < LB; ++b) acc[b] = 0.0;
#pragma unroll 12
      for (int p = 0; p < NC; ++p) {
        const double h = pb.H[p * pb.np + m];
#pragma unroll
        for (int b = 0; b < LB; ++b) acc[b] = __builtin_fma(h, w[b * NC + p], acc[b]);
      }
#pragma unroll
      for (int b = 0; b < LB; ++b)
        if (g * LB + b < nleaf) out[(leaf0 + g * LB + b) * NC + m] = (float)acc[b];
    }
  }
  __syncthreads();
}

// One item of degree D - 1: leaves [leaf0, leaf0 + nleaf) of problem p.
template <int D, int BLOCK, int LPI>
__device__ __forceinline__ void batch_item(const BatchProblem &pb, int parity, int64_t leaf0,
                                           int nleaf, BatchLds<BLOCK, LPI> &s) {
  constexpr int P = D * D * D;
  const TreeView &vel = pb.vel;
  const TreeView &conc = pb.conc[parity];
  VelSource vs{};
  vs.t[0] = vel;
  vs.kind = kVelTree;
  vs.ntree = 1;
  const int total = nleaf * P;
  const int tid = (int)threadIdx.x;
#pragma unroll 1
  for (int start = 0; start < total; start += BLOCK) {
    const bool live = start + tid < total;
    const int idx = live ? start + tid : total - 1;
    const int64_t leaf = leaf0 + idx / P;
    const int m = idx % P;
    const uint4 inf = conc.info[leaf];
    const double len = 1.0 / (double)(1u << inf.w);
    double x = (double)inf.x * len + len * pb.node[m % D];
    double y = (double)inf.y * len + len * pb.node[(m / D) % D];
    double z = (double)inf.z * len + len * pb.node[m / (D * D)];
    if (pb.bc == TBX_BC_PERIODIC) {
      x = wrap1(x);
      y = wrap1(y);
      z = wrap1(z);
    }
    int lf = locate(vel, x, y, z);
    // stage 1 from the nodal values; the order and contraction only in
    // workgroups holding a node of another depth's leaf, whose points keep
    // the nodal value where they have one (a point's result does not depend
    // on the workgroup it falls in)
    double v[3];
    bool got = false;
    if (pb.vnode) got = nodal_velocity<D>(pb.vnode, vel, inf, m, lf, P, 0, 1.0, v[0], v[1], v[2]);
    if (__syncthreads_or(!got)) {
      const int count = order_by_leaf(s.rows, live, lf);
      double u[3];
      rows_vec3<D, kFp32>(s.rows, vel, count, lf, x, y, z, u);
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = got ? v[c] : u[c];
    }
    const int count = rows_midpoint<D, kFp32, kVelTree>(s.rows, vs, pb.bc, pb.htau, pb.tau, 0, 1.0,
                                                        0.0, live, v, x, y, z);
    if (pb.bc == TBX_BC_PERIODIC) {
      x = wrap1(x);
      y = wrap1(y);
      z = wrap1(z);
    }
    lf = locate(conc, x, y, z);
    // a departure point lies mostly in its midpoint's leaf: the midpoints'
    // order serves the concentration too
    rows_dof<D, kFp32>(s.rows, conc, count, lf, x, y, z, [&](int, double u) {
      if (live) s.vals[start + tid] = (float)u;
    });
  }
  __syncthreads();
  batch_refit<D>(pb, pb.out32[parity], leaf0, nleaf, s);
}

template <int BLOCK, int LPI>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_batch(
    const BatchProblem *__restrict__ pb, int nprob, int parity, int64_t total_items,
    unsigned long long *counter) {
  __shared__ BatchLds<BLOCK, LPI> sh;
  while (true) {
    if (threadIdx.x == 0) sh.item = (long long)atomicAdd(counter, 1ull);
    __syncthreads();
    const int64_t item = sh.item;
    __syncthreads();
    if (item >= total_items) break;  // uniform over the workgroup
    const int p = find_problem(pb, nprob, item);
    const BatchProblem &b = pb[p];
    const int64_t leaf0 = (item - b.item0) * LPI;
    const int nleaf = (int)(b.L - leaf0 < LPI ? b.L - leaf0 : LPI);
    switch (b.q) {
      case 6:
        batch_item<7, BLOCK, LPI>(b, parity, leaf0, nleaf, sh);
        break;
      case 8:
        batch_item<9, BLOCK, LPI>(b, parity, leaf0, nleaf, sh);
        break;
      default:
        batch_item<11, BLOCK, LPI>(b, parity, leaf0, nleaf, sh);
        break;
    }
  }
}

__global__ void k_batch_reset(unsigned long long *counter) { *counter = 0ull; }

template <int BLOCK, int LPI>
hipError_t launch_cfg(const BatchProblem *pb, int nprob, int parity, int64_t total_items,
                      unsigned long long *counter, int grid, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_reset, dim3(1), dim3(1), 0, s, counter);
  hipLaunchKernelGGL((k_batch<BLOCK, LPI>), dim3(grid), dim3(BLOCK), 0, s, pb, nprob, parity,
                     total_items, counter);
  return hipGetLastError();
}

template <int BLOCK, int LPI>
int occupancy() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_batch<BLOCK, LPI>, BLOCK, 0) !=
      hipSuccess)
    return 1;
  return n > 0 ? n : 1;
}

}  // namespace

int batch_blocks_per_cu(int cfg) {
  switch (cfg) {
    case 0: return occupancy<256, 1>();
    case 1: return occupancy<256, 2>();
    case 2: return occupancy<512, 1>();
    case 3: return occupancy<512, 2>();
    case 4: return occupancy<512, 4>();
    default: return occupancy<1024, 1>();
  }
}

hipError_t launch_batch(int cfg, const BatchProblem *pb, int nprob, int parity,
                        int64_t total_items, unsigned long long *counter, int grid,
                        hipStream_t s) {
  switch (cfg) {
    case 0: return launch_cfg<256, 1>(pb, nprob, parity, total_items, counter, grid, s);
    case 1: return launch_cfg<256, 2>(pb, nprob, parity, total_items, counter, grid, s);
    case 2: return launch_cfg<512, 1>(pb, nprob, parity, total_items, counter, grid, s);
    case 3: return launch_cfg<512, 2>(pb, nprob, parity, total_items, counter, grid, s);
    case 4: return launch_cfg<512, 4>(pb, nprob, parity, total_items, counter, grid, s);
    default: return launch_cfg<1024, 1>(pb, nprob, parity, total_items, counter, grid, s);
  }
}

}  // namespace tbx
