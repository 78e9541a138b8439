// Degree-independent kernels of libtbx: point location, grid points and the
// FP32 coefficient mirror.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tbx_device.h"

namespace tbx {
namespace {

// EvalTree's wrap + keys + leaf assignment (tree_functor.h:442-489,
// :190-198) without evaluation; pts are left untouched.  A block takes
// kLocatePts x kBlock consecutive points: their coordinates (24 bytes a
// point) come in through LDS with 16-byte loads, consecutive per lane, and
// each thread then locates kLocatePts points a block apart, all their
// directory loads issued before the first search.  Coordinates and leaf ids
// are streamed (non-temporal), which leaves the caches to the directory and
// the keys.
constexpr int kLocatePts = 4;
typedef double stage2 __attribute__((ext_vector_type(2)));

__global__ __launch_bounds__(kBlock) void k_locate(TreeView t,
                                                   const double *__restrict__ pts,
                                                   int64_t n, int bc,
                                                   int32_t *__restrict__ leaf) {
  constexpr int NP = kBlock * kLocatePts;  // points of the block
  __shared__ stage2 stage[NP * 3 / 2];     // NP x 3 doubles
  const int64_t p0 = (int64_t)blockIdx.x * NP;
  const int64_t np = n - p0 < NP ? n - p0 : NP;
  const int tid = threadIdx.x;
  if (np == NP && (reinterpret_cast<uintptr_t>(pts) & 15u) == 0) {
    // the block's 3 NP doubles as NP * 3 / 2 16-byte pieces
    const stage2 *src = reinterpret_cast<const stage2 *>(pts + 3 * p0);
#pragma unroll
    for (int k = 0; k < NP * 3 / 2 / kBlock; ++k)
      stage[k * kBlock + tid] = __builtin_nontemporal_load(src + k * kBlock + tid);
  } else {
    double *dst = reinterpret_cast<double *>(stage);
    for (int k = tid; k < 3 * np; k += kBlock) dst[k] = pts[3 * p0 + k];
  }
  __syncthreads();
  const double *c = reinterpret_cast<const double *>(stage);
  uint64_t key[kLocatePts];
  int lo[kLocatePts], hi[kLocatePts];
#pragma unroll
  for (int k = 0; k < kLocatePts; ++k) {
    // lanes past the end locate the block's first point and store nothing
    const int j = k * kBlock + tid < np ? k * kBlock + tid : 0;
    double a = c[3 * j + 0], b = c[3 * j + 1], z = c[3 * j + 2];
    if (bc == TBX_BC_PERIODIC) {
      a = wrap1(a);
      b = wrap1(b);
      z = wrap1(z);
    }
    key[k] = point_key(a, b, z);
    lo[k] = dir_first(t, key[k]);
    hi[k] = dir_last(t, key[k]);
  }
#pragma unroll
  for (int k = 0; k < kLocatePts; ++k) {
    const int j = k * kBlock + tid;
    const int r = dir_search(t, key[k], lo[k], hi[k]);
    if (j < np) __builtin_nontemporal_store(r, leaf + p0 + j);
  }
}

struct NodeTable {
  double node[TBX_MAX_Q + 1];
  int d;
};

// CollectChebTreeGridPoints (tree_utils.h:478-491): corner + len * node,
// node index x fastest (cheb.h:60-67).
__global__ __launch_bounds__(kBlock) void k_grid_points(TreeView t,
                                                        NodeTable nt,
                                                        double *__restrict__ out) {
  const int d = nt.d, P = d * d * d;
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= t.L * P) return;
  const int64_t leaf = i / P;
  const int m = (int)(i - leaf * P);
  const uint4 inf = t.info[leaf];
  const double len = 1.0 / (double)(1u << inf.w);
  out[3 * i + 0] = (double)inf.x * len + len * nt.node[m % d];
  out[3 * i + 1] = (double)inf.y * len + len * nt.node[(m / d) % d];
  out[3 * i + 2] = (double)inf.z * len + len * nt.node[m / (d * d)];
}

__global__ __launch_bounds__(kBlock) void k_to_f32(const double *__restrict__ in,
                                                   float *__restrict__ out,
                                                   int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) out[i] = (float)in[i];
}

constexpr int kXcds = 8;
constexpr int kMetaStride = 32;  // words: a cache line each
constexpr int kMetaWords = 2 * kMetaStride;  // [0] scattered, [kMetaStride] places taken
constexpr int kFewLeaves = 1024;
constexpr int kProbeBlock = 1024;
constexpr int kProbes = kProbeBlock / 64;  // a wavefront each
constexpr int kOrderBlocks = 16384;  // a multiple of kXcds

// Order of a call's points by leaf (counting sort; order_words(n, L) words of
// scratch): leaf and rank of every point, hist, then perm.  Groups follow
// each other in no particular order; a point's place in its group depends on
// the run, its value does not.
//
// k_order_begin decides whether there is anything to order, from kProbes
// windows of 64 consecutive points spread over the call: scattered (meta[0])
// where more than a quarter of them hold more than run_leaves leaves.  Others
// are taken as they come (their accesses stay coalesced, a workgroup orders
// its few leaves by itself), and the kernels after this one return at once.
// Counting and placing every point before it was known took 20 us, and 20 to
// 60 per million points, of calls that gained nothing: 1 M points in leaf
// order on 512 leaves of degree 8 48 us, now 30; 4 M on 4,096 leaves of degree
// 4, three components, 123 us, now 71.  Points in the order of a tree's grid
// change leaf at every face and hold few all the same: 23.9 M departure points
// of 32,768 leaves of degree 8 1,937 us ordered, now 645.  Block 0 probes, the
// others clear the counters.
__global__ __launch_bounds__(kProbeBlock) void k_order_begin(TreeView t,
                                                             const double *__restrict__ pts,
                                                             int64_t n, int bc,
                                                             int32_t *__restrict__ meta,
                                                             int64_t words, int run_leaves) {
  if (blockIdx.x > 0) {
    const int64_t stride = (int64_t)(gridDim.x - 1) * kProbeBlock;
    for (int64_t i = kMetaStride + (int64_t)(blockIdx.x - 1) * kProbeBlock + threadIdx.x;
         i < words; i += stride)
      meta[i] = 0;
    return;
  }
  __shared__ int scattered;
  if (threadIdx.x == 0) scattered = 0;
  __syncthreads();
  const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
  int64_t i = (n > 64 ? n - 64 : 0) * wave / (kProbes - 1) + lane;
  i = i < n ? i : n - 1;
  double x = pts[3 * i + 0], y = pts[3 * i + 1], z = pts[3 * i + 2];
  if (bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
  }
  const int lf = locate(t, x, y, z);
  uint64_t rest = __builtin_amdgcn_ballot_w64(true);
#pragma unroll 1
  for (int k = 0; k < run_leaves && rest; ++k)
    rest &= ~__builtin_amdgcn_ballot_w64(lf == __builtin_amdgcn_readlane(lf, __builtin_ctzll(rest)));
  if (lane == 0 && rest) atomicAdd(&scattered, 1);
  __syncthreads();
  if (threadIdx.x == 0) meta[0] = 4 * scattered > kProbes;
}

// k_order_count: rank = the point's number in its leaf.  A wavefront adds
// once per leaf that several of its lanes share, so that many points of one
// leaf do not queue on its counter.  Each of the eight XCDs (workgroups go to
// them in turn) has its own counters, hist[x][L]: a line that the XCDs add to
// in turn travels between their L2s (1,000,003 scattered points of a call 172
// us with one array, 139 with eight).  FEW (L <= kFewLeaves): a workgroup
// counts in LDS and adds once per leaf, for many points on few leaves would
// all queue on the same counters (457,182 points on 512 leaves 90 us, 68 in
// LDS).  At most kOrderBlocks workgroups, so that a call whose points are not
// ordered does not wait for 62,500 empty ones (14 us); tile b of the points
// is on XCD b % kXcds in any case.
template <bool FEW>
__global__ __launch_bounds__(kBlock) void k_order_count(TreeView t,
                                                        const double *__restrict__ pts,
                                                        int64_t n, int bc,
                                                        int32_t *__restrict__ leaf,
                                                        int32_t *__restrict__ rank,
                                                        int32_t *__restrict__ hist,
                                                        const int32_t *__restrict__ meta) {
  if (meta[0] == 0) return;
  __shared__ int cnt[FEW ? kFewLeaves : 1];
  hist += (int)(blockIdx.x % kXcds) * t.L;
  for (int64_t i0 = (int64_t)blockIdx.x * kBlock; i0 < n; i0 += (int64_t)gridDim.x * kBlock) {
    const int64_t i = i0 + threadIdx.x;
    const bool live = i < n;
    int lf = 0;
    if (live) {
      double x = pts[3 * i + 0], y = pts[3 * i + 1], z = pts[3 * i + 2];
      if (bc == TBX_BC_PERIODIC) {
        x = wrap1(x);
        y = wrap1(y);
        z = wrap1(z);
      }
      lf = locate(t, x, y, z);
    }
    int r = 0;
    if constexpr (FEW) {
      for (int l = (int)threadIdx.x; l < t.L; l += kBlock) cnt[l] = 0;
      __syncthreads();
      if (live) r = atomicAdd(&cnt[lf], 1);
      __syncthreads();
      for (int l = (int)threadIdx.x; l < t.L; l += kBlock)
        if (cnt[l]) cnt[l] = atomicAdd(&hist[l], cnt[l]);
      __syncthreads();
      r += cnt[lf];
      __syncthreads();  // the next tile counts again
    } else {
      const int lane = (int)(threadIdx.x & 63u);
      uint64_t pending = __builtin_amdgcn_ballot_w64(live);
      bool todo = live;
      for (int it = 0; it < 3 && pending; ++it) {
        const int src = __builtin_ctzll(pending);
        const int k = __builtin_amdgcn_readlane(lf, src);
        const bool mine = todo && lf == k;
        const uint64_t m = __builtin_amdgcn_ballot_w64(mine);
        if (__builtin_popcountll(m) < 4) break;
        int base = 0;
        if (lane == src) base = atomicAdd(&hist[k], __builtin_popcountll(m));
        base = __builtin_amdgcn_readlane(base, src);
        if (mine) {
          r = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                               __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
          todo = false;
        }
        pending &= ~m;
      }
      if (todo) r = atomicAdd(&hist[lf], 1);
    }
    if (live) {
      leaf[i] = lf;
      rank[i] = r;
    }
  }
}

// hist[l] = first place of leaf l's points: a wavefront's 64 leaves take
// their places together.
__global__ __launch_bounds__(kBlock) void k_order_start(int32_t *__restrict__ hist, int64_t L,
                                                        int32_t *__restrict__ meta) {
  if (meta[0] == 0) return;
  const int64_t l = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int lane = (int)(threadIdx.x & 63u);
  int h[kXcds], c = 0;
#pragma unroll
  for (int x = 0; x < kXcds; ++x) {
    h[x] = l < L ? hist[x * L + l] : 0;
    c += h[x];
  }
  int incl = c;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(incl, d, 64);
    if (lane >= d) incl += o;
  }
  int base = 0;
  if (lane == 63 && incl) base = atomicAdd(&meta[kMetaStride], incl);
  base = __builtin_amdgcn_readlane(base, 63);
  if (l >= L) return;
  int start = base + incl - c;  // the leaf's places, XCD by XCD
#pragma unroll
  for (int x = 0; x < kXcds; ++x) {
    hist[x * L + l] = start;
    start += h[x];
  }
}

// perm[place] = point.
__global__ __launch_bounds__(kBlock) void k_order_place(const int32_t *__restrict__ leaf,
                                                        const int32_t *__restrict__ rank,
                                                        const int32_t *__restrict__ hist,
                                                        const int32_t *__restrict__ meta,
                                                        int64_t n, int64_t L,
                                                        int32_t *__restrict__ perm) {
  if (meta[0] == 0) return;
  hist += (int)(blockIdx.x % kXcds) * L;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    perm[hist[leaf[i]] + rank[i]] = (int32_t)i;
}

inline unsigned grid_for(int64_t n) {
  return (unsigned)((n + kBlock - 1) / kBlock);
}

}  // namespace

hipError_t launch_locate(const TreeView &t, const double *pts, int64_t n,
                         int bc, int32_t *leaf, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int64_t per = (int64_t)kBlock * kLocatePts;
  hipLaunchKernelGGL(k_locate, dim3((unsigned)((n + per - 1) / per)), dim3(kBlock), 0, s, t,
                     pts, n, bc, leaf);
  return hipGetLastError();
}

int64_t order_words(int64_t n, int64_t L) { return 3 * n + kXcds * L + kMetaWords; }

hipError_t launch_order_points(const TreeView &t, const double *pts, int64_t n, int bc,
                               double work, int32_t *words, PointPerm *perm, hipStream_t s) {
  int32_t *leaf = words, *rank = leaf + n, *meta = rank + n, *hist = meta + kMetaWords;
  perm->use = meta;
  perm->perm = hist + kXcds * t.L;
  const int64_t clear = kXcds * t.L + kMetaWords;
  const unsigned grid = std::min<unsigned>(grid_for(n), kOrderBlocks);
  // On few leaves counting is cheap and large triangles gain from whole runs:
  // grid points of 512 leaves of degree 14 119 us ordered and 131 as they come,
  // three components 223 and 258; of degree 8, three components (495
  // multiply-adds a point) 45.8 and 38.4; of 4,096 leaves of degree 14 1,526
  // and 829.
  const int run_leaves = t.L <= kFewLeaves && work >= 600 ? 2 : 8;
  hipLaunchKernelGGL(k_order_begin,
                     dim3(1 + (unsigned)std::min<int64_t>((clear + 4 * kProbeBlock - 1) /
                                                              (4 * kProbeBlock), kOrderBlocks)),
                     dim3(kProbeBlock), 0, s, t, pts, n, bc, meta, clear, run_leaves);
  hipLaunchKernelGGL(t.L <= kFewLeaves ? k_order_count<true> : k_order_count<false>, dim3(grid),
                     dim3(kBlock), 0, s, t, pts, n, bc, leaf, rank, hist, meta);
  hipLaunchKernelGGL(k_order_start, dim3(grid_for(t.L)), dim3(kBlock), 0, s, hist, t.L, meta);
  hipLaunchKernelGGL(k_order_place, dim3(grid), dim3(kBlock), 0, s, leaf, rank, hist, meta, n,
                     t.L, const_cast<int32_t *>(perm->perm));
  return hipGetLastError();
}

hipError_t launch_grid_points(const TreeView &t, const double *node, int d,
                              double *out, hipStream_t s) {
  const int64_t n = t.L * (int64_t)d * d * d;
  if (n <= 0) return hipSuccess;
  NodeTable nt{};
  for (int i = 0; i < d; ++i) nt.node[i] = node[i];
  nt.d = d;
  hipLaunchKernelGGL(k_grid_points, dim3(grid_for(n)), dim3(kBlock), 0, s, t,
                     nt, out);
  return hipGetLastError();
}

hipError_t launch_to_f32(const double *in, float *out, int64_t n,
                         hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_to_f32, dim3(grid_for(n)), dim3(kBlock), 0, s, in, out,
                     n);
  return hipGetLastError();
}

}  // namespace tbx
