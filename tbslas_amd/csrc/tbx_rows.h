// Leaf contraction for a workgroup's points, coefficients broadcast within
// DPP rows.
//
// A contraction of the packed triangle at one point is
//   u = sum_{i,j} T_i(z) T_j(y) sum_k c_ijk T_k(x),   i + j + k < D.
// The workgroup's points are first ordered by leaf, the points of a leaf
// padded to a multiple of 16, so that the 16 lanes of a DPP row share a
// leaf and every point is contracted once.  A vector register holds 16
// coefficients of the row's leaf, one per lane, and v_fmac with row_newbcast
// broadcasts one of them to the row: a coefficient reaches its multiply-add
// from one coalesced vector load per 16, several loads ahead.
// T_0(x) = T_0(y) = T_0(z) = 1 are not multiplied by: 799 operations for
// the 680 terms of degree 14.
//
// What it replaces (contract in tbx_device.h, which TBX_EXACT keeps): scalar
// operands through the scalar cache, which hits a third of the time at
// degree 14, and a wavefront of 64 repeated per distinct leaf (1.3 to 1.45
// passes after a regroup of 1,024).  The step kernel before and after: FP64 degree
// 14, 16.7 M points, 7.58 -> 3.5 ms; FP64 degree 8, 3.0 M points, 459 -> 297
// us; FP32 + FP64 head degree 14, 123 M points, 25.5 -> 18.4 ms.  Bound by
// the vector ALU's issue rate: an FP64 multiply-add issues every 2.4 ns per
// SIMD (measured; 4 clocks at the clock it sustains), an FP32 one every
// 1.7 ns.
//
// Also measured: the same contraction as MFMA tiles of 16 rows (i, j) x 16
// points x k.  The FP64 and FP32 MFMAs do not overlap with vector work on
// this part and pay for padding the triangle: 4.7 ms and 498 us in FP64.
//
// A point's sum depends on its own lane alone: it does not change with the
// points around it.
#pragma once

#include "tbx_device.h"
#include "tbx_mfma.h"  // static_for

namespace tbx {

// T_0 .. T_{D-1} at x as cheb_poly gives them, the recurrence fused.
template <int D, typename T>
__device__ __forceinline__ void row_cheb(double x, T *v) {
  const bool in = fabs(x) <= 1.0;
  const double xx = in ? x : 0.0, x2 = 2.0 * xx;
  double y0 = in ? 1.0 : 0.0, y1 = xx;
  v[0] = (T)y0;
  if constexpr (D > 1) v[1] = (T)xx;
#pragma unroll
  for (int k = 2; k < D; ++k) {
    const double y2 = __builtin_fma(x2, y1, -y0);
    v[k] = (T)y2;
    y0 = y1;
    y1 = y2;
  }
}

// A DPP row's 16 lanes hold c[0 .. 15]; all lanes active.
//   row_add<K, N>    w += sum_n c[K + n] p[n], n < N
//   row_start<K, N>  w = c[K] + sum_n c[K + 1 + n] p[n], n < N - 1
// A value written by the vector ALU may be read by a DPP instruction two
// wait states later at the earliest, hence the s_nop.  Volatile: kept in
// order, so that rows are not started ahead of their turn (hoisted, their
// partial sums spill).
#define TBX_F(n, k) "v_fmac_f64_dpp %0, %1, %" #n " row_newbcast:%2+" #k " row_mask:0xf bank_mask:0xf\n\t"
#define TBX_M "v_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf\n\t"
template <int K, int N>
__device__ __forceinline__ void row_add(double &w, double c, const double *p) {
  static_assert(N >= 1 && N <= 16 && K + N <= 16, "within a row");
  if constexpr (N >= 8) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4) TBX_F(8, 5) TBX_F(9, 6) TBX_F(10, 7)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]));
    if constexpr (N > 8) row_add<K + 8, N - 8>(w, c, p + 8);
  } else if constexpr (N == 7) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4) TBX_F(8, 5) TBX_F(9, 6)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]));
  } else if constexpr (N == 6) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4) TBX_F(8, 5)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]));
  } else if constexpr (N == 5) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]));
  } else if constexpr (N == 4) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
  } else if constexpr (N == 3) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]));
  } else if constexpr (N == 2) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]));
  } else {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]));
  }
}
template <int K, int N>
__device__ __forceinline__ void row_start(double &w, double c, const double *p) {
  static_assert(N >= 1 && N <= 16 && K + N <= 16, "within a row");
  if constexpr (N >= 8) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4) TBX_F(7, 5) TBX_F(8, 6) TBX_F(9, 7)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]));
    if constexpr (N > 8) row_add<K + 8, N - 8>(w, c, p + 7);
  } else if constexpr (N == 7) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4) TBX_F(7, 5) TBX_F(8, 6)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]));
  } else if constexpr (N == 6) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4) TBX_F(7, 5)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]));
  } else if constexpr (N == 5) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
  } else if constexpr (N == 4) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]));
  } else if constexpr (N == 3) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]));
  } else if constexpr (N == 2) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]));
  } else {
    asm volatile("s_nop 1\n\t" TBX_M 
                 : "=&v"(w)
                 : "v"(c), "n"(K));
  }
}
#undef TBX_F
#undef TBX_M
#define TBX_F(n, k) "v_fmac_f32_dpp %0, %1, %" #n " row_newbcast:%2+" #k " row_mask:0xf bank_mask:0xf\n\t"
#define TBX_M "v_mov_b32_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf\n\t"
template <int K, int N>
__device__ __forceinline__ void row_add(float &w, float c, const float *p) {
  static_assert(N >= 1 && N <= 16 && K + N <= 16, "within a row");
  if constexpr (N >= 8) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4) TBX_F(8, 5) TBX_F(9, 6) TBX_F(10, 7)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]));
    if constexpr (N > 8) row_add<K + 8, N - 8>(w, c, p + 8);
  } else if constexpr (N == 7) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4) TBX_F(8, 5) TBX_F(9, 6)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]));
  } else if constexpr (N == 6) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4) TBX_F(8, 5)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]));
  } else if constexpr (N == 5) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3) TBX_F(7, 4)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]));
  } else if constexpr (N == 4) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2) TBX_F(6, 3)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
  } else if constexpr (N == 3) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1) TBX_F(5, 2)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]));
  } else if constexpr (N == 2) {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0) TBX_F(4, 1)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]));
  } else {
    asm volatile("s_nop 1\n\t" TBX_F(3, 0)
                 : "+v"(w)
                 : "v"(c), "n"(K), "v"(p[0]));
  }
}
template <int K, int N>
__device__ __forceinline__ void row_start(float &w, float c, const float *p) {
  static_assert(N >= 1 && N <= 16 && K + N <= 16, "within a row");
  if constexpr (N >= 8) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4) TBX_F(7, 5) TBX_F(8, 6) TBX_F(9, 7)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]));
    if constexpr (N > 8) row_add<K + 8, N - 8>(w, c, p + 7);
  } else if constexpr (N == 7) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4) TBX_F(7, 5) TBX_F(8, 6)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]));
  } else if constexpr (N == 6) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4) TBX_F(7, 5)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]));
  } else if constexpr (N == 5) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3) TBX_F(6, 4)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
  } else if constexpr (N == 4) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2) TBX_F(5, 3)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]), "v"(p[2]));
  } else if constexpr (N == 3) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1) TBX_F(4, 2)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]), "v"(p[1]));
  } else if constexpr (N == 2) {
    asm volatile("s_nop 1\n\t" TBX_M TBX_F(3, 1)
                 : "=&v"(w)
                 : "v"(c), "n"(K), "v"(p[0]));
  } else {
    asm volatile("s_nop 1\n\t" TBX_M 
                 : "=&v"(w)
                 : "v"(c), "n"(K));
  }
}
#undef TBX_F
#undef TBX_M

// acc[n] += c[K + n] x, n < N: lanes K .. K + N - 1 of the DPP row's register
// c, one accumulator each (the s_nop as above).
template <int K, int N>
__device__ __forceinline__ void row_outer(double *acc, double c, double x) {
  static_assert(N >= 1 && N <= 16 && K + N <= 16, "within a row");
  if constexpr (N >= 8) {
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, %8, %9 row_newbcast:%10+0 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, %8, %9 row_newbcast:%10+1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, %8, %9 row_newbcast:%10+2 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, %8, %9 row_newbcast:%10+3 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %4, %8, %9 row_newbcast:%10+4 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %5, %8, %9 row_newbcast:%10+5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %6, %8, %9 row_newbcast:%10+6 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %7, %8, %9 row_newbcast:%10+7 row_mask:0xf bank_mask:0xf\n\t"
                 : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4]), "+v"(acc[5]), "+v"(acc[6]), "+v"(acc[7])
                 : "v"(c), "v"(x), "n"(K));
    if constexpr (N > 8) row_outer<K + 8, N - 8>(acc + 8, c, x);
  } else if constexpr (N >= 4) {
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, %4, %5 row_newbcast:%6+0 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, %4, %5 row_newbcast:%6+1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, %4, %5 row_newbcast:%6+2 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, %4, %5 row_newbcast:%6+3 row_mask:0xf bank_mask:0xf\n\t"
                 : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
                 : "v"(c), "v"(x), "n"(K));
    if constexpr (N > 4) row_outer<K + 4, N - 4>(acc + 4, c, x);
  } else if constexpr (N >= 2) {
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%4+0 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, %2, %3 row_newbcast:%4+1 row_mask:0xf bank_mask:0xf\n\t"
                 : "+v"(acc[0]), "+v"(acc[1])
                 : "v"(c), "v"(x), "n"(K));
    if constexpr (N > 2) row_outer<K + 2, N - 2>(acc + 2, c, x);
  } else {
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3+0 row_mask:0xf bank_mask:0xf\n\t"
                 : "+v"(acc[0])
                 : "v"(c), "v"(x), "n"(K));
  }
}

// w += a b in its place among the row operations: left to the scheduler, the
// outer sums gather at the end and every row's partial sum stays live.
__device__ __forceinline__ void fmac_here(double &w, double a, double b) {
  asm volatile("v_fmac_f64 %0, %1, %2" : "+v"(w) : "v"(a), "v"(b));
}
__device__ __forceinline__ void fmac_here(float &w, float a, float b) {
  asm volatile("v_fmac_f32 %0, %1, %2" : "+v"(w) : "v"(a), "v"(b));
}

// One leaf component at the lane's point, the lane's DPP row sharing the
// leaf: c its coefficients from lane & 15 on, px / py = T_1 .. T_{D-1} (x)
// / (y), z inside [-1, 1].  Up to 15 doubles past the last coefficient are
// read (the coefficient buffers are padded).  kRing loads are in flight.
template <int D, bool HEAD, typename T>
__device__ __forceinline__ T row_contract(const T *__restrict__ c, const T (&px)[D],
                                          const T (&py)[D], double z) {
  constexpr int NC = D * (D + 1) * (D + 2) / 6, NB = (NC + 15) / 16, kRing = 6;
  T r[kRing];
  static_for<(kRing - 1 < NB ? kRing - 1 : NB)>([&](auto bc) {
    constexpr int b = decltype(bc)::value;
    r[b] = c[16 * b];
  });
  T u = 0;
  double zm = 1.0, zc = z;
  const double z2 = 2.0 * z;
  static_for<D>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    T v = 0;
    static_for<D - i>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      constexpr int first = tri_start(D, i, j), len = D - i - j;
      T w = 0;
      // the row's coefficients, cut at multiples of 16
      static_for<2>([&](auto hc) {
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
          const T cb = r[b % kRing];
          // terms of the FP64 head (degree <= kHeadDeg) are skipped
          constexpr int skip = HEAD && i + j <= kHeadDeg ? kHeadDeg + 1 - i - j : 0;
          if constexpr (lo == first && skip == 0) {
            row_start<lo % 16, hi - lo>(w, cb, px + 1);
          } else if constexpr (lo == first) {
            static_assert(lo % 16 + skip <= 16, "");
            if constexpr (hi - lo > skip)
              row_add<lo % 16 + skip, hi - lo - skip>(w, cb, px + skip);
          } else {
            row_add<0, hi - lo>(w, cb, px + (lo - first));
          }
        }
      });
      if constexpr (j == 0)
        v = w;
      else
        fmac_here(v, py[j], w);
    });
    if constexpr (i == 0) {
      u = v;
    } else {
      if constexpr (i > 1) {
        const double zn = __builtin_fma(z2, zc, -zm);
        zm = zc;
        zc = zn;
      }
      fmac_here(u, (T)zc, v);
    }
  });
  return u;
}

// ---------------------------------------------------------------------------
// A workgroup's points.
// ---------------------------------------------------------------------------
// order's entries: a thread, with the bits above kPlaceMask set where the
// place is a copy that pads a run.
constexpr int kPlaceMask = 0x7fff;

// The leaf of the first pending lane of the lane's DPP row (of its first
// lane, if none is).
__device__ __forceinline__ int row_leaf(uint64_t pending, int leaf) {
  const int row = (int)(threadIdx.x & 48u);
  const uint32_t rest = (uint32_t)(pending >> row) & 0xffffu;
  return __builtin_amdgcn_ds_bpermute((row + (rest ? __builtin_ctz(rest) : 0)) << 2, leaf);
}

// Orders a wavefront's LDS writes before its other lanes' reads.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int BLOCK>
struct RowsLds {
  double e[3][BLOCK];  // leaf coordinates in, values out (per thread's point)
  double start[3][BLOCK];  // the threads' RK2 start points
  int leaf[BLOCK];
  uint16_t order[BLOCK + 16 * (kRgSlots + 1)];  // position -> thread
  int key[kRgSlots];
  int cnt[kRgSlots + 1];
  int total;
};

// Orders the active threads' points by leaf: afterwards order[0, count) are
// their threads, points of one leaf together and padded to a multiple of 16
// with copies of the last one; returns count, a multiple of 16.  Leaves
// that find no slot in eight probes share the last run.  A wavefront enters
// leaves that several of its lanes share once for them all, until it meets
// one of under three lanes (scattered points enter lane by lane, in
// parallel: one after another 64 leaves would take some 20,000 clocks).
// Every thread of the workgroup must call it; the caller synchronises
// before order is read.
template <int BLOCK>
__device__ __forceinline__ int order_by_leaf(RowsLds<BLOCK> &s, bool active, int leaf) {
  const int tid = (int)threadIdx.x, lane = tid & 63;
  for (int i = tid; i <= kRgSlots; i += BLOCK) {  // a block may hold 64 threads
    if (i < kRgSlots) s.key[i] = -1;
    s.cnt[i] = 0;
  }
  __syncthreads();
  int slot = kRgSlots, rank = 0;
  bool todo = active;
  auto insert = [&]() {  // the thread's leaf into the table: its slot
    uint32_t h = ((uint32_t)leaf * 0x9E3779B1u) >> 26;  // 6 bits: kRgSlots == 64
#pragma unroll 1
    for (int probe = 0; probe < 8; ++probe) {
      const int prev = atomicCAS(&s.key[h], -1, leaf);
      if (prev == -1 || prev == leaf) return (int)h;
      h = (h + 1) & (kRgSlots - 1);
    }
    return kRgSlots;
  };
  uint64_t pending = __builtin_amdgcn_ballot_w64(active);
#pragma unroll 1
  for (int it = 0; it < 6 && pending; ++it) {
    const int src = __builtin_ctzll(pending);
    const int k = __builtin_amdgcn_readlane(leaf, src);
    const bool mine = todo && leaf == k;
    const uint64_t m = __builtin_amdgcn_ballot_w64(mine);
    if (__builtin_popcountll(m) < 3) break;
    pending &= ~m;
    int sl = kRgSlots, base = 0;
    if (lane == src) {
      sl = insert();
      base = atomicAdd(&s.cnt[sl], __builtin_popcountll(m));
    }
    sl = __builtin_amdgcn_readlane(sl, src);
    base = __builtin_amdgcn_readlane(base, src);
    if (mine) {
      slot = sl;
      rank = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                              __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      todo = false;
    }
  }
  if (todo) {
    slot = insert();
    rank = atomicAdd(&s.cnt[slot], 1);
  }
  __syncthreads();
  const int mine = s.cnt[slot];  // points of the thread's run
  if (tid < 64) {  // exclusive scan of the 64 padded slot counts by wave 0
    const int c = (s.cnt[tid] + 15) & ~15;
    int incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (tid >= d) incl += o;
    }
    s.key[tid] = incl - c;
    if (tid == 63) s.total = incl;  // the overflow run goes last
  }
  __syncthreads();
  const int first = slot < kRgSlots ? s.key[slot] : s.total;
  const int count = s.total + ((s.cnt[kRgSlots] + 15) & ~15);
  if (active) {
    s.order[first + rank] = (uint16_t)tid;
    if (rank == mine - 1)
      for (int i = rank + 1; i & 15; ++i) s.order[first + i] = (uint16_t)(tid | ~kPlaceMask);
  }
  return count;
}

// A sum u over the basis at a point: outside the leaf's box, where the basis
// is zero (cheb_poly), it was taken at the box's middle instead, and counts as
// zero times every coefficient: a NaN where one of them is not finite.
__device__ __forceinline__ double in_box(bool in, double u) {
  return in ? u : __builtin_fma(0.0, u, 0.0);
}

// Components c0 .. c0 + nc - 1 (nc <= 3) of t at the points in order[0,
// count): s.e / s.leaf hold every point's leaf coordinates and leaf, and
// component c is returned in s.e[c] (the coordinates are gone).  The caller
// synchronises before and after.
//
// A wavefront takes 64 places, four DPP rows.  A row's lanes share a leaf
// except in the overflow run, where the pass repeats per leaf.
template <int D, int MODE, int BLOCK>
__device__ __forceinline__ void rows(RowsLds<BLOCK> &s, const TreeView &t, int c0,
                                     int nc, int count) {
  using T = typename ModeType<MODE>::T;
  constexpr int NC = D * (D + 1) * (D + 2) / 6;
  const int lane = (int)(threadIdx.x & 63u);
#pragma unroll 1
  for (int p0 = (int)(threadIdx.x & ~63u); p0 < count; p0 += BLOCK) {
    const int src = s.order[p0 + lane < count ? p0 + lane : count - 1] & kPlaceMask;
    const int leaf = s.leaf[src];
    const double ex = s.e[0][src], ey = s.e[1][src], ez = s.e[2][src];
    const bool in = fabs(ex) <= 1.0 && fabs(ey) <= 1.0 && fabs(ez) <= 1.0;
    T px[D], py[D];
    row_cheb<D>(in ? ex : 0.0, px);
    row_cheb<D>(in ? ey : 0.0, py);
    const double z = in ? ez : 0.0;
    uint64_t pending = __builtin_amdgcn_ballot_w64(true);
#pragma unroll 1
    while (pending) {
      const int lf = row_leaf(pending, leaf);
      const bool mine = leaf == lf;
      pending &= ~__builtin_amdgcn_ballot_w64(mine);
      const T *cb = coeff_base<MODE>(t) + ((size_t)lf * t.dof + c0) * NC + (lane & 15);
#pragma unroll 1
      for (int c = 0; c < nc; ++c) {
        const double u = (double)row_contract<D, MODE == kFp32h>(cb, px, py, z);
        if (mine) s.e[c][src] = in_box(in, u);
        cb += NC;
      }
    }
  }
}

// Leaf coordinates of a located point into the workgroup's buffers.
template <int BLOCK>
__device__ __forceinline__ void put_point(RowsLds<BLOCK> &s, const TreeView &t, int leaf,
                                          double x, double y, double z) {
  const int tid = (int)threadIdx.x;
  double ex, ey, ez;
  leaf_xi(t, leaf, x, y, z, ex, ey, ez);
  s.e[0][tid] = ex;
  s.e[1][tid] = ey;
  s.e[2][tid] = ez;
  s.leaf[tid] = leaf;
}

// The FP64 head (degree <= kHeadDeg) of one component at the thread's point.
template <int D>
__device__ __forceinline__ double head_value(const TreeView &t, int comp, int leaf, double ex,
                                             double ey, double ez) {
  constexpr int NC = D * (D + 1) * (D + 2) / 6;
  double hx[3], hy[3], hz[3];
  cheb_poly<3>(ex, hx);
  cheb_poly<3>(ey, hy);
  cheb_poly<3>(ez, hz);
  const double *c = t.coeff + ((size_t)leaf * t.dof + comp) * NC;
  Head<D> h;
  int n = 0;
#pragma unroll
  for (int i = 0; i <= Head<D>::H; ++i)
#pragma unroll
    for (int j = 0; i + j <= Head<D>::H; ++j)
#pragma unroll
      for (int k = 0; i + j + k <= Head<D>::H; ++k) h.c[n++] = c[tri_index(D, i, j, k)];
  return h.eval(hx, hy, hz);
}

// A velocity tree at the active threads' points (x, y, z), located in leaf:
// v.  count: the points in s.order.
template <int D, int MODE, int BLOCK>
__device__ __forceinline__ void rows_vec3(RowsLds<BLOCK> &s,
                                          const TreeView &t, int count, int leaf, double x,
                                          double y, double z, double (&v)[3]) {
  put_point(s, t, leaf, x, y, z);
  __syncthreads();
  rows<D, MODE>(s, t, 0, 3, count);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = s.e[c][threadIdx.x];
  if constexpr (MODE == kFp32h) {
    double ex, ey, ez;
    leaf_xi(t, leaf, x, y, z, ex, ey, ez);
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] += head_value<D>(t, c, leaf, ex, ey, ez);
  }
}

// All components of t at the threads' points, each through store(l, value)
// of the point's thread.
template <int D, int MODE, int BLOCK, typename Store>
__device__ __forceinline__ void rows_dof(RowsLds<BLOCK> &s, const TreeView &t, int count, int leaf, double x,
                                         double y, double z, Store store) {
  for (int c0 = 0; c0 < t.dof; c0 += 3) {
    const int nc = t.dof - c0 < 3 ? t.dof - c0 : 3;
    put_point(s, t, leaf, x, y, z);
    __syncthreads();
    rows<D, MODE>(s, t, c0, nc, count);
    __syncthreads();
    for (int c = 0; c < nc; ++c) {
      double v = s.e[c][threadIdx.x];
      if constexpr (MODE == kFp32h) {
        double ex, ey, ez;
        leaf_xi(t, leaf, x, y, z, ex, ey, ez);
        v += head_value<D>(t, c0 + c, leaf, ex, ey, ez);
      }
      store(c0 + c, v);
    }
  }
}

// Whether the 16 lanes of every DPP row of the wavefront hold points of at
// most two leaves, the row's first lane's and its last's: points that come in
// runs of a leaf.  They are contracted as they come (in_place_dof): the order
// in LDS and the second round that its padding takes bring such points nothing
// (1 M of them on 512 leaves of degree 8 36.7 us, in place 29.9; of degree 6
// 29.6, in place 25.2).  All lanes are active.
__device__ __forceinline__ bool rows_in_place(int leaf) {
  // row_newbcast:0 and row_newbcast:15
  const int first = __builtin_amdgcn_update_dpp(leaf, leaf, 0x150, 0xf, 0xf, false);
  const int last = __builtin_amdgcn_update_dpp(leaf, leaf, 0x15f, 0xf, 0xf, false);
  return __builtin_amdgcn_ballot_w64(leaf != first && leaf != last) == 0;
}

// All components of t at the thread's point, contracted in its own lane, each
// through store(l, value): the bits of rows_dof.
template <int D, int MODE, typename Store>
__device__ __forceinline__ void in_place_dof(const TreeView &t, int leaf, double x, double y,
                                             double z, Store store) {
  using T = typename ModeType<MODE>::T;
  constexpr int NC = D * (D + 1) * (D + 2) / 6;
  double ex, ey, ez;
  leaf_xi(t, leaf, x, y, z, ex, ey, ez);
  const bool in = fabs(ex) <= 1.0 && fabs(ey) <= 1.0 && fabs(ez) <= 1.0;
  T px[D], py[D];
  row_cheb<D>(in ? ex : 0.0, px);
  row_cheb<D>(in ? ey : 0.0, py);
  const double zx = in ? ez : 0.0;
  uint64_t pending = __builtin_amdgcn_ballot_w64(true);
#pragma unroll 1
  while (pending) {
    const int lf = row_leaf(pending, leaf);
    const bool mine = leaf == lf;
    pending &= ~__builtin_amdgcn_ballot_w64(mine);
    const T *cb = coeff_base<MODE>(t) + (size_t)lf * t.dof * NC + (threadIdx.x & 15);
#pragma unroll 1
    for (int l = 0; l < t.dof; ++l) {
      double u = (double)row_contract<D, MODE == kFp32h>(cb, px, py, zx);
      u = in_box(in, u);
      if constexpr (MODE == kFp32h) u += head_value<D>(t, l, leaf, ex, ey, ez);
      if (mine) store(l, u);
      cb += NC;
    }
  }
}

// eval_velocity for a workgroup: the functor at the active threads' points,
// ordered by their leaves in the first tree (hint0: the thread's point's).
// Idle threads' values are not defined.
template <int D, int MODE, int KIND, int BLOCK>
__device__ __forceinline__ void rows_velocity(RowsLds<BLOCK> &s, const VelSource &vs,
                                              int stage, double ts, int scaled, double g, int bc,
                                              int count, int hint0, double &x, double &y,
                                              double &z, double (&v)[3]) {
  if constexpr (KIND == kVelTree) {
    rows_vec3<D, MODE>(s, vs.t[0], count, hint0, x, y, z, v);
    if (scaled) {
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = v[c] * g;
    }
  } else {
    // both combinations are linear in the trees' values: a tree's weight at
    // a time, 1.5 / -0.5 (tree_extrap_functor.h:71-77) or the cubic Hermite
    // interpolation of a unit value (tree_set_functor.h:66-72)
    const int nt = KIND == kVelExtrap ? (stage == 1 ? 1 : 2) : 4;
    v[0] = v[1] = v[2] = 0.0;
#pragma unroll 1
    for (int k = 0; k < nt; ++k) {
      if (k > 0 && bc == TBX_BC_PERIODIC) {  // the array is wrapped in place per tree
        x = wrap1(x);
        y = wrap1(y);
        z = wrap1(z);
      }
      const TreeView &tk = k == 0 ? vs.t[0] : k == 1 ? vs.t[1] : k == 2 ? vs.t[2] : vs.t[3];
      double u[3], w;
      rows_vec3<D, MODE>(s, tk, count, k == 0 ? hint0 : locate(tk, x, y, z), x, y, z, u);
      if constexpr (KIND == kVelExtrap)
        w = stage == 1 ? 1.0 : k == 0 ? 1.5 : -0.5;
      else
        w = cubic1d(ts, vs.tt, k == 0 ? 1.0 : 0.0, k == 1 ? 1.0 : 0.0, k == 2 ? 1.0 : 0.0,
                    k == 3 ? 1.0 : 0.0);
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = __builtin_fma(w, u[c], v[c]);
    }
  }
}

// The second half of an IntegrateRK2 substep (rk2_finish) for a workgroup:
// the active threads' start points (x, y, z) with first-stage velocities v
// move to the substep's end.  Returns the count of the midpoints' order.
template <int D, int MODE, int KIND, int BLOCK>
__device__ __forceinline__ int rows_midpoint(RowsLds<BLOCK> &s, const VelSource &vel, int bc,
                                             double htau, double tau, int scaled, double g2,
                                             double ts2, bool active, double (&v)[3], double &x,
                                             double &y, double &z) {
  // midpoint xtmp = xinit + (0.5 * dt) * vtmp (traj.inc:36), wrapped for
  // its evaluation only
  double hx = x + htau * v[0], hy = y + htau * v[1], hz = z + htau * v[2];
  if (bc == TBX_BC_PERIODIC) {
    hx = wrap1(hx);
    hy = wrap1(hy);
    hz = wrap1(hz);
  }
  const int lf = locate(vel.t[0], hx, hy, hz);
  const int count = order_by_leaf(s, active, lf);
  // the start point waits in LDS, not in registers
  const int tid = (int)threadIdx.x;
  s.start[0][tid] = x;
  s.start[1][tid] = y;
  s.start[2][tid] = z;
  rows_velocity<D, MODE, KIND>(s, vel, 2, ts2, scaled, g2, bc, count, lf, hx, hy, hz, v);
  asm volatile("" ::: "memory");  // read back, not kept
  // xsol = xinit + dt * vtmp (traj.inc:41-42)
  x = s.start[0][tid] + tau * v[0];
  y = s.start[1][tid] + tau * v[1];
  z = s.start[2][tid] + tau * v[2];
  return count;
}

// One IntegrateRK2 substep (rk2_substep) for a workgroup, in place.
template <int D, int MODE, int KIND, int BLOCK>
__device__ __forceinline__ void rows_substep(RowsLds<BLOCK> &s, const VelSource &vel, int bc,
                                             double htau, double tau, int scaled, double g1,
                                             double g2, double ts1, double ts2, bool active,
                                             double &x, double &y, double &z) {
  if (bc == TBX_BC_PERIODIC) {
    x = wrap1(x);
    y = wrap1(y);
    z = wrap1(z);
  }
  const int lf = locate(vel.t[0], x, y, z);
  const int count = order_by_leaf(s, active, lf);
  double v[3];
  rows_velocity<D, MODE, KIND>(s, vel, 1, ts1, scaled, g1, bc, count, lf, x, y, z, v);
  rows_midpoint<D, MODE, KIND>(s, vel, bc, htau, tau, scaled, g2, ts2, active, v, x, y, z);
}

}  // namespace tbx
