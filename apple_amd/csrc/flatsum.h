// Fixed-order workgroup sums of FP64 tables (per-block energies, per-vertex-
// block dot products), shared by the finish pass, the solver's scalar
// kernels and the element passes that take a scalar step themselves.
#pragma once

#include <hip/hip_runtime.h>

#include "lanes.h"

namespace apl {

// LDS bytes the sums below may need
constexpr int SUMS_LDS = (16 + 1) * 16 * 8;

// Column sums of a row-major table of W doubles per row, p[0 .. n) with n a
// multiple of W, by one workgroup of NT threads (W divides 64).  Thread t
// adds the entries t, t + NT, t + 2 NT, ... -- all of column t % W -- in
// eight strands; lanes of equal column then combine by a fixed shuffle tree
// and the waves in order.  The sums are in sm[0 .. W) on return (sm:
// (NT / 64 + 1) W doubles; a barrier has passed).  The order depends only on
// n, so a table gives the same bits wherever it sits in a batch.
template <int W, int NT>
__device__ inline void flat_column_sums(const double* __restrict__ p, long long n, double* sm) {
  static_assert(64 % W == 0 && NT % 64 == 0, "column width must divide the wave");
  const int t = threadIdx.x;
  double a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (long long f = t; f < n; f += 8LL * NT) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = f + (long long)u * NT < n ? p[f + (long long)u * NT] : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] += v[u];
  }
  double s = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
#pragma unroll
  for (int off = 32; off >= W; off >>= 1) s += __shfl_down(s, off, 64);
  const int lane = t & 63, w = t >> 6;
  if (lane < W) sm[(1 + w) * W + lane] = s;
  __syncthreads();
  if (t < W) {
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) r += sm[(1 + i) * W + t];
    sm[t] = r;
  }
  __syncthreads();
}

// The same sums, bit for bit, of a short table (n <= 4 NV: four of the eight
// strands) by a workgroup of NT < NV threads, each of which stands for NV / NT
// threads of flat_column_sums<W, NV>.  sm: (NV / 64 + 1) W doubles.
template <int W, int NV, int NT>
__device__ inline void flat_column_sums_short(const double* __restrict__ p, int n, double* sm) {
  static_assert(64 % W == 0 && NT % 64 == 0 && NV % NT == 0, "column width must divide the wave");
  constexpr int M = NV / NT;
  const int t = threadIdx.x;
  const int lane = t & 63, w = t >> 6;
  double v[M][4];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int f = t + m * NT + u * NV;
      v[m][u] = f < n ? p[f] : 0.0;
    }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    double s = (v[m][0] + v[m][1]) + (v[m][2] + v[m][3]);
    s = add_xor<32>(s);
    if constexpr (W <= 16) s = add_xor<16>(s);
    if constexpr (W <= 8) s = add_xor<8>(s);
    if constexpr (W <= 4) s = add_xor<4>(s);
    if constexpr (W <= 2) s = add_xor<2>(s);
    if (lane < W) sm[(1 + w + m * (NT / 64)) * W + lane] = s;
  }
  __syncthreads();
  if (t < W) {
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < NV / 64; ++i) r += sm[(1 + i) * W + t];
    sm[t] = r;
  }
  __syncthreads();
}

// The sum that flat_column_sums<2, NV> gives for the second column of a
// two-column table, of that column alone (p[0 .. n), contiguous): the same
// additions in the same order.  There column 1 of row b goes to thread
// 2 (b mod NV/2) + 1, so here NV/2 threads hold the odd threads' sums and a
// group of 32 lanes stands for one of its waves.  Valid in every thread
// (sm: NV / 64 doubles).
template <int NV>
__device__ inline double flat_sum_odd(const double* __restrict__ p, long long n, double* sm) {
  constexpr int H = NV / 2;
  const int t = threadIdx.x;
  if (t < H) {
    double a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (long long f = t; f < n; f += 8LL * H) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = f + (long long)u * H < n ? p[f + (long long)u * H] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] += v[u];
    }
    double s = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
#pragma unroll
    for (int off = 16; off >= 1; off >>= 1) s += __shfl_down(s, off, 32);
    if ((t & 31) == 0) sm[t >> 5] = s;
  }
  __syncthreads();
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < H / 32; ++i) r += sm[i];
  __syncthreads();
  return r;
}

// The same sum of a short table (n <= 4 NV) by a workgroup of NT threads.
template <int NV, int NT>
__device__ inline double flat_sum_odd_short(const double* __restrict__ p, int n, double* sm) {
  constexpr int H = NV / 2, M = H / NT;
  static_assert(H % NT == 0, "each thread stands for M threads");
  const int t = threadIdx.x;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int f = t + m * NT + u * H;
      v[u] = f < n ? p[f] : 0.0;
    }
    double s = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    s = add_xor<1>(add_xor<2>(add_xor<4>(add_xor<8>(add_xor<16>(s)))));
    if ((t & 31) == 0) sm[(t >> 5) + m * (NT / 32)] = s;
  }
  __syncthreads();
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < H / 32; ++i) r += sm[i];
  return r;
}

}  // namespace apl
