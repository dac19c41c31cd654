// d/dy of a Chebyshev row held in LDS (ortho.rs:107-125): d_i = w_i + d_{i+2}, w_i = 2 (i+1) c_{i+1},
// d_0 = c_1 + d_2 / 2, a suffix sum along each parity chain, one wavefront per chain.
#pragma once
#include <hip/hip_runtime.h>

#include "chains.hpp"
#include "wave.hpp"

namespace rbc {
namespace rowdiff {

// buf: element i at pad(i + 2), zeros beyond the n values; p: the wavefront's chain, per its slice
// length.  Every thread of the block must call it (it holds barriers); buf receives the derivative.
template <int SLICE>
__device__ __forceinline__ void derive(double* buf, int n, int per, int lane, int p) {
#pragma clang fp contract(off)
  using chains::pad;
  const int len = p == 0 ? (n + 1) / 2 : n / 2;
  const int t0 = lane * per, cnt = max(0, min(per, len - t0));
  double v[SLICE], s = 0.0;
#pragma unroll
  for (int q = SLICE - 1; q >= 0; --q) {
    const int i = p + 2 * (t0 + q);
    v[q] = q < cnt ? (i == 0 ? buf[pad(3)] : 2.0 * (double)(i + 1) * buf[pad(i + 3)]) : 0.0;
    if (i > 0) s = s + v[q];
  }
  double above;
  wave::suffix_sum(s, lane, above);
#pragma unroll
  for (int q = SLICE - 1; q >= 0; --q) {
    if (q < cnt) {
      above = (p == 0 && t0 + q == 0) ? v[q] + above / 2.0 : v[q] + above;
      v[q] = above;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < SLICE; ++q)
    if (q < cnt) buf[pad(p + 2 * (t0 + q) + 2)] = v[q];
  __syncthreads();
}

// The same of a composite row, buf holding its n - 2 coefficients u of phi_k = T_k + l_k T_{k+2} (zeros
// beyond), low the l_k: phi_k' = a_k T_{k+1} + b_k (T_{k-1} + T_{k-3} + ..) with a_k = 2 (k + 2) l_k and
// b_k = 2 k + a_k, so d_i = a_{i-1} u_{i-1} + sum_{k > i, k - i odd} b_k u_k, at i = 0 half the sum.  The sum over
// the stencil's results, derive() of to_ortho, cancels their leading parts (b_k is -4 for Dirichlet, their
// weights 2 k), and rounds that much worse.
template <int SLICE>
__device__ __forceinline__ void derive_composite(double* buf, const double* __restrict__ low, int n, int per, int lane,
                                                 int p) {
#pragma clang fp contract(off)
  using chains::pad;
  const int len = p == 0 ? (n + 1) / 2 : n / 2, m = n - 2;
  const int t0 = lane * per, cnt = max(0, min(per, len - t0));
  double v[SLICE], own[SLICE], s = 0.0;
#pragma unroll
  for (int q = SLICE - 1; q >= 0; --q) {
    const int i = p + 2 * (t0 + q), k = i + 1, j = i - 1;
    v[q] = own[q] = 0.0;
    if (q < cnt && k < m) v[q] = __builtin_fma(2.0 * (double)(k + 2), low[k], 2.0 * (double)k) * buf[pad(k + 2)];
    if (q < cnt && j >= 0 && j < m) own[q] = 2.0 * (double)(j + 2) * low[j] * buf[pad(j + 2)];
    if (i > 0) s = s + v[q];
  }
  double above;
  wave::suffix_sum(s, lane, above);
#pragma unroll
  for (int q = SLICE - 1; q >= 0; --q) {
    if (q < cnt) {
      above = v[q] + above;
      v[q] = (p == 0 && t0 + q == 0) ? above / 2.0 : own[q] + above;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < SLICE; ++q)
    if (q < cnt) buf[pad(p + 2 * (t0 + q) + 2)] = v[q];
  __syncthreads();
}

// d2/dy2 of a composite row: T_k'' = sum_{i <= k - 2, k - i even} k (k^2 - i^2) T_i, half of it at i = 0, so
// e_i = c_i u_i + sum_{k > i, k - i even} (A_k - i^2 B_k) u_k, c_i = 4 (i + 1) (i + 2) l_i, A_k = k^3 + l_k (k + 2)^3,
// B_k = k + l_k (k + 2): two suffix sums along the row's own chain.  All terms of a Neumann row have one sign,
// of a Dirichlet row the first sum outweighs the other.  257 coefficients that fall off as k^-2, rounding
// against 64 bits: 2e-16; derive() twice of to_ortho 3e-15 (Dirichlet) and 6.6e-15, a dense product 3e-16.
template <int SLICE>
__device__ __forceinline__ void derive2_composite(double* buf, const double* __restrict__ low, int n, int per, int lane,
                                                  int p) {
#pragma clang fp contract(off)
  using chains::pad;
  const int len = p == 0 ? (n + 1) / 2 : n / 2, m = n - 2;
  const int t0 = lane * per, cnt = max(0, min(per, len - t0));
  double a[SLICE], b[SLICE], own[SLICE], sa = 0.0, sb = 0.0;
#pragma unroll
  for (int q = SLICE - 1; q >= 0; --q) {
    const int i = p + 2 * (t0 + q);
    a[q] = b[q] = own[q] = 0.0;
    if (q < cnt && i < m) {
      const double u = buf[pad(i + 2)], l = low[i], k = (double)i, k2 = (double)(i + 2);
      own[q] = 4.0 * (k + 1.0) * k2 * l * u;
      a[q] = __builtin_fma(l, k2 * k2 * k2, k * k * k) * u;
      b[q] = __builtin_fma(l, k2, k) * u;
    }
    sa = sa + a[q];
    sb = sb + b[q];
  }
  double abovea, aboveb;
  wave::suffix_sum(sa, lane, abovea);
  wave::suffix_sum(sb, lane, aboveb);
#pragma unroll
  for (int q = SLICE - 1; q >= 0; --q) {
    const double i = (double)(p + 2 * (t0 + q));
    const double e = own[q] + __builtin_fma(-(i * i), aboveb, abovea);
    abovea = a[q] + abovea;
    aboveb = b[q] + aboveb;
    a[q] = i == 0.0 ? e / 2.0 : e;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < SLICE; ++q)
    if (q < cnt) buf[pad(p + 2 * (t0 + q) + 2)] = a[q];
  __syncthreads();
}

}  // namespace rowdiff
}  // namespace rbc
