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

}  // namespace rowdiff
}  // namespace rbc
