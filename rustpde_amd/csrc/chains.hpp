// Recurrences along one parity chain of a row, held by one wavefront: lane l owns chain
// positions t in [t0, t0 + cnt), t0 = l * per, in registers v[q] (q = t - t0).  Each pass is
// a linear recurrence: the lane composes the affine map of its slice, the maps are scanned
// across the wavefront (wave.hpp), and each lane replays its slice with the reference's
// arithmetic from its incoming state (divisions by a diagonal taken as products with its
// tabulated reciprocal).  Used by the row kernels and the fused pressure stage.
#pragma once
#include <hip/hip_runtime.h>

#include "wave.hpp"

namespace rbc {
namespace chains {

constexpr int WAVE = 64;

// Workgroup barrier that orders LDS accesses only: the fences cover the local address
// space, so the wave's outstanding global loads (prefetched operands) and stores stay in
// flight across it (__syncthreads first waits for every outstanding global access of the
// wave).  For phases that exchange data between the threads of a workgroup through LDS
// only; data passed through global memory needs __syncthreads.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// padded LDS index of row element i (stored at pad(i + 2)): one pad double per 16
__host__ __device__ __forceinline__ int pad(int j) { return j + (j >> 4); }

// LDS doubles for a row of nr values with two guard zeros on each side
inline int buf_len(int nr) { return pad(nr + 6) + 1; }

// A row of nr values -> LDS (element i at pad(i + 2), zeros at i in [-2, 0) and
// [nr, nr + 4)) by the nthr threads of a group, thread tid; all loads are issued before the
// first store.  Needs MAXQ * nthr >= nr + 6.  The row's values lie INC apart.
template <int MAXQ, int INC = 1>
__device__ __forceinline__ void stage_row(double* buf, const double* __restrict__ row, bool valid, int nr, int tid,
                                          int nthr) {
  double v[MAXQ];
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int i = tid + q * nthr - 2;
    v[q] = (valid && i >= 0 && i < nr) ? row[i * INC] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int j = tid + q * nthr;
    if (j < nr + 6) buf[pad(j)] = v[q];
  }
}

// LDS row -> HBM: row[i] = x_i, or row[i] = x_i (-1) + row[i] with `subtract` (old values
// loaded first).  Needs MAXQ * nthr >= m.  The row's values lie INC apart.
template <int MAXQ, int INC = 1>
__device__ __forceinline__ void unstage_row(const double* buf, double* __restrict__ row, bool valid, int m, int tid,
                                            int nthr, bool subtract) {
#pragma clang fp contract(off)
  if (!valid) return;
  double old[MAXQ];
  if (subtract) {
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * nthr;
      old[q] = i < m ? row[i * INC] : 0.0;
    }
  }
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int i = tid + q * nthr;
    if (i < m) {
      const double x = buf[pad(i + 2)];
      row[i * INC] = subtract ? x * (-1.0) + old[q] : x;
    }
  }
}

// Every pass splits the lane's slice into a lower half L (q < H) and an upper half U
// (q >= H), H = SLICE / 2.  Their maps are composed side by side, the lane map is the
// composition of the two, and after the wavefront scan the entry state of the second half
// in the direction of the recurrence is the first half's map applied to the lane's entry
// state, so both halves are replayed side by side: two independent dependency chains per
// lane instead of one.

// Fdma forward elimination (fdma.rs:101-118): y_t = x_t - y_{t-1} lo_t (lo_t = low[i - 2]), of NR
// right-hand sides with the same multipliers
template <int SLICE, int NR>
__device__ __forceinline__ void fdma_forward(double (&v)[NR][SLICE], const double (&lo)[SLICE], int lane, int t0,
                                             int cnt) {
#pragma clang fp contract(off)
  static_assert(SLICE % 2 == 0, "two half slices");
  constexpr int H = SLICE / 2;
  double A1 = 1.0, A2 = 1.0, B1[NR] = {}, B2[NR] = {};  // half maps y_out = A y_in + B
#pragma unroll
  for (int j = 0; j < H; ++j) {
    if (j < cnt) {
      const bool start = t0 + j == 0;
      A1 = start ? 0.0 : -A1 * lo[j];
#pragma unroll
      for (int k = 0; k < NR; ++k) B1[k] = start ? v[k][j] : v[k][j] - B1[k] * lo[j];
    }
    const int q = H + j;
    if (q < cnt) {
      A2 = -A2 * lo[q];
#pragma unroll
      for (int k = 0; k < NR; ++k) B2[k] = v[k][q] - B2[k] * lo[q];
    }
  }
  double b[NR], y[NR];  // lane map
#pragma unroll
  for (int k = 0; k < NR; ++k) b[k] = A2 * B1[k] + B2[k];
  wave::scan_states<false>(A2 * A1, b, lane, y);
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    double y1 = y[k], y2 = A1 * y1 + B1[k];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      if (j < cnt) {
        y1 = (t0 + j == 0) ? v[k][j] : v[k][j] - y1 * lo[j];
        v[k][j] = y1;
      }
      const int q = H + j;
      if (q < cnt) {
        y2 = v[k][q] - y2 * lo[q];
        v[k][q] = y2;
      }
    }
  }
}

// Fdma back substitution: x_t = (y_t - x_{t+1} up1 - x_{t+2} up2) / dia over a chain of
// length len (g1, g2 zero where t + 1, t + 2 leave the chain).  rd holds 1 / dia: the
// division becomes a product with the tabulated reciprocal (one rounding apart).
using wave::Map2;  // s' = M s + w on the state s = (x_{t+1}, x_{t+2})
template <int SLICE, int NR>
__device__ __forceinline__ void fdma_backward(double (&v)[NR][SLICE], const double (&rd)[SLICE], const double (&g1)[SLICE],
                                              const double (&g2)[SLICE], int lane, int t0, int cnt, int len) {
#pragma clang fp contract(off)
  constexpr int H = SLICE / 2;
  Map2 h[2];  // lower and upper half, top-down: the upper first; their offsets per right-hand side
  double w[2][NR][2] = {};
  auto step = [&](int s, int q) {
    Map2& a = h[s];
    const double r = rd[q], c1 = -(g1[q] * r), c2 = -(g2[q] * r);
    const double n00 = c1 * a.m00 + c2 * a.m10, n01 = c1 * a.m01 + c2 * a.m11;
    a.m10 = a.m00;
    a.m11 = a.m01;
    a.m00 = n00;
    a.m01 = n01;
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const double n = c1 * w[s][k][0] + c2 * w[s][k][1] + v[k][q] * r;
      w[s][k][1] = w[s][k][0];
      w[s][k][0] = n;
    }
  };
#pragma unroll
  for (int j = H - 1; j >= 0; --j) {
    if (j < cnt) step(0, j);
    if (H + j < cnt) step(1, H + j);
  }
  const Map2 &L = h[0], &U = h[1];
  double b[NR][2], u[NR][2];
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    b[k][0] = __builtin_fma(L.m00, w[1][k][0], __builtin_fma(L.m01, w[1][k][1], w[0][k][0]));
    b[k][1] = __builtin_fma(L.m10, w[1][k][0], __builtin_fma(L.m11, w[1][k][1], w[0][k][1]));
  }
  wave::scan_states2(wave::compose(L, U), b, lane, u);
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    double u0 = u[k][0], u1 = u[k][1];
    double l0 = U.m00 * u0 + U.m01 * u1 + w[1][k][0], l1 = U.m10 * u0 + U.m11 * u1 + w[1][k][1];
#pragma unroll
    for (int j = H - 1; j >= 0; --j) {
      if (j < cnt) {
        const int t = t0 + j;
        double val = v[k][j];
        if (t + 1 < len) val = val - l0 * g1[j];
        if (t + 2 < len) val = val - l1 * g2[j];
        val = val * rd[j];
        l1 = l0;
        l0 = val;
        v[k][j] = val;
      }
      const int q = H + j;
      if (q < cnt) {
        const int t = t0 + q;
        double val = v[k][q];
        if (t + 1 < len) val = val - u0 * g1[q];
        if (t + 2 < len) val = val - u1 * g2[q];
        val = val * rd[q];
        u1 = u0;
        u0 = val;
        v[k][q] = val;
      }
    }
  }
}
// one right-hand side
template <int SLICE>
__device__ __forceinline__ void fdma_forward(double (&v)[SLICE], const double (&lo)[SLICE], int lane, int t0, int cnt) {
  fdma_forward(reinterpret_cast<double(&)[1][SLICE]>(v), lo, lane, t0, cnt);
}
template <int SLICE>
__device__ __forceinline__ void fdma_backward(double (&v)[SLICE], const double (&rd)[SLICE], const double (&g1)[SLICE],
                                              const double (&g2)[SLICE], int lane, int t0, int cnt, int len) {
  fdma_backward(reinterpret_cast<double(&)[1][SLICE]>(v), rd, g1, g2, lane, t0, cnt, len);
}

// tdma normal equations (linalg.rs:14-57), forward: g_i = (d_i - g_{i-2} off_{i-2}) / den_i,
// g_i = d_i / den_i at the chain start (of_q = off_{i-2}, rn_q = 1 / den_i: the divisions
// become products with the tabulated reciprocal)
template <int SLICE>
__device__ __forceinline__ void tdma_forward(double (&v)[SLICE], const double (&of)[SLICE], const double (&rn)[SLICE],
                                             int lane, int t0, int cnt) {
#pragma clang fp contract(off)
  constexpr int H = SLICE / 2;
  double A1 = 1.0, B1 = 0.0, A2 = 1.0, B2 = 0.0;
#pragma unroll
  for (int j = 0; j < H; ++j) {
    if (j < cnt) {
      if (t0 + j == 0) {
        A1 = 0.0;
        B1 = v[j] * rn[j];
      } else {
        A1 = -(of[j] * rn[j]) * A1;
        B1 = (v[j] - B1 * of[j]) * rn[j];
      }
    }
    const int q = H + j;
    if (q < cnt) {
      A2 = -(of[q] * rn[q]) * A2;
      B2 = (v[q] - B2 * of[q]) * rn[q];
    }
  }
  double b[1] = {A2 * B1 + B2}, y[1];
  wave::scan_states<false>(A2 * A1, b, lane, y);
  double g1v = y[0];
  double g2v = A1 * g1v + B1;
#pragma unroll
  for (int j = 0; j < H; ++j) {
    if (j < cnt) {
      g1v = (t0 + j == 0) ? v[j] * rn[j] : (v[j] - g1v * of[j]) * rn[j];
      v[j] = g1v;
    }
    const int q = H + j;
    if (q < cnt) {
      g2v = (v[q] - g2v * of[q]) * rn[q];
      v[q] = g2v;
    }
  }
}

// tdma back substitution: x_i = g_i for i >= m - 2, else x_i = g_i - x_{i+2} w_i (chain p)
template <int SLICE>
__device__ __forceinline__ void tdma_backward(double (&v)[SLICE], const double (&wv)[SLICE], int lane, int t0, int cnt,
                                              int p, int m) {
#pragma clang fp contract(off)
  constexpr int H = SLICE / 2;
  double A1 = 1.0, B1 = 0.0, A2 = 1.0, B2 = 0.0;  // L and U, top-down
#pragma unroll
  for (int j = H - 1; j >= 0; --j) {
    if (j < cnt) {
      if (p + 2 * (t0 + j) >= m - 2) {
        A1 = 0.0;
        B1 = v[j];
      } else {
        A1 = -wv[j] * A1;
        B1 = v[j] - B1 * wv[j];
      }
    }
    const int q = H + j;
    if (q < cnt) {
      if (p + 2 * (t0 + q) >= m - 2) {
        A2 = 0.0;
        B2 = v[q];
      } else {
        A2 = -wv[q] * A2;
        B2 = v[q] - B2 * wv[q];
      }
    }
  }
  double b[1] = {A1 * B2 + B1}, y[1];
  wave::scan_states<true>(A1 * A2, b, lane, y);
  double x2 = y[0];
  double x1 = A2 * x2 + B2;
#pragma unroll
  for (int j = H - 1; j >= 0; --j) {
    if (j < cnt) {
      x1 = (p + 2 * (t0 + j) >= m - 2) ? v[j] : v[j] - x1 * wv[j];
      v[j] = x1;
    }
    const int q = H + j;
    if (q < cnt) {
      x2 = (p + 2 * (t0 + q) >= m - 2) ? v[q] : v[q] - x2 * wv[q];
      v[q] = x2;
    }
  }
}

// The two tdma passes for two right-hand sides with the same tables at once (the x and y
// projections of the pressure stage): the maps' multipliers depend on the tables only, so
// they are composed and scanned once; each right-hand side keeps its own offset.  Every
// value is formed as by tdma_forward / tdma_backward.
template <int SLICE>
__device__ __forceinline__ void tdma_forward2(double (&v)[SLICE], double (&u)[SLICE], const double (&of)[SLICE],
                                              const double (&rn)[SLICE], int lane, int t0, int cnt) {
#pragma clang fp contract(off)
  constexpr int H = SLICE / 2;
  double A1 = 1.0, B1 = 0.0, C1 = 0.0, A2 = 1.0, B2 = 0.0, C2 = 0.0;
#pragma unroll
  for (int j = 0; j < H; ++j) {
    if (j < cnt) {
      if (t0 + j == 0) {
        A1 = 0.0;
        B1 = v[j] * rn[j];
        C1 = u[j] * rn[j];
      } else {
        A1 = -(of[j] * rn[j]) * A1;
        B1 = (v[j] - B1 * of[j]) * rn[j];
        C1 = (u[j] - C1 * of[j]) * rn[j];
      }
    }
    const int q = H + j;
    if (q < cnt) {
      A2 = -(of[q] * rn[q]) * A2;
      B2 = (v[q] - B2 * of[q]) * rn[q];
      C2 = (u[q] - C2 * of[q]) * rn[q];
    }
  }
  double b[2] = {A2 * B1 + B2, A2 * C1 + C2}, y[2];
  wave::scan_states<false>(A2 * A1, b, lane, y);
  double g1v = y[0], h1v = y[1];
  double g2v = A1 * g1v + B1, h2v = A1 * h1v + C1;
#pragma unroll
  for (int j = 0; j < H; ++j) {
    if (j < cnt) {
      g1v = (t0 + j == 0) ? v[j] * rn[j] : (v[j] - g1v * of[j]) * rn[j];
      h1v = (t0 + j == 0) ? u[j] * rn[j] : (u[j] - h1v * of[j]) * rn[j];
      v[j] = g1v;
      u[j] = h1v;
    }
    const int q = H + j;
    if (q < cnt) {
      g2v = (v[q] - g2v * of[q]) * rn[q];
      h2v = (u[q] - h2v * of[q]) * rn[q];
      v[q] = g2v;
      u[q] = h2v;
    }
  }
}

template <int SLICE>
__device__ __forceinline__ void tdma_backward2(double (&v)[SLICE], double (&u)[SLICE], const double (&wv)[SLICE],
                                               int lane, int t0, int cnt, int p, int m) {
#pragma clang fp contract(off)
  constexpr int H = SLICE / 2;
  double A1 = 1.0, B1 = 0.0, C1 = 0.0, A2 = 1.0, B2 = 0.0, C2 = 0.0;  // L and U, top-down
#pragma unroll
  for (int j = H - 1; j >= 0; --j) {
    if (j < cnt) {
      if (p + 2 * (t0 + j) >= m - 2) {
        A1 = 0.0;
        B1 = v[j];
        C1 = u[j];
      } else {
        A1 = -wv[j] * A1;
        B1 = v[j] - B1 * wv[j];
        C1 = u[j] - C1 * wv[j];
      }
    }
    const int q = H + j;
    if (q < cnt) {
      if (p + 2 * (t0 + q) >= m - 2) {
        A2 = 0.0;
        B2 = v[q];
        C2 = u[q];
      } else {
        A2 = -wv[q] * A2;
        B2 = v[q] - B2 * wv[q];
        C2 = u[q] - C2 * wv[q];
      }
    }
  }
  double b[2] = {A1 * B2 + B1, A1 * C2 + C1}, y[2];
  wave::scan_states<true>(A1 * A2, b, lane, y);
  double x2 = y[0], y2 = y[1];
  double x1 = A2 * x2 + B2, y1 = A2 * y2 + C2;
#pragma unroll
  for (int j = H - 1; j >= 0; --j) {
    if (j < cnt) {
      const bool top = p + 2 * (t0 + j) >= m - 2;
      x1 = top ? v[j] : v[j] - x1 * wv[j];
      y1 = top ? u[j] : u[j] - y1 * wv[j];
      v[j] = x1;
      u[j] = y1;
    }
    const int q = H + j;
    if (q < cnt) {
      const bool top = p + 2 * (t0 + q) >= m - 2;
      x2 = top ? v[q] : v[q] - x2 * wv[q];
      y2 = top ? u[q] : u[q] - y2 * wv[q];
      v[q] = x2;
      u[q] = y2;
    }
  }
}

// suffix sums along the chain: v_t <- v_t + v_{t+1} + ... (the derivative recurrence
// d_i = g_i + d_{i+2} of ortho.rs:107-125, summed from the top as the reference does)
template <int SLICE>
__device__ __forceinline__ void suffix_sum(double (&v)[SLICE], int lane, int cnt) {
#pragma clang fp contract(off)
  constexpr int H = SLICE / 2;
  double t1 = 0.0, t2 = 0.0;
#pragma unroll
  for (int j = H - 1; j >= 0; --j) {
    if (j < cnt) t1 = v[j] + t1;
    if (H + j < cnt) t2 = v[H + j] + t2;
  }
  double a2;
  wave::suffix_sum(t1 + t2, lane, a2);
  double a1 = t2 + a2;
#pragma unroll
  for (int j = H - 1; j >= 0; --j) {
    if (j < cnt) {
      a1 = v[j] + a1;
      v[j] = a1;
    }
    if (H + j < cnt) {
      a2 = v[H + j] + a2;
      v[H + j] = a2;
    }
  }
}

}  // namespace chains
}  // namespace rbc
