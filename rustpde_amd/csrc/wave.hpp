// Cross-lane sums and scans of affine maps inside one wavefront through DPP moves and lane reads: no LDS round trip.
#pragma once
#include <hip/hip_runtime.h>

namespace rbc {
namespace wave {

// DPP controls (GFX9 encoding): row_shl:n moves lane l + n of the lane's row of 16 into
// lane l (lanes whose source leaves the row keep the 0 given as `old`); wave_shl:1 moves
// lane l + 1 of the wavefront (lane 63 keeps the 0)
// (row_shr:n: lane l - n)
constexpr int ROW_SHL = 0x100, ROW_SHR = 0x110, WAVE_SHL1 = 0x130;

template <int CTRL, typename V>
__device__ __forceinline__ V dpp(V x) {
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(V, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
  } else {
    const long long u = __builtin_bit_cast(long long, x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(V, ((long long)hi << 32) | (unsigned)lo);
  }
}

// the same, lanes whose source leaves the row keep `old`
template <int CTRL>
__device__ __forceinline__ double dpp_or(double x, double old) {
  const long long u = __builtin_bit_cast(long long, x), o = __builtin_bit_cast(long long, old);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)u, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(u >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

template <typename V>
__device__ __forceinline__ V lane_value(V x, int l) {
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(V, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
  } else {
    const long long u = __builtin_bit_cast(long long, x);
    const int lo = __builtin_amdgcn_readlane((int)u, l), hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
    return __builtin_bit_cast(V, ((long long)hi << 32) | (unsigned)lo);
  }
}

// inclusive suffix sums over the 64 lanes, s_l = x_l + x_{l+1} + ... + x_63: suffix sums
// inside each row of 16 (steps 1, 2, 4, 8), then the totals of the rows above (read from
// their first lanes) added per row; excl receives s_{l+1} (0 for lane 63)
template <typename V>
__device__ __forceinline__ V suffix_sum(V x, int lane, V& excl) {
  x = x + dpp<ROW_SHL + 1>(x);
  x = x + dpp<ROW_SHL + 2>(x);
  x = x + dpp<ROW_SHL + 4>(x);
  x = x + dpp<ROW_SHL + 8>(x);
  const V t1 = lane_value(x, 16), t2 = lane_value(x, 32), t3 = lane_value(x, 48);
  const V s2 = t2 + t3, s1 = t1 + s2;
  const int row = lane >> 4;
  const V above = row == 0 ? s1 : row == 1 ? s2 : row == 2 ? t3 : (V)0;
  x = x + above;
  excl = dpp<WAVE_SHL1>(x);
  return x;
}

// Scans of the lanes' affine maps y_out = a y_in + b_j, j < NB, on a state that is zero before the first
// lane: composed inside each row of 16 in four steps, the rows' entry states then follow in turn from the
// row totals (lane reads), and each lane's from its row's.  y_j receives the lane's entry state.  (Against
// six steps of LDS permutes over the whole wavefront, and with two entries a lane for rows up to 258 in
// place of four: 256 x 257, pressure rows 13.7 -> 9.8 us, row solves of three fields 7.3 -> 4.9; with
// eight entries a lane, 1024 x 1025, 40.9 -> 38.1 and 21.7 -> 20.0.)
template <bool DOWN, int N, int NB>
__device__ __forceinline__ void scan_step(double& a, double (&b)[NB]) {
  constexpr int CTRL = (DOWN ? ROW_SHL : ROW_SHR) + N;
  const double q = dpp_or<CTRL>(a, 1.0);
#pragma unroll
  for (int j = 0; j < NB; ++j) b[j] = __builtin_fma(a, dpp_or<CTRL>(b[j], 0.0), b[j]);
  a = a * q;
}
// DOWN: from the last lane to the first
template <bool DOWN, int NB>
__device__ __forceinline__ void scan_states(double a, double (&b)[NB], int lane, double (&y)[NB]) {
  scan_step<DOWN, 1>(a, b);
  scan_step<DOWN, 2>(a, b);
  scan_step<DOWN, 4>(a, b);
  scan_step<DOWN, 8>(a, b);
  constexpr int L0 = DOWN ? 48 : 15, L1 = DOWN ? 32 : 31, L2 = DOWN ? 16 : 47;  // row totals, first to last
  constexpr int CTRL = (DOWN ? ROW_SHL : ROW_SHR) + 1;
  const double a1 = lane_value(a, L1), a2 = lane_value(a, L2), e = dpp_or<CTRL>(a, 1.0);
  const int row = DOWN ? 3 - (lane >> 4) : lane >> 4;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const double s1 = lane_value(b[j], L0), s2 = __builtin_fma(a1, s1, lane_value(b[j], L1)),
                 s3 = __builtin_fma(a2, s2, lane_value(b[j], L2));
    const double s = row == 0 ? 0.0 : row == 1 ? s1 : row == 2 ? s2 : s3;
    y[j] = __builtin_fma(e, s, dpp_or<CTRL>(b[j], 0.0));
  }
}

// The same from the last lane to the first for maps of a state of two values, s' = M s + w
struct Map2 {
  double m00 = 1.0, m01 = 0.0, m10 = 0.0, m11 = 1.0, w0 = 0.0, w1 = 0.0;
};
// a after b: M = M_a M_b, w = M_a w_b + w_a
__device__ __forceinline__ Map2 compose(const Map2& a, const Map2& b) {
  Map2 c;
  c.m00 = __builtin_fma(a.m00, b.m00, a.m01 * b.m10);
  c.m01 = __builtin_fma(a.m00, b.m01, a.m01 * b.m11);
  c.m10 = __builtin_fma(a.m10, b.m00, a.m11 * b.m10);
  c.m11 = __builtin_fma(a.m10, b.m01, a.m11 * b.m11);
  c.w0 = __builtin_fma(a.m00, b.w0, __builtin_fma(a.m01, b.w1, a.w0));
  c.w1 = __builtin_fma(a.m10, b.w0, __builtin_fma(a.m11, b.w1, a.w1));
  return c;
}
// The scan for NB right-hand sides with the same matrices (a's own w is not used): w_j the lane's offsets,
// u_j its entry states
template <int CTRL, int NB>
__device__ __forceinline__ void scan_step2(Map2& a, double (&w)[NB][2]) {
  Map2 q = a;
  q.m00 = dpp_or<CTRL>(a.m00, 1.0);
  q.m01 = dpp_or<CTRL>(a.m01, 0.0);
  q.m10 = dpp_or<CTRL>(a.m10, 0.0);
  q.m11 = dpp_or<CTRL>(a.m11, 1.0);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const double q0 = dpp_or<CTRL>(w[j][0], 0.0), q1 = dpp_or<CTRL>(w[j][1], 0.0);
    w[j][0] = __builtin_fma(a.m00, q0, __builtin_fma(a.m01, q1, w[j][0]));
    w[j][1] = __builtin_fma(a.m10, q0, __builtin_fma(a.m11, q1, w[j][1]));
  }
  const Map2 c = compose(a, q);
  a.m00 = c.m00;
  a.m01 = c.m01;
  a.m10 = c.m10;
  a.m11 = c.m11;
}
template <int NB>
__device__ __forceinline__ void scan_states2(Map2 a, double (&w)[NB][2], int lane, double (&u)[NB][2]) {
  scan_step2<ROW_SHL + 1>(a, w);
  scan_step2<ROW_SHL + 2>(a, w);
  scan_step2<ROW_SHL + 4>(a, w);
  scan_step2<ROW_SHL + 8>(a, w);
  const int row = 3 - (lane >> 4);
  const double x00 = dpp_or<ROW_SHL + 1>(a.m00, 1.0), x01 = dpp_or<ROW_SHL + 1>(a.m01, 0.0);
  const double x10 = dpp_or<ROW_SHL + 1>(a.m10, 0.0), x11 = dpp_or<ROW_SHL + 1>(a.m11, 1.0);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    double s0[4], s1[4];  // entry states of rows 3, 2, 1, 0
    s0[0] = s1[0] = 0.0;
    s0[1] = lane_value(w[j][0], 48);
    s1[1] = lane_value(w[j][1], 48);
#pragma unroll
    for (int r = 2; r < 4; ++r) {
      const int l = 64 - 16 * r;
      s0[r] = __builtin_fma(lane_value(a.m00, l), s0[r - 1], __builtin_fma(lane_value(a.m01, l), s1[r - 1], lane_value(w[j][0], l)));
      s1[r] = __builtin_fma(lane_value(a.m10, l), s0[r - 1], __builtin_fma(lane_value(a.m11, l), s1[r - 1], lane_value(w[j][1], l)));
    }
    const double e0 = row == 0 ? 0.0 : row == 1 ? s0[1] : row == 2 ? s0[2] : s0[3];
    const double e1 = row == 0 ? 0.0 : row == 1 ? s1[1] : row == 2 ? s1[2] : s1[3];
    u[j][0] = __builtin_fma(x00, e0, __builtin_fma(x01, e1, dpp_or<ROW_SHL + 1>(w[j][0], 0.0)));
    u[j][1] = __builtin_fma(x10, e0, __builtin_fma(x11, e1, dpp_or<ROW_SHL + 1>(w[j][1], 0.0)));
  }
}
__device__ __forceinline__ void scan_states2(Map2 a, int lane, double& u0, double& u1) {
  double w[1][2] = {{a.w0, a.w1}}, u[1][2];
  scan_states2(a, w, lane, u);
  u0 = u[0][0];
  u1 = u[0][1];
}

}  // namespace wave
}  // namespace rbc
