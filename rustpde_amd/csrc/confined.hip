// Row kernels of the confined step (Chebyshev x Chebyshev), one block per row and instance: what
// lies between the dense products along x and acts along y or point by point.  Each replaces two
// to four launches (stencil passes, derivative, element-wise sums): at 64^2, where a launch takes
// 2 us or more whatever it does, that is what they are for; at 257^2 they also save the passes
// over memory in between.
//   rhs_rows   the right-hand sides of ux, uy, temp (navier.rs:622-674): to_ortho of the field, the
//              pressure gradient (d/dy formed here), buoyancy, convective terms, boundary terms
//   div_rows   d/dx ux + d/dy uy (navier.rs:698-703) from d/dx ux in x-ortho space
//   proj_rows  the projection of ux and uy (navier.rs:683-695) from the x parts of the pseudo
//              pressure's gradient, and the pressure update (navier.rs:717-721) in further blocks
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

#include "chains.hpp"
#include "ops.hpp"
#include "rowdiff.hpp"

namespace rbc {

namespace {

using chains::buf_len;
using chains::pad;
using chains::WAVE;
constexpr int NT = 2 * WAVE;  // threads of a block: two parity chains

void check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// to_ortho along x of coefficient j of a field: rows r and r - 2 of q [mx, ld] (taps cx[n rows][2])
__device__ __forceinline__ double x_taps(const double* __restrict__ q, int ld, int mx, int r, int j, double c0,
                                         double c1) {
#pragma clang fp contract(off)
  const double a = q[(size_t)min(r, mx - 1) * ld + j], b = q[(size_t)max(r - 2, 0) * ld + j];
  return (r < mx ? a * c0 : 0.0) + (r >= 2 ? b * c1 : 0.0);
}
// to_ortho along both axes at (r, i): the x stencil first, then taps i and i - 2 along y
__device__ __forceinline__ double xy_taps(const double* __restrict__ q, int mx, int my, int r, int i, double cx0,
                                          double cx1, double cy0, double cy1) {
#pragma clang fp contract(off)
  const double v0 = x_taps(q, my, mx, r, min(i, my - 1), cx0, cx1);
  const double v2 = x_taps(q, my, mx, r, max(i - 2, 0), cx0, cx1);
  return (i < my ? v0 * cy0 : 0.0) + (i >= 2 ? v2 * cy1 : 0.0);
}

// one block per row and field: 128 x 129 3.5 us, 257 x 257 6.5 (5.7 and 8.6 with the three fields of a row
// in one block, two wavefronts a CU)
template <int SLICE>
__global__ __launch_bounds__(NT) void rhs_rows_kernel(ConfinedRows a, int per) {
#pragma clang fp contract(off)
  extern __shared__ double buf[];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), p = tid / WAVE;
  const int r = blockIdx.x, n = a.ny, f = a.f0 + blockIdx.z;
  const long o = a.stride * blockIdx.y, at = o + (long)r * n;
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + NT - 1) / NT;
  const double* U = a.U + f * a.field + o;
  double* out = a.RHS + f * a.field + at;
  const double* cv = a.CV + f * a.field + at;
  const double x0 = f == 2 ? a.sxt[r] : a.sxu[r], x1 = f == 2 ? a.sxt[a.nx + r] : a.sxu[a.nx + r];
  if (f == 1) {  // d/dy pres, buoyancy
    chains::stage_row<MAXQ>(buf, a.P0 + at, true, n, tid, NT);
    const double xt0 = a.sxt[r], xt1 = a.sxt[a.nx + r];
    double v[MAXQ], t[MAXQ];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * NT;
      v[q] = t[q] = 0.0;
      if (i >= n) continue;
      const double cy0 = a.sy[i], cy1 = a.sy[n + i];
      v[q] = xy_taps(U, a.mx, a.my, r, i, x0, x1, cy0, cy1);
      t[q] = xy_taps(a.U + 2 * a.field + o, a.mx, a.my, r, i, xt0, xt1, cy0, cy1) + a.that_bc[at + i];
    }
    __syncthreads();
    rowdiff::derive<SLICE>(buf, n, per, lane, p);
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * NT;
      if (i >= n) continue;
      double w = v[q] - (buf[pad(i + 2)] * a.inv_scy) * a.dt;
      w = w + t[q] * a.dt;
      out[i] = w - cv[i] * a.dt;
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int i = tid + q * NT;
    if (i >= n) continue;
    const double u = xy_taps(U, a.mx, a.my, r, i, x0, x1, a.sy[i], a.sy[n + i]);
    const double w = f == 0 ? u - a.G[at + i] * a.dt : (u + a.gxx[at + i]) + a.gyy[at + i];
    out[i] = w - cv[i] * a.dt;
  }
}

template <int SLICE>
__global__ __launch_bounds__(NT) void div_rows_kernel(ConfinedRows a, int per) {
#pragma clang fp contract(off)
  extern __shared__ double buf[];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), p = tid / WAVE;
  const int r = blockIdx.x, n = a.ny, my = a.my;
  const long o = a.stride * blockIdx.y;
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + NT - 1) / NT;
  const double x0 = a.sxu[r], x1 = a.sxu[a.nx + r];
  const double* uy = a.U + a.field + o;
  const double* tx = a.TX + o + (long)r * my;
  double v[MAXQ], w[MAXQ];
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {  // uy in ortho space; the x part's taps along y beside it
    const int i = tid + q * NT;
    v[q] = w[q] = 0.0;
    if (i < n) {
      const double cy0 = a.sy[i], cy1 = a.sy[n + i];
      v[q] = xy_taps(uy, a.mx, my, r, i, x0, x1, cy0, cy1);
      w[q] = (i < my ? tx[min(i, my - 1)] * cy0 : 0.0) + (i >= 2 ? tx[i - 2] * cy1 : 0.0);
    }
  }
  if (tid < 2) buf[pad(tid)] = 0.0;
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int j = tid + q * NT + 2;
    if (j < n + 6) buf[pad(j)] = v[q];
  }
  __syncthreads();
  rowdiff::derive<SLICE>(buf, n, per, lane, p);
  double* out = a.DIV + o + (long)r * n;
  double sum = 0.0;
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int i = tid + q * NT;
    if (i >= n) continue;
    const double d = buf[pad(i + 2)] * a.inv_scy + w[q];
    if (a.norm) sum += d * d;
    else out[i] = d;
  }
  if (!a.norm) return;
  // the sum of squares instead: the rows' sums are added by the last block to arrive, which leaves the
  // counter at zero
  __shared__ double red[NT];
  __shared__ bool last;
  auto add = [&](double v) {
    red[tid] = v;
    __syncthreads();
    for (int h = NT / 2; h > 0; h >>= 1) {
      if (tid < h) red[tid] += red[tid + h];
      __syncthreads();
    }
  };
  add(sum);
  unsigned* count = reinterpret_cast<unsigned*>(a.part);
  if (tid == 0) {
    __hip_atomic_store(a.part + 1 + r, red[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  sum = 0.0;
  for (int i = tid; i < (int)gridDim.x; i += NT)
    sum += __hip_atomic_load(a.part + 1 + i, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
  add(sum);
  if (tid == 0) {
    *a.norm = red[0];
    __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// blocks [0, f mx): row r of ux (f = 0) and uy (f = 1); then nx blocks of pressure rows
template <int SLICE>
__global__ __launch_bounds__(NT) void proj_rows_kernel(ConfinedRows a, int per_n, int per) {
#pragma clang fp contract(off)
  extern __shared__ double buf[];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), p = tid / WAVE;
  const int n = a.ny, m = a.my, b = blockIdx.x, nf = a.f1 - a.f0;
  const long o = a.stride * blockIdx.y;
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + NT - 1) / NT;
  if (b >= nf * a.mx) {  // pres = (pres - nu div) + to_ortho(pseu) / dt
    const int r = b - nf * a.mx;
    const double nu = a.nuarr ? a.nuarr[blockIdx.y] : a.nu;
    const double x0 = a.sxp[r], x1 = a.sxp[a.nx + r];
    for (int i = tid; i < n; i += NT) {
      const double phi = xy_taps(a.P1 + o, a.mx, m, r, i, x0, x1, a.syp[i], a.syp[n + i]);
      const long j = o + (long)r * n + i;
      const double q = a.P0[j] - a.DIV[j] * nu;
      a.P0[j] = q + phi * a.inv_dt;
    }
    return;
  }
  const int f = a.f0 + b / a.mx, r = b % a.mx;
  const double* g = (f == 0 ? a.GA : a.GB) + o + (long)r * m;
  double v[MAXQ];
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int i = tid + q * NT;
    v[q] = 0.0;
    if (i < n) v[q] = (i < m ? g[min(i, m - 1)] * a.syp[i] : 0.0) + (i >= 2 ? g[i - 2] * a.syp[n + i] : 0.0);
  }
  if (tid < 2) buf[pad(tid)] = 0.0;
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int j = tid + q * NT + 2;
    if (j < n + 6) buf[pad(j)] = v[q];
  }
  __syncthreads();
  if (f == 1) {
    rowdiff::derive<SLICE>(buf, n, per_n, lane, p);
    if (a.inv_scy != 1.0) {
      for (int i = tid; i < n; i += NT) buf[pad(i + 2)] = buf[pad(i + 2)] * a.inv_scy;
      __syncthreads();
    }
  }
  // from_ortho along y, the recurrences of tdma_rows_lds
  const int len = p == 0 ? (m + 1) / 2 : m / 2;
  const int t0 = lane * per, cnt = max(0, min(per, len - t0));
  double x[SLICE], c0[SLICE], c1[SLICE];
#define TB(k, q) a.tdma[((size_t)((k) * 2 + p) * per + (q)) * WAVE + lane]
#pragma unroll
  for (int q = 0; q < SLICE; ++q) {
    c0[q] = TB(0, q);
    c1[q] = TB(1, q);
  }
#pragma unroll
  for (int q = 0; q < SLICE; ++q) {
    const int j = p + 2 * (t0 + q) + 2;
    x[q] = q < cnt ? buf[pad(j)] * c0[q] + buf[pad(j + 2)] * c1[q] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < SLICE; ++q) {
    c0[q] = TB(2, q);
    c1[q] = TB(3, q);
  }
  chains::tdma_forward(x, c0, c1, lane, t0, cnt);
#pragma unroll
  for (int q = 0; q < SLICE; ++q) c0[q] = TB(4, q);
#undef TB
  chains::tdma_backward(x, c0, lane, t0, cnt, p, m);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < SLICE; ++q)
    if (q < cnt) buf[pad(p + 2 * (t0 + q) + 2)] = x[q];
  __syncthreads();
  chains::unstage_row<MAXQ>(buf, const_cast<double*>(a.U) + f * a.field + o + (long)r * m, true, m, tid, NT, true);
}

// One block per row and field (blockIdx.y).  PER: rows are split planes of a Fourier x axis.  The row's
// derivatives along y (the residual twice, for uy also pres once) run as suffix sums in LDS.
template <int SLICE, bool PER>
__global__ __launch_bounds__(NT) void adjoint_rows_kernel(AdjointRows a) {
#pragma clang fp contract(off)
  extern __shared__ double buf[];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), p = tid / WAVE;
  const int r = blockIdx.x, f = blockIdx.y, n = a.ny, m = a.my, nx = a.rows;
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + NT - 1) / NT;
  const double* sx = f == 2 ? a.sxt : a.sxu;
  const double x0 = PER ? 1.0 : sx[r], x1 = PER ? 0.0 : sx[nx + r];
  const double bx0 = PER ? 1.0 : a.sxu[r], bx1 = PER ? 0.0 : a.sxu[nx + r];  // uy's taps for the buoyancy
  const bool im = PER && r >= a.mx;
  const double kk = PER ? (double)(im ? r - a.mx : r) / a.kscale : 0.0;
  // to_ortho of a spectral field at (r, i)
  auto taps = [&](const double* q, int i, double c0, double c1, double cy0, double cy1) {
    if constexpr (PER) {
      const double* row = q + (long)r * m;
      return (i < m ? row[min(i, m - 1)] * cy0 : 0.0) + (i >= 2 ? row[i - 2] * cy1 : 0.0);
    } else {
      return xy_taps(q, a.mx, m, r, i, c0, c1, cy0, cy1);
    }
  };
  const double* F = a.F + f * a.field;
  double s[MAXQ], gp[MAXQ];
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {  // the residual in ortho space
    const int i = tid + q * NT;
    s[q] = gp[q] = 0.0;
    if (i < n) s[q] = taps(F, i, x0, x1, a.sy[i], a.sy[n + i]);
  }
  if (f == 1) {  // d/dy pres
    chains::stage_row<MAXQ>(buf, a.P0 + (long)r * n, true, n, tid, NT);
    __syncthreads();
    rowdiff::derive<SLICE>(buf, n, a.per, lane, p);
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * NT;
      if (i < n) gp[q] = buf[pad(i + 2)] * a.inv_scy;
    }
    __syncthreads();
  } else if (f == 0) {
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * NT;
      if (i >= n) continue;
      if constexpr (PER) gp[q] = (im ? a.P0[(long)(r - a.mx) * n + i] : -a.P0[(long)(r + a.mx) * n + i]) * kk;
      else gp[q] = a.GX[(long)r * n + i];
    }
  }
  if (tid < 2) buf[pad(tid)] = 0.0;
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int j = tid + q * NT + 2;
    if (j < n + 6) buf[pad(j)] = s[q];
  }
  __syncthreads();
  rowdiff::derive<SLICE>(buf, n, a.per, lane, p);
  rowdiff::derive<SLICE>(buf, n, a.per, lane, p);
  const double k = f == 2 ? a.ka : a.nu;
#pragma unroll
  for (int q = 0; q < MAXQ; ++q) {
    const int i = tid + q * NT;
    if (i >= n) continue;
    const double cy0 = a.sy[i], cy1 = a.sy[n + i];
    const long j = f * a.field + (long)r * n + i;
    double lx;
    if constexpr (PER) {
      lx = -(kk * kk) * s[q];
    } else {
      const double* row = a.LX + f * a.field + (long)r * m;
      lx = (i < m ? row[min(i, m - 1)] * cy0 : 0.0) + (i >= 2 ? row[i - 2] * cy1 : 0.0);
    }
    const double ly = (buf[pad(i + 2)] * a.inv_scy) * a.inv_scy;
    double v = taps(a.U + f * a.field, i, x0, x1, cy0, cy1);
    if (f < 2) v = v - gp[q] * a.dt;
    v = v + a.CV[j] * a.dt;
    if (f == 2) v = v + taps(a.F + a.field, i, bx0, bx1, cy0, cy1) * a.dt;
    v = v + (lx * a.dt) * k;
    a.RHS[j] = v + (ly * a.dt) * k;
  }
}

}  // namespace

bool confined_rows_supported(int nx, int ny) {
  return nx >= 8 && ny >= 8 && row_ops_supported(ny) && tdma_rows_lds_supported(ny - 2);
}

static void check_args(const ConfinedRows& a, int nb) {
  if (!confined_rows_supported(a.nx, a.ny) || a.mx != a.nx - 2 || a.my != a.ny - 2)
    throw std::invalid_argument("confined rows: unsupported sizes");
  if (nb < 1 || nb > 65535 || a.f0 < 0 || a.f1 > 3 || a.f0 > a.f1) throw std::invalid_argument("confined rows: bad batch");
}

#define RBC_CONFINED(KERNEL, per, blocks, fields, ...)                                       \
  do {                                                                                       \
    const dim3 grid((unsigned)(blocks), nb, fields), block(NT);                              \
    const size_t lds = buf_len(a.ny) * sizeof(double);                                       \
    if ((per) <= 2) RBC_LAUNCH(KERNEL<2>, grid, block, lds, s, __VA_ARGS__);                 \
    else if ((per) <= 4) RBC_LAUNCH(KERNEL<4>, grid, block, lds, s, __VA_ARGS__);                 \
    else if ((per) <= 8) RBC_LAUNCH(KERNEL<8>, grid, block, lds, s, __VA_ARGS__);            \
    else RBC_LAUNCH(KERNEL<16>, grid, block, lds, s, __VA_ARGS__);                           \
  } while (0)

void rhs_rows(hipStream_t s, const ConfinedRows& a, int nb) {
  check_args(a, nb);
  const int per = fdma_rows_lds_per(a.ny);
  if (a.f0 == a.f1) return;
  RBC_CONFINED(rhs_rows_kernel, per, a.nx, a.f1 - a.f0, a, per);
  check("rhs_rows");
}
void div_rows(hipStream_t s, const ConfinedRows& a, int nb) {
  check_args(a, nb);
  const int per = fdma_rows_lds_per(a.ny);
  if (a.norm && (nb != 1 || !a.part)) throw std::invalid_argument("div_rows: the norm of one instance");
  RBC_CONFINED(div_rows_kernel, per, a.nx, 1, a, per);
  check("div_rows");
}
void proj_rows(hipStream_t s, const ConfinedRows& a, int nb, bool pressure) {
  check_args(a, nb);
  if (a.f1 > 2) throw std::invalid_argument("proj_rows: fields 0 and 1");
  const int per_n = fdma_rows_lds_per(a.ny), per = fdma_rows_lds_per(a.my);
  const int blocks = (a.f1 - a.f0) * a.mx + (pressure ? a.nx : 0);
  if (blocks == 0) return;
  RBC_CONFINED(proj_rows_kernel, per_n, blocks, 1, a, per_n, per);
  check("proj_rows");
}

void adjoint_rows(hipStream_t s, const AdjointRows& in) {
  AdjointRows a = in;
  const bool fourier = !a.LX;
  if (!row_ops_supported(a.ny) || a.my != a.ny - 2 || a.mx < 1 || a.rows != (fourier ? 2 * a.mx : a.mx + 2))
    throw std::invalid_argument("adjoint_rows: unsupported sizes");
  a.per = fdma_rows_lds_per(a.ny);
  const dim3 grid((unsigned)a.rows, 3), block(NT);
  const size_t lds = buf_len(a.ny) * sizeof(double);
#define RBC_ADJOINT(SL)                                                                        \
  do {                                                                                         \
    if (fourier) RBC_LAUNCH((adjoint_rows_kernel<SL, true>), grid, block, lds, s, a);          \
    else RBC_LAUNCH((adjoint_rows_kernel<SL, false>), grid, block, lds, s, a);                 \
  } while (0)
  if (a.per <= 2) RBC_ADJOINT(2);
  else if (a.per <= 4) RBC_ADJOINT(4);
  else if (a.per <= 8) RBC_ADJOINT(8);
  else RBC_ADJOINT(16);
#undef RBC_ADJOINT
  check("adjoint_rows");
}

}  // namespace rbc
