// Row operators of Space2 along axis 1 (y): to_ortho and derivatives of a composite or plain
// Chebyshev row, and from_ortho, on real rows or on interleaved complex rows, FP64.
//
// A block of four wavefronts holds two value rows: two real rows, or the real and imaginary
// parts of one complex row (read and written as 16-byte pairs where both parts are at hand, so
// that the caller's interleaved arrays need no separate split pass).  Each row is two parity
// chains, one wavefront each (chains.hpp).  The operators are bound by memory: one read of the
// input and one write of the output.  At fourier_r2c(512) x cheb_dirichlet(513), 8 fields, one
// d/dx, d/dy, d2/dy2, to_ortho and from_ortho each take 2,834 us in all as split copies, dense
// FMA products and merge copies per field, and 114 us as one launch per operator over the batch
// (13 us a launch; the rest is each call's wait).
//
// The dense products' entries were rounded once from long double, so the rows' own forms are chosen for
// their rounding: derivatives of the composite basis itself (rowdiff.hpp), from_ortho by the stencil's null
// vector, not the reference's recurrences over intermediate results.
#include <hip/hip_runtime.h>

#include <cmath>
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
constexpr int WAVES = 4;

void check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// d1 derivatives (ortho.rs:107-125) of the to_ortho stencil (composite_stencil.rs:207-229) of
// every row, (i k)^d0 (r2c.rs:88-99) applied first and the division by sc last (complex rows;
// real rows multiply by sc, the caller's reciprocal).  in: mi values per row, out: n.
// COMP: the derivative of a composite row that is formed at once (0: to_ortho, then d1 plain derivatives); the
// second one's registers would cost the others a block per CU.
template <int SLICE, bool CPLX, int COMP>
__global__ __launch_bounds__(WAVE* WAVES) void ortho_rows_kernel(const double* __restrict__ in, double* __restrict__ out,
                                                                 long rows, int mi, int n, int per, int bl,
                                                                 const double* __restrict__ coef, int d1, int d0, int m0,
                                                                 double sc, double isc) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int slot = w >> 1, p = w & 1, tid = p * WAVE + lane;
  double* buf = lds + slot * bl;
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + 2 * WAVE - 1) / (2 * WAVE);
  const long row = CPLX ? (long)blockIdx.x : 2 * (long)blockIdx.x + slot;
  const bool valid = row < rows;
  const double kk = CPLX && d0 > 0 ? (double)(row % m0) : 0.0;
  {
    double v[MAXQ];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * 2 * WAVE - 2;
      v[q] = 0.0;
      if (valid && i >= 0 && i < mi) {
        if constexpr (CPLX) {
          const double2 c = reinterpret_cast<const double2*>(in)[row * mi + i];
          double a = c.x, b = c.y;
          for (int t = 0; t < d0; ++t) {  // (a + i b) (0 + i k) as num-complex
            const double na = a * 0.0 - b * kk, nb = a * kk + b * 0.0;
            a = na;
            b = nb;
          }
          v[q] = slot ? b : a;
        } else {
          v[q] = in[row * mi + i];
        }
      }
    }
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int j = tid + q * 2 * WAVE;
      if (j < n + 6) buf[pad(j)] = v[q];
    }
  }
  __syncthreads();
  if constexpr (COMP == 1) {
    rowdiff::derive_composite<SLICE>(buf, coef + n + 2, n, per, lane, p);
  } else if constexpr (COMP == 2) {
    rowdiff::derive2_composite<SLICE>(buf, coef + n + 2, n, per, lane, p);
  } else if (coef) {  // stencil taps, zero where absent
    double v[MAXQ];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * 2 * WAVE;
      v[q] = i < n ? buf[pad(i + 2)] * coef[i] + buf[pad(i)] * coef[n + i] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * 2 * WAVE;
      if (i < n) buf[pad(i + 2)] = v[q];
    }
    __syncthreads();
  }
  if constexpr (COMP == 0)
    for (int t = 0; t < d1; ++t) rowdiff::derive<SLICE>(buf, n, per, lane, p);
  if constexpr (CPLX) {
    const double ns = sc * sc + 0.0 * 0.0;
    for (int i = threadIdx.x; i < n; i += WAVE * WAVES) {
      double a = lds[pad(i + 2)], b = lds[bl + pad(i + 2)];
      if (isc != 0.0) {  // sc a power of two: the same value (and sign of a zero) without the division
        a = (a * sc + b * 0.0) * isc * isc;
        b = (b * sc - a * 0.0) * isc * isc;
      } else if (sc != 1.0) {  // num-complex division by (sc, 0)
        const double na = (a * sc + b * 0.0) / ns, nb = (b * sc - a * 0.0) / ns;
        a = na;
        b = nb;
      }
      reinterpret_cast<double2*>(out)[row * n + i] = double2{a, b};
    }
  } else {
    if (!valid) return;
    for (int i = tid; i < n; i += 2 * WAVE) out[row * n + i] = sc != 1.0 ? buf[pad(i + 2)] * sc : buf[pad(i + 2)];
  }
}

// from_ortho of every row (composite_stencil.rs:250-276): the least squares x of S x = q, S the stencil
// q_t = x_t + l_{t-1} x_{t-1} along a parity chain of one value more than x has.  What S x cannot reach is
// along w, S^T w = 0 (w_t = -l_t w_{t+1}); with it taken off, r = q - w (w q) / (w w), S x = r is solved from
// either end: Dirichlet (l = -1, w = 1: tab null) by suffix sums, x_t = -(r_{t+1} + r_{t+2} + ..), from the
// small coefficients down; Neumann (-1 < l <= 0) by x_t = r_t - l_{t-1} x_{t-1}, tab holding w and l_{t-1} in
// slice order.  iw: 1 / (w w) of the two chains.  w is taken off twice, the second time what rounding left.
// Rounding against 64 bits, rows of 257 coefficients that fall off as k^-2: Dirichlet 2e-16, Neumann 1e-16 of
// the result (dense product 6e-16 and 3e-16; the normal equations S^T S x = S^T q of linalg.rs:14-57, whose
// condition grows as the square, 1.2e-14 and 1.5e-15).  in: n = m + 2 values per row, out: m.
template <int SLICE, bool CPLX>
__global__ __launch_bounds__(WAVE* WAVES) void composite_rows_kernel(const double* __restrict__ in,
                                                                     double* __restrict__ out, long rows, int m, int per,
                                                                     int bl, const double* __restrict__ tab, double iw0,
                                                                     double iw1) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int slot = w >> 1, p = w & 1, tid = p * WAVE + lane, n = m + 2;
  double* buf = lds + slot * bl;
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + 2 * WAVE - 1) / (2 * WAVE);
  const long row = CPLX ? (long)blockIdx.x : 2 * (long)blockIdx.x + slot;
  const bool valid = row < rows;
  {
    double v[MAXQ];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int i = tid + q * 2 * WAVE - 2;
      v[q] = valid && i >= 0 && i < n ? (CPLX ? in[2 * (row * n + i) + slot] : in[row * n + i]) : 0.0;
    }
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      const int j = tid + q * 2 * WAVE;
      if (j < n + 6) buf[pad(j)] = v[q];
    }
  }
  __syncthreads();
  const int len = p == 0 ? (n + 1) / 2 : n / 2;  // values q of the chain; x has one less
  const int t0 = lane * per, cnt = max(0, min(per, len - t0));
  double v[SLICE], nw[SLICE], l[SLICE];
#pragma unroll
  for (int q = 0; q < SLICE; ++q) {
    v[q] = q < cnt ? buf[pad(p + 2 * (t0 + q) + 2)] : 0.0;
    nw[q] = q < cnt ? 1.0 : 0.0;
    l[q] = -1.0;
    if (tab) {
      nw[q] = tab[((size_t)p * per + q) * WAVE + lane];
      l[q] = tab[((size_t)(2 + p) * per + q) * WAVE + lane];
    }
  }
  const double iw = p ? iw1 : iw0;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    double s = 0.0, above;
#pragma unroll
    for (int q = 0; q < SLICE; ++q)
      if (q < cnt) s = s + nw[q] * v[q];
    const double a = wave::lane_value(wave::suffix_sum(s, lane, above), 0) * iw;
#pragma unroll
    for (int q = 0; q < SLICE; ++q)
      if (q < cnt) v[q] = __builtin_fma(-a, nw[q], v[q]);
  }
  if (tab) {
    chains::fdma_forward(v, l, lane, t0, cnt);
  } else {
    double s = 0.0, above;
#pragma unroll
    for (int q = SLICE - 1; q >= 0; --q) s = s + v[q];
    wave::suffix_sum(s, lane, above);
#pragma unroll
    for (int q = SLICE - 1; q >= 0; --q) {
      const double r = v[q];
      v[q] = -above;
      above = above + r;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < SLICE; ++q)
    if (q < cnt) buf[pad(p + 2 * (t0 + q) + 2)] = v[q];
  __syncthreads();
  if constexpr (CPLX) {
    for (int i = threadIdx.x; i < m; i += WAVE * WAVES)
      reinterpret_cast<double2*>(out)[row * m + i] = double2{lds[pad(i + 2)], lds[bl + pad(i + 2)]};
  } else {
    if (!valid) return;
    for (int i = tid; i < m; i += 2 * WAVE) out[row * m + i] = buf[pad(i + 2)];
  }
}

}  // namespace

// the slices of a row of n values: at most 16 entries per lane and chain
bool row_ops_supported(int n) { return n >= 6 && fdma_rows_lds_per(n) <= 16; }

#define RBC_ROW_OP(KERNEL, blocks, per, PARAMS, ...)                                             \
  do {                                                                                          \
    const dim3 grid((unsigned)(blocks)), block(WAVE * WAVES);                                   \
    const size_t sh = 2 * bl * sizeof(double);                                                  \
    if ((per) <= 2) RBC_LAUNCH((KERNEL<2, PARAMS>), grid, block, sh, s, __VA_ARGS__);           \
    else if ((per) <= 4) RBC_LAUNCH((KERNEL<4, PARAMS>), grid, block, sh, s, __VA_ARGS__);      \
    else if ((per) <= 6) RBC_LAUNCH((KERNEL<6, PARAMS>), grid, block, sh, s, __VA_ARGS__);      \
    else if ((per) <= 8) RBC_LAUNCH((KERNEL<8, PARAMS>), grid, block, sh, s, __VA_ARGS__);      \
    else RBC_LAUNCH((KERNEL<16, PARAMS>), grid, block, sh, s, __VA_ARGS__);                     \
  } while (0)

template <bool CPLX, int COMP>
static void launch_ortho(hipStream_t s, const double* in, double* out, long rows, int mi, int n, int per, int bl,
                         const double* coef, int d1, int d0, int m0, double sc, double isc) {
#define RBC_PARAMS CPLX, COMP
  RBC_ROW_OP(ortho_rows_kernel, CPLX ? rows : (rows + 1) / 2, per, RBC_PARAMS, in, out, rows, mi, n, per, bl, coef, d1, d0,
             m0, sc, isc);
#undef RBC_PARAMS
}

void ortho_rows(hipStream_t s, const double* in, double* out, long rows, bool cplx, int mi, int n, const double* coef,
                int d1, int d0, int m0, double sc) {
  if (!row_ops_supported(n) || mi > n || (!coef && mi != n) || d1 < 0 || (coef && d1 > 2) || d0 < 0 || (d0 > 0 && m0 < 1))
    throw std::invalid_argument("ortho_rows: bad arguments");
  if (rows < 1 || rows > 0x3fffffff) throw std::invalid_argument("ortho_rows: bad rows");
  const int per = fdma_rows_lds_per(n), bl = buf_len(n);
  int ex = 0;
  const double isc = sc > 0.0 && sc != 1.0 && std::frexp(sc, &ex) == 0.5 ? 1.0 / sc : 0.0;
  const int comp = coef ? d1 : 0;
  if (!cplx) {
    d0 = 0;
    m0 = 1;
  }
#define RBC_ORTHO(C, D) launch_ortho<C, D>(s, in, out, rows, mi, n, per, bl, coef, d1, d0, m0, sc, C ? isc : 0.0)
  if (comp == 0) cplx ? RBC_ORTHO(true, 0) : RBC_ORTHO(false, 0);
  else if (comp == 1) cplx ? RBC_ORTHO(true, 1) : RBC_ORTHO(false, 1);
  else cplx ? RBC_ORTHO(true, 2) : RBC_ORTHO(false, 2);
#undef RBC_ORTHO
  check("ortho_rows");
}

void composite_rows(hipStream_t s, const double* in, double* out, long rows, bool cplx, const Composite& c) {
  const int n = c.m + 2, m = c.m;
  if (!row_ops_supported(n)) throw std::invalid_argument("composite_rows: bad length");
  if (rows < 1 || rows > 0x3fffffff) throw std::invalid_argument("composite_rows: bad rows");
  const int per = fdma_rows_lds_per(n), bl = buf_len(n);
  if (cplx) RBC_ROW_OP(composite_rows_kernel, rows, per, true, in, out, rows, m, per, bl, c.tab, c.iw[0], c.iw[1]);
  else RBC_ROW_OP(composite_rows_kernel, (rows + 1) / 2, per, false, in, out, rows, m, per, bl, c.tab, c.iw[0], c.iw[1]);
  check("composite_rows");
}

}  // namespace rbc
