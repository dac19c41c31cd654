// Banded row solves of the tensor solvers (fdma_tensor.rs:195-234 with the per-row Fdma
// of fdma.rs:101-118), FP64, optionally fused with the preconditioner matvec that
// precedes them (MatVecFdma along y, matvec.rs:172-193): the row-solve kernel around the
// block body of rowsolve.hpp, and the from_ortho row kernel of the composite bases.
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

#include "chains.hpp"
#include "ops.hpp"
#include "rowsolve.hpp"

namespace rbc {

namespace {

using chains::buf_len;
using chains::pad;
using chains::WAVE;
using rowsolve::WAVES;

// Tables of up to four batch entries (blockIdx.y), or one shared by all entries.
struct RowTables {
  const double* band[4];
  const double* diag[4];
  int shared;
};

// One block per set (nrows = 2 nsets) or per two rows, blockIdx.y the batch entry.
// With pairg > 0 (one block per set, entries 0 and 1 on the same tables) the grid is 1-D:
// blocks [0, 16 pairg) hold entries 0 and 1 interleaved in groups of 16, block b of a group
// taking set 8 g + (b mod 8) of entry (b / 8) mod 2, so that the two blocks of a set are
// dispatched 8 apart and land on the same XCD (workgroups go round-robin over the 8 XCDs):
// the second reads the set's tables from that XCD's L2.  Blocks from 16 pairg on take the
// further entries, nsets blocks each.
template <int SLICE>
__global__ __launch_bounds__(WAVE* WAVES, SLICE <= 8 ? 4 : 2) void fdma_rows_lds_kernel(const double* __restrict__ R, int ldr, int nr,
                                                                    double* __restrict__ X, int ld, int nrows, int m,
                                                                    int nsets, int per, int bl, RowTables tb, long sr,
                                                                    long sx, int pairg) {
  extern __shared__ double lds[];
  int entry = blockIdx.y, bx = blockIdx.x;
  if (pairg > 0) {
    const int pb = 16 * pairg;
    if (bx < pb) {
      entry = (bx >> 3) & 1;
      bx = (bx >> 4) * 8 + (bx & 7);
      if (bx >= nsets) return;  // the whole block: no barrier reached
    } else {
      bx -= pb;
      entry = 2 + bx / nsets;
      bx -= (entry - 2) * nsets;
    }
  }
  const int ti = tb.shared ? 0 : entry;
  rowsolve::fdma_block<SLICE>(lds, R + sr * entry, ldr, nr, X + sx * entry, ld, nrows, m, nsets, per, bl, tb.band[ti],
                              tb.diag[ti], bx);
}

// ux and uy of the periodic step, a set's rows of both fields 8 blocks apart (as above), with the right-hand
// sides formed in place of a launch that writes and a pass that reads them: 256 x 257, 6.8 us where these
// took 4.0 and 4.9
template <int SLICE>
__global__ __launch_bounds__(WAVE* WAVES, 4) void step_rows_kernel(StepRhs a, double* X, int per, int bl,
                                                                   const double* __restrict__ bandp,
                                                                   const double* __restrict__ diagp) {
  extern __shared__ double lds[];
  const int bx = blockIdx.x, f = (bx >> 3) & 1, set = (bx >> 4) * 8 + (bx & 7);
  if (set >= a.mx) return;  // the whole block: no barrier reached
  rowsolve::step_block<SLICE>(lds, a, f, X + f * a.F, per, bl, bandp, diagp, set);
}

// The rows of blockIdx.y-th interleaved complex array [nsets, nr] -> [nsets, m], one block per
// set.  The caller's arrays are read and written once: at fourier_r2c(256) x cheb_neumann(257),
// 4 right-hand sides, 19 us a call with the wait for it, against 59 us with a split and a merge
// copy per right-hand side around the solve.
template <int SLICE>
__global__ __launch_bounds__(WAVE* WAVES, SLICE <= 8 ? 4 : 2) void fdma_rows_complex_kernel(
    const double* __restrict__ R, int ldr, int nr, double* __restrict__ X, int ld, int m, int nsets, int per, int bl,
    const double* __restrict__ bandp, const double* __restrict__ diagp) {
  extern __shared__ double lds[];
  R += 2 * (size_t)nsets * ldr * blockIdx.y;
  X += 2 * (size_t)nsets * ld * blockIdx.y;
  rowsolve::fdma_block<SLICE, true>(lds, R, ldr, nr, X, ld, 2 * nsets, m, nsets, per, bl, bandp, diagp, blockIdx.x);
}

// The rows of NR batch entries (from NR blockIdx.y on) with the same tables by one wavefront per (set,
// parity chain): the tables are read and the maps' matrices composed and scanned once for the NR right-hand
// sides.  One row per set and entry (nrows = nsets); a block holds two sets.  512 x 512, 64 right-hand sides:
// 89 us against 122 us with a wavefront per row; its 267 MB would take 54 us, the rest is the scans.
template <int SLICE, int NR>
__global__ __launch_bounds__(WAVE* WAVES, 2) void fdma_rows_batch_kernel(const double* __restrict__ R, int ldr, int nr,
                                                                         double* __restrict__ X, int ld, int m,
                                                                         int nsets, int per, int bl,
                                                                         const double* __restrict__ bandp,
                                                                         const double* __restrict__ diagp, int batch,
                                                                         long sr, long sx) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int slot = w >> 1, p = w & 1, tid = p * WAVE + lane;
  double* buf = lds + slot * NR * bl;
  const int set = blockIdx.x * (WAVES / 2) + slot, b0 = blockIdx.y * NR, s0 = min(set, nsets - 1);
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + 2 * WAVE - 1) / (2 * WAVE);
  auto valid = [&](int k) { return set < nsets && b0 + k < batch; };
#pragma unroll
  for (int k = 0; k < NR; ++k)
    chains::stage_row<MAXQ>(buf + k * bl, R + sr * (b0 + k) + (size_t)set * ldr, valid(k), nr, tid, 2 * WAVE);
  __syncthreads();
  const int len = p == 0 ? (m + 1) / 2 : m / 2, t0 = lane * per, cnt = max(0, min(per, len - t0));
  double v[NR][SLICE];
  if (bandp) {  // taps at offsets 0, -2, +2, +4, summed in that order
    const size_t tp = (size_t)2 * per * WAVE;
    double c[4][SLICE];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int q = 0; q < SLICE; ++q) c[t][q] = bandp[t * tp + ((size_t)p * per + q) * WAVE + lane];
#pragma unroll
    for (int k = 0; k < NR; ++k)
#pragma unroll
      for (int q = 0; q < SLICE; ++q) {
        double val = 0.0;
        if (q < cnt) {
          const int j = p + 2 * (t0 + q) + 2;
          const double* row = buf + k * bl;
          val = c[0][q] * row[pad(j)];
          val = val + c[1][q] * row[pad(j - 2)];
          val = val + c[2][q] * row[pad(j + 2)];
          val = val + c[3][q] * row[pad(j + 4)];
        }
        v[k][q] = val;
      }
  } else {
#pragma unroll
    for (int k = 0; k < NR; ++k)
#pragma unroll
      for (int q = 0; q < SLICE; ++q) v[k][q] = q < cnt ? buf[k * bl + pad(p + 2 * (t0 + q) + 2)] : 0.0;
  }
  const double* dg = diagp + (size_t)s0 * (8 * (size_t)per * WAVE);
  auto table = [&](int a, int q) { return dg[((size_t)(a * 2 + p) * per + q) * WAVE + lane]; };
  {
    double lo[SLICE];
#pragma unroll
    for (int q = 0; q < SLICE; ++q) lo[q] = table(0, q);
    chains::fdma_forward(v, lo, lane, t0, cnt);
  }
  {
    double rd[SLICE], g1[SLICE], g2[SLICE];  // 1 / dia, up1, up2
#pragma unroll
    for (int q = 0; q < SLICE; ++q) {
      rd[q] = table(1, q);
      g1[q] = table(2, q);
      g2[q] = table(3, q);
    }
    chains::fdma_backward(v, rd, g1, g2, lane, t0, cnt, len);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NR; ++k)
#pragma unroll
    for (int q = 0; q < SLICE; ++q)
      if (q < cnt) buf[k * bl + pad(p + 2 * (t0 + q) + 2)] = v[k][q];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NR; ++k)
    chains::unstage_row<MAXQ>(buf + k * bl, X + sx * (b0 + k) + (size_t)set * ld, valid(k), m, tid, 2 * WAVE, false);
}

// from_ortho of a composite basis per row (composite_stencil.rs:250-276, linalg.rs:14-57):
// d_i = p_i diag_i + p_{i+2} low2_i, then g_i = (d_i - g_{i-2} off_{i-2}) / den_i and
// x_i = g_i - x_{i+2} w_i (x_i = g_i for the last two i), arithmetic as tdma_y.  One
// wavefront per (row, parity chain).  With `project` the result is subtracted from X as
// the velocity projection does (navier.rs:683-695): X = x (-1) + X.
template <int SLICE>
__global__ __launch_bounds__(WAVE* WAVES) void tdma_rows_lds_kernel(const double* __restrict__ R, int ldr,
                                                                    double* __restrict__ X, int ld, int rows, int m,
                                                                    int per, int bl, const double* __restrict__ tab,
                                                                    long sr, long sx, int project) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int slot = w >> 1, p = w & 1;
  R += sr * blockIdx.y;
  X += sx * blockIdx.y;
  double* buf = lds + slot * bl;
  const int r = blockIdx.x * (WAVES / 2) + slot, nr = m + 2;
  const bool valid = r < rows;
  constexpr int MAXQ = (2 * SLICE * WAVE + 8 + 2 * WAVE - 1) / (2 * WAVE);
  chains::stage_row<MAXQ>(buf, R + (size_t)r * ldr, valid, nr, p * WAVE + lane, 2 * WAVE);
  __syncthreads();
  const int len = p == 0 ? (m + 1) / 2 : m / 2;
  const int t0 = lane * per;
  const int cnt = max(0, min(per, len - t0));
  double v[SLICE];
#define TB(a, q) tab[((size_t)((a) * 2 + p) * per + (q)) * WAVE + lane]
  {
    double dg[SLICE], l2[SLICE];
#pragma unroll
    for (int q = 0; q < SLICE; ++q) {
      dg[q] = TB(0, q);
      l2[q] = TB(1, q);
    }
#pragma unroll
    for (int q = 0; q < SLICE; ++q) {
      const int j = p + 2 * (t0 + q) + 2;
      v[q] = q < cnt ? buf[pad(j)] * dg[q] + buf[pad(j + 2)] * l2[q] : 0.0;
    }
  }
  {  // forward: g_i = (d_i - g_{i-2} off_{i-2}) / den_i  (i >= 2), g_i = d_i / den_i (i < 2)
    double of[SLICE], rn[SLICE];  // off_{i-2}, 1 / den_i
#pragma unroll
    for (int q = 0; q < SLICE; ++q) {
      of[q] = TB(2, q);
      rn[q] = TB(3, q);
    }
    chains::tdma_forward(v, of, rn, lane, t0, cnt);
  }
  {  // back: x_i = g_i for i >= m - 2, else x_i = g_i - x_{i+2} w_i
    double wv[SLICE];
#pragma unroll
    for (int q = 0; q < SLICE; ++q) wv[q] = TB(4, q);
    chains::tdma_backward(v, wv, lane, t0, cnt, p, m);
  }
#undef TB
  __syncthreads();
#pragma unroll
  for (int q = 0; q < SLICE; ++q)
    if (q < cnt) buf[pad(p + 2 * (t0 + q) + 2)] = v[q];
  __syncthreads();
  chains::unstage_row<MAXQ>(buf, X + (size_t)r * ld, valid, m, p * WAVE + lane, 2 * WAVE, project != 0);
}

void check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

}  // namespace

int fdma_rows_lds_per(int m) { return ((m + 1) / 2 + WAVE - 1) / WAVE; }

bool fdma_rows_lds_supported(int m, int nr) {
  return m >= 5 && fdma_rows_lds_per(m) <= 16 && nr >= m &&
         (size_t)(WAVES / 2) * buf_len(nr) * sizeof(double) <= 65536;
}

// entries per lane and chain that hold the row's solution and stage its right-hand side
static int slice_of(int m, int nr) {
  const int a = fdma_rows_lds_per(m), b = fdma_rows_lds_per(nr - 2);
  return a > b ? a : b;
}

static void launch_rows(hipStream_t s, const double* R, int ldr, int nr, double* X, int ld, int nrows, int m,
                        int nsets, const RowTables& tb, int batch, long sr, long sx) {
  if (!fdma_rows_lds_supported(m, nr)) throw std::invalid_argument("fdma_rows_lds: unsupported row length");
  if (nsets < 1 || nrows < 1 || batch < 1 || batch > 65535) throw std::invalid_argument("fdma_rows_lds: bad sizes");
  if (!tb.shared && batch > 4) throw std::invalid_argument("fdma_rows_lds: at most 4 entries with own tables");
  for (int k = 0; k < (tb.shared ? 1 : batch); ++k)
    if (!tb.band[k] && nr != m) throw std::invalid_argument("fdma_rows_lds: rhs length must equal m without a band");
  const int per = fdma_rows_lds_per(m), bl = buf_len(nr), sl = slice_of(m, nr);
  const unsigned blocks = nrows == 2 * nsets ? (unsigned)nsets : (unsigned)((nrows + 1) / 2);
  const size_t lds = (size_t)(WAVES / 2) * bl * sizeof(double);
  // entries 0 and 1 on the same tables, one block per set: interleaved 1-D grid
  const bool paired = !tb.shared && batch >= 2 && nrows == 2 * nsets && tb.band[0] == tb.band[1] &&
                      tb.diag[0] == tb.diag[1];
  const int pairg = paired ? (nsets + 7) / 8 : 0;
  const dim3 grid = paired ? dim3((unsigned)(16 * pairg + (batch - 2) * nsets), 1) : dim3(blocks, batch),
             block(WAVE * WAVES);
  // four right-hand sides per wavefront from two blocks per CU on (a whole solve, a row / four rows per
  // wavefront: 510 rows x 8 (510 blocks) 90.0 / 86.6 us, 126 x 64 (1,008) 48.8 / 43.9, 510 x 4 (255) 56.6 /
  // 57.2, 94 x 8 (94) 23.5 / 25.9)
  constexpr int NR = 4;
  if (tb.shared && nrows == nsets && batch >= NR && sl <= 8 && (size_t)NR * lds <= 65536 &&
      (long)blocks * (batch / NR) >= 500) {
    const dim3 g2(blocks, (batch + NR - 1) / NR);
    const size_t l2 = NR * lds;
#define RBC_BATCH(SL)                                                                                                \
  RBC_LAUNCH((fdma_rows_batch_kernel<SL, NR>), g2, block, l2, s, R, ldr, nr, X, ld, m, nsets, per, bl, tb.band[0], \
             tb.diag[0], batch, sr, sx)
    if (sl <= 2) RBC_BATCH(2);
    else if (sl <= 4) RBC_BATCH(4);
    else RBC_BATCH(8);
#undef RBC_BATCH
    check("fdma_rows_batch");
    return;
  }
  if (sl <= 2)
    RBC_LAUNCH(fdma_rows_lds_kernel<2>, grid, block, lds, s, R, ldr, nr, X, ld, nrows, m, nsets, per, bl, tb,
                       sr, sx, pairg);
  else if (sl <= 4)
    RBC_LAUNCH(fdma_rows_lds_kernel<4>, grid, block, lds, s, R, ldr, nr, X, ld, nrows, m, nsets, per, bl, tb,
                       sr, sx, pairg);
  else if (sl <= 8)
    RBC_LAUNCH(fdma_rows_lds_kernel<8>, grid, block, lds, s, R, ldr, nr, X, ld, nrows, m, nsets, per, bl, tb,
                       sr, sx, pairg);
  else
    RBC_LAUNCH(fdma_rows_lds_kernel<16>, grid, block, lds, s, R, ldr, nr, X, ld, nrows, m, nsets, per, bl, tb,
                       sr, sx, pairg);
  check("fdma_rows_lds");
}

void fdma_rows_lds(hipStream_t s, const double* R, int ldr, int nr, double* X, int ld, int nrows, int m, int nsets,
                   const double* bandp, const double* diagp, int batch, long sr, long sx) {
  RowTables tb{};
  tb.band[0] = bandp;
  tb.diag[0] = diagp;
  tb.shared = 1;
  if (batch == 1 && nrows >= 4L * nsets && nrows % nsets == 0 && nrows / nsets <= 65535) {  // entries of one row per set
    batch = nrows / nsets;
    nrows = nsets;
    sr = (long)nsets * ldr;
    sx = (long)nsets * ld;
  }
  launch_rows(s, R, ldr, nr, X, ld, nrows, m, nsets, tb, batch, sr, sx);
}

void fdma_rows_lds_multi(hipStream_t s, const double* R, int ldr, int nr, double* X, int ld, int nrows, int m,
                         int nsets, const double* const* bandps, const double* const* diagps, int batch, long sr,
                         long sx) {
  if (batch < 1 || batch > 4) throw std::invalid_argument("fdma_rows_lds_multi: 1 to 4 entries");
  RowTables tb{};
  for (int k = 0; k < batch; ++k) {
    tb.band[k] = bandps[k];
    tb.diag[k] = diagps[k];
  }
  tb.shared = 0;
  launch_rows(s, R, ldr, nr, X, ld, nrows, m, nsets, tb, batch, sr, sx);
}

bool step_rows_supported(int ny) {
  return ny >= 9 && fdma_rows_lds_supported(ny - 2, ny) && fdma_rows_lds_per(ny - 2) <= STEP_SLICE;
}
void step_rows(hipStream_t s, const StepRhs& a, double* X, const double* bandp, const double* diagp) {
  if (!step_rows_supported(a.ny) || a.my != a.ny - 2 || a.mx < 1 || !a.U || !bandp || !diagp)
    throw std::invalid_argument("step_rows: unsupported sizes");
  const int per = fdma_rows_lds_per(a.my), bl = buf_len(a.ny), sl = slice_of(a.my, a.ny);
  const dim3 grid(16 * ((a.mx + 7) / 8)), block(WAVE * WAVES);
  const size_t lds = (size_t)(WAVES / 2) * bl * sizeof(double);
  if (sl <= 2) RBC_LAUNCH(step_rows_kernel<2>, grid, block, lds, s, a, X, per, bl, bandp, diagp);
  else RBC_LAUNCH(step_rows_kernel<4>, grid, block, lds, s, a, X, per, bl, bandp, diagp);
  check("step_rows");
}

void fdma_rows_lds_complex(hipStream_t s, const double* R, int ldr, int nr, double* X, int ld, int m, int nsets,
                           const double* bandp, const double* diagp, int batch) {
  if (!fdma_rows_lds_supported(m, nr)) throw std::invalid_argument("fdma_rows_lds_complex: unsupported row length");
  if (nsets < 1 || batch < 1 || !bandp || !diagp) throw std::invalid_argument("fdma_rows_lds_complex: bad arguments");
  const int per = fdma_rows_lds_per(m), bl = buf_len(nr), sl = slice_of(m, nr);
  const size_t lds = (size_t)(WAVES / 2) * bl * sizeof(double);
  for (int b = 0; b < batch; b += 65535) {
    const dim3 grid(nsets, batch - b < 65535 ? batch - b : 65535), block(WAVE * WAVES);
    const double* Rb = R + 2 * (size_t)nsets * ldr * b;
    double* Xb = X + 2 * (size_t)nsets * ld * b;
    if (sl <= 2)
      RBC_LAUNCH(fdma_rows_complex_kernel<2>, grid, block, lds, s, Rb, ldr, nr, Xb, ld, m, nsets, per, bl, bandp, diagp);
    else if (sl <= 4)
      RBC_LAUNCH(fdma_rows_complex_kernel<4>, grid, block, lds, s, Rb, ldr, nr, Xb, ld, m, nsets, per, bl, bandp, diagp);
    else if (sl <= 8)
      RBC_LAUNCH(fdma_rows_complex_kernel<8>, grid, block, lds, s, Rb, ldr, nr, Xb, ld, m, nsets, per, bl, bandp, diagp);
    else
      RBC_LAUNCH(fdma_rows_complex_kernel<16>, grid, block, lds, s, Rb, ldr, nr, Xb, ld, m, nsets, per, bl, bandp, diagp);
  }
  check("fdma_rows_lds_complex");
}

bool tdma_rows_lds_supported(int m) {
  return m >= 4 && fdma_rows_lds_per(m) <= 16 && (size_t)(WAVES / 2) * buf_len(m + 2) * sizeof(double) <= 65536;
}

void tdma_rows_lds(hipStream_t s, const double* R, int ldr, double* X, int ld, int rows, int m, const double* tabp,
                   int batch, long sr, long sx, bool project) {
  if (!tdma_rows_lds_supported(m)) throw std::invalid_argument("tdma_rows_lds: unsupported row length");
  if (rows < 1 || batch < 1 || batch > 65535) throw std::invalid_argument("tdma_rows_lds: bad sizes");
  const int per = fdma_rows_lds_per(m), bl = buf_len(m + 2), pj = project ? 1 : 0;
  const dim3 grid((unsigned)((rows + 1) / 2), batch), block(WAVE * WAVES);
  const size_t lds = (size_t)(WAVES / 2) * bl * sizeof(double);
  if (per <= 2)
    RBC_LAUNCH(tdma_rows_lds_kernel<2>, grid, block, lds, s, R, ldr, X, ld, rows, m, per, bl, tabp, sr, sx, pj);
  else if (per <= 4)
    RBC_LAUNCH(tdma_rows_lds_kernel<4>, grid, block, lds, s, R, ldr, X, ld, rows, m, per, bl, tabp, sr, sx, pj);
  else if (per <= 8)
    RBC_LAUNCH(tdma_rows_lds_kernel<8>, grid, block, lds, s, R, ldr, X, ld, rows, m, per, bl, tabp, sr, sx, pj);
  else
    RBC_LAUNCH(tdma_rows_lds_kernel<16>, grid, block, lds, s, R, ldr, X, ld, rows, m, per, bl, tabp, sr, sx,
                       pj);
  check("tdma_rows_lds");
}

}  // namespace rbc
