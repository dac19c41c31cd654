// Products with dense left operators (along x) on the FP64 matrix cores, split by parity.
//
// Every dense x operator of the Chebyshev bases couples indices of one parity only (spectral
// to spectral: derivatives, projections, implicit solves, eigen-transforms), or is even or odd
// about the middle of the axis (to and from the points).  The two parity classes are products
// of half the size each, so half the multiplications of the full operator are left:
//   blocks    C[2m + c] = sum_k A_c[m, k] B[2k + c'],
//   fold in   C[2m + c] = sum_k A_c[m, k] (B[k] +- B[n - 1 - k]),
//   fold out  C[m], C[n - 1 - m] = E +- O with E, O the class products.
//
// The operators are packed once in the order in which the lanes of a wavefront feed them to the
// MFMAs (xop_index): a wavefront reads 16 rows x 8 k values as one contiguous KiB, straight into
// registers.  B's rows are read the same way, 16 columns at a time.  There is no LDS staging and
// no barrier in the product: a wavefront runs on its own, with a chunk of loads in flight while
// it consumes the one before (a first form, staged through LDS with __syncthreads per slab of 32,
// spent 1.2 us per slab on 0.2 us of MFMAs at 257^2).
// The sum over k is formed as (q0 + q1) + (q2 + q3) of its four quarters in every variant, so
// that the choice of variant, which depends on the batch, never changes a result bit.
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

#include "fft_lds.hpp"
#include "ops.hpp"

namespace rbc {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

template <int NG>
struct XArgs {
  XGemm g[NG];
  int end[NG];  // first block index beyond each group
  int tx[NG], ty[NG];
};

// one of two kernel arguments: both are read up front (an indexed read would wait for the index,
// then for its own round trip to the argument memory)
template <typename T>
__device__ __forceinline__ T pick(bool one, T a, T b) {
  return one ? b : a;
}

// A wavefront computes 16 FM x 16 FN values.  SPLIT: the four wavefronts of a block share one
// such tile, a quarter of the k range each; otherwise they hold 2 x 2 tiles and each runs the
// quarters in turn.  KIND: XOP_BLOCKS (and XOP_DENSE, one class), XOP_FOLD_IN or XOP_FOLD_OUT,
// the same for every group; NG groups.  CH: groups of 8 k values per chunk of loads.
template <int FM, int FN, bool SPLIT, int CH, int KIND, int NG>
__global__ __launch_bounds__(256) void xgemm_kernel(XArgs<NG> ar) {
  constexpr bool IN2 = KIND == XOP_FOLD_IN, OUT2 = KIND == XOP_FOLD_OUT;
  constexpr int NC = OUT2 ? 2 : 1;  // classes of a block
  constexpr int BM = 16 * FM * (SPLIT ? 1 : 2), BN = 16 * FN * (SPLIT ? 1 : 2);
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  // consecutive logical blocks on one XCD: the tiles of one entry share operand panels in its L2
  int t = fftlds::xcd_remap(blockIdx.x, gridDim.x);
  XGemm g = ar.g[0];
  int tx = ar.tx[0], ty = ar.ty[0];
  if constexpr (NG > 1) {
    int base = 0;
#pragma unroll
    for (int i = 1; i < NG; ++i)
      if (t >= ar.end[i - 1]) {
        g = ar.g[i];
        tx = ar.tx[i];
        ty = ar.ty[i];
        base = ar.end[i - 1];
      }
    t -= base;
  }
  int n0 = (t % tx) * BN;
  t /= tx;
  int m0 = (t % ty) * BM;
  t /= ty;
  if (!SPLIT) {
    m0 += (wid >> 1) * 16 * FM;
    n0 += (wid & 1) * 16 * FN;
  }
  const bool halves = !OUT2 && g.op.kind != XOP_DENSE;
  const bool c1 = halves && (t & 1);  // the block's class
  const int z = halves ? t >> 1 : t;
  const int M = pick(c1, g.op.M[0], g.op.M[1]), N = g.N;
  // the smaller class's or the last column's missing tile (no barrier follows without SPLIT; with
  // it the whole block leaves)
  if (m0 >= M || n0 >= N) return;
  const bool second = g.split > 0 && z >= g.split;
  const double* __restrict__ B = g.B + g.sB * z;
  double* __restrict__ C = g.C + g.sC * z;
  const int ldb = g.ldb, rs = g.op.rstep, last = g.op.cols - 1;
  const long aoff = g.amod ? g.sA * (z % g.amod) : 0;
  const double *a0 = second ? g.a2[0] : g.op.a[0], *a1 = second ? g.a2[1] : g.op.a[1];
  const int G = g.op.groups;  // groups of 8 k values of a packed row, a multiple of 4 CH
  // class c of the block (folding out: both, otherwise its own)
  const double* Ac[NC];
  int Kc[NC], r0[NC];
  bool any = false;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const bool one = OUT2 ? c == 1 : c1;
    any = any || m0 < pick(one, g.op.mnz[0], g.op.mnz[1]);  // else past a cut: zero rows
    Kc[c] = pick(one, g.op.K[0], g.op.K[1]);
    r0[c] = pick(one, g.op.r0[0], g.op.r0[1]);
    Ac[c] = pick(one, a0, a1) + aoff + ((size_t)(m0 >> 4) * G * 64 + lane) * 2;
  }
  const double* Bn[FN];  // this lane's columns (past N: a column inside, never stored)
#pragma unroll
  for (int j = 0; j < FN; ++j) Bn[j] = B + min(n0 + 16 * j + lr, N - 1);

  struct Chunk {
    double2 a[NC][CH][FM], b[NC][CH][FN], m[IN2 ? CH : 1][IN2 ? FN : 1];
  };
  auto load = [&](int g0, Chunk& x) {  // groups g0 .. g0 + CH - 1
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int h = 0; h < CH; ++h) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
          x.a[c][h][i] = *reinterpret_cast<const double2*>(Ac[c] + ((size_t)i * G + g0 + h) * 128);
        const int k = (g0 + h) * 8 + 2 * lk;
        const int q0 = r0[c] + rs * min(k, Kc[c] - 1), q1 = r0[c] + rs * min(k + 1, Kc[c] - 1);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          x.b[c][h][j].x = Bn[j][(long)q0 * ldb];
          x.b[c][h][j].y = Bn[j][(long)q1 * ldb];
          if constexpr (IN2) {
            x.m[h][j].x = Bn[j][(long)(last - q0) * ldb];
            x.m[h][j].y = Bn[j][(long)(last - q1) * ldb];
          }
        }
      }
  };
  v4d acc[NC][FM][FN];
  auto clear = [&]() {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[c][i][j] = v4d{0, 0, 0, 0};
  };
  auto mac = [&](int g0, const Chunk& x) {
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int k = (g0 + h) * 8 + 2 * lk;
        const bool ok0 = k < Kc[c], ok1 = k + 1 < Kc[c];  // the packed rows end in zeros, B does not
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          double2 b = x.b[c][h][j];
          if constexpr (IN2) {
            b.x = c1 ? b.x - x.m[h][j].x : b.x + x.m[h][j].x;
            b.y = c1 ? b.y - x.m[h][j].y : b.y + x.m[h][j].y;
          }
          b.x = ok0 ? b.x : 0.0;
          b.y = ok1 ? b.y : 0.0;
#pragma unroll
          for (int i = 0; i < FM; ++i) {
            acc[c][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.a[c][h][i].x, b.x, acc[c][i][j], 0, 0, 0);
            acc[c][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.a[c][h][i].y, b.y, acc[c][i][j], 0, 0, 0);
          }
        }
      }
  };
  // the chunks [g0, g0 + n CH) of one quarter, the next chunk's loads in flight; x holds the
  // first and receives the chunk after the last (clamped to the row)
  Chunk x, y;
  const int nch = G / (4 * CH), top = G - CH;
  auto quarter = [&](int g0) {
    clear();
    int n = 0;
    for (; n + 2 <= nch; n += 2) {
      load(min(g0 + (n + 1) * CH, top), y);
      mac(g0 + n * CH, x);
      load(min(g0 + (n + 2) * CH, top), x);
      mac(g0 + (n + 1) * CH, y);
    }
    if (n < nch) {
      if constexpr (SPLIT) {
        mac(g0 + n * CH, x);
      } else {
        load(min(g0 + (n + 1) * CH, top), y);
        mac(g0 + n * CH, x);
        x = y;
      }
    }
  };
  if constexpr (SPLIT) {
    // partial sums of the quarters through LDS, lanes side by side
    __shared__ v4d part[2][NC * FM * FN][64];
    const int g0 = wid * nch * CH;
    clear();
    if (any) {
      load(g0, x);
      quarter(g0);
    }
    auto put = [&](int s) {
#pragma unroll
      for (int e = 0; e < NC * FM * FN; ++e) part[s][e][lane] = acc[e / (FM * FN)][e / FN % FM][e % FN];
    };
    auto add = [&](int s) {
#pragma unroll
      for (int e = 0; e < NC * FM * FN; ++e) acc[e / (FM * FN)][e / FN % FM][e % FN] += part[s][e][lane];
    };
    if (wid & 1) put(wid >> 1);
    __syncthreads();
    if (!(wid & 1)) add(wid >> 1);
    __syncthreads();
    if (wid == 2) put(0);
    __syncthreads();
    if (wid != 0) return;
    add(0);
  } else {
    v4d sum[NC][FM][FN], pair[NC][FM][FN];
    if (any) {
      load(0, x);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        quarter(q * nch * CH);
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
              if (q == 0) sum[c][i][j] = acc[c][i][j];
              else if (q == 2) pair[c][i][j] = acc[c][i][j];
              else if (q == 1) sum[c][i][j] += acc[c][i][j];
              else acc[c][i][j] = sum[c][i][j] + (pair[c][i][j] + acc[c][i][j]);
            }
      }
    } else {
      clear();
    }
  }
  const int ldc = g.ldc, rows = g.op.rows, c0 = pick(c1, g.op.c0[0], g.op.c0[1]), cs = g.op.cstep;
  const bool pin = g.zero00 != 0;
  auto put = [&](int row, int col, double v) {
    if (pin && row == 0 && col == 0) v = 0.0;
    C[(size_t)row * ldc + col] = v;
  };
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + i * 16 + 4 * r + lk, n = n0 + j * 16 + lr;
        if (m >= M || n >= N) continue;
        const double v = acc[0][i][j][r];
        if constexpr (OUT2) {
          const double o = acc[1][i][j][r];
          const int mirror = rows - 1 - m;
          put(m, n, v + o);
          if (mirror != m) put(mirror, n, v - o);
        } else {
          put(c0 + cs * m, n, v);
        }
      }
}

template <int FM, int FN, bool SPLIT, int CH, int KIND, int NG>
void launch(hipStream_t s, const XGemm* groups) {
  constexpr int BM = 16 * FM * (SPLIT ? 1 : 2), BN = 16 * FN * (SPLIT ? 1 : 2);
  XArgs<NG> ar{};
  long total = 0;
  for (int i = 0; i < NG; ++i) {
    ar.g[i] = groups[i];
    ar.tx[i] = (groups[i].N + BN - 1) / BN;
    ar.ty[i] = (groups[i].op.M[0] + BM - 1) / BM;
    const int ncls = KIND == XOP_FOLD_OUT || groups[i].op.kind == XOP_DENSE ? 1 : 2;
    total += (long)ar.tx[i] * ar.ty[i] * ncls * groups[i].entries;
    if (total > 0x7fffffffL) throw std::invalid_argument("xgemm: too many tiles");
    ar.end[i] = (int)total;
  }
  RBC_LAUNCH((xgemm_kernel<FM, FN, SPLIT, CH, KIND, NG>), dim3((unsigned)total), dim3(256), 0, s, ar);
}

enum { TILE_16, TILE_32, TILE_64 };

template <int CH, int KIND, int NG>
void launch_tile(hipStream_t s, const XGemm* groups, int tile) {
  // the larger tiles take shorter chunks: fewer registers, more wavefronts per SIMD
  constexpr int CS = CH == 4 ? 2 : CH == 3 ? 1 : CH;
  switch (tile) {
    case TILE_16: launch<1, 1, true, CH, KIND, NG>(s, groups); break;
    case TILE_32: launch<2, 1, true, CS, KIND, NG>(s, groups); break;
    default: launch<2, 2, false, CS, KIND, NG>(s, groups); break;
  }
}

template <int CH, int KIND>
void launch_groups(hipStream_t s, const XGemm* groups, int ng, int tile) {
  switch (ng) {
    case 1: launch_tile<CH, KIND, 1>(s, groups, tile); break;
    case 2: launch_tile<CH, KIND, 2>(s, groups, tile); break;
    default: launch_tile<CH, KIND, 3>(s, groups, tile); break;
  }
}

template <int KIND>
void launch_chunk(hipStream_t s, const XGemm* groups, int ng, int tile, int ch) {
  switch (ch) {
    case 1: launch_groups<1, KIND>(s, groups, ng, tile); break;
    case 2: launch_groups<2, KIND>(s, groups, ng, tile); break;
    case 3: launch_groups<3, KIND>(s, groups, ng, tile); break;
    default: launch_groups<4, KIND>(s, groups, ng, tile); break;
  }
}

}  // namespace

// groups of 8 k values of a packed row with K values: four equal quarters of whole chunks
int xop_chunk(int K) {  // the chunk of 2, 3 or 4 groups that pads a quarter least
  const int q = (K + 31) / 32;  // groups of a quarter
  if (q <= 4) return q;
  int best = 4;
  for (int ch = 3; ch >= 2; --ch)
    if ((q + ch - 1) / ch * ch < (q + best - 1) / best * best) best = ch;
  return best;
}
int xop_groups(int K) {
  const int q = (K + 31) / 32, ch = xop_chunk(K);
  return 4 * ((q + ch - 1) / ch * ch);
}

// The tile follows from the launch's size, 16 x 16 tiles times groups of 8 k values (twice when
// folding out), us per launch on MI355X in a graph of such launches, 16 x 16 against 32 x 16 with the
// k range split over a block's four wavefronts, and the staged kernel it replaces (full operator):
//   128^2 x 12 entries, blocks (6,144):   3.41 / 3.51  (5.65)     192^2 x 3 (5,184):  3.54 / 3.74  (7.38)
//   128^2 x 36 (18,432):                  5.76 / 5.34  (9.04)     257^2 x 3 (22,032): 6.50 / 5.81  (10.3)
//   192^2 x 36 (62,208):                  12.3 / 10.2  (19.0)     257^2 x 36 (264,384): 36.8 / 28.8  (45.6)
//   64^2 x 3 (384): 2.67 / 2.79 (4.00), of which 1.66 is an empty launch.
// Beyond a million the wavefronts of a block take a tile of their own each, 64 x 64 together, which
// halves the loads per product: 510^2 x 64 (2.1 million) 179 us, 47 TFLOP/s, against 195 us.
void xgemm(hipStream_t s, const XGemm* groups, int ng) {
  if (ng < 1 || ng > XGEMM_GROUPS) throw std::invalid_argument("xgemm: bad group count");
  const int kind = groups[0].op.kind == XOP_DENSE ? XOP_BLOCKS : groups[0].op.kind;
  const int ch = xop_chunk(groups[0].op.K[0] > groups[0].op.K[1] ? groups[0].op.K[0] : groups[0].op.K[1]);
  long size = 0;
  for (int i = 0; i < ng; ++i) {
    const XGemm& g = groups[i];
    if (g.entries < 1 || g.N < 1 || g.op.M[0] < 1 || !g.B || !g.C || g.op.M[1] > g.op.M[0])
      throw std::invalid_argument("xgemm: bad sizes");
    if ((g.op.kind == XOP_DENSE ? XOP_BLOCKS : g.op.kind) != kind || g.op.groups != groups[0].op.groups)
      throw std::invalid_argument("xgemm: the groups' operators differ in kind or length");
    const int ncls = g.op.kind == XOP_DENSE ? 1 : 2;
    size += (long)((g.N + 15) / 16) * ((g.op.M[0] + 15) / 16) * ncls * g.entries * g.op.groups;
  }
  const int tile = size < 18000 ? TILE_16 : size < 1000000 ? TILE_32 : TILE_64;
  if (kind == XOP_FOLD_IN) launch_chunk<XOP_FOLD_IN>(s, groups, ng, tile, ch);
  else if (kind == XOP_FOLD_OUT) launch_chunk<XOP_FOLD_OUT>(s, groups, ng, tile, ch);
  else launch_chunk<XOP_BLOCKS>(s, groups, ng, tile, ch);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string("xgemm: ") + hipGetErrorString(e));
}

}  // namespace rbc
