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

// TR: the result is written transposed (C^T = op B, the operands of the MFMAs exchanged so that the
// stores stay contiguous).  A product along y is a product along x of the transposed field, so a
// two-dimensional transform is two such products, each reading and writing whole lines.
// NC: parity classes of a block.  Folding in, both classes use the same loads; folding out and
// transposed both classes' results share their lines of C.
template <int KIND, bool TR>
constexpr int classes_of() {
  return KIND == XOP_DENSE ? 1 : KIND == XOP_BLOCKS ? (TR ? 2 : 1) : 2;
}

// The values from element off on of an array whose valid part ends at element `end`, as a buffer: loads
// beyond it give zero.  Base and bound stay in scalar registers, so a load of row k of an operand costs no
// vector instruction but itself; 64-bit addresses, clamped rows and selects per value cost a tenth of the
// kernels' time (510^2 x 64 200 -> 186 us, the convective products of 257^2 15.3 -> 13.5).
using Buffer = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ Buffer rows_from(const double* base, long off, long end) {
  const long left = (end - off) * 8;
  const int n = left <= 0 ? 0 : left > 0x7ffffff8L ? 0x7ffffff8 : (int)left;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(base + off), 0, n, 0x00020000);
}
__device__ __forceinline__ double value_at(Buffer b, unsigned byte) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, byte, 0, 0));
}

// (q0 + q1) + (q2 + q3) of the four wavefronts' partial tiles e < NE, in LDS: get(e, r) gives the
// calling wavefront's register r of tile e, put(e, v) takes the sum of register wid.
template <int NE, class Get, class Put>
__device__ __forceinline__ void add_quarters(double* part, int wid, int lane, Get get, Put put) {
#pragma unroll
  for (int e = 0; e < NE; ++e)
#pragma unroll
    for (int r = 0; r < 4; ++r) part[((e * 4 + wid) * 4 + r) * 64 + lane] = get(e, r);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    double q[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) q[w] = part[((e * 4 + w) * 4 + wid) * 64 + lane];
    put(e, (q[0] + q[1]) + (q[2] + q[3]));
  }
}

// A wavefront computes 16 FM x 16 FN values.  SPLIT: the four wavefronts of a block share one
// such tile, a quarter of the k range each; otherwise they hold 2 x 2 tiles and each runs the
// quarters in turn.  KIND: the groups' operators' (folding out, a group may hold block
// operators too).  CH: groups of 8 k values per chunk of loads.
template <int FM, int FN, bool SPLIT, int CH, int KIND, int NG, bool TR>
__global__ __launch_bounds__(256, 2) void xgemm_kernel(XArgs<NG> ar) {
  constexpr bool IN2 = KIND == XOP_FOLD_IN;
  constexpr int NC = classes_of<KIND, TR>(), ND = IN2 ? 1 : NC;  // ND: distinct sets of data loads
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
  const bool halves = KIND == XOP_BLOCKS && NC == 1;
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
  // class c of the block (both, or its own)
  const double* Ac[NC];
  int Kc[NC], r0[NC];
  const double* Bc[NC];  // the class's first input row, and its extent
  long end[NC];
  bool any = false;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const bool one = NC == 2 ? c == 1 : c1;
    any = any || m0 < pick(one, g.op.mnz[0], g.op.mnz[1]);  // else past a cut: zero rows
    Kc[c] = pick(one, g.op.K[0], g.op.K[1]);
    r0[c] = pick(one, g.op.r0[0], g.op.r0[1]);
    Ac[c] = pick(one, a0, a1) + aoff + (size_t)(m0 >> 4) * G * 128;
    Bc[c] = B + (long)r0[c] * ldb;
    end[c] = (long)(Kc[c] - 1) * rs * ldb + N;
  }
  const double* Bn[FN];  // this lane's columns (past N: a column inside, never stored)
  unsigned at[FN][2];    // and its two k values of a group there
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = min(n0 + 16 * j + lr, N - 1);
    Bn[j] = B + col;
    at[j][0] = 8u * (unsigned)(2 * lk * rs * ldb + col);
    at[j][1] = at[j][0] + 8u * (unsigned)(rs * ldb);
  }
  const long kst = ldb;  // from one input row of the operator to the next

  struct Chunk {
    double2 a[NC][CH][FM], b[ND][CH][FN], m[IN2 ? CH : 1][IN2 ? FN : 1];
  };
  auto load = [&](int g0, Chunk& x) {  // groups g0 .. g0 + CH - 1
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int h = 0; h < CH; ++h) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
          x.a[c][h][i] = reinterpret_cast<const double2*>(Ac[c] + ((size_t)i * G + g0 + h) * 128)[lane];
        if (c >= ND) continue;
        if constexpr (IN2) {  // clamped rows: the mirrored ones run down, past no bound that a buffer has
          const int k = (g0 + h) * 8 + 2 * lk;
          const int q0 = r0[c] + rs * min(k, Kc[c] - 1), q1 = r0[c] + rs * min(k + 1, Kc[c] - 1);
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            x.b[c][h][j].x = Bn[j][q0 * kst];
            x.b[c][h][j].y = Bn[j][q1 * kst];
            x.m[h][j].x = Bn[j][(last - q0) * kst];
            x.m[h][j].y = Bn[j][(last - q1) * kst];
          }
        } else {
          const Buffer w = rows_from(Bc[c], (long)(g0 + h) * 8 * rs * ldb, end[c]);
#pragma unroll
          for (int j = 0; j < FN; ++j) x.b[c][h][j] = double2{value_at(w, at[j][0]), value_at(w, at[j][1])};
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
        const bool ok0 = k < Kc[c], ok1 = k + 1 < Kc[c];
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          double2 b = x.b[c < ND ? c : 0][h][j];
          if constexpr (IN2) {
            b.x = c ? b.x - x.m[h][j].x : b.x + x.m[h][j].x;
            b.y = c ? b.y - x.m[h][j].y : b.y + x.m[h][j].y;
            b.x = ok0 ? b.x : 0.0;  // the packed rows end in zeros, the clamped rows do not
            b.y = ok1 ? b.y : 0.0;
          }
#pragma unroll
          for (int i = 0; i < FM; ++i) {
            const double2 a = x.a[c][h][i];
            acc[c][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(TR ? b.x : a.x, TR ? a.x : b.x, acc[c][i][j], 0, 0, 0);
            acc[c][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(TR ? b.y : a.y, TR ? a.y : b.y, acc[c][i][j], 0, 0, 0);
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
  // the values a lane writes: register r of its MFMA results, all four of them or, with the k range
  // split, the wavefront's own r (each wavefront adds and stores a quarter of the tile)
  constexpr int RN = SPLIT ? 1 : 4;
  double res[NC][FM][FN][RN];
  if constexpr (SPLIT) {
    const int g0 = wid * nch * CH;
    clear();
    if (any) {
      load(g0, x);
      quarter(g0);
    }
    __shared__ double part[NC * FM * FN * 16 * 64];
    add_quarters<NC * FM * FN>(part, wid, lane, [&](int e, int r) { return acc[e / (FM * FN)][e / FN % FM][e % FN][r]; },
                               [&](int e, double v) { res[e / (FM * FN)][e / FN % FM][e % FN][0] = v; });
  } else {
    v4d pair[NC][FM][FN];
    __shared__ v4d sum[NC][FM][FN][256];
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
              if (q == 0) sum[c][i][j][tid] = acc[c][i][j];
              else if (q == 2) pair[c][i][j] = acc[c][i][j];
              else if (q == 1) sum[c][i][j][tid] += acc[c][i][j];
              else acc[c][i][j] = sum[c][i][j][tid] + (pair[c][i][j] + acc[c][i][j]);
            }
      }
    } else {
      clear();
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) res[c][i][j][SPLIT ? 0 : r] = acc[c][i][j][r];
  }
  const int ldc = g.ldc, rows = g.op.rows, cs = g.op.cstep;
  const bool pin = g.zero00 != 0, out2 = KIND == XOP_FOLD_OUT && g.op.kind == XOP_FOLD_OUT;
  const int e0 = pick(c1, g.op.c0[0], g.op.c0[1]), e1 = g.op.c0[1], M1 = g.op.M[1];
  auto put = [&](int row, int col, double v) {  // row of the operator, column of the data
    if (pin && row == 0 && col == 0) v = 0.0;
    C[TR && !g.plain ? (size_t)col * ldc + row : (size_t)row * ldc + col] = v;
  };
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < RN; ++q) {
        const int r = SPLIT ? wid : q;
        const int m = m0 + i * 16 + (TR ? lr : 4 * r + lk), n = n0 + j * 16 + (TR ? 4 * r + lk : lr);
        if (m >= M || n >= N) continue;
        const double v = res[0][i][j][q];
        if constexpr (NC == 2) {
          const double o = res[1][i][j][q];
          if (out2) {
            const int mirror = rows - 1 - m;
            put(m, n, v + o);
            if (mirror != m) put(mirror, n, v - o);
          } else {
            put(e0 + cs * m, n, v);
            if (m < M1) put(e1 + cs * m, n, o);
          }
        } else {
          put(e0 + cs * m, n, v);
        }
      }
}

// conv_products: a block computes rows [m0, m0 + 16) and their mirror rows of 16 columns, its four
// wavefronts a quarter of the k range each: the products
//   u = bs T_ux, v = bs T_uy, and per field d/dx q = bs D_q, d/dy q = bds T_q,
// of two parity classes each, combined point by point.  NF = 1: one field per block, u and v formed
// again for each; NF = 3: the three fields in one block (8 products in place of 12, on 16 tiles of
// accumulators per wavefront).  One launch in place of four (the velocity, two
// products with an epilogue, the boundary field's gradient).
template <int CH, int NF, int W>
__global__ __launch_bounds__(256, W) void conv_kernel(ConvArgs a, int tx, int ty) {
  constexpr int ND = NF == 3 ? 6 : 4, NP = NF == 3 ? 8 : 4;  // data arrays, products
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  int t = fftlds::xcd_remap(blockIdx.x, gridDim.x);
  const int n0 = (t % tx) * 16;
  t /= tx;
  const int m0 = (t % ty) * 16, z = t / ty, b = z % a.nb, f = NF == 3 ? 0 : a.f0 + z / a.nb, N = a.nx;
  const int col = min(n0 + lr, N - 1), G = a.bs.groups;
  // NF = 1: T_ux, T_uy, D_f, T_f; NF = 3: T and D of the three fields
  const double* src[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int ff = NF == 3 ? i % 3 : i < 2 ? i : f;
    src[i] = (NF == 3 ? i < 3 : i != 2) ? a.T : a.D;
    src[i] += a.stride * (ff * a.nb + b);
  }
  const unsigned at0 = 8u * (unsigned)(4 * lk * N + col), at1 = at0 + 16u * (unsigned)N;
  const double* opa[2][2];  // [bs, bds][class]
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    opa[0][c] = a.bs.a[c] + (size_t)(m0 >> 4) * G * 128;
    opa[1][c] = a.bds.a[c] + (size_t)(m0 >> 4) * G * 128;
  }
  // rows of row parity p: 2 k + p below cols; class c of bs takes parity rb[c], of bds rd[c]
  const int Kp[2] = {a.bs.r0[0] == 0 ? a.bs.K[0] : a.bs.K[1], a.bs.r0[0] == 0 ? a.bs.K[1] : a.bs.K[0]};
  const int pb = a.bs.r0[0], pd = a.bds.r0[0];  // parity of class 0
  struct Chunk {
    double2 o[2][2][CH], d[ND][2][CH];  // [operator][class], [array][row parity]
  };
  v4d acc[NP][2];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[p][c] = v4d{0, 0, 0, 0};
  auto load = [&](int g0, Chunk& x) {
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
          x.o[p][c][h] = reinterpret_cast<const double2*>(opa[p][c] + (size_t)(g0 + h) * 128)[lane];
#pragma unroll
        for (int i = 0; i < ND; ++i) {
          const Buffer w = rows_from(src[i] + c * N, (long)(g0 + h) * 16 * N, (long)(2 * Kp[c] - 1) * N);
          x.d[i][c][h] = double2{value_at(w, at0), value_at(w, at1)};
        }
      }
  };
  // operator and data array of product p
  auto op_of = [](int p) { return NF == 3 ? p >= 5 : p == 3; };
  auto data_of = [](int p) { return NF == 3 ? (p < 2 ? p : p < 5 ? p + 1 : p - 5) : p; };
  auto mac = [&](const Chunk& x) {
#pragma unroll
    for (int h = 0; h < CH; ++h) {
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const double2 o = x.o[op_of(p) ? 1 : 0][c][h];
          const bool odd = (c ^ (op_of(p) ? pd : pb)) != 0;
          const double2 &d0 = x.d[data_of(p)][0][h], &d1 = x.d[data_of(p)][1][h];
          const double v0 = odd ? d1.x : d0.x, v1 = odd ? d1.y : d0.y;
          acc[p][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.x, v0, acc[p][c], 0, 0, 0);
          acc[p][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.y, v1, acc[p][c], 0, 0, 0);
        }
    }
  };
  Chunk x, y;
  const int nch = G / (4 * CH), top = G - CH, g0 = wid * nch * CH;
  load(g0, x);
  int n = 0;
  for (; n + 2 <= nch; n += 2) {
    load(min(g0 + (n + 1) * CH, top), y);
    mac(x);
    load(min(g0 + (n + 2) * CH, top), x);
    mac(y);
  }
  if (n < nch) mac(x);
  const int ny = a.bs.rows;
  double res[NP][2];
  __shared__ double part[8 * 16 * 64];
#pragma unroll
  for (int h = 0; h < NP / 4; ++h) {  // four products at a time through LDS
    if (h) __syncthreads();
    add_quarters<8>(part, wid, lane, [&](int e, int r) { return acc[4 * h + (e >> 1)][e & 1][r]; },
                    [&](int e, double v) { res[4 * h + (e >> 1)][e & 1] = v; });
  }
  const int m = m0 + 4 * wid + lk, nn = n0 + lr;
  if (m >= a.bs.M[0] || nn >= N) return;
#pragma unroll
  for (int side = 0; side < 2; ++side) {
#pragma clang fp contract(off)
    const int row = side ? ny - 1 - m : m;
    if (side && row == m) continue;
    double v[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) v[p] = side ? res[p][0] - res[p][1] : res[p][0] + res[p][1];
    const size_t at = (size_t)row * N + nn;
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const int ff = NF == 3 ? i : f;
      double q = (NF == 3 ? v[2 + i] : v[2]) * v[0];
      q = q + (NF == 3 ? v[5 + i] : v[3]) * v[1];
      if (ff == 2) {
        q = q + v[0] * a.fx[a.sf * b + at];
        q = q + v[1] * a.fy[a.sf * b + at];
      }
      a.C[a.stride * (ff * a.nb + b) + at] = q;
    }
  }
}

// adjoint_products: as conv_kernel with one of the three terms per block, the four products
//   ux:   bs D_u, bds T_u, bs D_v, bs D_t      uy:   bs D_v, bds T_v, bds T_u, bds T_t
//   temp: bs D_t, bds T_t (the other two repeat them: its blocks end with the others')
// of the residuals' x-transformed values T and derivatives D, taken with the fields' values at the
// point: one launch in place of 14 terms of four launches each.
template <int CH>
__global__ __launch_bounds__(256, 2) void adjoint_kernel(AdjointConvArgs a, int tx, int ty) {
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  int t = fftlds::xcd_remap(blockIdx.x, gridDim.x);
  const int n0 = (t % tx) * 16;
  t /= tx;
  const int m0 = (t % ty) * 16, f = t / ty, N = a.nx;
  const int col = min(n0 + lr, N - 1), G = a.bs.groups;
  // product p: operator 0 bs, 1 bds; its array
  const int op[4] = {0, 1, f == 0 ? 0 : f == 1 ? 1 : 0, f == 0 ? 0 : 1};
  const int field[4] = {f, f, f == 2 ? 2 : 1 - f, 2};
  const double* opa[4][2];
  const double* src[4][2];
  int K[4][2];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const double* base = op[p] ? a.bds.a[c] : a.bs.a[c];
      opa[p][c] = base + (size_t)(m0 >> 4) * G * 128;
      const int r0 = op[p] ? a.bds.r0[c] : a.bs.r0[c];
      K[p][c] = op[p] ? a.bds.K[c] : a.bs.K[c];
      src[p][c] = (op[p] ? a.T : a.D) + a.stride * field[p] + (long)r0 * N;
    }
  const unsigned at0 = 8u * (unsigned)(4 * lk * N + col), at1 = at0 + 16u * (unsigned)N;
  struct Chunk {
    double2 o[4][2][CH], d[4][2][CH];
  };
  v4d acc[4][2];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[p][c] = v4d{0, 0, 0, 0};
  auto load = [&](int g0, Chunk& x) {
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          x.o[p][c][h] = reinterpret_cast<const double2*>(opa[p][c] + (size_t)(g0 + h) * 128)[lane];
          const Buffer w = rows_from(src[p][c], (long)(g0 + h) * 16 * N, (long)(2 * K[p][c] - 1) * N);
          x.d[p][c][h] = double2{value_at(w, at0), value_at(w, at1)};
        }
  };
  auto mac = [&](const Chunk& x) {
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          acc[p][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.o[p][c][h].x, x.d[p][c][h].x, acc[p][c], 0, 0, 0);
          acc[p][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.o[p][c][h].y, x.d[p][c][h].y, acc[p][c], 0, 0, 0);
        }
  };
  Chunk x, y;
  const int nch = G / (4 * CH), top = G - CH, g0 = wid * nch * CH;
  load(g0, x);
  int n = 0;
  for (; n + 2 <= nch; n += 2) {
    load(min(g0 + (n + 1) * CH, top), y);
    mac(x);
    load(min(g0 + (n + 2) * CH, top), x);
    mac(y);
  }
  if (n < nch) mac(x);
  const int ny = a.bs.rows;
  double res[4][2];
  __shared__ double part[8 * 16 * 64];
  add_quarters<8>(part, wid, lane, [&](int e, int r) { return acc[e >> 1][e & 1][r]; },
                  [&](int e, double v) { res[e >> 1][e & 1] = v; });
  const int m = m0 + 4 * wid + lk, nn = n0 + lr;
  if (m >= a.bs.M[0] || nn >= N) return;
#pragma unroll
  for (int side = 0; side < 2; ++side) {
#pragma clang fp contract(off)
    const int row = side ? ny - 1 - m : m;
    if (side && row == m) continue;
    double v[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) v[p] = side ? res[p][0] - res[p][1] : res[p][0] + res[p][1];
    const size_t at = (size_t)row * N + nn;
    const double U = a.V[at], V = a.V[a.stride + at];
    double q = U * v[0] + V * v[1];
    if (f < 2) {  // the terms in the order of navier_adjoint.rs:581-626
      q = q + U * (f == 0 ? v[0] : v[2]);
      q = q + V * (f == 0 ? v[2] : v[1]);
      q = q + a.V[2 * a.stride + at] * v[3];
      q = q + a.bc[at] * v[3];
    }
    a.C[a.stride * f + at] = q;
  }
}

template <int FM, int FN, bool SPLIT, int CH, int KIND, int NG, bool TR>
void launch(hipStream_t s, const XGemm* groups) {
  constexpr int BM = 16 * FM * (SPLIT ? 1 : 2), BN = 16 * FN * (SPLIT ? 1 : 2);
  XArgs<NG> ar{};
  long total = 0;
  for (int i = 0; i < NG; ++i) {
    ar.g[i] = groups[i];
    ar.tx[i] = (groups[i].N + BN - 1) / BN;
    ar.ty[i] = (groups[i].op.M[0] + BM - 1) / BM;
    const int ncls = KIND == XOP_BLOCKS && classes_of<KIND, TR>() == 1 ? 2 : 1;  // blocks per tile
    total += (long)ar.tx[i] * ar.ty[i] * ncls * groups[i].entries;
    if (total > 0x7fffffffL) throw std::invalid_argument("xgemm: too many tiles");
    ar.end[i] = (int)total;
  }
  RBC_LAUNCH((xgemm_kernel<FM, FN, SPLIT, CH, KIND, NG, TR>), dim3((unsigned)total), dim3(256), 0, s, ar);
}

enum { TILE_16, TILE_32, TILE_64 };

template <int CH, int KIND, int NG, bool TR>
void launch_tile(hipStream_t s, const XGemm* groups, int tile) {
  // the larger tiles take shorter chunks: fewer registers, more wavefronts per SIMD
  constexpr int CS = CH == 4 ? 2 : CH == 3 ? 1 : CH;
  switch (tile) {
    case TILE_16: launch<1, 1, true, CH, KIND, NG, TR>(s, groups); break;
    case TILE_32: launch<2, 1, true, CS, KIND, NG, TR>(s, groups); break;
    default: launch<2, 2, false, 1, KIND, NG, TR>(s, groups); break;
  }
}

template <int KIND, int NG, bool TR>
void launch_chunk(hipStream_t s, const XGemm* groups, int tile, int ch) {
  switch (ch) {
    case 1: launch_tile<1, KIND, NG, TR>(s, groups, tile); break;
    case 2: launch_tile<2, KIND, NG, TR>(s, groups, tile); break;
    case 3: launch_tile<3, KIND, NG, TR>(s, groups, tile); break;
    default: launch_tile<4, KIND, NG, TR>(s, groups, tile); break;
  }
}

template <bool TR>
void launch_kind(hipStream_t s, const XGemm* groups, int ng, int kind, int tile, int ch) {
  if (ng > 1) {
    if (kind == XOP_FOLD_OUT) launch_chunk<XOP_FOLD_OUT, XGEMM_GROUPS, TR>(s, groups, tile, ch);
    else if (kind == XOP_DENSE) launch_chunk<XOP_DENSE, XGEMM_GROUPS, TR>(s, groups, tile, ch);
    else launch_chunk<XOP_BLOCKS, XGEMM_GROUPS, TR>(s, groups, tile, ch);
    return;
  }
  switch (kind) {
    case XOP_FOLD_IN: launch_chunk<XOP_FOLD_IN, 1, TR>(s, groups, tile, ch); break;
    case XOP_FOLD_OUT: launch_chunk<XOP_FOLD_OUT, 1, TR>(s, groups, tile, ch); break;
    case XOP_BLOCKS: launch_chunk<XOP_BLOCKS, 1, TR>(s, groups, tile, ch); break;
    default: launch_chunk<XOP_DENSE, 1, TR>(s, groups, tile, ch); break;
  }
}

}  // namespace

// groups of 8 k values of a packed row with K values: four equal quarters of whole chunks
int xop_chunk(int groups) {  // the longest chunk of at most 4 groups that divides a quarter
  const int q = groups / 4;
  for (int ch = q < 4 ? q : 4; ch > 1; --ch)
    if (q % ch == 0) return ch;
  return 1;
}
int xop_groups(int K) {
  const int q = (K + 31) / 32;  // groups of a quarter
  if (q <= 4) return 4 * q;
  int best = 4;  // the chunk of 2, 3 or 4 groups that pads the quarter least
  for (int ch = 3; ch >= 2; --ch)
    if ((q + ch - 1) / ch * ch < (q + best - 1) / best * best) best = ch;
  return 4 * ((q + best - 1) / best * best);
}

void conv_products(hipStream_t s, const ConvArgs& a) {
  if (a.bs.kind != XOP_FOLD_OUT || a.bds.kind != XOP_FOLD_OUT || a.bs.groups != a.bds.groups ||
      a.bs.rows != a.bds.rows || a.bs.cols != a.bds.cols || a.f0 < 0 || a.f1 > 3 || a.f0 >= a.f1 || a.nx < 1 || a.nx > (1 << 24) || a.nb < 1)
    throw std::invalid_argument("conv_products: bad arguments");
  if (a.bs.rstep != 2 || a.bds.rstep != 2) throw std::invalid_argument("conv_products: bad operators");
  const int tx = (a.nx + 15) / 16, ty = (a.bs.M[0] + 15) / 16;
  const long tiles = (long)tx * ty * a.nb;
  // one field per block while these are at most two per CU, else the three in one (us, one / three: 64^2,
  // 12 instances (288 blocks of one field) 5.3 / 6.1, 36 (864) 9.6 / 7.6; 96^2, 6 (324) 7.1 / 8.9, 12 (648)
  // 10.6 / 8.8; 128^2, 6 (576) 10.6 / 9.6; 192^2, 2 (432) 9.2 / 11.0, 3 (648) 12.9 / 11.0; 257^2, 1 (459)
  // 13.2 / 13.5, 3 (1,377) 30.5 / 23.2, 12 98.6 / 71.3).  A wavefront per tile with the whole k range is no
  // faster (192^2, 36: 85 us against 67, 3: 30 against 11).
  const bool three = a.f0 == 0 && a.f1 == 3 && 3 * tiles > 512;
  const long total = tiles * (three ? 1 : a.f1 - a.f0);
  if (total > 0x7fffffffL) throw std::invalid_argument("conv_products: too many tiles");
  const dim3 grid((unsigned)total), block(256);
  // W blocks per CU: two hide each other's loads and sums (257^2, 12 instances: 87 us with one, 71 with
  // two; 128^2, 12: 16.0 / 14.2); where there is one per CU at most it takes all registers (153 blocks, 257^2:
  // 13.5 with one, 15.3 with two)
  if (three && tiles <= 256) RBC_LAUNCH((conv_kernel<1, 3, 1>), grid, block, 0, s, a, tx, ty);
  else if (three) RBC_LAUNCH((conv_kernel<1, 3, 2>), grid, block, 0, s, a, tx, ty);
  else if (a.bs.groups / 4 % 2 == 0) RBC_LAUNCH((conv_kernel<2, 1, 2>), grid, block, 0, s, a, tx, ty);
  else RBC_LAUNCH((conv_kernel<1, 1, 2>), grid, block, 0, s, a, tx, ty);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string("conv_products: ") + hipGetErrorString(e));
}

void adjoint_products(hipStream_t s, const AdjointConvArgs& a) {
  if (a.bs.kind != XOP_FOLD_OUT || a.bds.kind != XOP_FOLD_OUT || a.bs.groups != a.bds.groups ||
      a.bs.rows != a.bds.rows || a.bs.cols != a.bds.cols || a.bs.rstep != 2 || a.bds.rstep != 2 || a.nx < 1 || a.nx > (1 << 24))
    throw std::invalid_argument("adjoint_products: bad arguments");
  const int tx = (a.nx + 15) / 16, ty = (a.bs.M[0] + 15) / 16;
  const long total = 3L * tx * ty;
  if (total > 0x7fffffffL) throw std::invalid_argument("adjoint_products: too many tiles");
  RBC_LAUNCH((adjoint_kernel<1>), dim3((unsigned)total), dim3(256), 0, s, a, tx, ty);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string("adjoint_products: ") + hipGetErrorString(e));
}

// The tile follows from the launch's size, 16 x 16 tiles times groups of 8 k values (twice when
// folding out), us per launch on MI355X in a graph of such launches, 16 x 16 against 32 x 16 with the
// k range split over a block's four wavefronts, and the staged kernel it replaces (full operator):
//   128^2 x 12 entries, blocks (6,144):   3.41 / 3.51  (5.65)     192^2 x 3 (5,184):  3.54 / 3.74  (7.38)
//   128^2 x 36 (18,432):                  5.76 / 5.34  (9.04)     257^2 x 3 (22,032): 6.50 / 5.81  (10.3)
//   192^2 x 36 (62,208):                  12.3 / 10.2  (19.0)     257^2 x 36 (264,384): 36.8 / 28.8  (45.6)
//   64^2 x 3 (384): 2.47 / 2.79 (4.00), of which 1.66 is an empty launch.
// Beyond 400,000 the wavefronts of a block take a tile of their own each, 64 x 64 together, which halves
// the loads per product, unless the larger tiles are more than a tenth of padding (32 x 16 / 64 x 64:
// 510^2 x 64 (2.1 million) 216 / 168, 50.5 TFLOP/s, 510^2 x 16 (524,288) 51 / 40, 510^2 x 4 (131,072) 14.5 /
// 14.5, folding in 512^2 x 8 (262,144) 29.4 / 31.7; 300^2 x 36, a quarter of padding, 33 / 44).  The sum of
// their first two quarters waits in LDS and the registers are bounded for two blocks per CU: 510^2 x 64
// takes 186 us with the sum in registers, 182 without the bound.
static void xgemm_any(hipStream_t s, const XGemm* in, int ng, bool transposed) {
  if (ng < 1 || ng > XGEMM_GROUPS) throw std::invalid_argument("xgemm: bad group count");
  XGemm groups[XGEMM_GROUPS];
  bool out = false;
  long size = 0, size64 = 0;  // the latter with the padding of 64 x 64 tiles
  for (int i = 0; i < ng; ++i) {
    const XGemm& g = groups[i] = in[i];
    out = out || g.op.kind == XOP_FOLD_OUT;
    if (g.entries < 1 || g.N < 1 || g.op.M[0] < 1 || !g.B || !g.C || g.op.M[1] > g.op.M[0])
      throw std::invalid_argument("xgemm: bad sizes");
    if (g.ldb > (1 << 24) || g.ldb < g.N) throw std::invalid_argument("xgemm: rows too long");
    if (g.op.groups != in[0].op.groups) throw std::invalid_argument("xgemm: the groups' operators differ in length");
    const int ncls = g.op.kind == XOP_DENSE ? 1 : 2;
    const long per = (long)ncls * g.entries * g.op.groups;
    size += (long)((g.N + 15) / 16) * ((g.op.M[0] + 15) / 16) * per;
    size64 += 16L * ((g.N + 63) / 64) * ((g.op.M[0] + 63) / 64) * per;
  }
  if (ng > 1) {
    for (int i = 0; i < ng; ++i)
      if (in[i].op.kind == XOP_FOLD_IN || (in[i].op.kind == XOP_DENSE) != (in[0].op.kind == XOP_DENSE))
        throw std::invalid_argument("xgemm: these operators do not share a launch");
    for (int i = ng; i < XGEMM_GROUPS; ++i) {  // an empty group
      groups[i] = groups[0];
      groups[i].entries = 0;
    }
  }
  const int kind = out ? (int)XOP_FOLD_OUT : groups[0].op.kind, ch = xop_chunk(groups[0].op.groups);
  const int tile = size < 18000 ? TILE_16 : size < 400000 || 10 * size64 > 11 * size ? TILE_32 : TILE_64;
  if (transposed) launch_kind<true>(s, groups, ng, kind, tile, ch);
  else launch_kind<false>(s, groups, ng, kind, tile, ch);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string("xgemm: ") + hipGetErrorString(e));
}

void xgemm(hipStream_t s, const XGemm* groups, int ng) { xgemm_any(s, groups, ng, false); }
void xgemm_t(hipStream_t s, const XGemm* groups, int ng) { xgemm_any(s, groups, ng, true); }

}  // namespace rbc
