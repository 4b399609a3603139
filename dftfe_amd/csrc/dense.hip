// Dense FP64 steps of CholGS and Rayleigh-Ritz on the tall node-major block
// X (M x N, M ~ 10^6, N ~ 10^3) as FP64 MFMA kernels:
//   * gram:   C = A^T B over all M rows (the overlap X^T X and the projected
//             Hamiltonian X^T (H~X)), lower-triangle tiles only when asked,
//             split over M into chunks whose partial tiles are summed in a
//             fixed order (deterministic);
//   * rotate: Y = X R over row panels (R = Q, the Ritz rotation, or a column
//             block of R = L^{-T}, the Cholesky-Gram-Schmidt one, with the
//             inner extent cut at the block's last row: the blocks below the
//             diagonal are zero).
// Reference steps replaced: fillParallelOverlapMatScalapack
// (src/linAlg/linearAlgebraOperationsDevice.cc:3078-3240), XtHX
// (src/dftOperator/kohnShamDFTOperatorDevice.cc:4000-4157),
// subspaceRotationScalapack (linearAlgebraOperationsDevice.cc:1832-2242) and
// the rotations of pseudoGSDevice.cc / rayleighRitzDevice.cc, which call
// hipBLAS dgemm per block.

#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "dense.hpp"
#include "mfma.hpp"

namespace chfsi {

namespace {

constexpr int TT = kRotateTile;  // output tile edge
constexpr int KS = 16;    // K rows per LDS slab
constexpr int NT = 256;   // 4 waves (wi, wj): blocks of 16 (2a + wi, 2b + wj), a, b < 4
// rows of a gram chunk at least: gram of 64 columns on 110k rows 0.49 ms with 4096, 0.20
// with 1024, 0.13 with 512, 0.14 with 256
constexpr int kMinRows = 512;
constexpr int PADW = 16;  // LDS row padding of [k][128] slabs (doubles)

// Work items are spread over the 8 XCDs so that consecutive items (the tiles
// of one K chunk in gram, the column tiles of one row panel in rotate) share
// an XCD and its L2.
__device__ __forceinline__ int xcd_item(int per_xcd) {
  const int wid = blockIdx.x;
  return (wid & 7) * per_xcd + (wid >> 3);
}

// acc[a][b] += A block a x B block b over one slab, for the blocks in MASK (bit 4 a + b).
// A[k][row] is at as[k AK + row AR], B[k][column] at bs[k BK + column BR], from the lane's
// own k, row and column on.
template <unsigned MASK, int AK, int AR, int BK, int BR>
__device__ __forceinline__ void blocks(const double *as, const double *bs, f64x4 (&acc)[4][4]) {
#pragma unroll
  for (int kk = 0; kk < KS / 4; ++kk) {
    double av[4], bv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (MASK >> (4 * q) & 15) av[q] = as[kk * 4 * AK + q * 32 * AR];
      if (MASK >> q & 0x1111) bv[q] = bs[kk * 4 * BK + q * 32 * BR];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (MASK >> (4 * a + b) & 1) acc[a][b] = mfma16(av[a], bv[b], acc[a][b]);
  }
}

// Sets of blocks (bit 4 a + b) that the kernels are compiled for.  One set serves the
// four waves of a workgroup: branches around single MFMAs made the compiler copy
// accumulators (190 spilled registers).  gram: all; on and below the diagonal; tiles
// with 96 / 64 rows and their diagonal forms.  rotate: all columns, 96, 64, 32.
constexpr int kGramForms = 6;
constexpr unsigned kGramForm[kGramForms] = {0xffff, 0xf731, 0x0fff, 0x0731, 0x00ff, 0x0031};
constexpr unsigned kColumnForm[4] = {0x1111, 0x3333, 0x7777, 0xffff};

__host__ __device__ inline int gram_form(int I, int J, int m, int diag_off) {
  const int na = m - I > 96 ? 0 : (m - I > 64 ? 2 : 4);
  return na + (diag_off >= 0 && J + diag_off >= I ? 1 : 0);
}

// Pairs c + 32 e of a row of n into r, entries past its end read from entry 0.
// VEC: 16-byte loads (rows 16-byte aligned, c and n even, so that a pair lies
// inside or outside the row).
template <bool VEC>
__device__ __forceinline__ void load8(const double *row, int c, int n, double2 (&r)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = c + 32 * e;
    if (VEC)
      r[e] = *reinterpret_cast<const double2 *>(row + (i < n ? i : 0));
    else
      r[e] = double2{row[i < n ? i : 0], row[i + 1 < n ? i + 1 : 0]};
  }
}

// Pair c of the rows r0 + r + 32 e of n entries, those past the last row read from row r0.
template <bool VEC>
__device__ __forceinline__ void load_rows(const double *M, int64_t ld, int64_t r0, int r,
                                          int64_t rows, int c, int n, double2 (&v)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double *row = M + (r0 + r + 32 * e < rows ? r0 + r + 32 * e : r0) * ld;
    if (VEC)
      v[e] = *reinterpret_cast<const double2 *>(row + (c < n ? c : 0));
    else
      v[e] = double2{row[c < n ? c : 0], row[c + 1 < n ? c + 1 : 0]};
  }
}

}  // namespace

// Bound by the FP64 matrix cores.  The loads of slab s + 1 are issued before the MFMAs
// of slab s and first used when they are stored behind them; with the masks applied
// at the load every slab waited for them (500 columns on 216k rows: 1.77 ms, then 1.39;
// 1.33 with the blocks below, 1.19 with whole lines staged and shorter chunks).
//
// C_tile(I, J) = sum_{k in chunk} A[k, I + i] B[k, J + j], written to
// P[part][i + 128 j].  Blocks of 16 past the edge or above the diagonal are left out
// (zero in P); dealing the blocks to the waves alternately leaves each of them 10 of 16
// in a diagonal tile.
template <bool VEC>
__global__ __launch_bounds__(NT, 2) void gram_kernel(const double *A, int64_t lda, const double *B,
                                                     int64_t ldb, int m, int n, int64_t K,
                                                     int diag_off, const GramItem *items,
                                                     int per_xcd, int nitems, double *P) {
  __shared__ __align__(16) double As[2][KS][TT + PADW];
  __shared__ __align__(16) double Bs[2][KS][TT + PADW];
  const int item = xcd_item(per_xcd);
  if ((blockIdx.x >> 3) >= per_xcd || item >= nitems) return;
  const GramItem it = items[item];
  const int I = it.I * TT, J = it.J * TT;
  const int64_t kb = (int64_t)it.slab * KS;
  const int64_t ke = kb + (int64_t)it.nslab * KS < K ? kb + (int64_t)it.nslab * KS : K;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wi = w & 1, wj = w >> 1;

  // staging: thread t loads row t/16 of the slab, the column pairs 2 (t%16) + 32 e (16
  // lanes a line of memory and all banks of LDS).  Indices past the block are clamped
  // and the values dropped when they are stored, so nothing waits for a load before
  // the MFMAs of the slab in between.
  const int lr = tid >> 4, lc = (tid & 15) * 2;
  double2 ra[4], rb[4];
  auto load = [&](int64_t k0) {
    const int64_t k = k0 + lr < ke ? k0 + lr : ke - 1;
    const double *ap = A + k * lda, *bp = B + k * ldb;
    load8<VEC>(ap, I + lc, m, ra);
    load8<VEC>(bp, J + lc, n, rb);
  };
  auto store = [&](int buf, int64_t k0) {
    const bool kok = k0 + lr < ke;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = I + lc + 32 * e, j = J + lc + 32 * e;
      *reinterpret_cast<double2 *>(&As[buf][lr][lc + 32 * e]) =
          double2{kok & (i < m) ? ra[e].x : 0.0, kok & (i + 1 < m) ? ra[e].y : 0.0};
      *reinterpret_cast<double2 *>(&Bs[buf][lr][lc + 32 * e]) =
          double2{kok & (j < n) ? rb[e].x : 0.0, kok & (j + 1 < n) ? rb[e].y : 0.0};
    }
  };

  const int nslab = (int)((ke - kb + KS - 1) / KS);
  auto run = [&](auto form) {
    constexpr unsigned MASK = decltype(form)::value;
    f64x4 acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = f64x4{0, 0, 0, 0};
    if (nslab > 0) {
      load(kb);
      store(0, kb);
    }
    __syncthreads();
    for (int s = 0; s < nslab; ++s) {
      const int buf = s & 1;
      if (s + 1 < nslab) load(kb + (int64_t)(s + 1) * KS);
      blocks<MASK, TT + PADW, 1, TT + PADW, 1>(&As[buf][lane >> 4][wi * 16 + (lane & 15)],
                                               &Bs[buf][lane >> 4][wj * 16 + (lane & 15)], acc);
      if (s + 1 < nslab) store(buf ^ 1, kb + (int64_t)(s + 1) * KS);
      __syncthreads();
    }
    double *Pt = P + (int64_t)it.part * TT * TT;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = (2 * a + wi) * 16 + acc_row<double>(lane, r);
          const int j = (2 * b + wj) * 16 + (lane & 15);
          Pt[i + (int64_t)j * TT] = acc[a][b][r];
        }
  };
  switch (gram_form(I, J, m, diag_off)) {
    case 0: run(std::integral_constant<unsigned, kGramForm[0]>{}); break;
    case 1: run(std::integral_constant<unsigned, kGramForm[1]>{}); break;
    case 2: run(std::integral_constant<unsigned, kGramForm[2]>{}); break;
    case 3: run(std::integral_constant<unsigned, kGramForm[3]>{}); break;
    case 4: run(std::integral_constant<unsigned, kGramForm[4]>{}); break;
    default: run(std::integral_constant<unsigned, kGramForm[5]>{}); break;
  }
}

// C[I + i + (J + j) ldc] = sum over chunks of the partial tiles (chunk order)
__global__ void gram_reduce_kernel(const double *P, const GramItem *tiles, int m, int n, double *C,
                                   int64_t ldc) {
  const GramItem t = tiles[blockIdx.y];
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= TT * TT) return;
  const int i = e % TT, j = e / TT;
  const int gi = t.I * TT + i, gj = t.J * TT + j;
  if (gi >= m || gj >= n) return;
  double s = 0.0;
  for (int c = 0; c < t.nslab; ++c) s += P[(int64_t)(t.part + c) * TT * TT + e];
  C[gi + (int64_t)gj * ldc] = s;
}

// Rows of R past diag + 16 (column / 16) + 15 hold zeros: those blocks are left out.
//
// Y[k, J + j] = sum_{i < K} X[k, i] R[i, J + j] for the rows [r0, r0 + rows)
// of the panel and J + j < N; R[i][j] = Rm[i + j ldr] (TR = 0) or
// Rm[j + i ldr] (TR = 1).  LDS slabs: X as [128 rows][KS + 1] (odd stride:
// the 16 rows of an A-operand read fall in distinct banks); R as
// [128 columns][KS + 1] when its columns are contiguous in memory (TR = 0),
// else [KS rows][128 + PADW].
template <int TR, bool VEC>
__global__ __launch_bounds__(NT, 2) void rotate_kernel(const double *X, int64_t ldx,
                                                       const double *Rm, int64_t ldr, int K,
                                                       int diag, int N, int64_t rows, double *Y,
                                                       int64_t ldy, int ntj, int per_xcd,
                                                       int nitems) {
  constexpr int XS = KS + 1;
  constexpr int RSZ = TR ? KS * (TT + PADW) : TT * XS;
  __shared__ __align__(16) double Xs[2][TT * XS];
  __shared__ __align__(16) double Rs[2][RSZ];
  const int item = xcd_item(per_xcd);
  if ((blockIdx.x >> 3) >= per_xcd || item >= nitems) return;
  const int64_t R0 = (int64_t)(item / ntj) * TT;
  const int J = (item % ntj) * TT;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wi = w & 1, wj = w >> 1;
  const int nslab = (K + KS - 1) / KS;

  // X slab: thread t takes the rows t/8 + 32 e and one column pair (8 lanes a line); R
  // slab: TR = 1 row t/16 and the column pairs 2 (t%16) + 32 e, TR = 0 columns t/8 + 32 e
  // and one row pair.  As in gram_kernel, clamped and dropped at the store.
  const int xr = tid >> 3, xc = (tid & 7) * 2;
  const int rm = TR ? tid >> 4 : xr, rc = TR ? (tid & 15) * 2 : xc;
  double2 rx[4], rr[4];
  auto load = [&](int i0) {
    load_rows<VEC>(X, ldx, R0, xr, rows, i0 + xc, K, rx);
    if (TR)
      load8<VEC>(Rm + (int64_t)(i0 + rm < K ? i0 + rm : 0) * ldr, J + rc, N, rr);
    else
      load_rows<VEC>(Rm, ldr, J, rm, N, i0 + rc, K, rr);
  };
  auto store = [&](int buf, int i0) {
    const bool i0ok = i0 + xc < K, i1ok = i0 + xc + 1 < K;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool kok = R0 + xr + 32 * e < rows;
      double *x = &Xs[buf][(xr + 32 * e) * XS + xc];
      x[0] = kok & i0ok ? rx[e].x : 0.0;
      x[1] = kok & i1ok ? rx[e].y : 0.0;
      if (TR) {
        const bool iok = i0 + rm < K;
        const int j = J + rc + 32 * e;
        *reinterpret_cast<double2 *>(&Rs[buf][rm * (TT + PADW) + rc + 32 * e]) =
            double2{iok & (j < N) ? rr[e].x : 0.0, iok & (j + 1 < N) ? rr[e].y : 0.0};
      } else {
        const bool jok = J + rm + 32 * e < N;
        double *r = &Rs[buf][(rm + 32 * e) * XS + xc];
        r[0] = jok & i0ok ? rr[e].x : 0.0;
        r[1] = jok & i1ok ? rr[e].y : 0.0;
      }
    }
  };

  // slabs whose rows of R reach column block c end at (diag + J) / 16 + c + 1
  constexpr int RK = TR ? TT + PADW : 1, RB = TR ? 1 : XS;
  const int dslab = diag >= K ? nslab : (diag + J + KS - 1) / KS;
  auto run = [&](auto form) {
    constexpr unsigned MASK = decltype(form)::value;
    f64x4 acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = f64x4{0, 0, 0, 0};
    load(0);
    store(0, 0);
    __syncthreads();
    auto upto = [&](auto part, int s, int end) {
      end = end < nslab ? end : nslab;
      for (; s < end; ++s) {
        const int buf = s & 1;
        if (s + 1 < nslab) load((s + 1) * KS);
        blocks<MASK & decltype(part)::value, 1, XS, RK, RB>(
            &Xs[buf][(wi * 16 + (lane & 15)) * XS + (lane >> 4)],
            TR ? &Rs[buf][(lane >> 4) * (TT + PADW) + wj * 16 + (lane & 15)]
               : &Rs[buf][(wj * 16 + (lane & 15)) * XS + (lane >> 4)],
            acc);
        if (s + 1 < nslab) store(buf ^ 1, (s + 1) * KS);
        __syncthreads();
      }
    };
    upto(std::integral_constant<unsigned, 0xffff>{}, 0, diag >= K ? nslab : dslab + 2);
    if (diag < K) {
      upto(std::integral_constant<unsigned, 0xeeee>{}, dslab + 2, dslab + 4);
      upto(std::integral_constant<unsigned, 0xcccc>{}, dslab + 4, dslab + 6);
      upto(std::integral_constant<unsigned, 0x8888>{}, dslab + 6, dslab + 8);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t k = R0 + (2 * a + wi) * 16 + acc_row<double>(lane, r);
        if (k >= rows) continue;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int j = J + (2 * b + wj) * 16 + (lane & 15);
          if (j < N) Y[k * ldy + j] = acc[a][b][r];
        }
      }
  };
  switch (N - J > 96 ? 3 : (N - J - 1) / 32) {
    case 0: run(std::integral_constant<unsigned, kColumnForm[0]>{}); break;
    case 1: run(std::integral_constant<unsigned, kColumnForm[1]>{}); break;
    case 2: run(std::integral_constant<unsigned, kColumnForm[2]>{}); break;
    default: run(std::integral_constant<unsigned, kColumnForm[3]>{}); break;
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// 16-byte loads: rows of n entries, aligned, without a half pair at the end
static bool pairs(const double *p, int64_t ld, int n) {
  return ld % 2 == 0 && ((uintptr_t)p & 15) == 0 && n % 2 == 0;
}

// Work items of a gram call and, per tile, its partial sums.  At most one wave of
// items over the chip's 512 workgroup slots (256 CUs, two workgroups each): a second,
// partial wave would double the time.  A tile whose waves multiply fewer blocks (diagonal,
// edge) gets longer chunks, so that the items end together; chunks of at least kMinRows
// rows, at most 256 of them.  (216k rows, whole CholGS in ms, every block of every tile
// on equal chunks / so: 500 columns 4.94 / 4.73, 333 columns 3.60 / 3.35.)
// whole > 0: equal chunks instead, as many as the lower triangle of whole columns
// has room for, so that an entry's sum does not depend on the group of columns that
// the call covers.
static void gram_plan(int64_t K, int m, int n, int diag_off, int whole,
                      std::vector<GramItem> *items, std::vector<GramItem> *tiles) {
  const int tm = (m + TT - 1) / TT, tn = (n + TT - 1) / TT;
  items->clear();
  tiles->clear();
  std::vector<int> load;  // blocks of a wave, and 2 for the staging
  int sum = 0;
  for (int J = 0; J < tn; ++J)
    for (int I = 0; I < tm; ++I)
      if (diag_off < 0 || (I + 1) * TT - 1 >= J * TT + diag_off) {
        const int most = __builtin_popcount(kGramForm[gram_form(I * TT, J * TT, m, diag_off)]);
        tiles->push_back(GramItem{I, J, 0, 0, 0});
        load.push_back(most + 2);
        sum += most + 2;
      }
  const int nt = (int)tiles->size();
  if (nt == 0 || K <= 0) return;
  // slabs of a chunk of load 18, grown until the items fit
  const int64_t slabs = (K + KS - 1) / KS;
  const int64_t least = std::max<int64_t>((slabs + 255) / 256, kMinRows / KS);
  int64_t full = std::max<int64_t>(1, slabs * sum / (18 * 512));
  auto chunk = [&](int t) { return std::max<int64_t>(full * 18 / load[t], least); };
  if (whole > 0) {
    const int tw = (whole + TT - 1) / TT, nch = std::max(1, 512 / (tw * (tw + 1) / 2));
    full = (slabs + nch - 1) / nch;
    load.assign(nt, 18);
  } else {
    for (;; full += std::max<int64_t>(1, full / 256)) {
      int64_t count = 0;
      for (int t = 0; t < nt; ++t) count += (slabs + chunk(t) - 1) / chunk(t);
      if (count <= std::max(512, nt)) break;
    }
  }
  for (int t = 0; t < nt; ++t) {
    const int64_t c = chunk(t);
    const int nch = (int)((slabs + c - 1) / c);
    GramItem &tl = (*tiles)[t];
    tl.part = (int)items->size();
    tl.nslab = nch;
    for (int j = 0; j < nch; ++j)
      items->push_back(GramItem{tl.I, tl.J, (int)(j * c), (int)std::min(c, slabs - j * c),
                                tl.part + j});
  }
  // items that start on the same rows next to each other: they share an XCD's L2
  std::stable_sort(items->begin(), items->end(),
                   [](const GramItem &x, const GramItem &y) { return x.slab < y.slab; });
}

size_t gram_partial_bytes(int64_t K, int m, int n, int diag_off, int whole) {
  std::vector<GramItem> items, tiles;
  gram_plan(K, m, n, diag_off, whole, &items, &tiles);
  return sizeof(double) * items.size() * TT * TT;
}

hipError_t launch_gram(const double *A, int64_t lda, const double *B, int64_t ldb, int m, int n,
                       int64_t K, int diag_off, int whole, double *C, int64_t ldc, double *P,
                       GramItem *table_dev, hipStream_t s) {
  std::vector<GramItem> items, tiles;
  gram_plan(K, m, n, diag_off, whole, &items, &tiles);
  const int nt = (int)tiles.size(), nitems = (int)items.size();
  if (nitems == 0) return hipSuccess;
  if (nt > kGramMaxTiles || nt + nitems > kGramMaxTable) return hipErrorInvalidValue;
  tiles.insert(tiles.end(), items.begin(), items.end());
  hipError_t e = hipMemcpyAsync(table_dev, tiles.data(), sizeof(GramItem) * tiles.size(),
                                hipMemcpyHostToDevice, s);
  if (e != hipSuccess) return e;
  const int per_xcd = (nitems + 7) / 8;
  const bool vec = pairs(A, lda, m) && pairs(B, ldb, n);
  hipLaunchKernelGGL((vec ? gram_kernel<true> : gram_kernel<false>), dim3(8 * per_xcd), dim3(NT),
                     0, s, A, lda, B, ldb, m, n, K, diag_off, table_dev + nt, per_xcd, nitems, P);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(gram_reduce_kernel, dim3(TT * TT / 256, nt), dim3(256), 0, s, P, table_dev, m,
                     n, C, ldc);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  // the host table is read by the copy above before this call returns
  return hipStreamSynchronize(s);
}

hipError_t launch_rotate(const double *X, int64_t ldx, const double *Rm, int64_t ldr, int trans,
                         int K, int diag, int N, int64_t rows, double *Y, int64_t ldy,
                         hipStream_t s) {
  if (rows <= 0 || N <= 0 || K <= 0) return hipSuccess;
  const int ntj = (N + TT - 1) / TT;
  const int64_t nti = (rows + TT - 1) / TT;
  const int64_t nitems64 = nti * ntj;
  if (nitems64 > (int64_t(1) << 30)) return hipErrorInvalidValue;
  const int nitems = (int)nitems64;
  const int per_xcd = (nitems + 7) / 8;
  const bool vec = pairs(X, ldx, K) && pairs(Rm, ldr, trans ? N : K);
  hipLaunchKernelGGL((trans ? (vec ? rotate_kernel<1, true> : rotate_kernel<1, false>)
                            : (vec ? rotate_kernel<0, true> : rotate_kernel<0, false>)),
                     dim3(8 * per_xcd), dim3(NT), 0, s, X, ldx, Rm, ldr, K, diag, N, rows, Y, ldy,
                     ntj, per_xcd, nitems);
  return hipGetLastError();
}

}  // namespace chfsi
