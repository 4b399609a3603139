// FP64 MFMA kernels of the dense CholGS / Rayleigh-Ritz steps (dense.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace chfsi {

// largest number of 128 x 128 output tiles of one gram call (N <= 4096)
constexpr int kGramMaxTiles = 1024;
// entries of a gram call's table: its tiles, then its work items (at most 512, or one
// per tile)
constexpr int kGramMaxTable = 2 * kGramMaxTiles;

// a work item: K slabs [slab, slab + nslab) of 16 rows of tile (I, J), summed into
// partial tile `part`; a tile: partial tiles [part, part + nslab)
struct GramItem {
  int I, J, slab, nslab, part;
};

// C[i + j ldc] = sum_{k < K} A[k lda + i] B[k ldb + j] for i < m, j < n
// (A^T B of node-major blocks), split over K with partial tiles in P summed in
// a fixed order.  diag_off >= 0: only the tiles that reach the lower triangle
// of C, i >= j + diag_off (16 x 16 blocks above it read as zero there); -1: all.
// whole > 0: the call is one group of columns of the lower triangle of an
// m x whole product, whose entries have the same bits in every grouping.
// P holds gram_partial_bytes(K, m, n, diag_off, whole) bytes and table_dev
// kGramMaxTable entries; synchronises the stream (the table is copied
// from the host).
hipError_t launch_gram(const double *A, int64_t lda, const double *B, int64_t ldb, int m, int n,
                       int64_t K, int diag_off, int whole, double *C, int64_t ldc, double *P,
                       GramItem *table_dev, hipStream_t s);
size_t gram_partial_bytes(int64_t K, int m, int n, int diag_off, int whole);

// column tile of the rotation kernel
constexpr int kRotateTile = 128;

// Y[k ldy + j] = sum_{i < K} X[k ldx + i] R(i, j) for k < rows, j < N, with
// R(i, j) = Rm[i + j ldr] (trans = 0) or Rm[j + i ldr] (trans = 1).  R(i, j) is zero
// for i > diag + j (diag >= K: none need be).  Y must not overlap X unless N <= kRotateTile
// and Y's columns are among the K of X (row for row: in place).
hipError_t launch_rotate(const double *X, int64_t ldx, const double *Rm, int64_t ldr, int trans,
                         int K, int diag, int N, int64_t rows, double *Y, int64_t ldy,
                         hipStream_t s);

}  // namespace chfsi
