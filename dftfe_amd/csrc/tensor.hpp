// Tensor-product form of the cell operators: cells whose shape values and
// stiffness are products of one-dimensional tables (GLL Lagrange basis, Gauss
// quadrature, Cartesian cells) are applied direction by direction instead of
// through the dense n_e x n_e cell matrix.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "kernels.hpp"

namespace chfsi {

// (nodes per direction, Gauss points per direction) with an instantiation
bool tensor_shape(int ne, int nqc, int *n, int *q);

// Whether the tensor form is the faster one on B columns, from the cells of the
// largest colour; all: the operator can run all cells at once
bool tensor_wins(int n, bool fp64, int cells, int B, bool all);

// workgroups of a colour up to which one launch over all cells is the faster apply
constexpr int kAllCellsItems = 448;
// Whether all cells at once beat the colour launches on B columns
bool tensor_all_cells(int n, bool fp64, int cells, int B);
// The widest block for which they do (0: none)
int tensor_all_cells_columns(int n, bool fp64, int cells);

// Host check of an operator's shape values (nqc x ne) and stiffness (ne x ne):
// true when every entry is the product of one-dimensional, centro-symmetric
// tables (Gauss quadrature) to rounding.  Fills the kernels'
// tables, FP64 and FP32, and the products of the cell matrix build (n^2 q, or
// 4 n^2 q when the shape gradients G (nqc x ne x 3, nullable) have that form too).
bool tensor_tables(const double *Nq, const double *K, const double *G, int ne, int nqc,
                   std::vector<double> *tab, std::vector<float> *tab32,
                   std::vector<double> *products);

// Weights vJxW (C x nqc) in the kernels' order (scaled by exact powers of two)
hipError_t launch_tensor_potential(const double *vJxW, int C, int n, int q, double *v64,
                                   float *v32, hipStream_t s);

// Projector columns (layout of nl_C) in the x-parity rows of the kernels
hipError_t launch_tensor_projectors(const double *nlC, int64_t total, int n, int ne, int ne_pad,
                                    double *c64, float *c32, hipStream_t s);

// Touches of every DOF row by the cells' nodes in colour order: rows ptr[g] ..
// ptr[g + 1] of idx, each (position of the cell in the colour order) * n_e + node
struct TensorTouch {
  const uint32_t *ptr, *idx;
  int64_t M;
};

// One fused HX launch over a colour class (as launch_hx) on the tensor form;
// a.nl_C: the columns of launch_tensor_projectors.  With touch, all cells at once
// (a.cells: every colour's) through cells_out (cells x n_e x B) and a sum over
// the touches: the same result bit for bit
template <typename T>
hipError_t launch_hx_tensor(const HxLaunch<T> &a, const T *vq, const T *tab, int n, int q,
                            const TensorTouch *touch, T *cells_out, hipStream_t s);

// launch_quad_product on the tensor form (tab: the FP64 tables)
template <typename TIn>
hipError_t launch_quad_tensor(const uint32_t *map, int C, int n, int q, const double *JxW,
                              const TIn *a, int64_t lda, const TIn *b, int64_t ldb, int B,
                              const double *s_in, const double *w, int wshift, double wscale,
                              double *g, int accumulate, const double *tab, hipStream_t s);

// launch_build_h for one stiffness and geometry, from the products
hipError_t launch_build_tensor(const double *K, const double *P, const double *vJxW,
                               const double *gJxW, int C, int n, int q, int ne_pad, double *Ht64,
                               float *Ht32, uint16_t *Ht16, hipStream_t s);

}  // namespace chfsi
