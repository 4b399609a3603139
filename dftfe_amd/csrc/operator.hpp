// Device-resident operator state shared by the operator and solver sources.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <memory>
#include <vector>

#include "common.hpp"

namespace chfsi {

// hipMalloc; without room it gives back the kept workspaces and tries again
hipError_t device_malloc(void **p, size_t bytes);

// Grow-only device buffer.
struct Scratch {
  void *ptr = nullptr;
  size_t size = 0;
  chfsi_status ensure(size_t bytes);
  void release();
};

// One fused apply  dst <- base + alpha * S H S src  over all colour classes
// (see HxLaunch for base / beta_mode).  bf16 selects the BF16-input kernel
// (T = float only).  R (nullable, ld ldR) adds rcoef[v] * R[:, v] to every row
// once (the defect form of the filter; FP32, not with bf16).  choice (0: B):
// the block width that the kernels' choice goes by, the same for all the
// applies of a pass, so that a column's bits do not depend on the group that
// it is applied in.
// Layout of a caller-provided HX scratch: projection partials (n_slots x B),
// then the V-scaled projections (n_proj x B) at the next 256-byte boundary.
inline size_t noalloc_w_offset(size_t elem, int n_slots, int B) {
  return (elem * size_t(n_slots) * size_t(B) + 255) / 256 * 256;
}
inline size_t noalloc_scratch_bytes(size_t elem, int n_slots, int n_proj, int B) {
  return noalloc_w_offset(elem, n_slots, B) + elem * size_t(n_proj) * size_t(B);
}

template <typename T>
chfsi_status hx_fused(chfsi_operator *op, const T *src, int64_t ld_src, T *dst, int64_t ld_dst,
                      int B, T alpha, T beta, T gamma, int beta_mode, bool scaled, hipStream_t s,
                      bool bf16 = false, const T *R = nullptr, int64_t ldR = 0,
                      const T *rcoef = nullptr, void *ext_scratch = nullptr, int choice = 0,
                      size_t ext_bytes = 0);

// g (+)= wscale JxW sum_v w_v (N.(s a_v))(N.(s b_v)) per (cell, quadrature
// point), s = M^{-1/2} when scaled; with general constraints the rows of a and
// b are distributed for the interpolation and cleared after (a and b are
// written).  See launch_quad_product.
template <typename T>
chfsi_status quad_product(chfsi_operator *op, const T *a, int64_t lda, const T *b, int64_t ldb,
                          int B, bool scaled, const double *jxw, const double *w, double wscale,
                          double *g, int accumulate, hipStream_t st, int wshift);

}  // namespace chfsi

struct chfsi_solver;

struct chfsi_operator {
  int device = 0;
  int64_t M = 0;
  int C = 0, ne = 0, ne_pad = 0, nq = 0;
  // cell -> DOF map with first-touch flag (bit 31), cells sorted by colour
  uint32_t *d_map = nullptr;
  int *d_cells_by_color = nullptr;
  static constexpr int kMaxColors = 128;
  int ncolors = 0;
  int color_off[kMaxColors + 1] = {0};
  int max_color_cells = 0;
  // Loewdin scalings
  double *d_sqrt_mass = nullptr, *d_inv_sqrt_mass = nullptr;
  float *d_sqrt_mass32 = nullptr, *d_inv_sqrt_mass32 = nullptr;
  // shape data and cell Hamiltonians (padded K-tiled layout)
  double *d_K = nullptr, *d_Nq = nullptr, *d_Gq = nullptr, *d_jxw = nullptr;
  // per-cell geometry: stiffness per cell (d_K then holds C*n_e*n_e) and the
  // cells' inverse Jacobians (jac = 3 diagonal, 9 full; 0: none)
  bool K_per_cell = false;
  double *d_invJ = nullptr;
  int jac = 0;
  double *d_Ht64 = nullptr;
  float *d_Ht32 = nullptr;
  uint16_t *d_Ht16 = nullptr, *d_nlC16 = nullptr;  // BF16 copies
  bool has_H = false;
  bool h_sym = false;  // cell matrices exactly symmetric (built on the device)
  // nonlocal projector slots
  int n_proj = 0, n_slots = 0, n_nl_cells = 0;
  int *d_nl_off = nullptr, *d_slot_proj = nullptr, *d_proj_ptr = nullptr,
      *d_proj_slots = nullptr, *d_nl_cells = nullptr;
  double *d_nlC64 = nullptr, *d_nlCt64 = nullptr, *d_proj_V = nullptr;
  float *d_nlC32 = nullptr, *d_nlCt32 = nullptr;
  // owned-row form of the projection (projection variant 4): per nonlocal
  // cell the DOFs whose (DOF, projector) terms that cell forms (own_n[c] of
  // them, own_map[c * ne_pad + r]) and the assembled projector values on
  // those rows, in the slot layout of nlCt
  uint32_t *d_own_map = nullptr;
  int *d_own_n = nullptr;
  double *d_nlCto64 = nullptr;
  float *d_nlCto32 = nullptr;
  chfsi::Scratch partial64, partial32, W64, W32, tmp;
  // tensor-product form of the cell operators (tensor.hpp): nodes and Gauss
  // points per direction (0: the shape data is not of that form), the parity
  // tables, the potential's weights in the kernels' order
  // and the projector columns in their x-parity rows.  tensor_pot:
  // the cell matrices are those of the weights held here (an LDA potential)
  int tn = 0, tq = 0;
  bool tensor_pot = false;
  int *d_form = nullptr;  // the same on the device, for captured applies (operators with tn)
  // touches of every DOF in colour order and the cells' sums of one apply, for
  // small blocks (nullable).  The sums of each precision have a buffer of their
  // own, as the projections do: an FP64 and an FP32 apply may run at once.
  // It is never moved: a captured apply keeps its address.
  uint32_t *d_touch_ptr = nullptr, *d_touch_idx = nullptr;
  double *d_cells_out64 = nullptr;
  float *d_cells_out32 = nullptr;
  bool tensor_gga = false;  // the shape gradients are products too
  double *d_ttab64 = nullptr, *d_tprod = nullptr, *d_vq64 = nullptr, *d_nlCp64 = nullptr;
  float *d_ttab32 = nullptr, *d_vq32 = nullptr, *d_nlCp32 = nullptr;
  // HX tile variants per precision: the caller's (-1: none set), and the fastest
  // of the dense form (chfsi_operator_autotune).  Only a tile that the caller set
  // turns the tensor form off where the operator has it.
  int hx_variant64 = -1, hx_variant32 = -1;
  int hx_tuned64 = 0, hx_tuned32 = 0;
  int hx_variant16 = 0;  // BF16 apply: 0 K = 32 ring, 1 register-staged K = 16
  int proj_variant64 = -1, proj_variant32 = -1;  // -1: by size (proj_default)
  int max_srb = 1;  // largest slot count of any cell / 16
  // extra cell ids C .. C + n_extra_cells - 1: further projector groups of
  // cells with more than 128 slots (zero cell matrix, own colours, the nodes
  // of their real cell)
  int n_extra_cells = 0;
  // constraints (slave-major and master-major CSR)
  int64_t nc = 0, nm = 0;
  int64_t *d_idle_rows = nullptr;  // rows no cell writes (folded constraints)
  int64_t n_idle = 0;
  int64_t *d_c_rows = nullptr, *d_c_ptr = nullptr, *d_c_cols = nullptr;
  double *d_c_vals = nullptr;
  int64_t *d_m_rows = nullptr, *d_m_ptr = nullptr, *d_m_slaves = nullptr;
  double *d_m_vals = nullptr;
  // general (hanging-node) rows: not folded into the map; every apply
  // distributes into the constrained rows of its source (gathered with scale
  // 1: s_gather = M^{-1/2} with 1 on constrained rows) and sends the rows' sums
  // to their masters (output scale 0 marks them; ones_cons = 1 with 0 on
  // constrained rows for the unscaled apply)
  bool general_constraints = false;
  double *d_s_gather64 = nullptr, *d_ones_cons64 = nullptr;
  float *d_s_gather32 = nullptr, *d_ones_cons32 = nullptr;
  // Bloch k-points: complex cell matrices and projector tiles per k-point in
  // the paired (Re, Im) tile layout of the complex kernels
  int nk = 0, active_k = 0;
  std::vector<double> kpts;  // 3 per k-point
  double *d_Mc = nullptr, *d_Gd = nullptr;
  double *d_Hk64 = nullptr;
  float *d_Hk32 = nullptr;
  double *d_nlCk64 = nullptr, *d_nlCtk64 = nullptr;
  float *d_nlCk32 = nullptr, *d_nlCtk32 = nullptr;
  // owned-row form of the complex projector tiles (the rows of d_own_map),
  // per k-point; zproj_variant 0: cell form, 1: owned rows (the default)
  double *d_nlCtko64 = nullptr;
  float *d_nlCtko32 = nullptr;
  int zproj_variant = 1;
  int zhx_variant64 = 0, zhx_variant32 = 0;
  // workspace of the entry points without a solver (see Workspace), and its bytes
  // when it was last put down
  std::atomic<bool> work_busy{false};
  chfsi_solver *work = nullptr;
  size_t work_bytes = 0;
  hipEvent_t work_done = nullptr;
  chfsi::Scratch ztab_dev, ztab_W, ztab_P;  // tables and scratch of single complex applies

  ~chfsi_operator();
};

namespace chfsi {
// Frees the operator's kept workspace (no call may be using it)
void release_workspace(chfsi_operator *op);
// Frees the kept workspaces that no call is using; whether there were any
bool release_idle_workspaces();
// Rebuilds the complex cell matrices of every k-point from the real tiles.
chfsi_status rebuild_kpoint_matrices(chfsi_operator *op, hipStream_t s);
}  // namespace chfsi
