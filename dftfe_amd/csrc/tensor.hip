// Tensor-product cell operators (see tensor.hpp).
//
// A cell with n GLL nodes and q Gauss points per direction applies
//   y = 1/2 K x + N^T diag(v JxW) N x,   N = I (x) I (x) I,
//   K = a_x K1 (x) M1 (x) M1 + a_y M1 (x) K1 (x) M1 + a_z M1 (x) M1 (x) K1
// direction by direction: at n = 7, q = 8 about 2.4e4 operations per column
// against 2.4e5 of the dense 343 x 343 product.  All one-dimensional tables are
// centro-symmetric, so a line is split into its even and odd part
// (x_{+-i} = E_i +- O_i), which halves the products again and lets the even-x
// and odd-x halves of a plane live in different waves.
//
// Scaling: the input carries a factor 1/8 (one half per direction, so that
// E_i = x_i + x_{-i}, O_i = x_i - x_{-i} and a middle node enters alone), and
// the weights at the quadrature points the same factor for the way back
// (another half per direction whose quadrature index is the middle one).  All
// of these are powers of two, so nothing is rounded by them.

#include <algorithm>
#include <cmath>
#include <limits>

#include "mfma.hpp"
#include "scatter.hpp"
#include "tensor.hpp"

// Fused multiply-adds are written out: an instantiation for other widths must not
// contract other sums.  Within this form a column has the same bits in every
// block; the form, and the projection's tile, go by the columns of a whole pass.
#pragma clang fp contract(off)

namespace chfsi {

// ---------------------------------------------------------------------------
// One-dimensional tables (host): taken from the operator's own arrays, so that
// the apply agrees with its dense form to rounding
// ---------------------------------------------------------------------------
namespace {

typedef long double ld;

// Gauss weights on [0, 1] (Newton on the Legendre polynomial P_q)
std::vector<ld> gauss_weights(int q) {
  std::vector<ld> w(q);
  for (int i = 0; i < q; ++i) {
    ld t = cosl(acosl(-1.0L) * (q - i - 0.25L) / (q + 0.5L)), d = 1;
    for (int it = 0; it < 50; ++it) {
      ld p0 = 1, p1 = t;
      for (int k = 2; k <= q; ++k) {
        const ld p2 = ((2 * k - 1) * t * p1 - (k - 1) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      d = q * (t * p1 - p0) / (t * t - 1);
      t -= p1 / d;
    }
    w[i] = 1 / ((1 - t * t) * d * d);
  }
  return w;
}

// Mean of a rows x cols table and its point reflection
void symmetrise(std::vector<ld> &A) {
  for (size_t i = 0, j = A.size() - 1; i < j; ++i, --j) A[i] = A[j] = (A[i] + A[j]) / 2;
}

// v[j] = A[j] on the grid of FP32 values below `big`, with the sum over a
// constant (a middle value enters with one half) made `target` by entry `fix`
void balance(const double *A, int n, bool middle, double big, double target, int fix,
             double *out) {
  const double g = std::ldexp(1.0, std::ilogb(big) + 1 - 24);
  double sum = 0;
  for (int j = 0; j < n; ++j) {
    const double k = middle && j == n - 1 ? 0.5 : 1.0;
    const double r = std::nearbyint(A[j] * k / g) * g;
    out[j] = r / k;
    sum += r;
  }
  out[fix] += (target - sum) / (middle && fix == n - 1 ? 0.5 : 1.0);
}

}  // namespace

// FP64 tables: [parity][row][column] blocks over the first half of the rows and
// columns, even part A[r][c] + A[r][-c], odd part A[r][c] - A[r][-c] (padded
// with zeros to the size of the even one)
template <int N, int Q>
struct TensorTab {
  static constexpr int NE = (N + 1) / 2, NO = N / 2;  // even / odd nodal values of a line
  static constexpr int QE = (Q + 1) / 2, QO = Q / 2;  // even / odd quadrature values
  static constexpr int oI = 0, oM = oI + 2 * QE * NE;
  static constexpr int oKx = oM + 2 * NE * NE, oKy = oKx + 2 * NE * NE, oKz = oKy + 2 * NE * NE;
  static constexpr int oW = oKz + 2 * NE * NE;        // 1/2 w, the middle one 1/4 w
};

// FP32 operand tables of the 4 x 4 products: [table][row][column], zero beyond
// the blocks, then the weights.  L: what K's rounding leaves (see tensor_tables)
enum {
  kTabIe, kTabIo, kTabIeT, kTabIoT, kTabMe, kTabMo, kTabKx, kTabKxo, kTabKy, kTabKyo, kTabKz,
  kTabKzo, kTabLx, kTabLxo, kTabLy, kTabLyo, kTabLz, kTabLzo, kTabs
};

bool tensor_shape(int ne, int nqc, int *n, int *q) {
  static const int shapes[3][2] = {{5, 5}, {6, 6}, {7, 8}};
  for (auto &s : shapes)
    if (ne == s[0] * s[0] * s[0] && nqc == s[1] * s[1] * s[1]) {
      *n = s[0];
      *q = s[1];
      return true;
    }
  return false;
}

namespace {
// x, y, z index of each of n^3 nodes or points, x the fastest
struct Index3 {
  std::vector<int> x, y, z;
  explicit Index3(int n) {
    for (int c = 0; c < n; ++c)
      for (int b = 0; b < n; ++b)
        for (int a = 0; a < n; ++a) {
          x.push_back(a);
          y.push_back(b);
          z.push_back(c);
        }
  }
};

// Appends 2 (D_d I + I D_d) of each direction when every shape gradient is a
// product with one D_d to tol of the largest one
bool gradient_products(const double *G, const std::vector<ld> &I, int n, int q, double tol,
                       std::vector<double> *products) {
  const int ne = n * n * n, nqc = q * q * q;
  const Index3 in(n), iq(q);
  std::vector<ld> D[3];
  for (auto &d : D) d.assign(size_t(q) * n, 0);
  // means as for I (tensor_tables)
  double gmax = 0;
  for (int k = 0; k < nqc; ++k)
    for (int i = 0; i < ne; ++i) {
      const double *g = G + (size_t(k) * ne + i) * 3;
      for (int d = 0; d < 3; ++d) gmax = std::max(gmax, std::fabs(g[d]));
      if (iq.y[k] == iq.z[k]) D[0][iq.x[k] * n + in.x[i]] += g[0];
      if (iq.z[k] == iq.x[k]) D[1][iq.y[k] * n + in.y[i]] += g[1];
      if (iq.x[k] == iq.y[k]) D[2][iq.z[k] * n + in.z[i]] += g[2];
    }
  for (auto &d : D)
    for (ld &v : d) v /= q;
  const std::vector<double> Id(I.begin(), I.end());
  std::vector<double> Dd[3];
  for (int d = 0; d < 3; ++d) Dd[d].assign(D[d].begin(), D[d].end());
  for (int k = 0; k < nqc; ++k)
    for (int i = 0; i < ne; ++i) {
      const int ex = iq.x[k] * n + in.x[i], ey = iq.y[k] * n + in.y[i],
                ez = iq.z[k] * n + in.z[i];
      const double *g = G + (size_t(k) * ne + i) * 3;
      if (!(std::fabs(g[0] - Dd[0][ex] * Id[ey] * Id[ez]) <= tol * gmax &&
            std::fabs(g[1] - Id[ex] * Dd[1][ey] * Id[ez]) <= tol * gmax &&
            std::fabs(g[2] - Id[ex] * Id[ey] * Dd[2][ez]) <= tol * gmax))
        return false;
    }
  for (const auto &d : D)
    for (int a = 0; a < n; ++a)
      for (int b = 0; b < n; ++b)
        for (int k = 0; k < q; ++k)
          products->push_back(
              (double)(2 * (d[k * n + a] * I[k * n + b] + I[k * n + a] * d[k * n + b])));
  return true;
}
}  // namespace

namespace {
// Corrects the quadrature weights w so that I^T diag(w) I is closest to M: K_z is weighted
// by w at the points of x and y, where K_x and K_y take M itself, and an error of w
// acts alike in every cell.
void fit_weights(const std::vector<ld> &I, const std::vector<ld> &M, int n, int q,
                 std::vector<ld> &w) {
  // normal equations [q][q + 1]: A_kl = (I_k . I_l)^2, b_k = I_k^T M I_k - A w
  std::vector<ld> A(size_t(q) * (q + 1), 0);
  for (int k = 0; k < q; ++k) {
    ld *row = &A[k * (q + 1)];
    for (int a = 0; a < n; ++a)
      for (int b = 0; b < n; ++b) row[q] += I[k * n + a] * M[a * n + b] * I[k * n + b];
    for (int l = 0; l < q; ++l) {
      ld s = 0;
      for (int a = 0; a < n; ++a) s += I[k * n + a] * I[l * n + a];
      row[l] = s * s;
      row[q] -= row[l] * w[l];
    }
  }
  for (int c = 0; c < q; ++c) {
    int piv = c;
    for (int r = c + 1; r < q; ++r)
      if (fabsl(A[r * (q + 1) + c]) > fabsl(A[piv * (q + 1) + c])) piv = r;
    for (int k = 0; k <= q; ++k) std::swap(A[c * (q + 1) + k], A[piv * (q + 1) + k]);
    for (int r = 0; r < q; ++r) {
      if (r == c) continue;
      const ld f = A[r * (q + 1) + c] / A[c * (q + 1) + c];
      for (int k = c; k <= q; ++k) A[r * (q + 1) + k] -= f * A[c * (q + 1) + k];
    }
  }
  for (int c = 0; c < q; ++c) w[c] += A[c * (q + 1) + q] / A[c * (q + 1) + c];
}

// The mass and stiffness tables of K = D_x M M + M D_y M + M M D_z ([a * n + b]) that
// fit it best, from a start near them: K contracted with M in one direction and with M,
// or with the part of a D that is orthogonal to M, in another leaves the table of
// the third (the D up to multiples of M, which are fixed by a constant having no
// energy).  Two rounds reach rounding.
void fit_stiffness(const double *K, int n, std::vector<ld> &M, std::vector<ld> (&D)[3]) {
  const int nn = n * n, ne = nn * n;
  const Index3 in(n);
  // rows of A times b, columns of A times b (A: nn x nn)
  auto right = [nn](const std::vector<ld> &A, const std::vector<ld> &b, ld f,
                    std::vector<ld> &out) {
    for (int e = 0; e < nn; ++e)
      for (int k = 0; k < nn; ++k) out[e] += f * A[e * nn + k] * b[k];
  };
  auto left = [nn](const std::vector<ld> &A, const std::vector<ld> &b, ld f,
                   std::vector<ld> &out) {
    for (int k = 0; k < nn; ++k)
      for (int e = 0; e < nn; ++e) out[e] += f * A[k * nn + e] * b[k];
  };
  auto dot = [nn](const std::vector<ld> &a, const std::vector<ld> &b) {
    ld s = 0;
    for (int e = 0; e < nn; ++e) s += a[e] * b[e];
    return s;
  };
  const std::vector<ld> one(nn, 1);
  for (int round = 0; round < 2; ++round) {
    // K times M in z, y, x: [ex][ey], [ex][ez], [ey][ez]
    std::vector<ld> xy(nn * nn, 0), xz(nn * nn, 0), yz(nn * nn, 0);
    for (int i = 0; i < ne; ++i)
      for (int j = 0; j < ne; j += n) {
        const int xi = in.x[i] * n, ey = in.y[i] * n + in.y[j], ez = in.z[i] * n + in.z[j];
        const double *k = K + size_t(i) * ne + j;
        ld sum = 0;  // over x
        for (int x = 0; x < n; ++x) {
          const ld v = k[x];
          xy[(xi + x) * nn + ey] += v * M[ez];
          xz[(xi + x) * nn + ez] += v * M[ey];
          sum += v * M[xi + x];
        }
        yz[ey * nn + ez] += sum;
      }
    const ld mm = dot(M, M);
    for (auto &d : D) d.assign(nn, 0);
    right(xy, M, 1 / (mm * mm), D[0]);
    left(xy, M, 1 / (mm * mm), D[1]);
    left(xz, M, 1 / (mm * mm), D[2]);
    ld off[3], rest = 2 * dot(D[0], M) / mm;
    for (int d = 0; d < 3; ++d) rest -= off[d] = dot(D[d], one) / dot(M, one);
    std::vector<ld> P[3], next(nn, 0);
    for (int d = 0; d < 3; ++d) {
      for (int e = 0; e < nn; ++e) D[d][e] -= (off[d] + rest / 3) * M[e];
      const ld f = dot(D[d], M) / mm;
      P[d] = D[d];
      for (int e = 0; e < nn; ++e) P[d][e] -= f * M[e];
    }
    ld w[3];
    for (int d = 0; d < 3; ++d) w[d] = 1 / (6 * dot(P[d], P[d]) * mm);
    right(xy, P[1], w[1], next);
    right(xz, P[2], w[2], next);
    left(xy, P[0], w[0], next);
    right(yz, P[2], w[2], next);
    left(xz, P[0], w[0], next);
    left(yz, P[1], w[1], next);
    M = next;
  }
}
}  // namespace

bool tensor_tables(const double *Nq, const double *K, const double *G, int ne, int nqc,
                   std::vector<double> *tab, std::vector<float> *tab32,
                   std::vector<double> *products) {
  int n = 0, q = 0;
  if (!tensor_shape(ne, nqc, &n, &q)) return false;
  // rounding: products of three tables are within 5 eps of shape values and
  // gradients evaluated point by point, and within 2-6 eps of a stiffness from
  // one-dimensional tables or matrix products, 31 of one summed point after point
  // (512 points)
  const double eps = std::numeric_limits<double>::epsilon();
  const double tol = 32 * eps, tol_k = 128 * eps;
  const Index3 in(n), iq(q);
  std::vector<ld> w = gauss_weights(q);
  // I: sums of N over the nodes of the other two directions (which are one), mean
  // over their points with two equal indices (q n^2 entries: far below rounding)
  // and over the directions; x is the fastest index of nodes and points
  std::vector<ld> I(size_t(q) * n, 0), M(size_t(n) * n, 0), Kd[3];
  for (int k = 0; k < nqc; ++k) {
    const bool yz = iq.y[k] == iq.z[k], zx = iq.z[k] == iq.x[k], xy = iq.x[k] == iq.y[k];
    if (!(yz || zx || xy)) continue;
    for (int i = 0; i < ne; ++i) {
      const ld v = Nq[size_t(k) * ne + i];
      if (yz) I[iq.x[k] * n + in.x[i]] += v;
      if (zx) I[iq.y[k] * n + in.y[i]] += v;
      if (xy) I[iq.z[k] * n + in.z[i]] += v;
    }
  }
  for (ld &v : I) v /= 3 * q;
  // products of the cell matrix build: I I, and with shape gradients (nqc x ne x
  // 3, of the same form) 2 (D_d I + I D_d), [a][b][q], symmetric in a and b
  products->assign(size_t(n) * n * q, 0.0);
  for (int a = 0; a < n; ++a)
    for (int b = 0; b < n; ++b)
      for (int k = 0; k < q; ++k)
        (*products)[(size_t(a) * n + b) * q + k] = (double)(I[k * n + a] * I[k * n + b]);
  if (G && !gradient_products(G, I, n, q, tol, products)) products->resize(size_t(n) * n * q);
  symmetrise(I);
  for (int a = 0; a < n; ++a)
    for (int b = 0; b < n; ++b)
      for (int k = 0; k < q; ++k) M[a * n + b] += w[k] * I[k * n + a] * I[k * n + b];
  double kmax = 0;
  for (size_t i = 0; i < size_t(ne) * ne; ++i) kmax = std::max(kmax, std::fabs(K[i]));
  fit_stiffness(K, n, M, Kd);
  symmetrise(M);
  for (auto &A : Kd) symmetrise(A);
  fit_weights(I, M, n, q, w);
  const std::vector<double> Id(I.begin(), I.end()), Md(M.begin(), M.end());
  const std::vector<double> Kd0(Kd[0].begin(), Kd[0].end()), Kd1(Kd[1].begin(), Kd[1].end()),
      Kd2(Kd[2].begin(), Kd[2].end());
  for (int k = 0; k < nqc; ++k)
    for (int i = 0; i < ne; ++i) {
      const double v = Id[iq.x[k] * n + in.x[i]] * Id[iq.y[k] * n + in.y[i]] *
                       Id[iq.z[k] * n + in.z[i]];
      if (!(std::fabs(Nq[size_t(k) * ne + i] - v) <= tol)) return false;
    }
  for (int i = 0; i < ne; ++i)
    for (int j = 0; j < ne; ++j) {
      const int ex = in.x[i] * n + in.x[j], ey = in.y[i] * n + in.y[j],
                ez = in.z[i] * n + in.z[j];
      const double v =
          Kd0[ex] * Md[ey] * Md[ez] + Md[ex] * Kd1[ey] * Md[ez] + Md[ex] * Md[ey] * Kd2[ez];
      if (!(std::fabs(K[size_t(i) * ne + j] - v) <= tol_k * kmax)) return false;
    }
  // parity tables; the operator applies half the stiffness
  const int NE = (n + 1) / 2, NO = n / 2, QE = (q + 1) / 2, QO = q / 2;
  tab->clear();
  tab32->assign(kTabs * 16 + QE, 0.f);
  auto put = [&](const std::vector<ld> &A, int rows_e, int rows_o, ld f, int t32, int sums) {
    const size_t at = tab->size();
    for (int p = 0; p < 2; ++p)
      for (int r = 0; r < rows_e; ++r)
        for (int c = 0; c < NE; ++c) {
          const ld v = A[r * n + c], m = A[r * n + n - 1 - c];
          const bool in = p == 0 || (r < rows_o && c < NO);
          tab->push_back(in ? (double)(f * (p == 0 ? v + m : v - m)) : 0.0);
        }
    // FP32: a rounding error of a table acts alike in every cell, so it shifts
    // eigenvalues where the rounding of dense cell matrices averages out.  The
    // even part of I (sums = 1) is therefore rounded with its row sums kept
    // exact, so that a constant is interpolated to itself, and K (sums = 0)
    // is kept in two parts, the first with exact zero row sums (a constant has
    // no kinetic energy), the second the rest.  Plane waves of 0.5-1.2 Ha at
    // p = 5 and 6 shift by 3-7e-7 Ha with the first part alone (as any state
    // does, in proportion to its kinetic energy) and by at most 2e-8 with
    // both, which is the rounding of I, M and the weights; the dense FP32
    // matrices shift them by up to 1e-7.
    const double *e = tab->data() + at;
    double big = 0;
    for (int x = 0; x < rows_e * NE; ++x) big = std::max(big, std::fabs(e[x]));
    for (int r = 0; r < rows_e; ++r) {
      const double *er = e + r * NE;
      std::vector<double> v(er, er + NE);
      if (sums == 0) balance(er, NE, n & 1, big, 0.0, r, v.data());
      if (sums == 1) {
        const int fix = (int)(std::max_element(er, er + NE) - er);
        balance(er, NE, n & 1, er[fix], 1.0, fix, v.data());
      }
      for (int c = 0; c < NE; ++c) {
        float *d = tab32->data() + t32 * 16;
        const double ev = er[c], od = e[(rows_e + r) * NE + c];
        d[r * 4 + c] = (float)v[c];
        d[16 + r * 4 + c] = (float)od;
        if (sums == 0) {
          float *l = d + (kTabLx - kTabKx) * 16;
          l[r * 4 + c] = (float)(ev - d[r * 4 + c]);
          l[16 + r * 4 + c] = (float)(od - d[16 + r * 4 + c]);
        }
        if (t32 == kTabIe)
          for (int p = 0; p < 2; ++p) d[32 + p * 16 + c * 4 + r] = d[p * 16 + r * 4 + c];
      }
    }
  };
  put(I, QE, QO, 1, kTabIe, 1);
  put(M, NE, NO, 1, kTabMe, -1);
  for (int d = 0; d < 3; ++d) put(Kd[d], NE, NO, 0.5L, kTabKx + 2 * d, 0);
  for (int k = 0; k < QE; ++k) {
    tab->push_back((double)(w[k] * (2 * k + 1 == q ? 0.25L : 0.5L)));
    (*tab32)[kTabs * 16 + k] = (float)tab->back();
  }
  return true;
}

// ---------------------------------------------------------------------------
// Potential weights in the order of the pencil threads: per cell
// [group b * QE + a][mirror image s][z], s bit 0 mirroring x and bit 1 y, times
// 1/8 and another 1/2 per direction whose index is the middle one (its mirror
// image is the point itself and is counted twice; in z it enters once)
// ---------------------------------------------------------------------------
__global__ void tensor_potential_kernel(const double *v, int64_t total, int q, int qe, double *v64,
                                        float *v32) {
  const int per = qe * qe * 4 * q;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e / per;
    const int r = (int)(e % per);
    const int z = r % q, s = r / q % 4, a = r / (4 * q) % qe, b = r / (4 * q * qe);
    const int x = s & 1 ? q - 1 - a : a, y = s & 2 ? q - 1 - b : b;
    double f = 0.125;
    if (2 * a + 1 == q) f *= 0.5;
    if (2 * b + 1 == q) f *= 0.5;
    const double w = f * v[c * q * q * q + x + q * (y + q * z)];
    v64[e] = w;
    v32[e] = (float)w;
  }
}

// Projector columns in the rows of the kernels' kinetic stage: (z, y, x) with
// the even, then the odd values of y and x instead of the nodes
__global__ void tensor_projector_kernel(const double *c, int64_t total, int n, int ne, int ne_pad,
                                        double *c64, float *c32) {
  const int nev = (n + 1) / 2;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int row = (int)(e / 16 % ne_pad);
    double v = 0;
    if (row < ne) {
      const int kx = row % n, ky = row / n % n;
      const int x = kx < nev ? kx : kx - nev, y = ky < nev ? ky : ky - nev;
      const double *l = c + e - (int64_t)(row % (n * n)) * 16;  // the plane's first node
      auto at = [&](int yy) {
        const double p = l[(int64_t)(yy * n + x) * 16], m = l[(int64_t)(yy * n + n - 1 - x) * 16];
        return kx < nev ? (2 * x + 1 == n ? p : 0.5 * (p + m)) : 0.5 * (p - m);
      };
      const double p = at(y), m = at(n - 1 - y);
      v = ky < nev ? (2 * y + 1 == n ? p : 0.5 * (p + m)) : 0.5 * (p - m);
    }
    c64[e] = v;
    c32[e] = (float)v;
  }
}

hipError_t launch_tensor_projectors(const double *nlC, int64_t total, int n, int ne, int ne_pad,
                                    double *c64, float *c32, hipStream_t s) {
  const unsigned grid = (unsigned)std::min<int64_t>((total + 255) / 256, 1 << 16);
  hipLaunchKernelGGL(tensor_projector_kernel, dim3(grid), dim3(256), 0, s, nlC, total, n, ne,
                     ne_pad, c64, c32);
  return hipGetLastError();
}

hipError_t launch_tensor_potential(const double *vJxW, int C, int n, int q, double *v64,
                                   float *v32, hipStream_t s) {
  (void)n;
  const int qe = (q + 1) / 2;
  const int64_t total = int64_t(C) * qe * qe * 4 * q;
  const unsigned grid = (unsigned)std::min<int64_t>((total + 255) / 256, 1 << 16);
  hipLaunchKernelGGL(tensor_potential_kernel, dim3(grid), dim3(256), 0, s, vJxW, total, q, qe, v64,
                     v32);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Fused HX, tensor form
// ---------------------------------------------------------------------------
// One workgroup per (cell, TC columns).  A thread of the plane stages holds,
// for one column, the even-x or odd-x half of one z plane (28 values at
// n = 7), the parity uniform per wave so that all table entries are scalar
// operands; a thread of the pencil stages holds the four z lines mirrored in x
// and y.  The block goes through LDS between the stages:
//   gather (scaled rows) -> planes: b = (K_x M_y + M_x K_y) x -> z lines: M_z b
//   -> planes: u = I_x I_y x -> z lines: (I_z^T v I_z + w_x w_y K_z) u
//   -> planes: I_x^T I_y^T, sum -> rows: scatter.
// The nonlocal term C_e W (MFMA) joins M_z b.
// K_z runs on the lines interpolated in x and y (weighted there), K_x and K_y on
// nodal values: in FP32 the error is that of the dense product or below
// (stiffness tables at quadrature points would double it).
template <typename T, int N, int Q, int TC_, int VW>
struct TensorShape : TensorTab<N, Q> {
  static constexpr int TC = TC_, QE_ = (Q + 1) / 2;
  static constexpr int G = 64 / TC;              // column groups of a wave
  static constexpr int PW = (N + G - 1) / G;     // waves per x parity
  static constexpr int NW = 2 * PW, NT = 64 * NW, GR = NT / TC;
  static constexpr int ELEMS = (N * Q * Q > N * N * N ? N * Q * Q : N * N * N) * TC;
  static constexpr int NE3 = N * N * N;
  static constexpr int NRB = (NE3 + 15) / 16;
  static constexpr int RBW = (NRB + NW - 1) / NW;
  static constexpr int CBW = TC / 16;
  // gather and scatter: a thread takes VW columns of whole x lines; lanes of a
  // line, lines at once, lines per thread
  static constexpr int NV = QE_ * QE_ * 4 * Q;   // weights of a cell
  static constexpr int VT = (NV + NT - 1) / NT;
  static constexpr int LR = TC / VW, LG = NT / LR, LT = (N * N + LG - 1) / LG;
  // waves per SIMD the registers are limited for: two workgroups per CU at
  // n = 7 (their LDS allows no more), else what fits without spills
  static constexpr int WPE = sizeof(T) == 8 ? 2 : (N == 7 ? 4 : 3);
};

// FP64 tables are scalar operands
typedef const __attribute__((address_space(4))) double *ctab;

// (I_z^T diag(v) I_z + wk K_z) u on one line, in place
template <int N, int Q>
__device__ __forceinline__ void tensor_line(double (&u)[N], const double *v, double wk, ctab tab) {
  using S = TensorTab<N, Q>;
  constexpr int NE = S::NE, NO = S::NO, QE = S::QE, QO = S::QO;
  double E[NE], O[NE], rE[NE], rO[NE];
#pragma unroll
  for (int i = 0; i < NO; ++i) {
    E[i] = u[i] + u[N - 1 - i];
    O[i] = u[i] - u[N - 1 - i];
  }
  if constexpr (N & 1) E[NO] = u[NO];
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    double t = tab[S::oKz + i * NE] * E[0];
#pragma unroll
    for (int j = 1; j < NE; ++j) t = fmadd(tab[S::oKz + i * NE + j], E[j], t);
    rE[i] = wk * t;
  }
#pragma unroll
  for (int i = 0; i < NO; ++i) {
    double t = tab[S::oKz + (NE + i) * NE] * O[0];
#pragma unroll
    for (int j = 1; j < NO; ++j) t = fmadd(tab[S::oKz + (NE + i) * NE + j], O[j], t);
    rO[i] = wk * t;
  }
#pragma unroll
  for (int k = 0; k < QE; ++k) {
    double e = tab[S::oI + k * NE] * E[0], o = 0.0;
#pragma unroll
    for (int i = 1; i < NE; ++i) e = fmadd(tab[S::oI + k * NE + i], E[i], e);
    if (k < QO) {
      o = tab[S::oI + (QE + k) * NE] * O[0];
#pragma unroll
      for (int i = 1; i < NO; ++i) o = fmadd(tab[S::oI + (QE + k) * NE + i], O[i], o);
      const double p = v[k] * (e + o), m = v[Q - 1 - k] * (e - o);
      e = p + m;
      o = p - m;
    } else {
      e = v[k] * e;
    }
#pragma unroll
    for (int i = 0; i < NE; ++i) rE[i] = fmadd(tab[S::oI + k * NE + i], e, rE[i]);
    if (k < QO) {
#pragma unroll
      for (int i = 0; i < NO; ++i) rO[i] = fmadd(tab[S::oI + (QE + k) * NE + i], o, rO[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < NO; ++i) {
    u[i] = rE[i] + rO[i];
    u[N - 1 - i] = rE[i] - rO[i];
  }
  if constexpr (N & 1) u[NO] = rE[NO];
}

// Plane stages of x parity PX: the thread's values of plane k are NX x N nodal
// ones, [x][y], y as even part (s = 0) and odd part (s = 1).
template <typename T, int N, int Q, int TC, int PX>
struct Planes {
  using S = TensorTab<N, Q>;
  static constexpr int NE = S::NE, NO = S::NO, QE = S::QE, QO = S::QO;
  static constexpr int NX = PX ? NO : NE, QX = PX ? QO : QE;
  typedef T Plane[2][NE][NE];  // [y parity][y][x]
  typedef Plane Sums;
  ctab tab;
  __device__ __forceinline__ Planes(const double *t, const float *) : tab((ctab)t) {}
  // entries of parity p
  __device__ __forceinline__ double I(int p, int r, int c) const {
    return tab[S::oI + (p * QE + r) * NE + c];
  }
  __device__ __forceinline__ double M(int p, int r, int c) const {
    return tab[S::oM + (p * NE + r) * NE + c];
  }
  __device__ __forceinline__ double Kx(int r, int c) const {
    return tab[S::oKx + (PX * NE + r) * NE + c];
  }
  __device__ __forceinline__ double Ky(int p, int r, int c) const {
    return tab[S::oKy + (p * NE + r) * NE + c];
  }

  // x-parity values [z][y][x] (the plane's part of buf) -> parity values
  static __device__ __forceinline__ void read(const T *b, Plane &x) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const T *c = b + ((PX ? NE : 0) + i) * TC;
#pragma unroll
      for (int j = 0; j < NO; ++j) {
        const T p = c[j * N * TC], m = c[(N - 1 - j) * N * TC];
        x[0][j][i] = p + m;
        x[1][j][i] = p - m;
      }
      if constexpr (N & 1) x[0][NO][i] = c[NO * N * TC];
    }
  }

  // b = (K_x M_y + M_x K_y) x -> nodal parity values [z][y][x] at b
  __device__ __forceinline__ void kinetic(const Plane &x, bool act, T *b) const {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int ns = s ? NO : NE;
#pragma unroll
      for (int j = 0; j < ns; ++j) {
        T m[NE], q[NE];
#pragma unroll
        for (int i = 0; i < NX; ++i) {
          m[i] = M(s, j, 0) * x[s][0][i];
          q[i] = Ky(s, j, 0) * x[s][0][i];
#pragma unroll
          for (int jj = 1; jj < ns; ++jj) {
            m[i] = fmadd(M(s, j, jj), x[s][jj][i], m[i]);
            q[i] = fmadd(Ky(s, j, jj), x[s][jj][i], q[i]);
          }
        }
#pragma unroll
        for (int i = 0; i < NX; ++i) {
          T r = Kx(i, 0) * m[0];
#pragma unroll
          for (int ii = 1; ii < NX; ++ii) r = fmadd(Kx(i, ii), m[ii], r);
#pragma unroll
          for (int ii = 0; ii < NX; ++ii) r = fmadd(M(PX, i, ii), q[ii], r);
          if (act) b[((s ? NE + j : j) * N + (PX ? NE : 0) + i) * TC] = r;
        }
      }
    }
  }

  static __device__ __forceinline__ void load(const T *b, Plane &o) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < (s ? NO : NE); ++j)
#pragma unroll
        for (int i = 0; i < NX; ++i)
          o[s][j][i] = b[((s ? NE + j : j) * N + (PX ? NE : 0) + i) * TC];
  }

  // u = I_x I_y x -> quadrature parity values [z][y][x] at b
  __device__ __forceinline__ void interpolate(const Plane &x, bool act, T *b) const {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int qs = s ? QO : QE, ns = s ? NO : NE;
#pragma unroll
      for (int j = 0; j < qs; ++j) {
        T w[NE];
#pragma unroll
        for (int i = 0; i < NX; ++i) {
          w[i] = I(s, j, 0) * x[s][0][i];
#pragma unroll
          for (int jj = 1; jj < ns; ++jj) w[i] = fmadd(I(s, j, jj), x[s][jj][i], w[i]);
        }
#pragma unroll
        for (int i = 0; i < QX; ++i) {
          T r = I(PX, i, 0) * w[0];
#pragma unroll
          for (int ii = 1; ii < NX; ++ii) r = fmadd(I(PX, i, ii), w[ii], r);
          if (act) b[((s ? QE + j : j) * Q + (PX ? QE : 0) + i) * TC] = r;
        }
      }
    }
  }

  // o += I_x^T I_y^T r
  __device__ __forceinline__ void collect(const T *b, Plane &o) const {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int qs = s ? QO : QE, ns = s ? NO : NE;
#pragma unroll
      for (int j = 0; j < qs; ++j) {
        T r[QE], w[NE];
#pragma unroll
        for (int i = 0; i < QX; ++i) r[i] = b[((s ? QE + j : j) * Q + (PX ? QE : 0) + i) * TC];
#pragma unroll
        for (int i = 0; i < NX; ++i) {
          w[i] = I(PX, 0, i) * r[0];
#pragma unroll
          for (int ii = 1; ii < QX; ++ii) w[i] = fmadd(I(PX, ii, i), r[ii], w[i]);
        }
#pragma unroll
        for (int jj = 0; jj < ns; ++jj)
#pragma unroll
          for (int i = 0; i < NX; ++i)
            o[s][jj][i] = fmadd(I(s, j, jj), w[i], o[s][jj][i]);
      }
    }
  }

  // x-parity values of the nodes, [z][y][x parity value] at b
  static __device__ __forceinline__ void store(const Plane &o, bool act, T *b) {
    if (!act) return;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      T *c = b + ((PX ? NE : 0) + i) * TC;
#pragma unroll
      for (int j = 0; j < NO; ++j) {
        c[j * N * TC] = o[0][j][i] + o[1][j][i];
        c[(N - 1 - j) * N * TC] = o[0][j][i] - o[1][j][i];
      }
      if constexpr (N & 1) c[NO * N * TC] = o[0][NO][i];
    }
  }
};

// z line stages
template <typename T, int N, int Q>
struct Lines {
  using S = TensorTab<N, Q>;
  static constexpr int NE = S::NE, NO = S::NO;
  ctab tab;
  __device__ __forceinline__ Lines(const double *t, const float *) : tab((ctab)t) {}
  // M_z on one line of nodal values (stride st), in place
  __device__ __forceinline__ void mass(T *b, int st) const {
    T E[NE], O[NE];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      const T p = b[i * st], m = b[(N - 1 - i) * st];
      E[i] = p + m;
      O[i] = p - m;
    }
    if constexpr (N & 1) E[NO] = b[NO * st];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      T e = tab[S::oM + i * NE] * E[0];
#pragma unroll
      for (int j = 1; j < NE; ++j) e = fmadd(tab[S::oM + i * NE + j], E[j], e);
      if (i < NO) {
        T o = tab[S::oM + (NE + i) * NE] * O[0];
#pragma unroll
        for (int j = 1; j < NO; ++j) o = fmadd(tab[S::oM + (NE + i) * NE + j], O[j], o);
        b[i * st] = e + o;
        b[(N - 1 - i) * st] = e - o;
      } else {
        b[i * st] = e;
      }
    }
  }
  __device__ __forceinline__ T weight(int i) const { return tab[S::oW + i]; }
  __device__ __forceinline__ void potential(T (&u)[N], const T *v, T wk) const {
    tensor_line<N, Q>(u, v, wk, tab);
  }
};

// ---------------------------------------------------------------------------
// FP32 forms on v_mfma_f32_4x4x1: one instruction is 16 independent 4 x 4
// outer products, lane l holding column l % 4 of block l / 4 and the four rows
// of the result in four registers.  With the table entry A[l % 4][k] in the
// first operand, four of them multiply each lane's own 4-vector by a 4 x 4
// table: the parity blocks here, at twice the rate of 16 vector FMAs and beside
// the vector pipe.  The second part of the stiffness tables is 84 more of them a wave:
// 619 -> 657 us per colour launch on 1024 columns (512 cells, n = 7), the time of
// these instructions alone.
// ---------------------------------------------------------------------------
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

// c + A x over the first K entries of x (x(k): the k-th)
template <int K, typename F>
__device__ __forceinline__ f32x4 mat4(f32x4 a, F x, f32x4 c) {
#pragma unroll
  for (int k = 0; k < K; ++k) c = mfma4(a[k], x(k), c);
  return c;
}

template <int N, int Q, int TC, int PX>
struct Planes<float, N, Q, TC, PX> {
  using S = TensorTab<N, Q>;
  static constexpr int NE = S::NE, NO = S::NO, QE = S::QE, QO = S::QO;
  static constexpr int NX = PX ? NO : NE, QX = PX ? QO : QE;
  typedef float Plane[2][NE][NE];  // [y parity][y][x]
  typedef f32x4 Sums[2][NE];       // [y parity][x] over y
  const f32x4 *tab;                // this lane's rows of the operand tables
  __device__ __forceinline__ Planes(const float *, const float *t)
      : tab(reinterpret_cast<const f32x4 *>(t) + (threadIdx.x & 3)) {}
  __device__ __forceinline__ f32x4 operand(int k) const { return tab[4 * k]; }

  static __device__ __forceinline__ void read(const float *b, Plane &x) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const float *c = b + ((PX ? NE : 0) + i) * TC;
#pragma unroll
      for (int j = 0; j < NO; ++j) {
        const float p = c[j * N * TC], m = c[(N - 1 - j) * N * TC];
        x[0][j][i] = p + m;
        x[1][j][i] = p - m;
      }
      if constexpr (N & 1) x[0][NO][i] = c[NO * N * TC];
    }
  }

  template <int s>
  __device__ __forceinline__ void kinetic_s(const Plane &x, bool act, float *b) const {
    constexpr int ns = s ? NO : NE;
    const f32x4 z = {0, 0, 0, 0};
    const f32x4 my = operand(kTabMe + s), ky = operand(kTabKy + s);
    const f32x4 mx = operand(kTabMe + PX), kx = operand(kTabKx + PX);
    const f32x4 ly = operand(kTabLy + s), lx = operand(kTabLx + PX);
    f32x4 m[NE], q[NE];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      auto l = [&](int j) { return x[s][j][i]; };
      m[i] = mat4<ns>(my, l, z);
      q[i] = mat4<ns>(ky, l, mat4<ns>(ly, l, z));
    }
#pragma unroll
    for (int j = 0; j < ns; ++j) {
      auto mj = [&](int i) { return m[i][j]; };
      const f32x4 r = mat4<NX>(mx, [&](int i) { return q[i][j]; },
                               mat4<NX>(kx, mj, mat4<NX>(lx, mj, z)));
#pragma unroll
      for (int i = 0; i < NX; ++i)
        if (act) b[((s ? NE + j : j) * N + (PX ? NE : 0) + i) * TC] = r[i];
    }
  }
  __device__ __forceinline__ void kinetic(const Plane &x, bool act, float *b) const {
    kinetic_s<0>(x, act, b);
    kinetic_s<1>(x, act, b);
  }

  static __device__ __forceinline__ void load(const float *b, Sums &o) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NX; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[s][i][j] = j < (s ? NO : NE) ? b[((s ? NE + j : j) * N + (PX ? NE : 0) + i) * TC] : 0.f;
  }

  template <int s>
  __device__ __forceinline__ void interpolate_s(const Plane &x, bool act, float *b) const {
    constexpr int ns = s ? NO : NE, qs = s ? QO : QE;
    const f32x4 z = {0, 0, 0, 0};
    const f32x4 iy = operand(kTabIe + s), ix = operand(kTabIe + PX);
    f32x4 w[NE];
#pragma unroll
    for (int i = 0; i < NX; ++i) w[i] = mat4<ns>(iy, [&](int j) { return x[s][j][i]; }, z);
#pragma unroll
    for (int j = 0; j < qs; ++j) {
      const f32x4 r = mat4<NX>(ix, [&](int i) { return w[i][j]; }, z);
#pragma unroll
      for (int i = 0; i < QX; ++i)
        if (act) b[((s ? QE + j : j) * Q + (PX ? QE : 0) + i) * TC] = r[i];
    }
  }
  __device__ __forceinline__ void interpolate(const Plane &x, bool act, float *b) const {
    interpolate_s<0>(x, act, b);
    interpolate_s<1>(x, act, b);
  }

  template <int s>
  __device__ __forceinline__ void collect_s(const float *b, Sums &o) const {
    constexpr int qs = s ? QO : QE;
    const f32x4 z = {0, 0, 0, 0};
    const f32x4 iy = operand(kTabIeT + s), ix = operand(kTabIeT + PX);
    f32x4 w[QE];
#pragma unroll
    for (int j = 0; j < qs; ++j)
      w[j] = mat4<QX>(ix, [&](int i) { return b[((s ? QE + j : j) * Q + (PX ? QE : 0) + i) * TC]; },
                      z);
#pragma unroll
    for (int i = 0; i < NX; ++i)
      o[s][i] = mat4<qs>(iy, [&](int j) { return w[j][i]; }, o[s][i]);
  }
  __device__ __forceinline__ void collect(const float *b, Sums &o) const {
    collect_s<0>(b, o);
    collect_s<1>(b, o);
  }

  static __device__ __forceinline__ void store(const Sums &o, bool act, float *b) {
    if (!act) return;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      float *c = b + ((PX ? NE : 0) + i) * TC;
#pragma unroll
      for (int j = 0; j < NO; ++j) {
        c[j * N * TC] = o[0][i][j] + o[1][i][j];
        c[(N - 1 - j) * N * TC] = o[0][i][j] - o[1][i][j];
      }
      if constexpr (N & 1) c[NO * N * TC] = o[0][i][NO];
    }
  }
};

template <int N, int Q>
struct Lines<float, N, Q> {
  using S = TensorTab<N, Q>;
  static constexpr int NE = S::NE, NO = S::NO, QE = S::QE, QO = S::QO;
  const f32x4 *tab;
  const float *weights;
  __device__ __forceinline__ Lines(const float *, const float *t)
      : tab(reinterpret_cast<const f32x4 *>(t) + (threadIdx.x & 3)), weights(t + kTabs * 16) {}
  __device__ __forceinline__ float weight(int i) const { return weights[i]; }
  __device__ __forceinline__ f32x4 operand(int k) const { return tab[4 * k]; }

  __device__ __forceinline__ void mass(float *b, int st) const {
    const f32x4 z = {0, 0, 0, 0};
    float E[NE], O[NE];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      const float p = b[i * st], m = b[(N - 1 - i) * st];
      E[i] = p + m;
      O[i] = p - m;
    }
    if constexpr (N & 1) E[NO] = b[NO * st];
    const f32x4 e = mat4<NE>(operand(kTabMe), [&](int k) { return E[k]; }, z);
    const f32x4 o = mat4<NO>(operand(kTabMo), [&](int k) { return O[k]; }, z);
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      b[i * st] = e[i] + o[i];
      b[(N - 1 - i) * st] = e[i] - o[i];
    }
    if constexpr (N & 1) b[NO * st] = e[NO];
  }

  __device__ __forceinline__ void potential(float (&u)[N], const float *v, float wk) const {
    const f32x4 z = {0, 0, 0, 0};
    float E[NE], O[NE];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      E[i] = u[i] + u[N - 1 - i];
      O[i] = u[i] - u[N - 1 - i];
    }
    if constexpr (N & 1) E[NO] = u[NO];
    auto Ek = [&](int k) { return E[k]; };
    auto Ok = [&](int k) { return O[k]; };
    f32x4 rE = mat4<NE>(operand(kTabKz), Ek, mat4<NE>(operand(kTabLz), Ek, z)) * wk;
    f32x4 rO = mat4<NO>(operand(kTabKzo), Ok, mat4<NO>(operand(kTabLzo), Ok, z)) * wk;
    f32x4 e = mat4<NE>(operand(kTabIe), Ek, z);
    f32x4 o = mat4<NO>(operand(kTabIo), Ok, z);
#pragma unroll
    for (int k = 0; k < QE; ++k) {
      if (k < QO) {
        const float p = v[k] * (e[k] + o[k]), m = v[Q - 1 - k] * (e[k] - o[k]);
        e[k] = p + m;
        o[k] = p - m;
      } else {
        e[k] = v[k] * e[k];
      }
    }
    rE = mat4<QE>(operand(kTabIeT), [&](int k) { return e[k]; }, rE);
    rO = mat4<QO>(operand(kTabIoT), [&](int k) { return o[k]; }, rO);
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      u[i] = rE[i] + rO[i];
      u[N - 1 - i] = rE[i] - rO[i];
    }
    if constexpr (N & 1) u[NO] = rE[NO];
  }
};

// VW neighbouring columns of a row
template <typename T, int VW>
using tvec = T __attribute__((ext_vector_type(VW)));
template <typename T, int VW>
__device__ __forceinline__ tvec<T, VW> vload(const T *p) {
  return *(const __attribute__((address_space(1))) tvec<T, VW> *)p;
}
template <typename T, int VW>
__device__ __forceinline__ void vstore(T *p, tvec<T, VW> v) {
  *(__attribute__((address_space(1))) tvec<T, VW> *)p = v;
}
// p + row g of a block whose rows are ldb bytes apart
template <typename T>
__device__ __forceinline__ T *row_ptr(T *p, uint32_t g, uint32_t ldb) {
  return (T *)((char *)p + (uint64_t)g * ldb);
}
// The four z lines mirrored in x and y, from their parity values at b<y><x>; hx, hy:
// whether the index has an odd value (a middle one does not, it counts as zero)
template <typename T, int N, int Q, int TC>
__device__ __forceinline__ void pencil(const T *b00, const T *b01, const T *b10, const T *b11,
                                       bool hx, bool hy, T (&u)[4][N]) {
#pragma unroll
  for (int z = 0; z < N; ++z) {
    const int f = z * Q * Q * TC;
    const T ee = b00[f];
    const T oe = (Q & 1) && !hx ? T(0) : b01[f];
    const T eo = (Q & 1) && !hy ? T(0) : b10[f];
    const T oo = (Q & 1) && !(hx && hy) ? T(0) : b11[f];
    const T s0 = ee + oe, d0 = ee - oe, s1 = eo + oo, d1 = eo - oo;
    u[0][z] = s0 + s1;
    u[1][z] = d0 + d1;
    u[2][z] = s0 - s1;
    u[3][z] = d0 - d1;
  }
}

// CELLS: all cells in one launch, each writing its own sums to cells_out
// [cell position in a.cells][node][column]; hx_assemble_kernel adds them up
template <typename T, int N, int Q, int TC, int VW, bool CELLS>
__global__ __launch_bounds__((TensorShape<T, N, Q, TC, VW>::NT))
__attribute__((amdgpu_waves_per_eu(TensorShape<T, N, Q, TC, VW>::WPE))) void hx_tensor_kernel(
    HxLaunch<T> a, const T *vq, const T *tabp, T *cells_out) {
  using S = TensorShape<T, N, Q, TC, VW>;
  using vec = tvec<T, VW>;
  const uint32_t lds_b = (uint32_t)(a.ld_src * sizeof(T)), ldd_b = (uint32_t)(a.ld_dst * sizeof(T)),
                 ldr_b = (uint32_t)(a.ldR * sizeof(T));
  constexpr int NE = S::NE, NO = S::NO, QE = S::QE, QO = S::QO, NE3 = S::NE3;
  constexpr int GR = S::GR, NW = S::NW, PW = S::PW;
  using v4 = typename V4<T>::t;
  using P0 = Planes<T, N, Q, TC, 0>;
  using P1 = Planes<T, N, Q, TC, 1>;
  __shared__ __align__(16) T buf[S::ELEMS];
  // per node: DOF and first-touch bit, input scale / 8, output scale; the
  // weights at the cell's quadrature points take the input scales' place
  __shared__ uint32_t smap[NE3];
  __shared__ T sout[NE3];
  __shared__ __align__(16) T svq[S::NV > NE3 ? S::NV : NE3];
  T *const ssin = svq;
  // the 4 x 4 operand tables of the FP32 form
  __shared__ __align__(16) float tabs[sizeof(T) == 4 ? kTabs * 16 + QE : 4];

  // consecutive items (the column tiles of a cell first) on one XCD
  const int item = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
  if (item >= a.ncells * a.ntiles || other_form(a)) return;
  const int cell = a.cells[item / a.ntiles];
  const int v0 = (item % a.ntiles) * TC;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int col = t % TC, grp = t / TC;
  // projector slots of the cell; the projectors of its first 16
  const int s0 = a.nl_off ? a.nl_off[cell] : 0;
  const int ns = a.nl_off ? a.nl_off[cell + 1] - s0 : 0;
  int slot0[4];
  if (ns > 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) slot0[r] = gload(a.slot_proj, s0 + 4 * (lane >> 4) + r);
  }
  if constexpr (sizeof(T) == 4) {
    static_assert(kTabs * 16 + QE <= S::NT, "one table entry per thread");
    if (t < kTabs * 16 + QE) tabs[t] = tabp[t];
  }

  // ---- gather: x lines of the cell's nodes, scaled, as x-parity values into
  // buf[z][y][even, odd][col]
  const int rl = t % S::LR, lg = t / S::LR;     // lane of a line, first line
  const int vr = v0 + rl * VW;
  const bool vin = vr < a.B;                    // VW > 1: B is a multiple of it
  const int vc = vin ? vr : a.B - VW;
  // W rows of 16 slots (four per lane), from the slots' projectors
  auto projectors = [&](const int (&p)[4], T(&w)[4][S::CBW]) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int cb = 0; cb < S::CBW; ++cb) {
        const int v = v0 + cb * 16 + (lane & 15);
        w[r][cb] = gload(a.W, (int64_t)(p[r] < 0 ? 0 : p[r]) * a.ldW + (v < a.B ? v : a.B - 1));
      }
  };
  // projector columns of 16 slots: this wave's row blocks, four slots a lane
  auto columns = [&](int kt, T(&c)[S::RBW][4]) {
    const T *cm = a.nl_C + ((int64_t)s0 + kt) * a.ne_pad;
#pragma unroll
    for (int j = 0; j < S::RBW; ++j) {
      const int rb = wave + NW * j < S::NRB ? wave + NW * j : 0;
      const T *p = cm + (rb * 16 + (lane & 15)) * 16 + 4 * (lane >> 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) c[j][r] = gload(p, r);
    }
  };
  T c0[S::RBW][4], w0[4][S::CBW];

  // the cell's map and scales go through LDS: read by every lane of a line
  // they cost more than the rows themselves (28 loads per thread at n = 7)
  T vreg[S::VT];
  {
    constexpr int MT = (NE3 + S::NT - 1) / S::NT;
    uint32_t w[MT];
#pragma unroll
    for (int e = 0; e < MT; ++e) {
      const int i = t + e * S::NT;
      w[e] = gload(a.map, (int64_t)cell * NE3 + (i < NE3 ? i : 0));
      if (i < NE3) smap[i] = w[e];
    }
    __syncthreads();
    vec x[S::LT][N];
#pragma unroll
    for (int l = 0; l < S::LT; ++l) {
      const int line = lg + l * S::LG, lc = line < N * N ? line : N * N - 1;
#pragma unroll
      for (int i = 0; i < N; ++i)
        x[l][i] = vload<T, VW>(row_ptr(a.src + vc, smap[lc * N + i] & 0x7fffffffu, lds_b));
    }
    T si[MT], so[MT];
#pragma unroll
    for (int e = 0; e < MT; ++e) {
      si[e] = a.s_in ? gload(a.s_in, w[e] & 0x7fffffffu) : T(1);
      so[e] = a.s_out == a.s_in ? si[e] : (a.s_out ? gload(a.s_out, w[e] & 0x7fffffffu) : T(1));
    }
#pragma unroll
    for (int e = 0; e < S::VT; ++e) {
      const int i = t + e * S::NT;
      vreg[e] = gload(vq, (int64_t)cell * S::NV + (i < S::NV ? i : 0));
    }
    if (ns > 0) {
      projectors(slot0, w0);
      columns(0, c0);
    }
#pragma unroll
    for (int e = 0; e < MT; ++e) {
      const int i = t + e * S::NT;
      if (i < NE3) {
        ssin[i] = T(0.125) * si[e];
        sout[i] = so[e];
      }
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < S::LT; ++l) {
      const int line = lg + l * S::LG;
      if (line >= N * N) continue;
      T *b = buf + line * N * TC + rl * VW;
#pragma unroll
      for (int i = 0; i < N; ++i) x[l][i] *= ssin[line * N + i];
#pragma unroll
      for (int i = 0; i < NO; ++i) {
        *reinterpret_cast<vec *>(b + i * TC) = x[l][i] + x[l][N - 1 - i];
        *reinterpret_cast<vec *>(b + (NE + i) * TC) = x[l][i] - x[l][N - 1 - i];
      }
      if constexpr (N & 1) *reinterpret_cast<vec *>(b + NO * TC) = x[l][NO];
    }
  }
  __syncthreads();

  // ---- plane stages: this wave's x parity and the thread's plane
  const bool px = wave >= PW;
  const int kk = (wave - (px ? PW : 0)) * S::G + lane / TC;
  const bool act = kk < N;
  const int k = act ? kk : N - 1;
  T *const bn = buf + k * (N * N) * TC + col;   // the plane's nodal values
  T *const bq = buf + k * (Q * Q) * TC + col;   // its quadrature values
  const P0 p0(tabp, tabs);
  const P1 p1(tabp, tabs);
  const Lines<T, N, Q> lines(tabp, tabs);
  typename P0::Plane x;
  typename P0::Sums o;
  if (px) P1::read(bn, x); else P0::read(bn, x);
#pragma unroll
  for (int e = 0; e < S::VT; ++e) {
    const int i = t + e * S::NT;
    if (i < S::NV) svq[i] = vreg[e];
  }
  __syncthreads();
  if (px) p1.kinetic(x, act, bn); else p0.kinetic(x, act, bn);
  __syncthreads();
  // the nonlocal term C_e W runs on the matrix pipe beside the mass lines and
  // joins the in-plane kinetic part in its rows
  v4 acc[S::RBW][S::CBW];
  if (ns > 0) {
#pragma unroll
    for (int j = 0; j < S::RBW; ++j)
#pragma unroll
      for (int cb = 0; cb < S::CBW; ++cb) acc[j][cb] = v4{T(0), T(0), T(0), T(0)};
    for (int kt = 0; kt < ns; kt += 16) {
      if (kt > 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) slot0[r] = gload(a.slot_proj, s0 + kt + 4 * (lane >> 4) + r);
        projectors(slot0, w0);
        columns(kt, c0);
      }
      // a slot without projector (padding) has a zero column; its row of W is
      // another slot's, which need not be finite
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int cb = 0; cb < S::CBW; ++cb) w0[r][cb] = slot0[r] < 0 ? T(0) : w0[r][cb];
#pragma unroll
      for (int j = 0; j < S::RBW; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int cb = 0; cb < S::CBW; ++cb) acc[j][cb] = mfma16(c0[j][r], w0[r][cb], acc[j][cb]);
    }
  }
  for (int id = grp; id < N * N; id += GR) lines.mass(buf + id * TC + col, N * N * TC);
  __syncthreads();
  if (ns > 0) {
#pragma unroll
    for (int j = 0; j < S::RBW; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = (wave + NW * j) * 16 + acc_row<T>(lane, r);
        if (row < NE3)
#pragma unroll
          for (int cb = 0; cb < S::CBW; ++cb)
            buf[row * TC + cb * 16 + (lane & 15)] += acc[j][cb][r];
      }
    __syncthreads();
  }
  if (px) P1::load(bn, o); else P0::load(bn, o);
  __syncthreads();
  if (px) p1.interpolate(x, act, bq); else p0.interpolate(x, act, bq);
  __syncthreads();

  // ---- z lines of u: four mirrored lines per thread
  for (int id = grp; id < QE * QE; id += GR) {
    const int ix = id % QE, iy = id / QE;
    const bool hx = ix < QO, hy = iy < QO;
    T *b00 = buf + (iy * Q + ix) * TC + col;
    T *b01 = b00 + (hx ? QE : 0) * TC, *b10 = b00 + (hy ? QE : 0) * Q * TC,
      *b11 = b10 + (hx ? QE : 0) * TC;
    T u[4][N];
    pencil<T, N, Q, TC>(b00, b01, b10, b11, hx, hy, u);
    const T wk = lines.weight(ix) * lines.weight(iy);
    const T *v = svq + id * (4 * Q);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      T vv[Q];
#pragma unroll
      for (int z = 0; z < Q; ++z) vv[z] = v[s * Q + z];
      lines.potential(u[s], vv, wk);
    }
#pragma unroll
    for (int z = 0; z < N; ++z) {
      const int f = z * Q * Q * TC;
      const T s0 = u[0][z] + u[1][z], d0 = u[0][z] - u[1][z], s1 = u[2][z] + u[3][z],
              d1 = u[2][z] - u[3][z];
      b00[f] = s0 + s1;
      if (!(Q & 1) || hx) b01[f] = d0 + d1;
      if (!(Q & 1) || hy) b10[f] = s0 - s1;
      if (!(Q & 1) || (hx && hy)) b11[f] = d0 - d1;
    }
  }

  // ---- the destination's rows: loaded here so that they arrive while the last
  // plane stages run
  vec dv[S::LT][N];
  if constexpr (!CELLS) {
#pragma unroll
    for (int l = 0; l < S::LT; ++l) {
      const int line = lg + l * S::LG, lc = line < N * N ? line : N * N - 1;
#pragma unroll
      for (int i = 0; i < N; ++i)
        dv[l][i] = vload<T, VW>(row_ptr(a.dst + vc, smap[lc * N + i] & 0x7fffffffu, ldd_b));
    }
  }
  __syncthreads();
  if (px) p1.collect(bq, o); else p0.collect(bq, o);
  __syncthreads();
  if (px) P1::store(o, act, bn); else P0::store(o, act, bn);
  // what the combine adds on first touch: gamma times the source's row, and in
  // the defect form rcoef times the row of R.  Other rows read the block's first
  // row: one line for all of them
  T gamma = a.gamma;
  vec sv[S::LT][N];
#pragma unroll
  for (int l = 0; l < S::LT; ++l) {
    if constexpr (CELLS) continue;
    const bool any_src = a.gamma != T(0);
    const int line = lg + l * S::LG, lc = line < N * N ? line : N * N - 1;
    if (any_src) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const uint32_t w = smap[lc * N + i];
        sv[l][i] = vload<T, VW>(row_ptr(a.src + vc, w >> 31 ? w & 0x7fffffffu : 0, lds_b));
      }
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) sv[l][i] = T(0);
    }
  }
  if constexpr (sizeof(T) == 4 && !CELLS) {
    if (a.R) {
      const vec rc = vload<T, VW>(a.rcoef + vc);
#pragma unroll
      for (int l = 0; l < S::LT; ++l) {
        const int line = lg + l * S::LG, lc = line < N * N ? line : N * N - 1;
        vec rv[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const uint32_t w = smap[lc * N + i];
          rv[i] = vload<T, VW>(row_ptr(a.R + vc, w >> 31 ? w & 0x7fffffffu : 0, ldr_b));
        }
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int e = 0; e < VW; ++e)
            sv[l][i][e] = fmadd(rc[e], rv[i][e], gamma * sv[l][i][e]);
      }
      gamma = T(1);
    }
  }

  __syncthreads();

  // ---- scatter (the combine of hx_scatter)
#pragma unroll
  for (int l = 0; l < S::LT; ++l) {
    const int line = lg + l * S::LG;
    if (line >= N * N) continue;
    const T *b = buf + line * N * TC + rl * VW;
    vec y[N];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      const vec e = *reinterpret_cast<const vec *>(b + i * TC),
                f = *reinterpret_cast<const vec *>(b + (NE + i) * TC);
      y[i] = e + f;
      y[N - 1 - i] = e - f;
    }
    if constexpr (N & 1) y[NO] = *reinterpret_cast<const vec *>(b + NO * TC);
    if constexpr (CELLS) {
      T *out = cells_out + ((int64_t)(item / a.ntiles) * NE3 + line * N) * a.B + vc;
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (vin) vstore<T, VW>(out + (int64_t)i * a.B, y[i]);
      continue;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t w = smap[line * N + i], g = w & 0x7fffffffu;
      const bool first = (w >> 31) != 0;
      const T so = sout[line * N + i];
      // a zero output scale marks a constrained row (hanging node): it takes
      // the plain sums, nothing else on first touch
      const bool cons = so == T(0);
      const T sa = a.alpha * (cons ? T(1) : so);
      const T kf = a.beta_mode == 2 ? a.beta * so : a.beta;
      vec base;
#pragma unroll
      for (int e = 0; e < VW; ++e) {
        const T d = dv[l][i][e];
        T c = fmadd(gamma, sv[l][i][e], a.beta_mode == 1 ? T(0) : kf * d);
        c = first ? (cons ? T(0) : c) : d;
        base[e] = fmadd(sa, y[i][e], c);
      }
      if (vin) vstore<T, VW>(row_ptr(a.dst + vc, g, ldd_b), base);
    }
  }
}

// ---------------------------------------------------------------------------
// Sum of the cells' contributions, row by row in colour order: the same
// multiply-adds in the same order as the colour launches, so the same bits.
// ---------------------------------------------------------------------------
template <typename T, int VW>
__global__ __launch_bounds__(256) void hx_assemble_kernel(HxLaunch<T> a, const uint32_t *ptr,
                                                          const uint32_t *idx, int64_t M,
                                                          const T *cells_out) {
  using vec = tvec<T, VW>;
  const int per = a.B / VW;
  const int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x;
  const int64_t g = e / per;
  if (g >= M || other_form(a)) return;
  const int v = (int)(e % per) * VW;
  const uint32_t k0 = ptr[g], k1 = ptr[g + 1];
  if (k0 == k1) return;  // a folded row: no cell writes it
  const vec d = vload<T, VW>(a.dst + g * a.ld_dst + v);
  vec x, r;
#pragma unroll
  for (int i = 0; i < VW; ++i) x[i] = r[i] = T(0);
  if (a.gamma != T(0)) x = vload<T, VW>(a.src + g * a.ld_src + v);
  T gamma = a.gamma;
  if constexpr (sizeof(T) == 4) {
    if (a.R) {
      r = vload<T, VW>(a.R + g * a.ldR + v);
      const vec rc = vload<T, VW>(a.rcoef + v);
#pragma unroll
      for (int i = 0; i < VW; ++i) x[i] = fmadd(rc[i], r[i], gamma * x[i]);
      gamma = T(1);
    }
  }
  const T so = a.s_out ? a.s_out[g] : T(1);
  const bool cons = so == T(0);
  const T sa = a.alpha * (cons ? T(1) : so);
  const T kf = a.beta_mode == 2 ? a.beta * so : a.beta;
  vec y;
#pragma unroll
  for (int i = 0; i < VW; ++i)
    y[i] = cons ? T(0) : fmadd(gamma, x[i], a.beta_mode == 1 ? T(0) : kf * d[i]);
  for (uint32_t k = k0; k < k1; ++k) {
    const vec c = vload<T, VW>(cells_out + (int64_t)idx[k] * a.B + v);
#pragma unroll
    for (int i = 0; i < VW; ++i) y[i] = fmadd(sa, c[i], y[i]);
  }
  vstore<T, VW>(a.dst + g * a.ld_dst + v, y);
}

template <typename T, int N, int Q, int TC, int VW>
static hipError_t hx_tensor_go(HxLaunch<T> a, const T *vq, const T *tab, const TensorTouch *touch,
                               T *cells_out, hipStream_t s) {
  using S = TensorShape<T, N, Q, TC, VW>;
  a.ntiles = (a.B + TC - 1) / TC;
  const int items = a.ncells * a.ntiles;
  if (items == 0) return hipSuccess;
  a.per_xcd = (items + 7) / 8;
  if (!touch) {
    hipLaunchKernelGGL((hx_tensor_kernel<T, N, Q, TC, VW, false>), dim3(8 * a.per_xcd),
                       dim3(S::NT), 0, s, a, vq, tab, nullptr);
    return hipGetLastError();
  }
  hipLaunchKernelGGL((hx_tensor_kernel<T, N, Q, TC, VW, true>), dim3(8 * a.per_xcd), dim3(S::NT),
                     0, s, a, vq, tab, cells_out);
  const int64_t n = touch->M * (a.B / VW);
  hipLaunchKernelGGL((hx_assemble_kernel<T, VW>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     s, a, touch->ptr, touch->idx, touch->M, cells_out);
  return hipGetLastError();
}

// 16 bytes per lane (FP32: four columns, FP64: two) need whole, aligned groups
// of columns in every block; FP32 falls back to pairs, both to single columns.
template <typename T, int N, int Q, int TC>
static hipError_t hx_tensor_vec(const HxLaunch<T> &a, const T *vq, const T *tab,
                                const TensorTouch *touch, T *cells_out, hipStream_t s) {
  auto whole = [&](int w) {
    auto ok = [w](const T *p, int64_t ld) {
      return reinterpret_cast<uintptr_t>(p) % (w * sizeof(T)) == 0 && ld % w == 0;
    };
    return a.B % w == 0 && ok(a.src, a.ld_src) && ok(a.dst, a.ld_dst) && ok(a.R, a.ldR) &&
           ok(a.rcoef, 0);
  };
  if constexpr (sizeof(T) == 4)
    if (whole(4)) return hx_tensor_go<T, N, Q, TC, 4>(a, vq, tab, touch, cells_out, s);
  return whole(2) ? hx_tensor_go<T, N, Q, TC, 2>(a, vq, tab, touch, cells_out, s)
                  : hx_tensor_go<T, N, Q, TC, 1>(a, vq, tab, touch, cells_out, s);
}

// Where the tensor form is taken (cells: of the largest colour; one MI355X, ms per
// apply, tensor / best tile variant or, for one column, the matrix-vector kernel):
//   n = 7: 4096 cells x 1024 columns 6.1 / 11.0 FP32, 1728 x 1024 5.2 / 9.9 FP64,
//          1728 x 16 0.21 / 0.86, x 1 0.16 / 0.48
//   n = 6: 1728 cells x 256 columns 1.07 / 1.34 FP64, 0.61 / 0.79 FP32, x 1 0.16 / 0.29
//   n = 5: the dense product is only 1.7 times the operations, on the matrix
//          pipe; the tensor form has fewer bytes in flight behind its barriers
//          and wins while a colour does not fill the chip.  us per apply, tensor /
//          dense at workgroups a colour: FP64 256 141 / 196, 384 194 / 210, 432
//          215 / 204, 512 253 / 216; FP32 432 133 / 203, 640 213 / 220, 768
//          220 / 223, 864 275 / 230, 1024 301 / 229; without projectors FP64
//          432 150 / 167, 448 149 / 152.  One column, all cells at once:
//          64 cells a colour 50 / 120; colour by colour (no projectors) the
//          matrix-vector kernel is faster on few cells: FP64 27 92 / 83, 64 89 / 93;
//          FP32 64 70 / 69, 216 71 / 83
static int tile_columns(int n, bool fp64) { return n == 7 && fp64 ? 16 : 32; }

static int64_t colour_items(int n, bool fp64, int cells, int B) {
  const int tc = tile_columns(n, fp64);
  return int64_t(cells) * ((B + tc - 1) / tc);
}

bool tensor_wins(int n, bool fp64, int cells, int B, bool all) {
  if (n > 5) return true;
  const int64_t items = colour_items(n, fp64, cells, B);
  if (B == 1) return items <= kAllCellsItems && (all || cells >= (fp64 ? 64 : 128));
  return items <= (fp64 ? (all ? 400 : 448) : 640);
}

// One launch over all cells and a sum (all) against the colour launches: a launch
// lasts as long as one workgroup (12-20 us) however few it has, and eight of
// them in turn leave a small apply waiting; beyond about 450 workgroups a colour
// the extra pass over the cells' sums costs what the waiting did.  ms per apply,
// colours / all, FP64: n = 5, 512 cells x 1 column 0.140 / 0.051, x 64 0.146 / 0.092,
// x 128 0.154 / 0.142, x 400 0.416 / 0.408; n = 7, 512 cells x 1 0.215 / 0.070,
// x 64 0.228 / 0.177, x 128 0.304 / 0.306; 1728 x 16 0.264 / 0.213
bool tensor_all_cells(int n, bool fp64, int cells, int B) {
  return colour_items(n, fp64, cells, B) <= kAllCellsItems;
}

int tensor_all_cells_columns(int n, bool fp64, int cells) {
  return kAllCellsItems / cells * tile_columns(n, fp64);
}

template <typename T>
hipError_t launch_hx_tensor(const HxLaunch<T> &a, const T *vq, const T *tab, int n, int q,
                            const TensorTouch *touch, T *cells_out, hipStream_t s) {
  constexpr int W7 = sizeof(T) == 8 ? 16 : 32;
  if (n == 7 && q == 8) return hx_tensor_vec<T, 7, 8, W7>(a, vq, tab, touch, cells_out, s);
  if (n == 6 && q == 6) return hx_tensor_vec<T, 6, 6, 32>(a, vq, tab, touch, cells_out, s);
  if (n == 5 && q == 5) return hx_tensor_vec<T, 5, 5, 32>(a, vq, tab, touch, cells_out, s);
  return hipErrorInvalidValue;
}
template hipError_t launch_hx_tensor<double>(const HxLaunch<double> &, const double *,
                                             const double *, int, int, const TensorTouch *,
                                             double *, hipStream_t);
template hipError_t launch_hx_tensor<float>(const HxLaunch<float> &, const float *, const float *,
                                            int, int, const TensorTouch *, float *, hipStream_t);

// ---------------------------------------------------------------------------
// Products of two blocks at the quadrature points, tensor form (see
// launch_quad_product): one workgroup per cell walks over the column tiles.  The
// plane and line stages are those of the apply, one way and in FP64; a thread
// of the line stage keeps the sums of its 4 Q points over its column, which are
// added over the TC columns at the end, in a fixed order.  The next block's rows
// are on their way while the lines run.  Bound by the gather: 4096 cells x 1024
// columns (11.5 GB) 42 -> 2.8 ms for the density, 72 -> 7.7 ms for two blocks,
// against the dense interpolation on FP64 MFMA.
// ---------------------------------------------------------------------------
template <bool SAME, typename TIn, int N, int Q, int TC, int VW>
__global__ __launch_bounds__((TensorShape<double, N, Q, TC, VW>::NT))
__attribute__((amdgpu_waves_per_eu(2))) void quad_tensor_kernel(
    const uint32_t *map, const double *JxW, const TIn *a, int64_t lda, const TIn *b, int64_t ldb,
    int B, const double *s_in, const double *w, int wshift, double wscale, double *g,
    int accumulate, const double *tabp) {
  using S = TensorShape<double, N, Q, TC, VW>;
  constexpr int NE = S::NE, NO = S::NO, QE = S::QE, QO = S::QO, NE3 = S::NE3;
  static_assert(QE * QE <= S::GR, "one group of lines per thread");
  using P0 = Planes<double, N, Q, TC, 0>;
  using P1 = Planes<double, N, Q, TC, 1>;
  using vec = tvec<TIn, VW>;
  __shared__ __align__(16) double buf[S::ELEMS];
  __shared__ uint32_t smap[NE3];
  __shared__ double ssin[NE3];
  const int cell = blockIdx.x;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int col = t % TC, grp = t / TC;
  for (int i = t; i < NE3; i += S::NT) {
    const uint32_t d = gload(map, (int64_t)cell * NE3 + i) & 0x7fffffffu;
    smap[i] = d;
    ssin[i] = 0.125 * (s_in ? gload(s_in, d) : 1.0);
  }
  __syncthreads();

  const int rl = t % S::LR, lg = t / S::LR;
  const uint32_t lda_b = (uint32_t)(lda * sizeof(TIn)), ldb_b = (uint32_t)(ldb * sizeof(TIn));
  vec x[S::LT][N];
  // rows of one column tile; columns beyond the block are zero
  auto load = [&](const TIn *p, uint32_t ldp, int v0) {
    const int v = v0 + rl * VW, vc = v < B ? v : B - VW;  // VW > 1: B is a multiple of it
#pragma unroll
    for (int l = 0; l < S::LT; ++l) {
      const int line = lg + l * S::LG, lc = line < N * N ? line : N * N - 1;
#pragma unroll
      for (int i = 0; i < N; ++i) x[l][i] = vload<TIn, VW>(row_ptr(p + vc, smap[lc * N + i], ldp));
    }
  };
  const bool px = wave >= S::PW;
  const int kk = (wave - (px ? S::PW : 0)) * S::G + lane / TC;
  const bool act = kk < N;
  const int k = act ? kk : N - 1;
  double *const bn = buf + k * (N * N) * TC + col;
  double *const bq = buf + k * (Q * Q) * TC + col;
  const P0 p0(tabp, nullptr);
  const P1 p1(tabp, nullptr);
  const ctab tab = (ctab)tabp;
  const int ix = grp % QE, iy = grp / QE;
  const bool line_in = grp < QE * QE, hx = ix < QO, hy = iy < QO;
  double acc[4][Q];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int z = 0; z < Q; ++z) acc[s][z] = 0.0;

  load(a, lda_b, 0);
  for (int v0 = 0; v0 < B; v0 += TC) {
    const int v = v0 + col;
    const double wv = v < B ? (w ? gload(w, v >> wshift) : 1.0) : 0.0;
    double ua[SAME ? 1 : 4][SAME ? 1 : Q];
#pragma unroll
    for (int side = 0; side < (SAME ? 1 : 2); ++side) {
      const bool cin = v0 + rl * VW < B;
#pragma unroll
      for (int l = 0; l < S::LT; ++l) {
        const int line = lg + l * S::LG;
        if (line >= N * N) continue;
        double *d = buf + line * N * TC + rl * VW;
#pragma unroll
        for (int e = 0; e < VW; ++e) {
          double y[N];
#pragma unroll
          for (int i = 0; i < N; ++i)
            y[i] = cin ? (double)x[l][i][e] * ssin[line * N + i] : 0.0;
#pragma unroll
          for (int i = 0; i < NO; ++i) {
            d[i * TC + e] = y[i] + y[N - 1 - i];
            d[(NE + i) * TC + e] = y[i] - y[N - 1 - i];
          }
          if constexpr (N & 1) d[NO * TC + e] = y[NO];
        }
      }
      __syncthreads();
      typename P0::Plane pl;
      if (px) P1::read(bn, pl); else P0::read(bn, pl);
      __syncthreads();
      if (px) p1.interpolate(pl, act, bq); else p0.interpolate(pl, act, bq);
      if constexpr (SAME) {
        if (v0 + TC < B) load(a, lda_b, v0 + TC);
      }
      __syncthreads();
      if (line_in) {
        const double *b00 = buf + (iy * Q + ix) * TC + col;
        const double *b01 = b00 + (hx ? QE : 0) * TC, *b10 = b00 + (hy ? QE : 0) * Q * TC,
                     *b11 = b10 + (hx ? QE : 0) * TC;
        double u[4][N];
        pencil<double, N, Q, TC>(b00, b01, b10, b11, hx, hy, u);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          double E[NE], O[NE];
#pragma unroll
          for (int i = 0; i < NO; ++i) {
            E[i] = u[s][i] + u[s][N - 1 - i];
            O[i] = u[s][i] - u[s][N - 1 - i];
          }
          if constexpr (N & 1) E[NO] = u[s][NO];
#pragma unroll
          for (int z = 0; z < QE; ++z) {
            double e = tab[S::oI + z * NE] * E[0], o = 0.0;
#pragma unroll
            for (int i = 1; i < NE; ++i) e = fmadd(tab[S::oI + z * NE + i], E[i], e);
            if (z < QO) {
              o = tab[S::oI + (QE + z) * NE] * O[0];
#pragma unroll
              for (int i = 1; i < NO; ++i) o = fmadd(tab[S::oI + (QE + z) * NE + i], O[i], o);
            }
            const double p = z < QO ? e + o : e, m = e - o;
            if constexpr (SAME) {
              acc[s][z] = fmadd(wv * p, p, acc[s][z]);
              if (z < QO) acc[s][Q - 1 - z] = fmadd(wv * m, m, acc[s][Q - 1 - z]);
            } else if (side == 0) {
              ua[s][z] = wv * p;
              if (z < QO) ua[s][Q - 1 - z] = wv * m;
            } else {
              acc[s][z] = fmadd(ua[s][z], p, acc[s][z]);
              if (z < QO) acc[s][Q - 1 - z] = fmadd(ua[s][Q - 1 - z], m, acc[s][Q - 1 - z]);
            }
          }
        }
      }
      if constexpr (!SAME) {
        if (side == 0) load(b, ldb_b, v0);
        else if (v0 + TC < B) load(a, lda_b, v0 + TC);
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int z = 0; z < Q; ++z) {
      double r = acc[s][z];
#pragma unroll
      for (int off = TC / 2; off >= 1; off >>= 1) r += __shfl_xor(r, off);
      acc[s][z] = r;
    }
  if (line_in && col == 0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if ((Q & 1) && ((s & 1 && !hx) || (s & 2 && !hy))) continue;  // the same line again
      const int qx = s & 1 ? Q - 1 - ix : ix, qy = s & 2 ? Q - 1 - iy : iy;
#pragma unroll
      for (int z = 0; z < Q; ++z) {
        const int64_t o = (int64_t)cell * (Q * Q * Q) + qx + Q * (qy + Q * z);
        g[o] = (accumulate ? g[o] : 0.0) + (JxW ? JxW[o] : 1.0) * wscale * acc[s][z];
      }
    }
  }
}

template <typename TIn, int N, int Q, int TC>
static hipError_t quad_tensor_go(const uint32_t *map, int C, const double *JxW, const TIn *a,
                                 int64_t lda, const TIn *b, int64_t ldb, int B,
                                 const double *s_in, const double *w, int wshift, double wscale,
                                 double *g, int accumulate, const double *tab, hipStream_t s) {
  constexpr int V = 16 / sizeof(TIn);
  auto ok = [](const TIn *p, int64_t ld) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0 && ld % V == 0;
  };
  const bool wide = B % V == 0 && ok(a, lda) && ok(b, ldb);
  const bool same = a == b && lda == ldb;
#define CHFSI_QUAD(SAME, VW)                                                                  \
  hipLaunchKernelGGL((quad_tensor_kernel<SAME, TIn, N, Q, TC, VW>), dim3(C),                  \
                     dim3(TensorShape<double, N, Q, TC, VW>::NT), 0, s, map, JxW, a, lda, b,  \
                     ldb, B, s_in, w, wshift, wscale, g, accumulate, tab)
  if (wide && same) CHFSI_QUAD(true, V);
  else if (wide) CHFSI_QUAD(false, V);
  else if (same) CHFSI_QUAD(true, 1);
  else CHFSI_QUAD(false, 1);
#undef CHFSI_QUAD
  return hipGetLastError();
}

template <typename TIn>
hipError_t launch_quad_tensor(const uint32_t *map, int C, int n, int q, const double *JxW,
                              const TIn *a, int64_t lda, const TIn *b, int64_t ldb, int B,
                              const double *s_in, const double *w, int wshift, double wscale,
                              double *g, int accumulate, const double *tab, hipStream_t s) {
  if (n == 7 && q == 8)
    return quad_tensor_go<TIn, 7, 8, 16>(map, C, JxW, a, lda, b, ldb, B, s_in, w, wshift, wscale,
                                         g, accumulate, tab, s);
  if (n == 6 && q == 6)
    return quad_tensor_go<TIn, 6, 6, 32>(map, C, JxW, a, lda, b, ldb, B, s_in, w, wshift, wscale,
                                         g, accumulate, tab, s);
  if (n == 5 && q == 5)
    return quad_tensor_go<TIn, 5, 5, 32>(map, C, JxW, a, lda, b, ldb, B, s_in, w, wshift, wscale,
                                         g, accumulate, tab, s);
  return hipErrorInvalidValue;
}
template hipError_t launch_quad_tensor<double>(const uint32_t *, int, int, int, const double *,
                                               const double *, int64_t, const double *, int64_t,
                                               int, const double *, const double *, int, double,
                                               double *, int, const double *, hipStream_t);
template hipError_t launch_quad_tensor<float>(const uint32_t *, int, int, int, const double *,
                                              const float *, int64_t, const float *, int64_t, int,
                                              const double *, const double *, int, double,
                                              double *, int, const double *, hipStream_t);

// ---------------------------------------------------------------------------
// Cell matrices, tensor form: H_e = 1/2 K + sum_q N_i N_j v_q (+ the GGA term), as
// launch_build_h writes them.  A column (i', j', k') is contracted direction by
// direction with the products P[a][b][q] of the tables: over z for its k', over
// y for its (j', k') (shared by the n columns of a run), over x with 8 products
// per entry, where the dense build took 512 (2048 with GGA).  A workgroup takes
// one cell and a range of 16-column tiles; wave w writes the rows with i = w, two
// columns per lane, so every 128-byte row of a tile is stored whole.  Entries
// are sums over the same products in the same order for (i, j) and (j, i):
// exactly symmetric.  Bound by the stores (7.1 GB of FP64, FP32 and BF16 copies
// at 4096 cells, p = 6): LDA 5.5 -> 2.8 ms, GGA 20.1 -> 4.4 ms.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  auto r = [](float x) {
    uint32_t u = __float_as_uint(x);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
  };
  return r(a) | (r(b) << 16);
}

template <int N, int Q, bool GGA>
__global__ __launch_bounds__(64 * N) void build_tensor_kernel(const double *K, const double *P,
                                                             const double *vJxW,
                                                             const double *gJxW, int ne_pad,
                                                             int tiles, double *Ht64, float *Ht32,
                                                             uint16_t *Ht16) {
  constexpr int NT = 64 * N, NN = N * N, NE3 = NN * N, QQ = Q * Q, RUNS = 4;
  constexpr int F = GGA ? 3 : 1, G2 = GGA ? 2 : 1, NP = GGA ? 4 : 1;
  constexpr int SB = Q == 8 ? 10 : 6;  // row of y-contracted values, 16-byte aligned
  static_assert(16 <= (RUNS - 1) * N + 1, "runs of a tile");
  __shared__ double sP[NP][NN][Q];               // products
  __shared__ double sV[GGA ? 4 : 1][Q * QQ];     // weights (V, then g of each direction)
  __shared__ double sA[2][F][N][QQ];             // z-contracted, for k' and the next
  __shared__ __align__(16) double sB[RUNS][G2][NN][SB];
  const int64_t cell = blockIdx.x;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  for (int e = t; e < NP * NN * Q; e += NT) (&sP[0][0][0])[e] = P[e];
  for (int e = t; e < Q * QQ; e += NT) {
    sV[0][e] = vJxW[cell * (Q * QQ) + e];
    if constexpr (GGA) {
#pragma unroll
      for (int d = 0; d < 3; ++d) sV[GGA ? 1 + d : 0][e] = gJxW[(cell * (Q * QQ) + e) * 3 + d];
    }
  }
  __syncthreads();
  int have[2] = {-1, -1};
  const int kt1 = min((int)(blockIdx.y + 1) * tiles, ne_pad / 16);
  for (int kt = blockIdx.y * tiles; kt < kt1; ++kt) {
    const int c0 = kt * 16, r0 = c0 / N;
    const int cl = min(c0 + 15, NE3 - 1), nrun = cl / N - r0 + 1;
    for (int kp = r0 / N; kp <= cl / NN; ++kp) {
      if (have[kp & 1] == kp) continue;
      have[kp & 1] = kp;
      for (int e = t; e < N * QQ; e += NT) {
        const int k = e / QQ, yx = e % QQ;
        const double *p = sP[0][k * N + kp];
        double v = 0.0, x = 0.0, y = 0.0;
#pragma unroll
        for (int z = 0; z < Q; ++z) {
          v = fmadd(p[z], sV[0][z * QQ + yx], v);
          if constexpr (GGA) {
            v = fmadd(sP[GGA ? 3 : 0][k * N + kp][z], sV[GGA ? 3 : 0][z * QQ + yx], v);
            x = fmadd(p[z], sV[GGA ? 1 : 0][z * QQ + yx], x);
            y = fmadd(p[z], sV[GGA ? 2 : 0][z * QQ + yx], y);
          }
        }
        sA[kp & 1][0][k][yx] = v;
        if constexpr (GGA) {
          sA[kp & 1][GGA ? 1 : 0][k][yx] = x;
          sA[kp & 1][GGA ? 2 : 0][k][yx] = y;
        }
      }
    }
    __syncthreads();
    for (int e = t; e < nrun * NN * Q; e += NT) {
      const int x = e % Q, jk = e / Q % NN, rr = e / (Q * NN);
      const int jp = (r0 + rr) % N, kp = (r0 + rr) / N, j = jk % N, k = jk / N;
      const double *p = sP[0][j * N + jp], *a = sA[kp & 1][0][k];
      double v = 0.0, w = 0.0;
#pragma unroll
      for (int y = 0; y < Q; ++y) {
        v = fmadd(p[y], a[y * Q + x], v);
        if constexpr (GGA) {
          v = fmadd(sP[GGA ? 2 : 0][j * N + jp][y], sA[kp & 1][GGA ? 2 : 0][k][y * Q + x], v);
          w = fmadd(p[y], sA[kp & 1][GGA ? 1 : 0][k][y * Q + x], w);
        }
      }
      sB[rr][0][jk][x] = v;
      if constexpr (GGA) sB[rr][GGA ? 1 : 0][jk][x] = w;
    }
    __syncthreads();
    // rows of i = wave: lane = (row group, column pair)
    const int c = c0 + 2 * (lane & 7);
    const int ca = min(c, NE3 - 1), cb = min(c + 1, NE3 - 1);
    const int ra = ca / N - r0, rb = cb / N - r0;
    double pa[G2][Q], pb[G2][Q];
#pragma unroll
    for (int s = 0; s < G2; ++s)
#pragma unroll
      for (int x = 0; x < Q; ++x) {
        pa[s][x] = sP[s][wave * N + ca % N][x];
        pb[s][x] = sP[s][wave * N + cb % N][x];
      }
    const int64_t base = (cell * (ne_pad / 16) + kt) * (int64_t)ne_pad * 16 + 2 * (lane & 7);
    for (int jk = lane >> 3; jk < NN; jk += 8) {
      const int row = wave + N * jk;
      double va = 0.0, vb = 0.0;
#pragma unroll
      for (int s = 0; s < G2; ++s)
#pragma unroll
        for (int x = 0; x < Q; ++x) {
          va = fmadd(pa[s][x], sB[ra][s][jk][x], va);
          vb = fmadd(pb[s][x], sB[rb][s][jk][x], vb);
        }
      va = c < NE3 ? fmadd(0.5, K[row * NE3 + ca], va) : 0.0;
      vb = c + 1 < NE3 ? fmadd(0.5, K[row * NE3 + cb], vb) : 0.0;
      const int64_t o = base + (int64_t)row * 16;
      *reinterpret_cast<double2 *>(Ht64 + o) = make_double2(va, vb);
      *reinterpret_cast<float2 *>(Ht32 + o) = make_float2((float)va, (float)vb);
      *reinterpret_cast<uint32_t *>(Ht16 + o) = bf16_pair((float)va, (float)vb);
    }
    for (int e = t; e < (ne_pad - NE3) * 16; e += NT) {  // padded rows
      const int64_t o = (cell * (ne_pad / 16) + kt) * (int64_t)ne_pad * 16 + NE3 * 16 + e;
      Ht64[o] = 0.0;
      Ht32[o] = 0.f;
      Ht16[o] = 0;
    }
    __syncthreads();
  }
}

hipError_t launch_build_tensor(const double *K, const double *P, const double *vJxW,
                               const double *gJxW, int C, int n, int q, int ne_pad, double *Ht64,
                               float *Ht32, uint16_t *Ht16, hipStream_t s) {
  // at least about four workgroups per CU
  const int nt = ne_pad / 16, split = std::min(nt, std::max(1, 1024 / C));
  const int tiles = (nt + split - 1) / split;
  const dim3 grid(C, (nt + tiles - 1) / tiles);
#define CHFSI_BUILD(N, Q)                                                                       \
  if (n == N && q == Q) {                                                                       \
    if (gJxW)                                                                                   \
      hipLaunchKernelGGL((build_tensor_kernel<N, Q, true>), grid, dim3(64 * N), 0, s, K, P,     \
                         vJxW, gJxW, ne_pad, tiles, Ht64, Ht32, Ht16);                          \
    else                                                                                        \
      hipLaunchKernelGGL((build_tensor_kernel<N, Q, false>), grid, dim3(64 * N), 0, s, K, P,    \
                         vJxW, gJxW, ne_pad, tiles, Ht64, Ht32, Ht16);                          \
    return hipGetLastError();                                                                   \
  }
  CHFSI_BUILD(7, 8)
  CHFSI_BUILD(6, 6)
  CHFSI_BUILD(5, 5)
#undef CHFSI_BUILD
  return hipErrorInvalidValue;
}

}  // namespace chfsi
