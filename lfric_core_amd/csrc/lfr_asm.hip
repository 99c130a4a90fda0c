// Local-matrix assembly by quadrature on the device, lowest-order W0.
//
// Mass matrix: compute_mass_matrix_w_scalar_code
// (components/science/source/kernel/fem/sci_compute_mass_matrix_kernel_w_scalar_mod.F90:150-174)
// with w_scalar = W0 and the coordinate field chi on W0, Cartesian (X, Y, Z)
// coordinates: the Jacobian of the reference-cube map
// (components/science/source/kernel/geometry/sci_coordinate_jacobian_mod.F90:330-345,
// jac(i, dir) = sum_df chi_i(df) dphi_df/dxi_dir, df in order) and its
// cofactor determinant (:430-440); mm(ik, df, df2) for df >= df2 is the sum,
// qp_v outer and qp_h inner, of ((((w_h w_v) phi_df) phi_df2) detJ), then
// mirrored.
//
// Stiffness (no reference kernel; used for the assembled diffusion operator):
// K(a, b) = sum_q w_h w_v (J^-T grad phi_a) . (J^-T grad phi_b) |detJ|, with
// J^-T from the cofactors.
//
// Quadrature: nq-point Gauss-Legendre on [0, 1] in each direction (the
// published rule: roots of P_nq by Newton's method from the Chebyshev
// guesses, weights 1/((1 - t^2) P'(t)^2)), horizontal points x outer, y inner
// (quadrature_xyoz_mod.F90:235-242).  W0 basis: trilinear, local dofs in the
// reference element's vertex order (bottom SW, SE, NE, NW, then top).
//
// One thread per (row a, cell-layer ik), ik fastest, so the 8 values a thread
// writes, M(ik, a, b) at ik + n3 (a + 8 b), are coalesced across a wavefront.
#include <cmath>
#include <cstring>
#include <vector>

#include "lfr_internal.h"

namespace {

constexpr int kMaxQ = 6;
constexpr int kMaxQp = kMaxQ * kMaxQ * kMaxQ;
constexpr int kCxThreads = 64;    // threads of the shared-Jacobian kernels

// per quadrature point (v outer, h = (x outer, y inner) inner): basis[8],
// gradient[3][8], w_h, w_v
struct QpTable {
  double b[8];
  double g[3][8];
  double wh, wv;
};

void gauss_legendre01(int n, double* x, double* w) {
  for (int i = 0; i < n; ++i) {
    double t = std::cos(M_PI * (i + 0.75) / (n + 0.5));
    double dp = 1.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = t;
      for (int k = 2; k <= n; ++k) {
        const double p2 = ((2.0 * k - 1.0) * t * p1 - (k - 1.0) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      const double pn = n == 0 ? 1.0 : p1;
      const double pm = n == 1 ? 1.0 : p0;
      dp = n * (t * pn - pm) / (t * t - 1.0);
      const double dt = pn / dp;
      t -= dt;
      if (std::fabs(dt) < 1e-16) break;
    }
    // ascending points on [0, 1]
    x[n - 1 - i] = 0.5 * (t + 1.0);
    w[n - 1 - i] = 0.5 * 2.0 / ((1.0 - t * t) * dp * dp);
  }
}

__global__ void __launch_bounds__(256)
k_w0_assemble(double* __restrict__ mass, double* __restrict__ stiff, const double* __restrict__ chi1,
              const double* __restrict__ chi2, const double* __restrict__ chi3, const int32_t* __restrict__ map0,
              const QpTable* __restrict__ tab, int nqp, int ncell, int nl) {
  const int64_t n3 = (int64_t)ncell * nl;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= 8 * n3) return;
  const int a = (int)(t / n3);
  const int64_t ik = t - (int64_t)a * n3;
  const int c = (int)(ik / nl);
  const int k = (int)(ik - (int64_t)c * nl);
  double x1[8], x2[8], x3[8];
#pragma unroll
  for (int df = 0; df < 8; ++df) {
    const int64_t d = (int64_t)map0[(int64_t)c * 8 + df] + k;
    x1[df] = chi1[d];
    x2[df] = chi2[d];
    x3[df] = chi3[d];
  }
  double m[8], s[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    m[b] = 0.0;
    s[b] = 0.0;
  }
  for (int q = 0; q < nqp; ++q) {
    const QpTable& T = tab[q];
    double j[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int dir = 0; dir < 3; ++dir) j[i][dir] = 0.0;
#pragma unroll
    for (int df = 0; df < 8; ++df)
#pragma unroll
      for (int dir = 0; dir < 3; ++dir) {
        const double gd = T.g[dir][df];
        j[0][dir] = j[0][dir] + x1[df] * gd;
        j[1][dir] = j[1][dir] + x2[df] * gd;
        j[2][dir] = j[2][dir] + x3[df] * gd;
      }
    const double c00 = j[1][1] * j[2][2] - j[1][2] * j[2][1];
    const double c01 = j[1][0] * j[2][2] - j[1][2] * j[2][0];
    const double c02 = j[1][0] * j[2][1] - j[1][1] * j[2][0];
    const double dj = j[0][0] * c00 - j[0][1] * c01 + j[0][2] * c02;
    const double wq = T.wh * T.wv;
    // mass: df = max(a, b), df2 = min(a, b) as the mirrored lower triangle
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int df = a > b ? a : b, df2 = a > b ? b : a;
      const double v = ((wq * T.b[df]) * T.b[df2]) * dj;
      m[b] = m[b] + v;
    }
    if (stiff) {
      // J^-T = cof(J) / det: physical gradient g = J^-T ghat
      double inv[3][3];   // inv[i][dir] = (J^-1)[dir][i]
      inv[0][0] = c00;
      inv[0][1] = -(j[0][1] * j[2][2] - j[0][2] * j[2][1]);
      inv[0][2] = j[0][1] * j[1][2] - j[0][2] * j[1][1];
      inv[1][0] = -c01;
      inv[1][1] = j[0][0] * j[2][2] - j[0][2] * j[2][0];
      inv[1][2] = -(j[0][0] * j[1][2] - j[0][2] * j[1][0]);
      inv[2][0] = c02;
      inv[2][1] = -(j[0][0] * j[2][1] - j[0][1] * j[2][0]);
      inv[2][2] = j[0][0] * j[1][1] - j[0][1] * j[1][0];
      const double rd = 1.0 / dj;
      double ga[3];
#pragma unroll
      for (int i = 0; i < 3; ++i)
        ga[i] = (inv[0][i] * T.g[0][a] + inv[1][i] * T.g[1][a] + inv[2][i] * T.g[2][a]) * rd;
      const double wa = wq * fabs(dj);
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        double dot = 0.0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const double gb = (inv[0][i] * T.g[0][b] + inv[1][i] * T.g[1][b] + inv[2][i] * T.g[2][b]) * rd;
          dot = dot + ga[i] * gb;
        }
        s[b] = s[b] + wa * dot;
      }
    }
  }
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    mass[ik + n3 * (a + 8 * b)] = m[b];
    if (stiff) stiff[ik + n3 * (a + 8 * b)] = s[b];
  }
}

}  // namespace

extern "C" int lfr_compute_mass_matrix_w0(lfr_ctx* ctx, int nq, const void* chi1_d, const void* chi2_d,
                                          const void* chi3_d, const lfr_space* space, void* mass_d,
                                          void* stiff_d) {
  if (!ctx) return LFR_ERR_ARG;
  LFR_REQUIRE(ctx, chi1_d && chi2_d && chi3_d && space && mass_d, "lfr_compute_mass_matrix_w0: null argument");
  LFR_REQUIRE(ctx, nq >= 1 && nq <= kMaxQ, "lfr_compute_mass_matrix_w0: nq must be 1..%d, got %d", kMaxQ, nq);
  LFR_REQUIRE(ctx, space->ndf == 8, "lfr_compute_mass_matrix_w0: lowest-order W0 only (ndf %d, expected 8)",
              space->ndf);
  // the four top dofs must follow their bottom dofs (vertex columns)
  for (int c = 0; c < space->ncell; ++c)
    for (int v = 0; v < 4; ++v)
      LFR_REQUIRE(ctx, space->map_h[(size_t)c * 8 + 4 + v] == space->map_h[(size_t)c * 8 + v] + 1,
                  "lfr_compute_mass_matrix_w0: cell %d is not a lowest-order W0 dofmap", c + 1);
  double x[kMaxQ], w[kMaxQ];
  gauss_legendre01(nq, x, w);
  static const int vtx[8][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {0, 1, 0},
                                {0, 0, 1}, {1, 0, 1}, {1, 1, 1}, {0, 1, 1}};
  std::vector<QpTable> tab;
  for (int qv = 0; qv < nq; ++qv)
    for (int qx = 0; qx < nq; ++qx)
      for (int qy = 0; qy < nq; ++qy) {
        QpTable T;
        const double p[3] = {x[qx], x[qy], x[qv]};
        for (int df = 0; df < 8; ++df) {
          double f[3], d[3];
          for (int e = 0; e < 3; ++e) {
            f[e] = vtx[df][e] ? p[e] : 1.0 - p[e];
            d[e] = vtx[df][e] ? 1.0 : -1.0;
          }
          T.b[df] = f[0] * f[1] * f[2];
          T.g[0][df] = d[0] * f[1] * f[2];
          T.g[1][df] = f[0] * d[1] * f[2];
          T.g[2][df] = f[0] * f[1] * d[2];
        }
        T.wh = w[qx] * w[qy];
        T.wv = w[qv];
        tab.push_back(T);
      }
  const size_t tb = tab.size() * sizeof(QpTable);
  int rc = lfr_work_reserve(ctx, tb);
  if (rc) return rc;
  LFR_HIP(ctx, hipMemcpyAsync(ctx->work, tab.data(), tb, hipMemcpyHostToDevice, ctx->stream));
  const int64_t n = 8 * (int64_t)space->ncell * space->nlayers;
  hipLaunchKernelGGL(k_w0_assemble, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, (double*)mass_d,
                     (double*)stiff_d, (const double*)chi1_d, (const double*)chi2_d, (const double*)chi3_d,
                     space->map0_d, (const QpTable*)ctx->work, (int)tab.size(), space->ncell, space->nlayers);
  LFR_CHECK_LAUNCH(ctx);
  // the table is host memory of this call: finish the copy before it goes
  LFR_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LFR_OK;
}

// ---------------------------------------------------------------------------
// Bilinear forms of the lowest-order de Rham complex from basis tables given
// by the caller (as the PSy layer hands them to the reference kernels):
//
//   out(ik, df, df2) = sum_{qp_v} sum_{qp_h} integrand(df, df2, qp)
//
// with, wt = w_h w_v, L the row table and R the column table,
//   scalar masses   ((wt L_df) R_df2) detJ
//   kMapCov         (wt (Jt L_df).(Jt R_df2)) detJ      W1 mass, grad
//   kMapContra      (wt (J L_df).(J R_df2)) / detJ      W2 mass, curl
//   div             (wt L_df) R_df2                     (no metric)
// Jt = transpose of the cofactor inverse
// (pointwise_coordinate_jacobian_inverse, sci_coordinate_jacobian_mod.F90:1140-1161),
// J and detJ from the chi gradients (:993-1103, Cartesian).  The statements
// of k_form follow compute_derham_matrices_code
// (components/science/source/kernel/fem/sci_compute_derham_matrices_kernel_mod.F90:241-352)
// and compute_mass_matrix_w2_code
// (sci_compute_mass_matrix_kernel_w2_mod.F90:131-162), those of the scalar
// masses compute_mass_matrix_w_scalar_code
// (sci_compute_mass_matrix_kernel_w_scalar_mod.F90:150-174).
// Symmetric forms (the masses) are computed for df >= df2 and mirrored
// (in k_form the dot product has the same bits either way: products commute
// exactly).
// ---------------------------------------------------------------------------
namespace {

enum { kMapCov = 1, kMapContra = 2 };

template <int NR, int NC>
struct FormQp {
  double l[3][NR];    // row basis (component, dof) at the point
  double r[3][NC];    // column basis
  double g[3][8];     // chi reference gradients
  double wh, wv;
};

// A vector form by itself, for tables without the structure that the
// shared-Jacobian kernels below need: a workgroup holds CPB = 256 / NR
// cell-layers, thread (li, a) = (cell-layer, row), li fastest, so output
// stores are coalesced.  Per quadrature point the row-0 thread of a
// cell-layer forms J, detJ and the map (J or Jt) into LDS; then every thread
// maps its share of the column vectors (columns a, a + NR, ...) into LDS and
// its own row vector into registers; then each thread sums its row.  LDS is
// double-buffered by point parity.
template <int NR, int NC, int MAP>
__global__ void __launch_bounds__(256)
k_form(double* __restrict__ out, const double* __restrict__ chi1, const double* __restrict__ chi2,
              const double* __restrict__ chi3, const int32_t* __restrict__ map0,
              const FormQp<NR, NC>* __restrict__ tab, int nqp, int ncell, int nl) {
  constexpr int CPB = 256 / NR;
  __shared__ double sm[2][CPB][10];             // map (9) and detJ
  __shared__ double srv[2][CPB][NC][3];         // mapped column vectors
  const int64_t n3 = (int64_t)ncell * nl;
  const int li = threadIdx.x % CPB;
  const int a = threadIdx.x / CPB;              // row; a == NR: idle thread
  const int64_t ik = (int64_t)blockIdx.x * CPB + li;
  const bool valid = a < NR && ik < n3;
  const int64_t ikc = ik < n3 ? ik : n3 - 1;    // idle lanes work on a real cell-layer
  double x1[8], x2[8], x3[8];
  if (a == 0) {
    const int c = (int)(ikc / nl);
    const int k = (int)(ikc - (int64_t)c * nl);
#pragma unroll
    for (int df = 0; df < 8; ++df) {
      const int64_t d = (int64_t)map0[(int64_t)c * 8 + df] + k;
      x1[df] = chi1[d];
      x2[df] = chi2[d];
      x3[df] = chi3[d];
    }
  }
  double acc[NC];
#pragma unroll
  for (int b = 0; b < NC; ++b) acc[b] = 0.0;
  const int ar = a < NR ? a : 0;
  for (int q = 0; q < nqp; ++q) {
    const FormQp<NR, NC>& T = tab[q];
    const int pb = q & 1;
    if (a == 0) {
      double j[3][3];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int dir = 0; dir < 3; ++dir) j[i][dir] = 0.0;
#pragma unroll
      for (int df = 0; df < 8; ++df)
#pragma unroll
        for (int dir = 0; dir < 3; ++dir) {
          const double gd = T.g[dir][df];
          j[0][dir] = j[0][dir] + x1[df] * gd;
          j[1][dir] = j[1][dir] + x2[df] * gd;
          j[2][dir] = j[2][dir] + x3[df] * gd;
        }
      const double dj = j[0][0] * (j[1][1] * j[2][2] - j[1][2] * j[2][1]) -
                        j[0][1] * (j[1][0] * j[2][2] - j[1][2] * j[2][0]) +
                        j[0][2] * (j[1][0] * j[2][1] - j[1][1] * j[2][0]);
      double m[3][3];
      if (MAP == kMapContra) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int d = 0; d < 3; ++d) m[i][d] = j[i][d];
      } else {
        const double idj = 1.0 / dj;
        double inv[3][3];
        inv[0][0] = (j[1][1] * j[2][2] - j[1][2] * j[2][1]) * idj;
        inv[0][1] = -(j[0][1] * j[2][2] - j[0][2] * j[2][1]) * idj;
        inv[0][2] = (j[0][1] * j[1][2] - j[0][2] * j[1][1]) * idj;
        inv[1][0] = -(j[1][0] * j[2][2] - j[1][2] * j[2][0]) * idj;
        inv[1][1] = (j[0][0] * j[2][2] - j[0][2] * j[2][0]) * idj;
        inv[1][2] = -(j[0][0] * j[1][2] - j[0][2] * j[1][0]) * idj;
        inv[2][0] = (j[1][0] * j[2][1] - j[1][1] * j[2][0]) * idj;
        inv[2][1] = -(j[0][0] * j[2][1] - j[0][1] * j[2][0]) * idj;
        inv[2][2] = (j[0][0] * j[1][1] - j[0][1] * j[1][0]) * idj;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int d = 0; d < 3; ++d) m[i][d] = inv[d][i];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int d = 0; d < 3; ++d) sm[pb][li][3 * i + d] = m[i][d];
      sm[pb][li][9] = dj;
    }
    __syncthreads();
    double m[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int d = 0; d < 3; ++d) m[i][d] = sm[pb][li][3 * i + d];
    const double dj = sm[pb][li][9];
    double lv[3];
    // this thread's share of the column vectors, and its row vector
    for (int b = ar; b < NC && a < NR; b += NR) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        double sacc = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) sacc = sacc + m[i][d] * T.r[d][b];
        srv[pb][li][b][i] = sacc;
      }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double sacc = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) sacc = sacc + m[i][d] * T.l[d][ar];
      lv[i] = sacc;
    }
    __syncthreads();
    const double wt = T.wh * T.wv;
#pragma unroll
    for (int b = 0; b < NC; ++b) {
      double dot = 0.0;
#pragma unroll
      for (int i = 0; i < 3; ++i) dot = dot + lv[i] * srv[pb][li][b][i];
      acc[b] = acc[b] + (MAP == kMapCov ? (wt * dot) * dj : (wt * dot) / dj);
    }
  }
  if (valid) {
#pragma unroll
    for (int b = 0; b < NC; ++b) out[ik + n3 * (a + (int64_t)NR * b)] = acc[b];
  }
}

// ---------------------------------------------------------------------------
// Shared-Jacobian kernels of the lowest-order complex on the reference cell.
//
// The lowest-order vector bases lie along one axis each (W1: its edge's
// direction, W2: its face's normal) and the complex is exact on the reference
// cell: grad of a W0 function is a signed sum of three W1 functions (one edge
// per axis at the vertex) and curl of a W1 function one of two W2 functions
// (the two faces at the edge).  With those table properties, which the host
// checks entry by entry at every point,
//
//   mm1(a, b)  = sum_q (wt l_a l_b) H(axis a, axis b),  H = C C^T / detJ
//   mm2(a, b)  = sum_q (wt l_a l_b) G(axis a, axis b),  G = J^T J / detJ
//   grad(a, b) = sum over the axes of +- mm1(a, edge at vertex b)
//   curl(a, e) = sum over its faces of +- mm2(a, face at edge e)
//
// (C the cofactors of J), so a point costs one multiply-add per distinct
// entry of the two masses and nothing for grad and curl, and div has the same
// value in every cell.  One thread owns one cell-layer: J is formed once per
// point for all the outputs of a kernel, the tables are uniform across the
// wavefront and few enough (36 doubles a point for W1) for one batch of
// scalar loads, the accumulators stay in registers, and a wavefront's store
// of one entry is 512 contiguous bytes, written past the caches.  All ten
// outputs in one kernel would need 139 accumulators (278 registers); two
// kernels (W1 mass and grad; the others) keep two waves on each SIMD and form
// J twice.  One-wave workgroups let a SIMD start the next wave's sums under
// another's stores.  All ten outputs at C48L70 (3.6 GB written, 27 points):
// 11.3 ms with one kernel a form and a thread a row (k_form), 1.09 ms with
// this split and a table entry per product (102 doubles a point, 256-thread
// workgroups), 1.03 ms with streaming stores and one-wave workgroups, 0.84-0.92 ms
// (4.3-3.9 TB/s) with the functions' own values as the table.
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int axis1(int e) { return e >= 4 && e < 8 ? 2 : (e & 1) ? 0 : 1; }
__host__ __device__ constexpr int axis2(int f) { return f >= 4 ? 2 : f & 1; }
// edge of axis d at vertex v and the sign of its W1 function in grad of v's
__host__ __device__ constexpr int grad_edge(int d, int v) {
  const int b = v & 3, top = v >> 2;
  return d == 2 ? 4 + b : d == 0 ? (b < 2 ? 1 : 3) + 8 * top : (b == 1 || b == 2 ? 2 : 0) + 8 * top;
}
__host__ __device__ constexpr int grad_sign(int d, int v) {
  const int b = v & 3;
  return (d == 2 ? v >= 4 : d == 0 ? (b == 1 || b == 2) : b >= 2) ? 1 : -1;
}
// face s (0, 1) of edge e and the sign of its W2 function in curl of e's
__host__ __device__ constexpr int curl_face(int s, int e) {
  return e < 4 ? (s ? 4 : e) : e >= 8 ? (s ? 5 : e - 8) : e == 4 ? s : e == 5 ? 2 - s : e == 6 ? 2 + s : 3 * s;
}
__host__ __device__ constexpr int curl_sign(int s, int e) {
  return e == 0 || e == 3 ? (s ? -1 : 1)
         : e == 1 || e == 2 || e == 6 ? 1
         : e == 4 || e == 8 || e == 11 ? -1
         : e == 7 ? (s ? -1 : 1)
                  : (s ? 1 : -1);
}
// lower-triangle index of a symmetric entry, and of a symmetric 3x3
__host__ __device__ constexpr int tri_ix(int a, int b) { return a >= b ? a * (a + 1) / 2 + b : b * (b + 1) / 2 + a; }

struct QpEdge {       // W1 mass and grad
  double g[3][8];     // chi reference gradients
  double l[12];       // W1 functions along their axes, and wt
  double wt;
};
struct QpFace {       // W0, W3 and Wtheta masses, W2 mass and curl
  double g[3][8];
  double t0[36], tt[3], t3;
  double l2[6], wt;   // W2 functions along their axes
};

struct ComplexOut {
  double *mm0, *mmt, *mm3, *mm2, *mm2b, *curl;   // k_complex_face
  double *mm1, *grad;                            // k_complex_edge
};

// J (the statements of k_form) and its determinant
__device__ __forceinline__ double cell_jacobian(const double (&g)[3][8], const double (&x1)[8], const double (&x2)[8],
                                                const double (&x3)[8], double (&j)[3][3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int dir = 0; dir < 3; ++dir) j[i][dir] = 0.0;
#pragma unroll
  for (int df = 0; df < 8; ++df)
#pragma unroll
    for (int dir = 0; dir < 3; ++dir) {
      const double gd = g[dir][df];
      j[0][dir] = j[0][dir] + x1[df] * gd;
      j[1][dir] = j[1][dir] + x2[df] * gd;
      j[2][dir] = j[2][dir] + x3[df] * gd;
    }
  return j[0][0] * (j[1][1] * j[2][2] - j[1][2] * j[2][1]) - j[0][1] * (j[1][0] * j[2][2] - j[1][2] * j[2][0]) +
         j[0][2] * (j[1][0] * j[2][1] - j[1][1] * j[2][0]);
}

__device__ __forceinline__ void cell_corners(const double* __restrict__ chi1, const double* __restrict__ chi2,
                                             const double* __restrict__ chi3, const int32_t* __restrict__ map0,
                                             int64_t ik, int nl, double (&x1)[8], double (&x2)[8], double (&x3)[8]) {
  const int c = (int)(ik / nl);
  const int k = (int)(ik - (int64_t)c * nl);
#pragma unroll
  for (int df = 0; df < 8; ++df) {
    const int64_t d = (int64_t)map0[(int64_t)c * 8 + df] + k;
    x1[df] = chi1[d];
    x2[df] = chi2[d];
    x3[df] = chi3[d];
  }
}

__global__ void __launch_bounds__(kCxThreads, 2)
k_complex_edge(ComplexOut o, const double* __restrict__ chi1, const double* __restrict__ chi2,
               const double* __restrict__ chi3, const int32_t* __restrict__ map0, const QpEdge* __restrict__ tab,
               int nqp, int ncell, int nl, unsigned nb_pad) {
  const int64_t n3 = (int64_t)ncell * nl;
  const int64_t ik = (int64_t)lfr_xcd_block(blockIdx.x, nb_pad) * kCxThreads + threadIdx.x;
  double x1[8], x2[8], x3[8];
  cell_corners(chi1, chi2, chi3, map0, ik < n3 ? ik : n3 - 1, nl, x1, x2, x3);
  double m1[78];
#pragma unroll
  for (int i = 0; i < 78; ++i) m1[i] = 0.0;
  for (int q = 0; q < nqp; ++q) {
    const QpEdge& T = tab[q];
    double j[3][3];
    const double dj = cell_jacobian(T.g, x1, x2, x3, j);
    const double idj = T.wt / dj;
    double c[3][3];   // cofactors: row i is the image of reference covector i, times detJ
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int d1 = (d + 1) % 3, d2 = (d + 2) % 3, i1 = (i + 1) % 3, i2 = (i + 2) % 3;
        c[i][d] = j[d1][i1] * j[d2][i2] - j[d1][i2] * j[d2][i1];
      }
    double h[6];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      // 1 / detJ on one side first: the square of the cofactors goes with the
      // fourth power of a length and leaves the range long before H does
      const double c0 = c[a][0] * idj, c1 = c[a][1] * idj, c2 = c[a][2] * idj;
#pragma unroll
      for (int b = 0; b <= a; ++b)
        h[tri_ix(a, b)] = __builtin_fma(c2, c[b][2], __builtin_fma(c1, c[b][1], c0 * c[b][0]));
    }
#pragma unroll
    for (int b = 0; b < 12; ++b) {
      double hl[3];   // the column function mapped onto the three axes
#pragma unroll
      for (int d = 0; d < 3; ++d) hl[d] = h[tri_ix(d, axis1(b))] * T.l[b];
#pragma unroll
      for (int a = b; a < 12; ++a) m1[tri_ix(a, b)] = __builtin_fma(T.l[a], hl[axis1(a)], m1[tri_ix(a, b)]);
    }
  }
  if (ik >= n3) return;
  if (o.mm1) {
#pragma unroll
    for (int b = 0; b < 12; ++b)
#pragma unroll
      for (int a = 0; a < 12; ++a) __builtin_nontemporal_store(m1[tri_ix(a, b)], o.mm1 + (ik + n3 * (a + 12 * b)));
  }
  if (o.grad) {
#pragma unroll
    for (int v = 0; v < 8; ++v)
#pragma unroll
      for (int a = 0; a < 12; ++a) {
        const double p = grad_sign(0, v) * m1[tri_ix(a, grad_edge(0, v))];
        const double r = p + grad_sign(1, v) * m1[tri_ix(a, grad_edge(1, v))];
        __builtin_nontemporal_store(r + grad_sign(2, v) * m1[tri_ix(a, grad_edge(2, v))], o.grad + (ik + n3 * (a + 12 * v)));
      }
  }
}

// S0: W0 mass, ST: Wtheta and W3 masses (the statements of k_form's scalar
// masses: same bits), S2: W2 mass and curl
template <bool S0, bool ST, bool S2>
__global__ void __launch_bounds__(kCxThreads, 2)
k_complex_face(ComplexOut o, const double* __restrict__ chi1, const double* __restrict__ chi2,
               const double* __restrict__ chi3, const int32_t* __restrict__ map0, const QpFace* __restrict__ tab,
               int nqp, int ncell, int nl, unsigned nb_pad) {
  const int64_t n3 = (int64_t)ncell * nl;
  const int64_t ik = (int64_t)lfr_xcd_block(blockIdx.x, nb_pad) * kCxThreads + threadIdx.x;
  double x1[8], x2[8], x3[8];
  cell_corners(chi1, chi2, chi3, map0, ik < n3 ? ik : n3 - 1, nl, x1, x2, x3);
  double m0[S0 ? 36 : 1], mt[ST ? 3 : 1], m3 = 0.0, m2[S2 ? 21 : 1];
  if constexpr (S0) {
#pragma unroll
    for (int i = 0; i < 36; ++i) m0[i] = 0.0;
  }
  if constexpr (ST) {
#pragma unroll
    for (int i = 0; i < 3; ++i) mt[i] = 0.0;
  }
  if constexpr (S2) {
#pragma unroll
    for (int i = 0; i < 21; ++i) m2[i] = 0.0;
  }
  for (int q = 0; q < nqp; ++q) {
    const QpFace& T = tab[q];
    double j[3][3];
    const double dj = cell_jacobian(T.g, x1, x2, x3, j);
    if constexpr (S0) {
#pragma unroll
      for (int i = 0; i < 36; ++i) m0[i] = m0[i] + T.t0[i] * dj;
    }
    if constexpr (ST) {
#pragma unroll
      for (int i = 0; i < 3; ++i) mt[i] = mt[i] + T.tt[i] * dj;
      m3 = m3 + T.t3 * dj;
    }
    if constexpr (S2) {
      const double idj = T.wt / dj;
      double g[6];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b <= a; ++b)
          g[tri_ix(a, b)] =
              __builtin_fma(j[2][a], j[2][b], __builtin_fma(j[1][a], j[1][b], j[0][a] * j[0][b])) * idj;
#pragma unroll
      for (int b = 0; b < 6; ++b) {
        double gl[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) gl[d] = g[tri_ix(d, axis2(b))] * T.l2[b];
#pragma unroll
        for (int a = b; a < 6; ++a) m2[tri_ix(a, b)] = __builtin_fma(T.l2[a], gl[axis2(a)], m2[tri_ix(a, b)]);
      }
    }
  }
  if (ik >= n3) return;
  if constexpr (S0) {
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
      for (int a = 0; a < 8; ++a) __builtin_nontemporal_store(m0[tri_ix(a, b)], o.mm0 + (ik + n3 * (a + 8 * b)));
  }
  if constexpr (ST) {
    if (o.mmt) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a) __builtin_nontemporal_store(mt[tri_ix(a, b)], o.mmt + (ik + n3 * (a + 2 * b)));
    }
    if (o.mm3) __builtin_nontemporal_store(m3, o.mm3 + (ik));
  }
  if constexpr (S2) {
#pragma unroll
    for (int b = 0; b < 6; ++b)
#pragma unroll
      for (int a = 0; a < 6; ++a) {
        if (o.mm2) __builtin_nontemporal_store(m2[tri_ix(a, b)], o.mm2 + (ik + n3 * (a + 6 * b)));
        if (o.mm2b) __builtin_nontemporal_store(m2[tri_ix(a, b)], o.mm2b + (ik + n3 * (a + 6 * b)));
      }
    if (o.curl) {
#pragma unroll
      for (int e = 0; e < 12; ++e)
#pragma unroll
        for (int a = 0; a < 6; ++a) {
          const double p = curl_sign(0, e) * m2[tri_ix(a, curl_face(0, e))];
          __builtin_nontemporal_store(p + curl_sign(1, e) * m2[tri_ix(a, curl_face(1, e))], o.curl + (ik + n3 * (a + 6 * e)));
        }
    }
  }
}

// The six planes of div (and of broken div), each one value in every cell
struct DivFill {
  double v[6];
  double w[6];
};
__global__ void __launch_bounds__(256)
k_fill_div(double* __restrict__ div, double* __restrict__ bdiv, DivFill f, int64_t n3) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n3; i += (int64_t)gridDim.x * 256) {
#pragma unroll
    for (int p = 0; p < 6; ++p) {
      if (div) __builtin_nontemporal_store(f.v[p], div + (i + n3 * p));
      if (bdiv) __builtin_nontemporal_store(f.w[p], bdiv + (i + n3 * p));
    }
  }
}

// Fortran-order host table (ncomp, ndf, nqp_h, nqp_v) element
inline double tab_at(const double* t, int ncomp, int ndf, int nqp_h, int c, int df, int qh, int qv) {
  return t[c + ncomp * (df + (size_t)ndf * (qh + (size_t)nqp_h * qv))];
}

// Every function of the vector table lies along its axis at every point
// (components off it are zero; a NaN is not).
bool on_axes(const double* t, int ndf, int (*axis)(int), int nqp) {
  for (int q = 0; q < nqp; ++q)
    for (int df = 0; df < ndf; ++df)
      for (int c = 0; c < 3; ++c)
        if (c != axis(df) && t[c + 3 * (df + (size_t)ndf * q)] != 0.0) return false;
  return true;
}

// diff_basis_w0 is the signed sum of W1 functions of grad_edge / grad_sign
bool grad_of_w1(const double* dw0, const double* w1, int nqp) {
  for (int q = 0; q < nqp; ++q)
    for (int v = 0; v < 8; ++v)
      for (int d = 0; d < 3; ++d)
        if (dw0[d + 3 * (v + (size_t)8 * q)] != grad_sign(d, v) * w1[d + 3 * (grad_edge(d, v) + (size_t)12 * q)])
          return false;
  return true;
}

// diff_basis_w1 is the signed sum of W2 functions of curl_face / curl_sign
// (an edge's two faces lie along different axes)
bool curl_of_w2(const double* dw1, const double* w2, int nqp) {
  for (int q = 0; q < nqp; ++q)
    for (int e = 0; e < 12; ++e)
      for (int d = 0; d < 3; ++d) {
        double want = 0.0;
        for (int s = 0; s < 2; ++s) {
          const int f = curl_face(s, e);
          if (axis2(f) == d) want = curl_sign(s, e) * w2[d + 3 * (f + (size_t)6 * q)];
        }
        if (dw1[d + 3 * (e + (size_t)12 * q)] != want) return false;
      }
  return true;
}

template <int NR, int NC, int MAP>
int form_assemble(lfr_ctx* ctx, int nqp_h, int nqp_v, const double* L, const double* R, const double* dchi,
                  const double* wh, const double* wv, const void* chi1, const void* chi2, const void* chi3,
                  const lfr_space* sp, void* out) {
  using Q = FormQp<NR, NC>;
  std::vector<Q> tab;
  for (int qv = 0; qv < nqp_v; ++qv)
    for (int qh = 0; qh < nqp_h; ++qh) {
      Q T;
      for (int c = 0; c < 3; ++c)
        for (int df = 0; df < NR; ++df) T.l[c][df] = tab_at(L, 3, NR, nqp_h, c, df, qh, qv);
      for (int c = 0; c < 3; ++c)
        for (int df = 0; df < NC; ++df) T.r[c][df] = tab_at(R, 3, NC, nqp_h, c, df, qh, qv);
      for (int dir = 0; dir < 3; ++dir)
        for (int df = 0; df < 8; ++df) T.g[dir][df] = tab_at(dchi, 3, 8, nqp_h, dir, df, qh, qv);
      T.wh = wh[qh];
      T.wv = wv[qv];
      tab.push_back(T);
    }
  const size_t tb = tab.size() * sizeof(Q);
  int rc = lfr_work_reserve(ctx, tb);
  if (rc) return rc;
  LFR_HIP(ctx, hipMemcpyAsync(ctx->work, tab.data(), tb, hipMemcpyHostToDevice, ctx->stream));
  const int64_t n3 = (int64_t)sp->ncell * sp->nlayers;
  constexpr int CPB = 256 / NR;
  hipLaunchKernelGGL((k_form<NR, NC, MAP>), dim3((unsigned)((n3 + CPB - 1) / CPB)), dim3(256),
                     0, ctx->stream, (double*)out, (const double*)chi1, (const double*)chi2, (const double*)chi3,
                     sp->map0_d, (const Q*)ctx->work, (int)tab.size(), sp->ncell, sp->nlayers);
  LFR_CHECK_LAUNCH(ctx);
  // the table lives in ctx->work and comes from this call's host memory:
  // finish before the next form reuses either
  LFR_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LFR_OK;
}

int check_chi(lfr_ctx* ctx, const lfr_space* sp, const char* who) {
  LFR_REQUIRE(ctx, sp->ndf == 8, "%s: the chi space must be lowest-order W0 (ndf %d)", who, sp->ndf);
  for (int c = 0; c < sp->ncell; ++c)
    for (int v = 0; v < 4; ++v)
      LFR_REQUIRE(ctx, sp->map_h[(size_t)c * 8 + 4 + v] == sp->map_h[(size_t)c * 8 + v] + 1,
                  "%s: cell %d is not a lowest-order W0 dofmap", who, c + 1);
  return LFR_OK;
}

// What a call wants from the shared-Jacobian kernels: outputs and the tables
// they come from (null: not wanted).
struct ComplexCall {
  int nqp_h, nqp_v;
  const double *wh, *wv, *dchi;
  const double *w0, *wt, *w3, *w2, *w1;
  ComplexOut out;
};

template <typename Q, typename Fill>
int upload_points(lfr_ctx* ctx, const ComplexCall& k, std::vector<Q>& tab, size_t at, const Fill& fill) {
  for (int qv = 0; qv < k.nqp_v; ++qv)
    for (int qh = 0; qh < k.nqp_h; ++qh) {
      Q T = {};
      for (int dir = 0; dir < 3; ++dir)
        for (int df = 0; df < 8; ++df) T.g[dir][df] = tab_at(k.dchi, 3, 8, k.nqp_h, dir, df, qh, qv);
      fill(T, k.wh[qh] * k.wv[qv], qh, qv);
      tab.push_back(T);
    }
  LFR_HIP(ctx, hipMemcpyAsync((char*)ctx->work + at, tab.data(), tab.size() * sizeof(Q), hipMemcpyHostToDevice,
                              ctx->stream));
  return LFR_OK;
}

int complex_assemble(lfr_ctx* ctx, const ComplexCall& k, const void* chi1, const void* chi2, const void* chi3,
                     const lfr_space* sp) {
  const bool edge = k.out.mm1 || k.out.grad;
  const bool s0 = k.out.mm0, st = k.out.mmt || k.out.mm3, s2 = k.out.mm2 || k.out.mm2b || k.out.curl;
  if (!edge && !s0 && !st && !s2) return LFR_OK;
  const int nqp = k.nqp_h * k.nqp_v, h = k.nqp_h;
  const size_t at = (nqp * sizeof(QpEdge) + 255) & ~(size_t)255;
  int rc = lfr_work_reserve(ctx, at + nqp * sizeof(QpFace));
  if (rc) return rc;
  const double *c1 = (const double*)chi1, *c2 = (const double*)chi2, *c3 = (const double*)chi3;
  const int64_t n3 = (int64_t)sp->ncell * sp->nlayers;
  const unsigned nb = (unsigned)((((n3 + kCxThreads - 1) / kCxThreads) + 7) & ~(int64_t)7);
  std::vector<QpEdge> te;
  std::vector<QpFace> tf;
  if (edge) {
    rc = upload_points(ctx, k, te, 0, [&](QpEdge& T, double wt, int qh, int qv) {
      for (int a = 0; a < 12; ++a) T.l[a] = tab_at(k.w1, 3, 12, h, axis1(a), a, qh, qv);
      T.wt = wt;
    });
    if (rc) return rc;
    hipLaunchKernelGGL(k_complex_edge, dim3(nb), dim3(kCxThreads), 0, ctx->stream, k.out, c1, c2, c3, sp->map0_d,
                       (const QpEdge*)ctx->work, nqp, sp->ncell, sp->nlayers, nb);
    LFR_CHECK_LAUNCH(ctx);
  }
  if (s0 || st || s2) {
    rc = upload_points(ctx, k, tf, at, [&](QpFace& T, double wt, int qh, int qv) {
      if (s0)
        for (int a = 0; a < 8; ++a)
          for (int b = 0; b <= a; ++b)
            T.t0[tri_ix(a, b)] = (wt * tab_at(k.w0, 1, 8, h, 0, a, qh, qv)) * tab_at(k.w0, 1, 8, h, 0, b, qh, qv);
      if (k.out.mmt)
        for (int a = 0; a < 2; ++a)
          for (int b = 0; b <= a; ++b)
            T.tt[tri_ix(a, b)] = (wt * tab_at(k.wt, 1, 2, h, 0, a, qh, qv)) * tab_at(k.wt, 1, 2, h, 0, b, qh, qv);
      if (k.out.mm3) T.t3 = (wt * tab_at(k.w3, 1, 1, h, 0, 0, qh, qv)) * tab_at(k.w3, 1, 1, h, 0, 0, qh, qv);
      if (s2)
        for (int a = 0; a < 6; ++a) T.l2[a] = tab_at(k.w2, 3, 6, h, axis2(a), a, qh, qv);
      T.wt = wt;
    });
    if (rc) return rc;
#define LFR_FACE(A, B, C)                                                                                     \
  hipLaunchKernelGGL((k_complex_face<A, B, C>), dim3(nb), dim3(kCxThreads), 0, ctx->stream, k.out, c1, c2, c3,  \
                     sp->map0_d, (const QpFace*)((char*)ctx->work + at), nqp, sp->ncell, sp->nlayers, nb)
    switch ((s0 ? 4 : 0) | (st ? 2 : 0) | (s2 ? 1 : 0)) {
      case 1: LFR_FACE(false, false, true); break;
      case 2: LFR_FACE(false, true, false); break;
      case 3: LFR_FACE(false, true, true); break;
      case 4: LFR_FACE(true, false, false); break;
      case 5: LFR_FACE(true, false, true); break;
      case 6: LFR_FACE(true, true, false); break;
      default: LFR_FACE(true, true, true); break;
    }
#undef LFR_FACE
    LFR_CHECK_LAUNCH(ctx);
  }
  // the tables come from this call's host memory: finish before they go
  LFR_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LFR_OK;
}

// The divergence forms: sum over the points of (wt l) r, the same in every
// cell, formed here in the order of the reference loop.
void div_values(const double* w3, const double* dw2, const double* wh, const double* wv, int nqp_h, int nqp_v,
                double (&v)[6]) {
  for (int b = 0; b < 6; ++b) {
    double acc = 0.0;
    for (int qv = 0; qv < nqp_v; ++qv)
      for (int qh = 0; qh < nqp_h; ++qh) {
        const double wt = wh[qh] * wv[qv];
        const double p = (wt * tab_at(w3, 1, 1, nqp_h, 0, 0, qh, qv)) * tab_at(dw2, 1, 6, nqp_h, 0, b, qh, qv);
        acc = acc + p;
      }
    v[b] = acc;
  }
}

}  // namespace

extern "C" int lfr_compute_mass_matrix(lfr_ctx* ctx, int kind, int ndf, int nqp_h, int nqp_v, const double* basis,
                                       const double* diff_basis_chi, const double* wqp_h, const double* wqp_v,
                                       const void* chi1_d, const void* chi2_d, const void* chi3_d,
                                       const lfr_space* chi_space, void* mass_d) {
  if (!ctx) return LFR_ERR_ARG;
  LFR_REQUIRE(ctx, basis && diff_basis_chi && wqp_h && wqp_v && chi1_d && chi2_d && chi3_d && chi_space && mass_d,
              "lfr_compute_mass_matrix: null argument");
  LFR_REQUIRE(ctx, kind == 0 || kind == 1, "lfr_compute_mass_matrix: kind must be 0 (scalar) or 1 (W2), got %d",
              kind);
  LFR_REQUIRE(ctx, nqp_h >= 1 && nqp_v >= 1 && nqp_h * nqp_v <= 4096, "lfr_compute_mass_matrix: bad point counts");
  int rc = check_chi(ctx, chi_space, "lfr_compute_mass_matrix");
  if (rc) return rc;
  const double *B = basis, *G = diff_basis_chi;
  // scalar masses, and the W2 mass when its functions lie along the axes,
  // take the shared-Jacobian kernel
  ComplexCall k = {};
  k.nqp_h = nqp_h;
  k.nqp_v = nqp_v;
  k.wh = wqp_h;
  k.wv = wqp_v;
  k.dchi = G;
  double* out = (double*)mass_d;
  if (kind == 0 && ndf == 8) k.w0 = B, k.out.mm0 = out;
  if (kind == 0 && ndf == 2) k.wt = B, k.out.mmt = out;
  if (kind == 0 && ndf == 1) k.w3 = B, k.out.mm3 = out;
  if (kind == 1 && ndf == 6 && on_axes(B, 6, axis2, nqp_h * nqp_v)) k.w2 = B, k.out.mm2 = out;
  if (k.w0 || k.wt || k.w3 || k.w2) return complex_assemble(ctx, k, chi1_d, chi2_d, chi3_d, chi_space);
#define LFR_MASS(N)                                                                                           \
  return form_assemble<N, N, kMapContra>(ctx, nqp_h, nqp_v, B, B, G, wqp_h, wqp_v, chi1_d, chi2_d, chi3_d,      \
                                         chi_space, mass_d)
  if (kind == 1) {
    switch (ndf) {
      case 2: LFR_MASS(2);
      case 4: LFR_MASS(4);
      case 6: LFR_MASS(6);
      default: break;
    }
  }
#undef LFR_MASS
  return lfr_set_error(ctx, LFR_ERR_ARG, "lfr_compute_mass_matrix: no kernel for kind %d with %d dofs per cell",
                       kind, ndf);
}

extern "C" int lfr_compute_derham_matrices(lfr_ctx* ctx, const lfr_derham_tables* t, const void* chi1_d,
                                           const void* chi2_d, const void* chi3_d, const lfr_space* chi_space,
                                           void* mm0, void* mm1, void* mm2, void* mm2b, void* mm3, void* mmt,
                                           void* grad, void* curl, void* div, void* broken_div) {
  if (!ctx) return LFR_ERR_ARG;
  LFR_REQUIRE(ctx, t && chi1_d && chi2_d && chi3_d && chi_space, "lfr_compute_derham_matrices: null argument");
  LFR_REQUIRE(ctx, t->nqp_h >= 1 && t->nqp_v >= 1 && t->nqp_h * t->nqp_v <= 4096 && t->wqp_h && t->wqp_v &&
                       t->diff_basis_chi,
              "lfr_compute_derham_matrices: bad quadrature");
  int rc = check_chi(ctx, chi_space, "lfr_compute_derham_matrices");
  if (rc) return rc;
  const int h = t->nqp_h, v = t->nqp_v;
  const double *G = t->diff_basis_chi, *wh = t->wqp_h, *wv = t->wqp_v;
  struct Need {
    void* out;
    const double* a;
    const double* b;
    const char* what;
  };
  const Need need[10] = {{mm0, t->basis_w0, t->basis_w0, "basis_w0"},
                         {mm1, t->basis_w1, t->basis_w1, "basis_w1"},
                         {mm2, t->basis_w2, t->basis_w2, "basis_w2"},
                         {mm2b, t->basis_w2b, t->basis_w2b, "basis_w2b"},
                         {mm3, t->basis_w3, t->basis_w3, "basis_w3"},
                         {mmt, t->basis_wt, t->basis_wt, "basis_wt"},
                         {grad, t->basis_w1, t->diff_basis_w0, "basis_w1 and diff_basis_w0"},
                         {curl, t->basis_w2, t->diff_basis_w1, "basis_w2 and diff_basis_w1"},
                         {div, t->basis_w3, t->diff_basis_w2, "basis_w3 and diff_basis_w2"},
                         {broken_div, t->basis_w3, t->diff_basis_w2b, "basis_w3 and diff_basis_w2b"}};
  for (const Need& n : need)
    LFR_REQUIRE(ctx, !n.out || (n.a && n.b), "lfr_compute_derham_matrices: an output needs %s", n.what);
  // Outputs whose tables have the lowest-order structure share one Jacobian
  // a point (complex_assemble); a vector form of other tables is formed by
  // itself (k_form).
  const int nqp = h * v;
  ComplexCall k = {};
  k.nqp_h = h;
  k.nqp_v = v;
  k.wh = wh;
  k.wv = wv;
  k.dchi = G;
  k.w0 = t->basis_w0;
  k.wt = t->basis_wt;
  k.w3 = t->basis_w3;
  k.w1 = t->basis_w1;
  k.w2 = t->basis_w2;
  k.out.mm0 = (double*)mm0;
  k.out.mmt = (double*)mmt;
  k.out.mm3 = (double*)mm3;
  if ((mm1 || grad) && on_axes(t->basis_w1, 12, axis1, nqp)) {
    k.out.mm1 = (double*)mm1;
    if (grad && grad_of_w1(t->diff_basis_w0, t->basis_w1, nqp)) k.out.grad = (double*)grad;
  }
  if ((mm2 || curl) && on_axes(t->basis_w2, 6, axis2, nqp)) {
    k.out.mm2 = (double*)mm2;
    if (curl && curl_of_w2(t->diff_basis_w1, t->basis_w2, nqp)) k.out.curl = (double*)curl;
  }
  ComplexCall kb = {};   // the broken W2 mass, when its table is another one
  if (mm2b && on_axes(t->basis_w2b, 6, axis2, nqp)) {
    const bool same = (k.out.mm2 || k.out.curl) &&
                      std::memcmp(t->basis_w2b, t->basis_w2, sizeof(double) * 18 * nqp) == 0;
    if (same) {
      k.out.mm2b = (double*)mm2b;
    } else {
      kb = k;
      kb.out = {};
      kb.w2 = t->basis_w2b;
      kb.out.mm2 = (double*)mm2b;
    }
  }
  if (div || broken_div) {
    DivFill f = {};
    if (div) div_values(t->basis_w3, t->diff_basis_w2, wh, wv, h, v, f.v);
    if (broken_div) div_values(t->basis_w3, t->diff_basis_w2b, wh, wv, h, v, f.w);
    const int64_t n3 = (int64_t)chi_space->ncell * chi_space->nlayers;
    hipLaunchKernelGGL(k_fill_div, dim3(lfr_blocks(n3, 256, 8192)), dim3(256), 0, ctx->stream, (double*)div,
                       (double*)broken_div, f, n3);
    LFR_CHECK_LAUNCH(ctx);
  }
  rc = complex_assemble(ctx, k, chi1_d, chi2_d, chi3_d, chi_space);
  if (rc) return rc;
  rc = complex_assemble(ctx, kb, chi1_d, chi2_d, chi3_d, chi_space);
  if (rc) return rc;
#define LFR_FORM(OUT, DONE, NR, NC, MAP, L, R)                                                                  \
  if (OUT && !DONE) {                                                                                         \
    rc = form_assemble<NR, NC, MAP>(ctx, h, v, L, R, G, wh, wv, chi1_d, chi2_d, chi3_d, chi_space, OUT); \
    if (rc) return rc;                                                                                        \
  }
  LFR_FORM(mm1, k.out.mm1, 12, 12, kMapCov, t->basis_w1, t->basis_w1)
  LFR_FORM(mm2, k.out.mm2, 6, 6, kMapContra, t->basis_w2, t->basis_w2)
  LFR_FORM(mm2b, (k.out.mm2b || kb.out.mm2), 6, 6, kMapContra, t->basis_w2b, t->basis_w2b)
  LFR_FORM(grad, k.out.grad, 12, 8, kMapCov, t->basis_w1, t->diff_basis_w0)
  LFR_FORM(curl, k.out.curl, 6, 12, kMapContra, t->basis_w2, t->diff_basis_w1)
#undef LFR_FORM
  return LFR_OK;
}
