// k_assemble.hip - device-side re-assembly of the Oseen velocity blocks (gfx950): the
// element matrices of NSType4Galerkin3D (src/FE/NSE3D_FixPo.C:1919-2071) with the
// convection field of the fixed-point linearisation, and the evaluation of a Q2 velocity
// field at the quadrature points (the 'param' values the reference's assembly framework
// hands to it, src/FE/Assemble3D.C).
//
// Q2 hexahedra (27 nodes, xi fastest, include/FE3D/NF_C_H_Q2_3D.h), trilinear cell map from
// the 8 corners (corner index a + 2b + 4c), 3x3x3 Gauss rule (point q: xi = g[q % 3],
// eta = g[q / 3 % 3], zeta = g[q / 9]).  Element entry (test i, ansatz j):
//   sum_q w_q |det J| ( nu grad phi_i . grad phi_j + (b_q . grad phi_j) phi_i + sigma phi_j phi_i )
// added to A11, A22 and A33 of the active rows; A12..A32 are zero for this Galerkin form.
// Cells of one color share no velocity dof, so one launch per color scatters without
// atomics.
#include "pmg_internal.hpp"

namespace pmg {

namespace {

__device__ const double kGP[3] = {-0.7745966692414833770358531, 0.0, 0.7745966692414833770358531};
__device__ const double kGW[3] = {5.0 / 9.0, 8.0 / 9.0, 5.0 / 9.0};

__device__ inline void lag1(double t, double v[3], double d[3]) {
  v[0] = 0.5 * t * (t - 1.0); v[1] = 1.0 - t * t; v[2] = 0.5 * t * (t + 1.0);
  d[0] = t - 0.5; d[1] = -2.0 * t; d[2] = t + 0.5;
}

// value and reference gradient of Q2 basis i at quadrature point q
__device__ inline void q2_at(int q, int i, double &v, double &dx, double &dy, double &dz) {
  double vx[3], ax[3], vy[3], ay[3], vz[3], az[3];
  lag1(kGP[q % 3], vx, ax);
  lag1(kGP[(q / 3) % 3], vy, ay);
  lag1(kGP[q / 9], vz, az);
  const int a = i % 3, b = (i / 3) % 3, c = i / 9;
  v = vx[a] * vy[b] * vz[c];
  dx = ax[a] * vy[b] * vz[c];
  dy = vx[a] * ay[b] * vz[c];
  dz = vx[a] * vy[b] * az[c];
}

// block 0 of the active rows (entries [0, a_rowptr[n_active])) to zero before the colors add to it
__global__ void k_zero_active(double *__restrict__ a, long n_act_entries) {
  for (long k = blockIdx.x * long(blockDim.x) + threadIdx.x; k < n_act_entries; k += long(gridDim.x) * blockDim.x)
    a[k] = 0.0;
}
// the other eight blocks after them: A22 = A33 = A11, the rest zero.  The colors add to one block
// only (three would be 107 MB read and written per color of 3072 cells), and this pass writes what
// the zeroing of nine blocks wrote before: 16 us as before at 24576 cells.
__global__ void k_spread_active(double *__restrict__ a, long nnz, long n_act_entries) {
  for (long k = blockIdx.x * long(blockDim.x) + threadIdx.x; k < n_act_entries; k += long(gridDim.x) * blockDim.x) {
    const double v = a[k];
#pragma unroll
    for (int b = 1; b < 9; ++b) a[b * nnz + k] = b % 4 == 0 ? v : 0.0;
  }
}

// Geometry and basis data of one cell in LDS: weights w_q |det J| (W), values Vq[q][i] and
// physical gradients G*[q][i] of the 27 Q2 basis functions at the 27 Gauss points, and the
// convection at the points (Bc) and times the gradients (Bg).  Called by all CELL_T threads;
// ends with a barrier.
constexpr int CELL_T = 128;
struct CellData {
  double X[8][3], Bc[27][3], Ji[27][9], W[27];
  double Vq[27][27], Gx[27][27], Gy[27][27], Gz[27][27], Bg[27][27];
};

__device__ void cell_setup(CellData &D, int cell, const double *__restrict__ geom, const double *__restrict__ bq) {
  const int t = threadIdx.x;
  if (t < 24) D.X[t / 3][t % 3] = geom[long(cell) * 24 + t];
  if (t < 81) D.Bc[t / 3][t % 3] = bq[long(cell) * 81 + t];
  __syncthreads();
  if (t < 27) {
    const double xi = kGP[t % 3], eta = kGP[(t / 3) % 3], zeta = kGP[t / 9];
    double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    for (int c = 0; c < 2; ++c)
      for (int b = 0; b < 2; ++b)
        for (int aa = 0; aa < 2; ++aa) {
          const double sx = aa ? 1 : -1, sy = b ? 1 : -1, sz = c ? 1 : -1;
          const double nx = 0.5 * (1 + sx * xi), ny = 0.5 * (1 + sy * eta), nz = 0.5 * (1 + sz * zeta);
          const double dNx = 0.5 * sx * ny * nz, dNy = 0.5 * sy * nx * nz, dNz = 0.5 * sz * nx * ny;
          const double *P = D.X[aa + 2 * b + 4 * c];
          for (int r = 0; r < 3; ++r) {
            J[r][0] += dNx * P[r];
            J[r][1] += dNy * P[r];
            J[r][2] += dNz * P[r];
          }
        }
    const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                       J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                       J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    const double id = 1.0 / det;
    double *I = D.Ji[t];
    I[0] = (J[1][1] * J[2][2] - J[1][2] * J[2][1]) * id;
    I[1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
    I[2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
    I[3] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * id;
    I[4] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    I[5] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    I[6] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * id;
    I[7] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    I[8] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    D.W[t] = kGW[t % 3] * kGW[(t / 3) % 3] * kGW[t / 9] * fabs(det);
  }
  __syncthreads();
  // physical gradients: J^{-T} times the reference gradient
  for (int idx = t; idx < 27 * 27; idx += CELL_T) {
    const int q = idx / 27, i = idx - 27 * q;
    double v, dx, dy, dz;
    q2_at(q, i, v, dx, dy, dz);
    const double *I = D.Ji[q];
    const double gx = I[0] * dx + I[3] * dy + I[6] * dz;
    const double gy = I[1] * dx + I[4] * dy + I[7] * dz;
    const double gz = I[2] * dx + I[5] * dy + I[8] * dz;
    D.Vq[q][i] = v;
    D.Gx[q][i] = gx;
    D.Gy[q][i] = gy;
    D.Gz[q][i] = gz;
    D.Bg[q][i] = D.Bc[q][0] * gx + D.Bc[q][1] * gy + D.Bc[q][2] * gz;
  }
  __syncthreads();
}

// Element entries (test i, ansatz j) of NSType4Galerkin3D with the mass term sigma: thread t < 81 takes
// the nine with i = t / 9 + 9 r, j = t % 9 + 9 c.
// Bounds: one entry per thread at a time read eleven values from LDS per point and entry and,
// unrolled over the points, took the whole register file, so one cell was in work per CU and
// waited at each of its steps; nine per thread read three, and five cells share a CU.  3072 cells:
// k_assemble_oseen 248 -> 76 us, k_theta_rhs 172 -> 65 us, the same values bit for bit.
constexpr int TILES = 81;
__device__ __forceinline__ void element_entries(const CellData &D, int t, double nu, double sigma, double (&s)[3][3]) {
  const int i0 = t / 9, j0 = t - 9 * i0;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) s[r][c] = 0.0;
#pragma unroll 1
  for (int q = 0; q < 27; ++q) {
    const double w = D.W[q];
    double xi[3], yi[3], zi[3], vi[3], xj[3], yj[3], zj[3], vj[3], bj[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      xi[r] = D.Gx[q][i0 + 9 * r];
      yi[r] = D.Gy[q][i0 + 9 * r];
      zi[r] = D.Gz[q][i0 + 9 * r];
      vi[r] = D.Vq[q][i0 + 9 * r];
      xj[r] = D.Gx[q][j0 + 9 * r];
      yj[r] = D.Gy[q][j0 + 9 * r];
      zj[r] = D.Gz[q][j0 + 9 * r];
      vj[r] = D.Vq[q][j0 + 9 * r];
      bj[r] = D.Bg[q][j0 + 9 * r];
    }
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double val = fma(nu, fma(zi[r], zj[c], fma(xi[r], xj[c], yi[r] * yj[c])), bj[c] * vi[r]);
        if (sigma != 0.0) val = fma(sigma * vj[c], vi[r], val);
        s[r][c] = fma(w, val, s[r][c]);
      }
  }
}

__global__ __launch_bounds__(CELL_T) void k_assemble_oseen(const int *__restrict__ cells, int ncells,
                                                           const double *__restrict__ geom,
                                                           const double *__restrict__ bq,
                                                           const int *__restrict__ u_global,
                                                           const int *__restrict__ pmap,
                                                           const int *__restrict__ a_rowptr, int n_active,
                                                           double *__restrict__ a, double nu, double sigma) {
  __shared__ CellData D;
  if (int(blockIdx.x) >= ncells) return;
  const int cell = cells[blockIdx.x], t = threadIdx.x;
  const int *ug = u_global + long(cell) * NU_LOC;
  const int *mp = pmap + long(cell) * PM_STRIDE;
  // entry (row, col j) in the CSR: the gather map holds its row-blocked offset 9 k0 + (k - k0) of
  // block 0; Dirichlet rows keep their identity
  long k[3][3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int i = min(t, TILES - 1) / 9 + 9 * r, row = ug[i];
    const long k0 = row < n_active ? 8L * a_rowptr[row] : 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int off = mp[PM_A + i * NU_LOC + min(t, TILES - 1) % 9 + 9 * c];
      k[r][c] = t < TILES && row < n_active && off >= 0 ? off - k0 : -1;
    }
  }
  cell_setup(D, cell, geom, bq);
  if (t >= TILES) return;
  double s[3][3], old[3][3];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) old[r][c] = k[r][c] >= 0 ? a[k[r][c]] : 0.0;
  element_entries(D, t, nu, sigma, s);
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (k[r][c] >= 0) a[k[r][c]] = old[r][c] + s[r][c];
}

// rhs_c(row i) -= sum_j E_ij(nu, sigma') u_c(j) for the active rows of one color's cells:
// with sigma' = -sigma, sigma M u - A u of the theta scheme's right-hand side
__global__ __launch_bounds__(CELL_T) void k_theta_rhs(const int *__restrict__ cells, int ncells,
                                                      const double *__restrict__ geom, const double *__restrict__ bq,
                                                      const int *__restrict__ u_global, int n_udof, int n_active,
                                                      const double *__restrict__ u, double *__restrict__ rhs,
                                                      double nu, double sigma_neg) {
  __shared__ CellData D;
  __shared__ double ul[81];
  if (int(blockIdx.x) >= ncells) return;
  const int cell = cells[blockIdx.x], t = threadIdx.x;
  const int *ug = u_global + long(cell) * NU_LOC;
  if (t < 81) ul[t] = u[long(t / 27) * n_udof + ug[t % 27]];
  cell_setup(D, cell, geom, bq);
  double s[3][3];
  if (t < TILES) element_entries(D, t, nu, sigma_neg, s);
  __syncthreads();
  double(*const E)[27] = D.Gx;   // no longer needed
  if (t < TILES)
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) E[t / 9 + 9 * r][t % 9 + 9 * c] = s[r][c];
  __syncthreads();
  if (t < 81) {
    const int i = t / 3, c = t - 3 * i;
    const int row = ug[i];
    if (row < n_active) {
      double v = 0.0;
      for (int j = 0; j < 27; ++j) v += E[i][j] * ul[27 * c + j];
      rhs[long(c) * n_udof + row] -= v;
    }
  }
}

// theta-scheme right-hand side outside the active velocity rows: Dirichlet values from g
// (velocity rows >= n_active), zero pressure rows; the active velocity rows start at 0
__global__ void k_theta_rhs_init(double *__restrict__ rhs, const double *__restrict__ g, int n_udof, int n_active,
                                 int n_pdof) {
  const long i = blockIdx.x * long(blockDim.x) + threadIdx.x;
  const long n = 3L * n_udof + n_pdof;
  if (i >= n) return;
  if (i < 3L * n_udof) {
    const int r = int(i % n_udof);
    rhs[i] = r < n_active ? 0.0 : g[i];
  } else {
    rhs[i] = 0.0;
  }
}

// b[cell][q][c] = sum_i u_c(UDOF_i) phi_i(q)
__global__ void k_eval_velocity(int ncells, const double *__restrict__ u, int N, const int *__restrict__ u_global,
                                double *__restrict__ bq) {
  const long idx = blockIdx.x * long(blockDim.x) + threadIdx.x;
  if (idx >= long(ncells) * 27) return;
  const int cell = int(idx / 27), q = int(idx - 27L * cell);
  const int *ug = u_global + long(cell) * NU_LOC;
  double s0 = 0, s1 = 0, s2 = 0;
  for (int i = 0; i < 27; ++i) {
    double v, dx, dy, dz;
    q2_at(q, i, v, dx, dy, dz);
    const int g = ug[i];
    s0 += v * u[g];
    s1 += v * u[N + g];
    s2 += v * u[2L * N + g];
  }
  bq[idx * 3 + 0] = s0;
  bq[idx * 3 + 1] = s1;
  bq[idx * 3 + 2] = s2;
}

}  // namespace

void launch_assemble_oseen(const DevLevel &L, const double *geom, const double *bq, double nu, double sigma,
                           hipStream_t s) {
  std::vector<int> rp(2);
  PMG_HIP_CHECK(hipMemcpyAsync(rp.data(), L.a_rowptr + L.n_active, sizeof(int), hipMemcpyDeviceToHost, s));
  PMG_HIP_CHECK(hipStreamSynchronize(s));
  const long n_act = rp[0];
  k_zero_active<<<2048, 256, 0, s>>>(L.a, n_act);
  PMG_HIP_CHECK(hipGetLastError());
  for (int col = 0; col + 1 < int(L.ptr_colors.size()); ++col) {
    const int p0 = L.ptr_colors[col], nc = L.ptr_colors[col + 1] - p0;
    if (nc <= 0) continue;
    k_assemble_oseen<<<nc, CELL_T, 0, s>>>(L.cell_reorder + p0, nc, geom, bq, L.u_global, L.pmap, L.a_rowptr,
                                           L.n_active, L.a, nu, sigma);
    PMG_HIP_CHECK(hipGetLastError());
  }
  k_spread_active<<<2048, 256, 0, s>>>(L.a, L.a_nnz, n_act);
  PMG_HIP_CHECK(hipGetLastError());
}

void launch_theta_rhs(const DevLevel &L, const double *geom, const double *bq, double nu, double sigma,
                      const double *u, const double *g, double *rhs, hipStream_t s) {
  const long n = 3L * L.n_udof + L.n_pdof;
  k_theta_rhs_init<<<int((n + 255) / 256), 256, 0, s>>>(rhs, g, L.n_udof, L.n_active, L.n_pdof);
  PMG_HIP_CHECK(hipGetLastError());
  for (int col = 0; col + 1 < int(L.ptr_colors.size()); ++col) {
    const int p0 = L.ptr_colors[col], nc = L.ptr_colors[col + 1] - p0;
    if (nc <= 0) continue;
    k_theta_rhs<<<nc, CELL_T, 0, s>>>(L.cell_reorder + p0, nc, geom, bq, L.u_global, L.n_udof, L.n_active, u, rhs, nu,
                                   -sigma);
    PMG_HIP_CHECK(hipGetLastError());
  }
}

void launch_eval_velocity(const DevLevel &L, const double *u, double *bq, hipStream_t s) {
  const long n = long(L.n_cells) * 27;
  k_eval_velocity<<<int((n + 255) / 256), 256, 0, s>>>(L.n_cells, u, L.n_udof, L.u_global, bq);
  PMG_HIP_CHECK(hipGetLastError());
}

}  // namespace pmg
