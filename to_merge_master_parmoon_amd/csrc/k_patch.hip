// k_patch.hip - one color of the FP32 cell-Vanka sweep in one launch (gfx950).
//
// Residual, local solve and update of a patch by one workgroup.  The two-launch form
// (k_vanka_res, k_vanka_apply*) needs the second launch because patches of one color read
// dofs that other patches of the color update; here the updated velocity goes to another copy
// of the vector than the old one (patch_tables.hpp), so every read of the launch sees the
// state from before the color whatever order the workgroups run in.
//
// Bounds.  Small colors (8^3 to 16^3 cells): two dependent memory round trips (record, then
// rows and halo) and the launch; large ones: the stream of rows and stored data, about 21 KB
// of the operator per patch.  The residual of a patch reads 343 velocities 2197 times: they go
// to LDS once (16 bytes each) instead of through 16-byte gathers from L1, and the column
// indices (8.8 KB per patch) become 16-bit positions in the halo that the cells of the same
// structure share (575 structures among 32^3 = 32768 cells; 4 MB, in L2).  Four wavefronts of
// fixed roles (a role's rows have a fixed number of steps) keep every load of a patch in flight
// at once; with the row loops tested per row instead, the loads waited for each other and a
// color took 28.9 us at 32^3, 20.1 at 24^3 and 6.0 at 8^3.  Times per color (kernel trace, BF16
// stored data), the two launches before and this one: 32^3 30.5 + 8.8 -> 20.4 us, 24^3 (full
// inverses) 14.4 + 8.7 -> 13.0 us, 16^3 6.4 + 4.9 -> 6.2 us, 8^3 4.7 + 4.4 -> 4.4 us; the same
// sums in the same order, so the same results bit for bit.
//
// With nine velocity blocks a patch streams 79 KB of rows and 29 KB of inverse (FP32): 512
// patches of a 16^3 color take 12 us at the rate of a large copy.  A thread holds up to 99 row
// values and 88 of the inverse; limited to 256 registers (24 bytes of scratch) two workgroups
// share a CU.  Two launches before -> this one, FP32: 16^3 12.7 + 5.5 -> 12.3 us, 8^3
// 5.6 + 4.7 -> 6.3 us, the same results bit for bit.
#include "lu_sweeps.hpp"
#include "pmg_internal.hpp"
#include "pmg_rows.hpp"

namespace pmg {

namespace {

typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// What a thread holds of its group's row: the entries lane + 16 step, loaded before the
// workgroup waits for the halo.  NA, NB: steps of the A (B) and the BT row.  No load or LDS read
// stands behind a branch of its own, so that all of a thread's are in flight together.
template <int NA, int NB>
struct RowRegs {
  int n, m, row;
  float a[NA], b[3][NB], f;
  uint32_t ia[(NA + 1) / 2], ib;
};
__device__ __forceinline__ int clamp_entry(int j, int n) { return max(min(j, n - 1), 0); }

// velocity row of quad QD; d: its descriptor
template <class SH, int QD>
struct VelRow {
  static constexpr int NA = SH::a(QD), NB = SH::bt(QD), OA = 64 * SH::off_a(QD), OB = 64 * SH::off_bt(QD);
  RowRegs<NA, NB> R;
  __device__ __forceinline__ void load(const PatchStep &P, const int4 d, const uint32_t *__restrict__ pat, int l64) {
    const int lane = l64 & 15;
    R.n = d.z & 255;
    R.m = (d.z >> 8) & 255;
    R.row = (d.z >> 16) & 255;
#pragma unroll
    for (int p = 0; p < (NA + 1) / 2; ++p) R.ia[p] = pat[OA + 64 * p + l64];
    R.ib = pat[OB + l64];
    const float *v = P.a1 + d.x;
#pragma unroll
    for (int u = 0; u < NA; ++u) R.a[u] = v[clamp_entry(lane + 16 * u, R.n)];
    const float *w = P.btv + 3L * d.y;
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) R.b[c][u] = w[c * R.m + clamp_entry(lane + 16 * u, R.m)];
    R.f = P.f[long(lane < 3 ? lane : 0) * P.N + d.w];
  }
  // the residual into rs, in the natural local order; a lane's entries are added in the order
  // of row_a1_aos and row_bt_s
  __device__ __forceinline__ void residual(const float4 *hv, const float *hp, float *rs, int l64) const {
    const int lane = l64 & 15;
    float4 y[NA];
    float q[NB];
#pragma unroll
    for (int u = 0; u < NA; ++u) y[u] = hv[(R.ia[u / 2] >> (16 * (u % 2))) & 0xffffu];
#pragma unroll
    for (int u = 0; u < NB; ++u) q[u] = hp[(R.ib >> (16 * u)) & 0xffffu];
    float s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const float w = lane + 16 * u < R.n ? R.a[u] : 0.0f;
      s1 += w * y[u].x;
      s2 += w * y[u].y;
      s3 += w * y[u].z;
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const float z = lane + 16 * u < R.m ? q[u] : 0.0f;
      s1 += R.b[0][u] * z;
      s2 += R.b[1][u] * z;
      s3 += R.b[2][u] * z;
    }
    s1 = red16(s1);
    s2 = red16(s2);
    s3 = red16(s3);
    if (lane < 3 && R.row != PT_NOROW) rs[lane * NU_LOC + R.row] = R.f - (lane == 0 ? s1 : lane == 1 ? s2 : s3);
  }
};
// pressure row (quad 1): three values per entry, in the order of row_b_aos
template <class SH>
struct VelRow<SH, 1> {
  static constexpr int OA = 64 * SH::off_a(1);
  RowRegs<1, 2> R;
  __device__ __forceinline__ void load(const PatchStep &P, const int4 d, const uint32_t *__restrict__ pat, int l64) {
    const int lane = l64 & 15;
    R.n = d.z & 255;
    R.row = (d.z >> 16) & 255;
    R.ib = pat[OA + l64];
    const float *v = P.bv + 3L * d.x;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) R.b[c][u] = v[c * R.n + clamp_entry(lane + 16 * u, R.n)];
    R.f = P.f[3L * P.N + d.w];
  }
  __device__ __forceinline__ float sum(const float4 *hv, int l64) const {
    const int lane = l64 & 15;
    const float4 y[2] = {hv[R.ib & 0xffffu], hv[R.ib >> 16]};
    float s = 0.0f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bool ok = lane + 16 * u < R.n;
      const float z1 = ok ? y[u].x : 0.0f, z2 = ok ? y[u].y : 0.0f, z3 = ok ? y[u].z : 0.0f;
      s += fmaf(R.b[2][u], z3, fmaf(R.b[0][u], z1, R.b[1][u] * z2));   // as row_b_aos is compiled
    }
    return red16(s);
  }
  __device__ __forceinline__ void residual(const float4 *hv, const float *, float *rs, int l64) const {
    const float s = sum(hv, l64);
    if ((l64 & 15) == 0 && R.row != PT_NOROW) rs[2 * NU_LOC + R.row] = R.f - s;
  }
};

// velocity row of quad QD with nine velocity blocks, value b of entry j at 9 k0 + b n + j; the
// local residual in the row order of the stored inverse (invperm)
template <class SH, int QD>
struct VelRow9 {
  static constexpr int NA = SH::a(QD), NB = SH::bt(QD), OA = 64 * SH::off_a(QD), OB = 64 * SH::off_bt(QD);
  int n, m, row, perm;
  bool diag;   // Dirichlet row: the blocks A12 .. A32 are dropped
  float a[9][NA], b[3][NB], f;
  uint32_t ia[(NA + 1) / 2], ib;
  __device__ __forceinline__ void load(const PatchStep &P, const int4 d, const uint32_t *__restrict__ pat,
                                       const uint8_t *__restrict__ ip, int l64) {
    const int lane = l64 & 15;
    n = d.z & 255;
    m = (d.z >> 8) & 255;
    row = (d.z >> 16) & 255;
    diag = d.w >= P.n_active;
#pragma unroll
    for (int p = 0; p < (NA + 1) / 2; ++p) ia[p] = pat[OA + 64 * p + l64];
    ib = pat[OB + l64];
    const float *v = P.av + 9L * d.x;
#pragma unroll
    for (int u = 0; u < NA; ++u)
#pragma unroll
      for (int c = 0; c < 9; ++c) a[c][u] = v[c * n + clamp_entry(lane + 16 * u, n)];
    const float *w = P.btv + 3L * d.y;
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) b[c][u] = w[c * m + clamp_entry(lane + 16 * u, m)];
    f = P.f[long(lane < 3 ? lane : 0) * P.N + d.w];
    perm = ip[min(row + NU_LOC * (lane < 3 ? lane : 0), NLOC - 1)];
  }
  // sums in the order of row_a9_s (row_a_diag on Dirichlet rows) and row_bt_s
  __device__ __forceinline__ void residual(const float4 *hv, const float *hp, float *rs, int l64) const {
    const int lane = l64 & 15;
    float4 y[NA];
    float q[NB];
#pragma unroll
    for (int u = 0; u < NA; ++u) y[u] = hv[(ia[u / 2] >> (16 * (u % 2))) & 0xffffu];
#pragma unroll
    for (int u = 0; u < NB; ++u) q[u] = hp[(ib >> (16 * u)) & 0xffffu];
    float s[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const bool ok = lane + 16 * u < n;
      const float z[3] = {ok ? y[u].x : 0.0f, ok ? y[u].y : 0.0f, ok ? y[u].z : 0.0f};
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const float all = s[r] + fmaf(a[3 * r + 2][u], z[2], fmaf(a[3 * r][u], z[0], a[3 * r + 1][u] * z[1]));
        const float own = fmaf(a[4 * r][u], z[r], s[r]);
        s[r] = diag ? own : all;
      }
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const float z = lane + 16 * u < m ? q[u] : 0.0f;
#pragma unroll
      for (int r = 0; r < 3; ++r) s[r] += b[r][u] * z;
    }
#pragma unroll
    for (int r = 0; r < 3; ++r) s[r] = red16(s[r]);
    if (lane < 3 && row != PT_NOROW) rs[perm] = f - (lane == 0 ? s[0] : lane == 1 ? s[1] : s[2]);
  }
};
template <class SH>
struct VelRow9<SH, 1> {
  VelRow<SH, 1> V;
  int perm;
  __device__ __forceinline__ void load(const PatchStep &P, const int4 d, const uint32_t *__restrict__ pat,
                                       const uint8_t *__restrict__ ip, int l64) {
    V.load(P, d, pat, l64);
    perm = ip[min(V.R.row + 2 * NU_LOC, NLOC - 1)];
  }
  __device__ __forceinline__ void residual(const float4 *hv, const float *, float *rs, int l64) const {
    const float s = V.sum(hv, l64);
    if ((l64 & 15) == 0 && V.R.row != PT_NOROW) rs[perm] = V.R.f - s;
  }
};

template <typename F, bool FULL>
struct PatchLds {
  float4 hv[PT_HALO + 1];                   // the halo, and zeros at PT_ZERO
  float hp[4 * PT_RUNS];
  float rs[RLOC_STRIDE], xs[RLOC_STRIDE];   // local residual and solution
  float M[FULL ? 4 : SCH_STRIDE];           // stored block form
  float pp[NP_LOC];
};

// the barrier of the workgroup, for code of one wavefront each (every wavefront passes it the
// same number of times)
__device__ __forceinline__ void patch_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The part of wavefront W: its two row quads, its share of the halo and of the stored data, then
// of the local solve.
template <typename F, bool FULL, bool GRID, bool NINE, int W>
__device__ __forceinline__ void patch_wave(const PatchStep &P, const F *__restrict__ stored, long pos, int l64,
                                           PatchLds<F, FULL> &S) {
  using SH = PatchShape<GRID>;
  constexpr int PER = 16 / int(sizeof(F));
  constexpr int NV = MINV_LD / PER;            // 16-byte vectors of a row of the full inverse
  constexpr int NS = SCH_STRIDE / PER;         // of the block form
  constexpr int NSQ = FULL ? 0 : (NS - 64 * W + 255) / 256;   // this wavefront's share of it
  const int t = 64 * W + l64;
  const int *__restrict__ rc = P.rec + pos * P.stride;
  // Loads in the order of their use, since a wait for one is a wait for all before it: first
  // what the record alone gives, then the halo, the rows, and last the stored data.
  const int pid = rc[PR_HEAD];
  const int nh = P.stride - PR_HALO;   // records are padded to the level's largest halo
  const int loc0 = rc[PR_HALO + min(t, nh - 1)];
  int loc1 = 0, run = 0;
  if constexpr (W < 2) {
    loc1 = rc[PR_HALO + min(t + 256, nh - 1)];
    run = rc[PR_RUN + t / 4];
  }
  const int4 *__restrict__ ds = reinterpret_cast<const int4 *>(rc + PR_DESC) + 8 * W + (l64 >> 4);
  const int4 d0 = ds[0], d1 = ds[4];
  int dof = 0, out = 0, own = 0;
  if constexpr (W == 0) {
    dof = rc[PR_DOFS + min(t, NU_LOC + NP_LOC - 1)];
    out = rc[PR_OUT + min(t, NU_LOC - 1)];
  }
  const uint32_t *__restrict__ pat = P.pat + long(pid) * SH::words;
  const float4 *__restrict__ ua = reinterpret_cast<const float4 *>(P.ua);
  const float4 h0 = ua[loc0];
  float4 h1;
  float hq = 0.0f, pv = 0.0f;
  if constexpr (W < 2) {
    h1 = ua[loc1];
    hq = P.u[3L * P.N + run + t % 4];
  }
  std::conditional_t<NINE, VelRow9<SH, 2 * W>, VelRow<SH, 2 * W>> A;
  std::conditional_t<NINE, VelRow9<SH, 2 * W + 1>, VelRow<SH, 2 * W + 1>> B;
  if constexpr (NINE) {
    const uint8_t *__restrict__ ip = P.invperm + pos * PERM_STRIDE;
    A.load(P, d0, pat, ip, l64);
    B.load(P, d1, pat, ip, l64);
  } else {
    A.load(P, d0, pat, l64);
    B.load(P, d1, pat, l64);
  }
  if constexpr (W == 0) {
    own = pat[SH::own + min(t, NU_LOC - 1) / 2] >> (16 * (t & 1));
    pv = P.u[3L * P.N + (t < NU_LOC ? 0 : dof)];   // (lanes of velocity dofs: unused)
  }
  // the stored local data (non-temporal: read once per sweep)
  v4u mv[FULL ? NV : NSQ > 0 ? NSQ : 1];
  if constexpr (FULL && W < 2) {
    const F *src = stored + pos * MINV_STRIDE;
    const int r = min(t, NLOC - 1);
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const int off = W == 0 ? (q * 64 + r) * PER : 64 * MINV_LD + (q * (NLOC - 64) + r - 64) * PER;
      mv[q] = __builtin_nontemporal_load(reinterpret_cast<const v4u *>(src + off));
    }
  }
  if constexpr (!FULL) {
    const v4u *src = reinterpret_cast<const v4u *>(stored + pos * SCH_STRIDE);
#pragma unroll
    for (int q = 0; q < NSQ; ++q) mv[q] = __builtin_nontemporal_load(src + min(t + 256 * q, NS - 1));
  }
  S.hv[t] = h0;
  if constexpr (W < 2) {
    S.hv[t + 256] = h1;
    S.hp[t] = hq;
  }
  if constexpr (W == 3) {
    if (l64 < RLOC_STRIDE - NLOC) S.rs[NLOC + l64] = 0.0f;
    if (l64 == 63) S.hv[PT_ZERO] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  patch_barrier();
  A.residual(S.hv, S.hp, S.rs, l64);
  B.residual(S.hv, S.hp, S.rs, l64);
  if constexpr (!FULL) {
#pragma unroll
    for (int q = 0; q < NSQ; ++q)
      if (t + 256 * q < NS) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          if constexpr (sizeof(F) == 2) {
            S.M[(t + 256 * q) * PER + 2 * h] = __uint_as_float(mv[q][h] << 16);
            S.M[(t + 256 * q) * PER + 2 * h + 1] = __uint_as_float(mv[q][h] & 0xffff0000u);
          } else {
            S.M[(t + 256 * q) * PER + h] = __uint_as_float(mv[q][h]);
          }
        }
      }
  }
  patch_barrier();
  if constexpr (FULL && W < 2) {
    // x = M r, a row per thread, the products in the order of k_vanka_apply
    float acc = 0.0f;
#pragma unroll
    for (int j0 = 0; j0 < MINV_LD; j0 += 4) {
      const v4f r4 = *reinterpret_cast<const v4f *>(S.rs + j0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int j = j0 + k;
        float a;
        if constexpr (sizeof(F) == 2) {
          const unsigned w = mv[j / 8][(j % 8) / 2];
          a = __uint_as_float(j % 2 ? (w & 0xffff0000u) : (w << 16));
        } else {
          a = __uint_as_float(mv[j / 4][j % 4]);
        }
        acc = fmaf(a, r4[k], acc);
      }
    }
    if (t < NLOC) S.xs[t] = acc;
  }
  // block form: p = P1 r on wavefront 1 beside y_c = A^{-1} r_c on wavefront 0, then
  // x_c = y_c - W_c p, the products in the order of k_vanka_apply_schur
  float y[3] = {0.0f, 0.0f, 0.0f};
  if constexpr (!FULL && W == 1) {
    const int k = l64 >> 4, part = l64 & 15;
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < (NLOC + 15) / 16; ++i) {
      const int q = part + 16 * i;
      const float m = S.M[SCH_P1 + k * NLOC + min(q, NLOC - 1)], r = S.rs[q];
      acc = q < NLOC ? fmaf(m, r, acc) : acc;
    }
    acc = red16(acc);
    if (part == 0) S.pp[k] = acc;
  }
  if constexpr (!FULL && W == 0) {
    const int i = min(t, NU_LOC - 1);
#pragma unroll 9
    for (int m = 0; m < NU_LOC; ++m) {
      const float w = S.M[SCH_AINV + i * NU_LOC + m];
      y[0] = fmaf(w, S.rs[m], y[0]);
      y[1] = fmaf(w, S.rs[NU_LOC + m], y[1]);
      y[2] = fmaf(w, S.rs[2 * NU_LOC + m], y[2]);
    }
  }
  patch_barrier();
  if constexpr (W == 0) {
    if (t < NU_LOC) {
      float x[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if constexpr (FULL) {
          x[c] = S.xs[c * NU_LOC + t];
        } else {
          x[c] = y[c];
#pragma unroll
          for (int k = 0; k < NP_LOC; ++k) x[c] = fmaf(-S.M[SCH_W + (c * NU_LOC + t) * NP_LOC + k], S.pp[k], x[c]);
        }
      }
      const float4 v = S.hv[own & 0xffff];
      const float n0 = v.x + P.damp * x[0], n1 = v.y + P.damp * x[1], n2 = v.z + P.damp * x[2];
      reinterpret_cast<float4 *>(P.ua)[out] = make_float4(n0, n1, n2, 0.0f);
      if (P.mirror) {
        P.u[dof] = n0;
        P.u[long(P.N) + dof] = n1;
        P.u[2L * P.N + dof] = n2;
      }
    } else if (t < NU_LOC + NP_LOC) {
      P.u[3L * P.N + dof] = pv + P.damp * (FULL ? S.xs[2 * NU_LOC + t] : S.pp[t - NU_LOC]);
    }
  }
}

// the patch of this workgroup (-1: none)
template <class Step>
__device__ __forceinline__ int patch_slot(const Step &P) {
  int slot = blockIdx.x;
  if (P.grouped) {
    // workgroup b runs on XCD b % 8 and takes its share of the b % 8-th eighth of the color's
    // consecutive cells, so that an XCD's L2 holds the vectors of one compact part of the mesh
    const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
    const int b0 = int(long(P.ncells) * x / 8), b1 = int(long(P.ncells) * (x + 1) / 8);
    if (k >= b1 - b0) return -1;
    slot = b0 + k;
  }
  return P.slots ? P.slots[slot] : slot;
}

// FULL: stored 85 x 85 inverse (minv layout), else the block form (SCH_* layout).  GRID: shape
// of the records' patterns.  NINE: nine velocity blocks, else the shared one.
template <typename F, bool FULL, bool GRID, bool NINE>
__global__ __launch_bounds__(256, NINE ? 2 : 1) void k_patch_step(PatchStep P, const F *__restrict__ stored) {
  __shared__ __align__(16) PatchLds<F, FULL> S;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l64 = threadIdx.x & 63;
  const int slot = patch_slot(P);
  if (slot < 0) return;
  const long pos = long(P.pos0) + slot;
  if (wave == 0)
    patch_wave<F, FULL, GRID, NINE, 0>(P, stored, pos, l64, S);
  else if (wave == 1)
    patch_wave<F, FULL, GRID, NINE, 1>(P, stored, pos, l64, S);
  else if (wave == 2)
    patch_wave<F, FULL, GRID, NINE, 2>(P, stored, pos, l64, S);
  else
    patch_wave<F, FULL, GRID, NINE, 3>(P, stored, pos, l64, S);
}

// ------------------------------------------------------------------ FP64
// The same step with the FP64 operator and the stored LU factors of dgetf2 (k_patch_lu).  The
// velocity stays in the component vectors: copy 0 is u itself, the others follow in P.alt.
// Bounds: small colors the chain of 170 steps of the two sweeps (lu_sweeps.hpp); large ones the
// stream of factors and rows, 100 KB per patch (226 registers allow two workgroups per CU, whose
// loads in flight cover the latency).  Residual and solve launches before -> this one, per color:
// 8^3 5.8 + 9.5 -> 9.2 us, 16^3 11.5 + 13.8 -> 15.8 us, 12 x 16 x 20 10.9 + 13.2 -> 15.9 us; the
// set-up and solve at 32^3 72.0 -> 54.7 ms.  The same results bit for bit.
__device__ __forceinline__ double *velocity_at(const PatchStep64 &P, int loc) {
  double *p = P.u + loc;
  if (loc >= P.N) {
    loc -= P.N;
    p = P.alt + loc;
    if (loc >= P.N) p = P.alt + 2L * P.N + loc;   // 3 N + (loc - N)
  }
  return p;
}

// between the components of the halo in LDS (PT_ZERO behind it; a multiple of 64, so that one
// instruction reads two components)
constexpr int HSTRIDE = PT_HALO + 64;

// four consecutive entries from p on (8-byte aligned)
__device__ __forceinline__ void ld4d(const double *p, double (&o)[4]) { ld4(p, o); }
__device__ __forceinline__ int window(int jb, int n) { return n >= 4 ? min(jb, n - 4) : 0; }

template <class SH, int QD>
struct Row64 {
  static constexpr int NB = QD == 1 ? 0 : SH::a(QD), OA = SH::off_a(QD), OB = SH::off_bt(QD);
  int n, m, row;
  double a[NB > 0 ? NB : 1][4], b[3][4], f;
  uint2 ia[NB > 0 ? NB : 1], ib;
  int perm;
  __device__ __forceinline__ void load(const PatchStep64 &P, const int4 d, const uint32_t *__restrict__ pat,
                                       const uint8_t *__restrict__ ip, int l64) {
    const int lane = l64 & 15;
    n = d.z & 255;
    m = (d.z >> 8) & 255;
    row = (d.z >> 16) & 255;
    if constexpr (QD == 1) {
      // pressure row: the three blocks of B
      ib = reinterpret_cast<const uint2 *>(pat + OA)[l64];
      const double *v = P.bv + 3L * d.x + window(4 * lane, n);
#pragma unroll
      for (int c = 0; c < 3; ++c) ld4d(v + c * n, b[c]);
      f = P.f[3L * P.N + d.w];
      perm = ip[min(row + 2 * NU_LOC, NLOC - 1)];
    } else {
#pragma unroll
      for (int k = 0; k < NB; ++k) ia[k] = reinterpret_cast<const uint2 *>(pat + OA + 128 * k)[l64];
      ib = reinterpret_cast<const uint2 *>(pat + OB)[l64];
#pragma unroll
      for (int k = 0; k < NB; ++k) ld4d(P.a1 + d.x + window(64 * k + 4 * lane, n), a[k]);
      const double *w = P.btv + 3L * d.y + window(4 * lane, m);
#pragma unroll
      for (int c = 0; c < 3; ++c) ld4d(w + c * m, b[c]);
      f = P.f[long(lane < 3 ? lane : 0) * P.N + d.w];
      perm = ip[min(row + NU_LOC * (lane < 3 ? lane : 0), NLOC - 1)];
    }
  }
  static __device__ __forceinline__ int at(uint2 w, int u) { return ((u < 2 ? w.x : w.y) >> (16 * (u & 1))) & 0xffffu; }
  // the entries of a lane's window that are its own (row_window)
  static __device__ __forceinline__ bool own(int jb, int len, int u) {
    const int e = window(jb, len) + u;
    return e >= jb && e < len;
  }
  // sums in the order of row_a1_v, row_bt_v and row_b_v
  __device__ __forceinline__ void residual(const double *hv, const double *hp, double *rs, int l64) const {
    const int lane = l64 & 15;
    if constexpr (QD == 1) {
      double s = 0.0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double *y = hv + at(ib, u);
        const bool ok = own(4 * lane, n, u);
        const double z1 = ok ? y[0] : 0.0, z2 = ok ? y[HSTRIDE] : 0.0, z3 = ok ? y[2 * HSTRIDE] : 0.0;
        // contracted as row_b_v is compiled in k_vanka_res
        s += fma(b[2][u], z3, u == 0 ? fma(b[1][u], z2, b[0][u] * z1) : fma(b[0][u], z1, b[1][u] * z2));
      }
      s = red16(s);
      if (lane == 0 && row != PT_NOROW) rs[perm] = f - s;
    } else {
      double s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const double *y = hv + at(ia[k], u);
          const double w = own(64 * k + 4 * lane, n, u) ? a[k][u] : 0.0;
          s1 += w * y[0];
          s2 += w * y[HSTRIDE];
          s3 += w * y[2 * HSTRIDE];
        }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double z = own(4 * lane, m, u) ? hp[at(ib, u)] : 0.0;
        s1 += b[0][u] * z;
        s2 += b[1][u] * z;
        s3 += b[2][u] * z;
      }
      s1 = red16(s1);
      s2 = red16(s2);
      s3 = red16(s3);
      if (lane < 3 && row != PT_NOROW) rs[perm] = f - (lane == 0 ? s1 : lane == 1 ? s2 : s3);
    }
  }
};

struct Patch64Lds {
  double hv[3 * HSTRIDE], hp[4 * PT_RUNS], rs[RLOC_STRIDE];
  v4u fac[32 + 64 * 29];   // a factor part after 64 entries of padding (k_vanka_solve)
};

template <bool GRID, int W>
__device__ __forceinline__ void patch_wave64(const PatchStep64 &P, long pos, int l64, Patch64Lds &S) {
  using SH = PatchShape64<GRID>;
  // 16-byte vectors of the two factor parts, dealt to the four wavefronts in runs of 64
  constexpr int RL = 28, RU = 29, NL = (RL - W + 3) / 4, NU = (RU - W + 3) / 4;
  static_assert(64 * RL * 2 >= LU_L && 64 * RU * 2 >= LU_U, "factor parts");
  static_assert(lu_uoff(NLOC - 1) + 127 < 2 * 64 * RU, "the sweeps read past the copy");
  const int t = 64 * W + l64;
  const int *__restrict__ rc = P.rec + pos * P.stride;
  const int pid = rc[PR_HEAD];
  const int nh = P.stride - PR_HALO;
  const int loc0 = rc[PR_HALO + min(t, nh - 1)];
  int loc1 = 0, run = 0;
  if constexpr (W < 2) {
    loc1 = rc[PR_HALO + min(t + 256, nh - 1)];
    run = rc[PR_RUN + t / 4];
  }
  const int4 *__restrict__ ds = reinterpret_cast<const int4 *>(rc + PR_DESC) + 8 * W + (l64 >> 4);
  const int4 d0 = ds[0], d1 = ds[4];
  const uint8_t *__restrict__ ip = P.invperm + pos * PERM_STRIDE;
  // wavefront 0 solves: lane i owns rows i and 64 + i; rows c * 27 + j of dof j, 81 + k of
  // pressure dof k
  int out0 = 0, out1 = 0, own0 = 0, own1 = 0;
  const bool two = l64 < NLOC - 64;
  const int c0 = l64 / NU_LOC, j0 = l64 - c0 * NU_LOC;             // row l64 < 64
  const int i1 = min(64 + l64, NLOC - 1), j1 = i1 - 2 * NU_LOC;    // row 64 + l64: component 2 or pressure
  if constexpr (W == 0) {
    out0 = rc[PR_OUT + j0];
    out1 = j1 < NU_LOC ? rc[PR_OUT + j1] : rc[PR_DOFS + j1];
  }
  const uint32_t *__restrict__ pat = P.pat + long(pid) * SH::words;
  const double *const q0 = velocity_at(P, loc0);
  const double h0[3] = {q0[0], q0[P.N], q0[2L * P.N]};
  double h1[3] = {0.0, 0.0, 0.0}, hq = 0.0;
  if constexpr (W < 2) {
    const double *const q1 = velocity_at(P, loc1);
    h1[0] = q1[0];
    h1[1] = q1[P.N];
    h1[2] = q1[2L * P.N];
    hq = P.u[3L * P.N + run + t % 4];
  }
  Row64<SH, 2 * W> A;
  Row64<SH, 2 * W + 1> B;
  A.load(P, d0, pat, ip, l64);
  B.load(P, d1, pat, ip, l64);
  if constexpr (W == 0) {
    own0 = (pat[SH::own + j0 / 2] >> (16 * (j0 & 1))) & 0xffffu;
    own1 = (pat[SH::own + min(j1, NU_LOC - 1) / 2] >> (16 * (j1 & 1))) & 0xffffu;
  }
  double v1 = 0.0;
  if constexpr (W == 0) v1 = P.u[3L * P.N + (j1 < NU_LOC ? 0 : out1)];   // (velocity rows: unused)
  // the factors last: they are needed last
  const v4u *__restrict__ gL = reinterpret_cast<const v4u *>(P.lu + pos * LU_STRIDE);
  const v4u *__restrict__ gU = reinterpret_cast<const v4u *>(P.lu + pos * LU_STRIDE + LU_UOFF);
  v4u rL[NL], rU[NU];
#pragma unroll
  for (int q = 0; q < NL; ++q) rL[q] = gL[l64 + 64 * (4 * q + W)];
#pragma unroll
  for (int q = 0; q < NU; ++q) rU[q] = gU[l64 + 64 * (4 * q + W)];
#pragma unroll
  for (int c = 0; c < 3; ++c) S.hv[c * HSTRIDE + t] = h0[c];
  if constexpr (W < 2) {
#pragma unroll
    for (int c = 0; c < 3; ++c) S.hv[c * HSTRIDE + t + 256] = h1[c];
    S.hp[t] = hq;
  }
  if constexpr (W == 3)
    if (l64 < 3) S.hv[l64 * HSTRIDE + PT_ZERO] = 0.0;
  patch_barrier();
  A.residual(S.hv, S.hp, S.rs, l64);
  B.residual(S.hv, S.hp, S.rs, l64);
  v4u *const s4 = S.fac + 32;
#pragma unroll
  for (int q = 0; q < NL; ++q) s4[l64 + 64 * (4 * q + W)] = rL[q];
  patch_barrier();
  // the sweeps of k_vanka_solve, on wavefront 0; the others put the U part in place between them
  const double *const fac = reinterpret_cast<const double *>(s4);
  double x0 = 0.0, x1 = 0.0;
  if constexpr (W == 0) {
    x0 = S.rs[l64];
    x1 = two ? S.rs[64 + l64] : 0.0;
    lower_sweep<double, double>(fac, l64, x0, x1);
  }
  patch_barrier();
#pragma unroll
  for (int q = 0; q < NU; ++q) s4[l64 + 64 * (4 * q + W)] = rU[q];
  patch_barrier();
  if constexpr (W == 0) {
    upper_sweep<double, double>(fac, l64, two, x0, x1);
    velocity_at(P, out0)[long(c0) * P.N] = S.hv[c0 * HSTRIDE + own0] + P.damp * x0;
    if (two) {
      if (j1 < NU_LOC)
        velocity_at(P, out1)[2L * P.N] = S.hv[2 * HSTRIDE + own1] + P.damp * x1;
      else
        P.u[3L * P.N + out1] = v1 + P.damp * x1;
    }
  }
}

template <bool GRID>
__global__ __launch_bounds__(256) void k_patch_step64(PatchStep64 P) {
  __shared__ Patch64Lds S;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l64 = threadIdx.x & 63;
  const int slot = patch_slot(P);
  if (slot < 0) return;
  const long pos = long(P.pos0) + slot;
  if (wave == 0)
    patch_wave64<GRID, 0>(P, pos, l64, S);
  else if (wave == 1)
    patch_wave64<GRID, 1>(P, pos, l64, S);
  else if (wave == 2)
    patch_wave64<GRID, 2>(P, pos, l64, S);
  else
    patch_wave64<GRID, 3>(P, pos, l64, S);
}

}  // namespace

void launch_patch_step64(const PatchStep64 &P, hipStream_t s) {
  if (P.ncells <= 0) return;
  const int grid = P.grouped ? 8 * ((P.ncells + 7) / 8) : P.ncells;
  if (P.grid)
    k_patch_step64<true><<<grid, 256, 0, s>>>(P);
  else
    k_patch_step64<false><<<grid, 256, 0, s>>>(P);
  PMG_HIP_CHECK(hipGetLastError());
}

void launch_patch_step(const PatchStep &P, const float *stored32, const uint16_t *stored16, bool full, hipStream_t s) {
  if (P.ncells <= 0) return;
  const int grid = P.grouped ? 8 * ((P.ncells + 7) / 8) : P.ncells;
  auto go = [&](auto f_c, const auto *stored) {
    constexpr bool FULL = decltype(f_c)::value;
    using F = std::remove_const_t<std::remove_pointer_t<decltype(stored)>>;
    if constexpr (FULL)
      if (P.av) {
        k_patch_step<F, true, true, true><<<grid, 256, 0, s>>>(P, stored);
        return;
      }
    if (P.grid)
      k_patch_step<F, FULL, true, false><<<grid, 256, 0, s>>>(P, stored);
    else
      k_patch_step<F, FULL, false, false><<<grid, 256, 0, s>>>(P, stored);
  };
  if (P.av && !(full && P.grid)) throw DeviceError("launch_patch_step: nine blocks without full inverses on a grid");
  if (stored16 && full)
    go(std::true_type{}, stored16);
  else if (stored16)
    go(std::false_type{}, stored16);
  else if (full)
    go(std::true_type{}, stored32);
  else
    go(std::false_type{}, stored32);
  PMG_HIP_CHECK(hipGetLastError());
}

}  // namespace pmg
