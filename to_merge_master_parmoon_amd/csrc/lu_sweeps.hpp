// lu_sweeps.hpp - the triangular sweeps of one patch's packed LU factors by one wavefront.
//
// Lane i owns rows i and 64 + i (i < 21) of the 85 unknowns.  Each sweep is a chain of steps: the
// finished unknown of step k goes to all lanes (readlane) and column k is subtracted from the
// rows it reaches.  A column's entries are read from LDS one block of steps ahead of the
// block in work (the compiler left to itself reads one step ahead and waits for LDS at every
// step: about 105 cycles a step), and the entries of rows that a column does not reach are
// replaced by zero ahead of the chain, so that no select stands in it (putting every unknown aside
// at its step instead costs 3 % of a color).  FP64, one color of the fused step (k_patch.hip): 8^3
// 11.6 -> 9.2 us, 16^3 17.7 -> 15.8 us, the same results bit for bit.
// An unknown that is not finite would come to the rows that its column does not reach as zero
// times it.  Its own row shows it at the end; the sweep is then run again with selects.  (In FP64 the
// upper sweep only: one in the lower sweep makes all later rows and, from the last row's quotient
// on, all unknowns NaN with selects too.)
#pragma once
#include <hip/hip_runtime.h>

#include "pmg_internal.hpp"

namespace pmg {

__device__ inline double bcast(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}
__device__ inline float bcast(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__device__ inline double tfma(double a, double b, double c) { return fma(a, b, c); }
__device__ inline float tfma(float a, float b, float c) { return fmaf(a, b, c); }

template <typename T, typename F>
struct Ld;
template <typename T>
struct Ld<T, T> {
  static __device__ inline T get(const T *p, int i) { return p[i]; }
};
template <>
struct Ld<float, double> {
  static __device__ inline float get(const double *p, int i) { return float(p[i]); }
};
template <>
struct Ld<float, uint16_t> {
  static __device__ inline float get(const uint16_t *p, int i) {
    return __uint_as_float(uint32_t(p[i]) << 16);
  }
};

// some unknown of the patch is not finite (row 64 + lane exists on the first 21 lanes)
template <typename T>
__device__ __forceinline__ bool any_not_finite(int lane, T x0, T x1) {
  return __any(!(fabs(x0) < T(INFINITY)) || (lane < NLOC - 64 && !(fabs(x1) < T(INFINITY))));
}

constexpr int LU_STEPS = 6;   // steps of a block; two blocks of entries are in registers

// x := L^{-1} x; s: the packed L part in LDS, L(r, k) at lu_loff(k) + r - k - 1, with 64 readable
// entries before it
template <typename T, typename F>
__device__ __forceinline__ void lower_sweep(const F *s, int lane, T &x0, T &x1) {
  constexpr int N = NLOC - 1, NB = (N + LU_STEPS - 1) / LU_STEPS;
  const F *const sl0 = s + lane, *const sl1 = sl0 + 64;
  const T r0 = x0, r1 = x1;
  T a[2][LU_STEPS], b[2][LU_STEPS];
  auto fetch = [&](int blk, T (&p)[LU_STEPS], T (&q)[LU_STEPS]) {
#pragma unroll
    for (int i = 0; i < LU_STEPS; ++i) {
      const int k = blk * LU_STEPS + i, o = lu_loff(k) - k - 1;
      if (k >= N) continue;
      if (k < 64) p[i] = Ld<T, F>::get(sl0, o);
      q[i] = Ld<T, F>::get(sl1, o);
    }
  };
  fetch(0, a[0], b[0]);
#pragma unroll
  for (int blk = 0; blk < NB; ++blk) {
    if (blk + 1 < NB) fetch(blk + 1, a[(blk + 1) & 1], b[(blk + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < LU_STEPS; ++i) {
      const int k = blk * LU_STEPS + i;
      if (k >= N) continue;
      T &p = a[blk & 1][i], &q = b[blk & 1][i];
      // row lane is below the diagonal for lane > k, row 64 + lane for every k < 64
      if (k < 64) {
        p = lane > k ? p : T(0);
        const T xk = bcast(x0, k);
        x0 = tfma(-xk, p, x0);
        x1 = tfma(-xk, q, x1);
      } else {
        q = lane + 64 > k ? q : T(0);
        x1 = tfma(-bcast(x1, k - 64), q, x1);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (sizeof(T) == 8 || !any_not_finite(lane, x0, x1)) return;
  x0 = r0;
  x1 = r1;
#pragma unroll 1
  for (int k = 0; k < N; ++k) {
    const int o = lu_loff(k) - k - 1;
    const T xk = k < 64 ? bcast(x0, k) : bcast(x1, k - 64);
    if (lane > k) x0 = tfma(-xk, Ld<T, F>::get(sl0, o), x0);
    if (lane + 64 > k) x1 = tfma(-xk, Ld<T, F>::get(sl1, o), x1);
  }
}

// x := U^{-1} x; s: the packed U part, U(r, k) at lu_uoff(k) + r.  A row's value is final once its
// own step is passed, so its quotient is formed with all others after the chain.  The
// quotient: with rc the correctly rounded reciprocal, q = x rc, q' = fma(fma(-q, U, x), rc, q)
// is the correctly rounded x / U (Markstein), the division of the column-oriented dtrsm, in
// three dependent steps; FP32 takes q.
template <typename T, typename F>
__device__ __forceinline__ void upper_sweep(const F *s, int lane, bool two, T &x0, T &x1) {
  constexpr int NB = (NLOC + LU_STEPS - 1) / LU_STEPS;
  const F *const sl0 = s + lane, *const sl1 = sl0 + 64;
  const T r0 = x0, r1 = x1;
  const T dg0 = Ld<T, F>::get(s, lu_uoff(lane) + lane);
  const T dg1 = two ? Ld<T, F>::get(s, lu_uoff(64 + lane) + 64 + lane) : T(1);
  const T rc0 = T(1) / dg0, rc1 = T(1) / dg1;
  auto quotient = [](T x, T d, T rc) {
    T q = x * rc;
    if constexpr (sizeof(T) == 8) q = tfma(tfma(-q, d, x), rc, q);
    return q;
  };
  T a[2][LU_STEPS], b[2][LU_STEPS];
  auto fetch = [&](int blk, T (&p)[LU_STEPS], T (&q)[LU_STEPS]) {
#pragma unroll
    for (int i = 0; i < LU_STEPS; ++i) {
      const int k = NLOC - 1 - (blk * LU_STEPS + i);
      if (k < 0) continue;
      p[i] = Ld<T, F>::get(sl0, lu_uoff(k));
      if (k >= 64) q[i] = Ld<T, F>::get(sl1, lu_uoff(k));
    }
  };
  fetch(0, a[0], b[0]);
#pragma unroll
  for (int blk = 0; blk < NB; ++blk) {
    if (blk + 1 < NB) fetch(blk + 1, a[(blk + 1) & 1], b[(blk + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < LU_STEPS; ++i) {
      const int k = NLOC - 1 - (blk * LU_STEPS + i);
      if (k < 0) continue;
      T &p = a[blk & 1][i], &q = b[blk & 1][i];
      // row lane is above the diagonal for every k >= 64, row 64 + lane for none below 64
      if (k >= 64) {
        q = lane + 64 < k ? q : T(0);
        const T xk = bcast(quotient(x1, dg1, rc1), k - 64);
        x0 = tfma(-xk, p, x0);
        x1 = tfma(-xk, q, x1);
      } else {
        p = lane < k ? p : T(0);
        x0 = tfma(-bcast(quotient(x0, dg0, rc0), k), p, x0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  x0 = quotient(x0, dg0, rc0);
  x1 = quotient(x1, dg1, rc1);
  if (!any_not_finite(lane, x0, x1)) return;
  x0 = r0;
  x1 = r1;
#pragma unroll 1
  for (int k = NLOC - 1; k >= 0; --k) {
    const int o = lu_uoff(k);
    const T q0 = quotient(x0, dg0, rc0), q1 = quotient(x1, dg1, rc1);
    const T xk = k < 64 ? bcast(q0, k) : bcast(q1, k - 64);
    if (lane == k) x0 = q0;
    if (lane + 64 == k) x1 = q1;
    if (lane < k) x0 = tfma(-xk, Ld<T, F>::get(sl0, o), x0);
    if (lane + 64 < k) x1 = tfma(-xk, Ld<T, F>::get(sl1, o), x1);
  }
}

}  // namespace pmg
