// wave_argmax.hpp - pivot search of the LU kernels: the largest |a(i, j)| and the lowest i among
// equals (the rule of dgetf2).
//
// The value alone is reduced first (v_max_f64 over DPP patterns, three instructions a round),
// then the lowest index of the lanes that hold it: reducing (value, index) pairs takes two
// comparisons and three selects a round, each waiting for the one before, and was a good part of
// a pivot step.  16 columns of a panel of up to 256 rows 28 -> 20 us, of up to 768 rows 43 -> 38 us;
// the one-workgroup LU of 499 unknowns 2.17 -> 1.94 ms.
#pragma once
#include <hip/hip_runtime.h>

namespace pmg {

// the larger value; a NaN gives way to a number
__device__ inline double max_f64(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// one round with the lanes that the DPP pattern CTRL selects, in the rows of 16 lanes of ROWS
template <int CTRL, int ROWS>
__device__ inline double max_dpp(double v) {
  const int h = __double2hiint(v), l = __double2loint(v);
  const int hi = __builtin_amdgcn_update_dpp(h, h, CTRL, ROWS, 0xF, false);
  const int lo = __builtin_amdgcn_update_dpp(l, l, CTRL, ROWS, 0xF, false);
  return max_f64(v, __hiloint2double(hi, lo));
}
template <int CTRL, int ROWS>
__device__ inline int min_dpp(int v) {
  return min(v, __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xF, false));
}
// (bv, bi) := the wavefront's largest bv and the lowest bi among the lanes that hold it, in every
// lane (all 64 active; lanes without a candidate hold bv = -1; bi is no row if all are NaN).
// ASC: bi ascends with the lane.
template <bool ASC>
__device__ inline void wave_argmax(double &bv, int &bi) {
  // quad xor 1, quad xor 2, half-row mirror, row mirror, row 0 to 1 and 2 to 3, row 1 to 2 and 3
  double m = max_dpp<0xB1, 0xF>(bv);
  m = max_dpp<0x4E, 0xF>(m);
  m = max_dpp<0x141, 0xF>(m);
  m = max_dpp<0x140, 0xF>(m);
  m = max_dpp<0x142, 0xA>(m);
  m = max_dpp<0x143, 0xC>(m);
  m = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(m), 63), __builtin_amdgcn_readlane(__double2loint(m), 63));
  if (ASC) {
    const int f = __ffsll((long long)__ballot(bv == m));
    bi = f ? __builtin_amdgcn_readlane(bi, f - 1) : 0x7fffffff;
  } else {
    // no loop over the lanes of the ballot: it would keep the caller's column loop from unrolling
    int i = bv == m ? bi : 0x7fffffff;
    i = min_dpp<0xB1, 0xF>(i);
    i = min_dpp<0x4E, 0xF>(i);
    i = min_dpp<0x141, 0xF>(i);
    i = min_dpp<0x140, 0xF>(i);
    i = min_dpp<0x142, 0xA>(i);
    i = min_dpp<0x143, 0xC>(i);
    bi = __builtin_amdgcn_readlane(i, 63);
  }
  bv = m;
}
// the same over the results of W wavefronts (v, i in LDS)
template <int W>
__device__ inline void block_argmax(const double *v, const int *i, double &bv, int &bi) {
  double cv[W];
  int ci[W];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    cv[w] = v[w];
    ci[w] = i[w];
  }
  bv = cv[0];
#pragma unroll
  for (int w = 1; w < W; ++w) bv = max_f64(bv, cv[w]);
  bi = 0x7fffffff;
#pragma unroll
  for (int w = 0; w < W; ++w) bi = min(bi, cv[w] == bv ? ci[w] : 0x7fffffff);
}

}  // namespace pmg
