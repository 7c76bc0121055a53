// wave_argmax.hpp - pivot search of the LU kernels inside one wavefront: DPP within the rows of 16
// lanes instead of six rounds of LDS permutes (a 16-column panel of up to 768 rows 45 -> 43 us, of up
// to 256 rows 34 -> 28 us, the same pivots).
#pragma once
#include <hip/hip_runtime.h>

namespace pmg {

// (bv, bi) := the larger value, the lower index among equals (the pivot rule of dgetf2)
__device__ inline void amax_take(double &bv, int &bi, double ov, int oi) {
  const bool take = ov > bv || (ov == bv && oi < bi);
  bv = take ? ov : bv;
  bi = take ? oi : bi;
}
// one step of the reduction with the partner lane that the DPP pattern CTRL selects
template <int CTRL>
__device__ inline void amax_dpp(double &bv, int &bi) {
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(bv), CTRL, 0xF, 0xF, false);
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(bv), CTRL, 0xF, 0xF, false);
  const int oi = __builtin_amdgcn_mov_dpp(bi, CTRL, 0xF, 0xF, false);
  amax_take(bv, bi, __hiloint2double(hi, lo), oi);
}
// the wavefront's largest value and its lowest index in every lane (all 64 lanes active):
// within each row of 16 lanes by DPP (quad xor 1, quad xor 2, half-row mirror, row
// mirror), then the four rows' results by readlane, taken in lane order
__device__ inline void wave_argmax(double &bv, int &bi) {
  amax_dpp<0xB1>(bv, bi);
  amax_dpp<0x4E>(bv, bi);
  amax_dpp<0x141>(bv, bi);
  amax_dpp<0x140>(bv, bi);
  const int h = __double2hiint(bv), l = __double2loint(bv);
  double v = __hiloint2double(__builtin_amdgcn_readlane(h, 0), __builtin_amdgcn_readlane(l, 0));
  int i = __builtin_amdgcn_readlane(bi, 0);
#pragma unroll
  for (int r = 1; r < 4; ++r)
    amax_take(v, i, __hiloint2double(__builtin_amdgcn_readlane(h, 16 * r), __builtin_amdgcn_readlane(l, 16 * r)),
              __builtin_amdgcn_readlane(bi, 16 * r));
  bv = v;
  bi = i;
}

}  // namespace pmg
