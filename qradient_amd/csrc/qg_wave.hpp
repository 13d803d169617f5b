// Sums and prefix sums of FP64 values across a wave.
#pragma once
#include <hip/hip_runtime.h>

namespace qg {

// x moved across lanes by the DPP control CTRL (each 32-bit half with one
// v_mov_b32_dpp); lanes of rows outside ROWM get 0.
template <int CTRL, int ROWM>
__device__ __forceinline__ double dpp_d(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWM, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWM, 0xF, false);
  return __builtin_bit_cast(double, (unsigned long long)(unsigned)lo | ((unsigned long long)(unsigned)hi << 32));
}

// The sum of v over the wave (width lanes), returned in every lane, in a fixed
// order.  A full wave reduces with DPP moves, which stay in the vector ALU:
// pairs (quad_perm 1,0,3,2), quads (2,3,0,1), groups of 8 (row_half_mirror)
// and 16 (row_mirror) in every lane, then row_bcast:15 into rows 1 and 3 and
// row_bcast:31 into rows 2 and 3, which leaves the total in lane 63.  The
// shuffle tree it replaces (a chain of six ds_bpermute pairs per sum) had the
// complex128 adjoint passes at 24 qubits at 197 / 136 / 138 us against 167 /
// 131 / 134 us, and the complex64 one at 100.6 against 97.2 us per pass.
// Narrower waves (passes of fewer than 64 threads) keep the shuffle tree.
__device__ __forceinline__ double wave_sum(double v, int width) {
  if (width == 64) {
    v += dpp_d<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
    v += dpp_d<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
    v += dpp_d<0x141, 0xF>(v);  // row_half_mirror
    v += dpp_d<0x140, 0xF>(v);  // row_mirror
    v += dpp_d<0x142, 0xA>(v);  // row_bcast:15
    v += dpp_d<0x143, 0xC>(v);  // row_bcast:31
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, 63);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), 63);
    return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
  }
  for (int off = width >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, width);
  return v;
}

// The inclusive prefix sum of v over the 64 lanes, in a fixed order: row_shr
// by 1, 2, 4, 8 inside each row of 16, then row_bcast:15 and row_bcast:31
// carry the rows' totals on.
__device__ __forceinline__ double wave_scan(double v) {
  v += dpp_d<0x111, 0xF>(v);
  v += dpp_d<0x112, 0xF>(v);
  v += dpp_d<0x114, 0xF>(v);
  v += dpp_d<0x118, 0xF>(v);
  v += dpp_d<0x142, 0xA>(v);
  v += dpp_d<0x143, 0xC>(v);
  return v;
}

// Lane l's value of v (l uniform), in every lane.
__device__ __forceinline__ double wave_lane(double v, int l) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
}

}  // namespace qg
