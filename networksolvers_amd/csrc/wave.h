// Wave-level helpers shared by the factorisation and Krylov kernels: DPP sums of doubles
// across a 64-lane wave, lane broadcasts.
#pragma once
#include <hip/hip_runtime.h>

namespace nsmi {
namespace {

// DPP lane move of a double (two 32-bit moves); lanes disabled by the row mask or
// reading outside the row take 0
template <int CTRL, int ROWM>
__device__ inline double dpp_mov(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, ROWM, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, ROWM, 0xF, true);
  return __hiloint2double(hi, lo);
}

__device__ inline double read_lane63(double x) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 63),
                          __builtin_amdgcn_readlane(__double2loint(x), 63));
}

// Wave-wide sums of R values at once (the R chains interleave); every lane gets
// the totals.  Pair, quad, half-row and row sums by quad permutes and mirrors,
// then rows 1 and 3 take row 0 and 2 (row_bcast:15) and rows 2 and 3 take the
// sum of rows 0 and 1 (row_bcast:31): lane 63 holds the total.
template <int R>
__device__ inline void wave_totals(double (&a)[R]) {
#pragma unroll
  for (int s = 0; s < R; ++s) a[s] += dpp_mov<0xB1, 0xF>(a[s]);  // quad_perm [1,0,3,2]
#pragma unroll
  for (int s = 0; s < R; ++s) a[s] += dpp_mov<0x4E, 0xF>(a[s]);  // quad_perm [2,3,0,1]
#pragma unroll
  for (int s = 0; s < R; ++s) a[s] += dpp_mov<0x141, 0xF>(a[s]);  // row_half_mirror
#pragma unroll
  for (int s = 0; s < R; ++s) a[s] += dpp_mov<0x140, 0xF>(a[s]);  // row_mirror
#pragma unroll
  for (int s = 0; s < R; ++s) a[s] += dpp_mov<0x142, 0xA>(a[s]);  // row_bcast:15
#pragma unroll
  for (int s = 0; s < R; ++s) a[s] += dpp_mov<0x143, 0xC>(a[s]);  // row_bcast:31
#pragma unroll
  for (int s = 0; s < R; ++s) a[s] = read_lane63(a[s]);
}

__device__ inline double wave_total(double x) {
  double a[1] = {x};
  wave_totals<1>(a);
  return a[0];
}

// orders a wave's own LDS writes before its later LDS reads of other lanes' entries
__device__ inline void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline double lane_bcast(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

// largest value over the wave (every lane gets it)
__device__ inline double wave_max(double x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o, 64));
  return x;
}

}  // namespace
}  // namespace nsmi
