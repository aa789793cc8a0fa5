// Device helpers shared by the solver's translation units (solver.hip,
// direct.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace rpgo {

// DPP row rotation of an FP64 value (both halves), all lanes of the row valid
template <int N>
__device__ __forceinline__ double row_ror_f64(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, 0x120 + N, 0xF, 0xF, false),
                          __builtin_amdgcn_update_dpp(0, lo, 0x120 + N, 0xF, 0xF, false));
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the 64 lanes of a converged wavefront, in every lane: rotations
// within each row of 16 lanes by DPP (VALU, a few cycles each), then the four
// row sums by v_readlane.  A six-step shuffle reduction went through the LDS
// crossbar (ds_bpermute) at every step, on the critical path of each PCG
// launch.
__device__ __forceinline__ double wave_sum_pre(double v) {
  v += row_ror_f64<8>(v);
  v += row_ror_f64<4>(v);
  v += row_ror_f64<2>(v);
  v += row_ror_f64<1>(v);
  return (readlane_f64(v, 0) + readlane_f64(v, 16)) + (readlane_f64(v, 32) + readlane_f64(v, 48));
}

// block-wide FP64 sum (all threads call it; the result is valid in thread 0)
__device__ __forceinline__ double block_sum(double v, double* lds16) {
  v = wave_sum_pre(v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) lds16[wid] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x < 64) {
    t = threadIdx.x < (blockDim.x >> 6) ? lds16[threadIdx.x] : 0.0;
    t = wave_sum_pre(t);
  }
  return t;  // valid in thread 0
}

}  // namespace rpgo
