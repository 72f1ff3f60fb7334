// Sums across the lanes of a DPP row, lane reads, and a workgroup
// barrier for LDS alone (gfx950).
#pragma once
#include <hip/hip_runtime.h>

namespace rf {

// 32-bit DPP move of both halves of a double (CTRL: a DPP control code)
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  // every control used here names a lane of the row for each lane: there is
  // no old value to keep (and no register to set to it)
  const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(b), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(b >> 32), CTRL, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// sum over the 16 lanes of a DPP row, returned in every lane of the row:
// quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_ror:4, row_ror:8
__device__ __forceinline__ double row16_sum(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x124>(v);
  v += dpp_d<0x128>(v);
  return v;
}

// the value of one lane (a uniform index), in every lane
__device__ __forceinline__ double readlane_d(double v, int lane) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), lane);
  const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), lane);
  return __builtin_bit_cast(double, (static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// workgroup barrier that orders LDS only: the loads in flight stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// sum over 8 consecutive lanes, in every lane: quad_perm [1,0,3,2], quad_perm
// [2,3,0,1], row_half_mirror
__device__ __forceinline__ double half_row_sum(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x141>(v);
  return v;
}

}  // namespace rf
