// MFMA operand traits for gfx950.
#pragma once
#include <hip/hip_runtime.h>

namespace rf {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;

// v_mfma_f64_16x16x4f64: lane l supplies A[l%16][l/16], B[l/16][l%16]; output
// register r of lane l is D[l/16 + 4r][l%16] (checked on gfx950).
template <>
struct Mfma<double> {
  using acc_t = v4d;
  __device__ static acc_t op(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ static int orow(int lane, int r) { return lane / 16 + 4 * r; }
};

}  // namespace rf
