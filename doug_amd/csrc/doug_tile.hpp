// Device helpers shared by the kernel files.
#pragma once
#include "doug_kernels.hpp"

#pragma clang fp contract(off)

namespace doug {
namespace {

// Matrix-core tile product for each element type.  Both forms take A[l%16][l/16]
// and B[l/16][l%16] from lane l.  Result register r of lane l holds
//   f64 16x16x4: D[l/16 + 4r][l%16]   (single-row groups strided by 4)
//   f32 16x16x4: D[4(l/16) + r][l%16] (groups of four consecutive rows)
template <typename T>
struct Mma;
template <>
struct Mma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct Mma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

template <typename V>
__device__ __forceinline__ void zero_acc(V (&acc)[2][2]) {
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[a][b] = V{0, 0, 0, 0};
}

// orders this wavefront's LDS writes before its later LDS reads of them
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int local_col(const int32_t* __restrict__ occ_ptr,
                                         const int32_t* __restrict__ occ_pos, int c, int s0, int s) {
  for (int k = occ_ptr[c]; k < occ_ptr[c + 1]; k++) {
    const int q = occ_pos[k];
    if (q >= s0 + s) break;
    if (q >= s0) return q - s0;
  }
  return -1;
}

// Lets a kernel's workgroups take this much dynamic LDS: the most that any
// launch may ask for, since the limit belongs to the kernel and one context's
// need would take away another's.
template <typename K>
hipError_t allow_lds(K* kernel, int bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

}  // namespace
}  // namespace doug
