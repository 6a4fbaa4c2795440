// Small 3-vector helpers of the contact kernels, without FMA contraction whatever file includes
// them (most are built with -ffp-contract=off; division and square root are correctly rounded
// everywhere), so the same expression gives the same bits in the forward kernels, in the fused
// sweep and in their adjoint replays.
#pragma once
#include <hip/hip_runtime.h>

#define XRT_NO_FMA _Pragma("clang fp contract(off)")  // first in a function's body

namespace xrt {
namespace cm {

constexpr float kEpsC = 1e-6f;                 // EPSILON
constexpr float kScalarMax = 3.402823466e38f;  // SCALAR_MAX

struct F3 {
  float x, y, z;
};
__device__ __forceinline__ F3 L3(float4 a) { XRT_NO_FMA return F3{a.x, a.y, a.z}; }
__device__ __forceinline__ F3 A(F3 a, F3 b) { XRT_NO_FMA return F3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ F3 S(F3 a, F3 b) { XRT_NO_FMA return F3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ F3 M(F3 a, float s) { XRT_NO_FMA return F3{a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ float D(F3 a, F3 b) { XRT_NO_FMA return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ F3 C(F3 a, F3 b) { XRT_NO_FMA
  return F3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float Len(F3 a) { XRT_NO_FMA return sqrtf(D(a, a)); }
__device__ __forceinline__ F3 Nz(F3 a) { XRT_NO_FMA return M(a, 1.0f / Len(a)); }
__device__ __forceinline__ float Mixed(F3 a, F3 b, F3 c) { XRT_NO_FMA return D(a, C(b, c)); }
__device__ __forceinline__ float Cl(float x, float a, float b) { XRT_NO_FMA return x < a ? a : (x > b ? b : x); }
__device__ __forceinline__ F3 FaceNormal(F3 a, F3 b, F3 c) { XRT_NO_FMA return Nz(C(S(b, a), S(c, a))); }

}  // namespace cm
}  // namespace xrt
