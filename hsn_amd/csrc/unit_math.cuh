// The unit bank's activation, shared by its kernels (units.hip, unit_gemm.hip).
#pragma once

#include "common.cuh"

namespace hsn {
namespace units {

constexpr float kRsqrt2 = 0.70710678118654752f;
constexpr float kRsqrt2Pi = 0.39894228040143268f;

// The exact GELU x/2 (1 + erf(x / sqrt 2)) and its derivative Phi(x) + x phi(x)
// (kernels/include/hsn_ops.h:104-113), from the device library's erff / expf.
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * kRsqrt2)); }
__device__ __forceinline__ float gelu_grad(float x) {
    return 0.5f * (1.0f + erff(x * kRsqrt2)) + x * expf(-0.5f * x * x) * kRsqrt2Pi;
}

}  // namespace units
}  // namespace hsn
