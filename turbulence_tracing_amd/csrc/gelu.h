// GELU of the surrogate network, shared by its training and inference kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace tt {

// GELU, tanh form: 0.5 x (1 + tanh(u)), u = sqrt(2/pi) (x + 0.044715 x^3),
// evaluated as x * s with s = 0.5 (1 + tanh(u)) = 1 / (1 + exp(-2u)) and
// exp(-2u) = 2^(x (a + b x^2)), a = -2 sqrt(2/pi) log2(e), b = 0.044715 a.
// Saturates correctly: s -> 0 (exp2 -> inf) and s -> 1 (exp2 -> 0).
__device__ __forceinline__ float gelu_s(float x) {
    const float e = __builtin_amdgcn_exp2f(x * fmaf(-0.1029432395800235f, x * x, -2.302208198144325f));
    return __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu_f(float x) { return x * gelu_s(x); }
// d/dx [x s(2u)] = s + x 2 s (1 - s) u', u' = sqrt(2/pi) (1 + 3 * 0.044715 x^2)
__device__ __forceinline__ float gelu_grad(float x) {
    const float s = gelu_s(x);
    const float du = 0.7978845608028654f * fmaf(0.134145f, x * x, 1.0f);
    return fmaf(2.0f * x * s * (1.0f - s), du, s);
}

}  // namespace tt
