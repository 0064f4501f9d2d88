// Element-wise device functions shared by the ops library's kernels: the reference
// CPU backend's GELU, in forms that lose less. The library is compiled without
// FMA contraction; what is fused is written so.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#pragma clang fp contract(off)

namespace gpt_ops {

// GELU in its tanh form, 0.5 x (1 + tanh u), u = sqrt(2/pi) (x + 0.044715 x^3) with
// the constants as the reference writes them (cpu_backend.cpp:234, :281). With
// e = exp(-2|u|) and r = e / (1 + e) it is x - x r where x >= 0 and x r elsewhere,
// and its derivative 1 - r or r, plus 2 x r / (1 + e) u': no 1 + tanh or 1 - tanh^2
// whose cancellation would be left, and r, at most a half, is all that carries the
// rounding of exp. Against 64 bits, N(0, 3): 2-norm 2.1e-8 (x / (1 + exp(-2u)):
// 3.5e-8, 0.5 x (1 + tanh u): 2.8e-8), the derivative 3.6e-8 (3.6e-7, 1.4e-7).
constexpr float kGeluE = -2.88539008f * 0.79788456f;  // -2 log2(e) sqrt(2/pi)
constexpr float kGeluE3 = kGeluE * 0.044715f;
constexpr float kGeluD = 2.0f * 0.79788456f;
constexpr float kGeluD3 = 2.0f * 0.107032f;  // 2 * 3 * 0.044715 * sqrt(2/pi)

// r and 1 / (1 + e); past the largest float of x^3, e = 0.
__device__ __forceinline__ float gelu_rest(float x, float *q)
{
    const float e = __builtin_amdgcn_exp2f(-fabsf(x * fmaf(kGeluE3, x * x, kGeluE)));
    const float d = 1.0f + e, i = __builtin_amdgcn_rcpf(d);
    *q = fmaf(i, fmaf(-d, i, 1.0f), i);  // d in [1, 2]: one Newton step
    return e * *q;
}

__device__ __forceinline__ float gelu(float x)
{
    float q;
    const float r = gelu_rest(x, &q);
    // (infinity keeps its value: -FLT_MAX * 0 + inf)
    return x >= 0.0f ? fmaf(-fminf(x, 3.40282347e38f), r, x) : x * r;
}

__device__ __forceinline__ float gelu_grad(float x)
{
    float q;
    const float r = gelu_rest(x, &q);
    const float s = fmaf(x * (r * q), fmaf(kGeluD3, x * x, kGeluD), x >= 0.0f ? -r : r);
    return x >= 0.0f ? 1.0f + s : s;
}

}  // namespace gpt_ops
