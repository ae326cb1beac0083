// The exact (erf) GELU as the kernels of this library evaluate it.
#pragma once

#include "common.hpp"

namespace clusten {

// GELU(v) = v * Phi(v) with Phi(v) = erfc(-v / sqrt 2) / 2, and erfc(z) for z >= 0 as t * exp(-z^2 + P(t)), t = 1 / (1 + z/2),
// P a degree-9 polynomial: the classic Chebyshev fit whose fractional error stays below 1.2e-7 for every z.  No
// branches (eight of these interleave in the epilogue), and since it is erfc that is approximated to a relative
// bound the negative tail keeps its accuracy, which 0.5 * v * (1 + erf(v / sqrt 2)) loses to cancellation there:
// rounded to fp16 the result equals the exactly rounded GELU for all but a handful of the 63488 finite fp16 inputs
// (1 ulp), and differs from the erf formula only where that one is off (v < -2.5, by up to 6 ulp of values below
// 2e-4 in magnitude).
__device__ __forceinline__ float gelu_erf(float v) {
    const float z = fabsf(v) * 0.70710678118654752440f;
    const float t = __builtin_amdgcn_rcpf(1.f + 0.5f * z);
    float p = 0.17087277f;
    p = p * t - 0.82215223f;
    p = p * t + 1.48851587f;
    p = p * t - 1.13520398f;
    p = p * t + 0.27886807f;
    p = p * t - 0.18628806f;
    p = p * t + 0.09678418f;
    p = p * t + 0.37409196f;
    p = p * t + 1.00002368f;
    p = p * t - 1.26551223f;
    const float half_erfc = 0.5f * t * __expf(p - z * z);
    return v * (v < 0.f ? half_erfc : 1.f - half_erfc);
}

// The same for results that are rounded to 16 bits, in two thirds of the instructions: Phi(-a) = exp2(Q(a)) with Q a
// polynomial of degree 10 for log2 Phi(-a) on [0, 6.5] (minimax in log2, so the bound is relative: 1.3e-6 of Phi over the
// whole range, fp32 evaluation included; half a unit in the last place of fp16 is 4.9e-4), and GELU(v) = max(v, 0) - a Phi(-a)
// with a = |v|.  a stops at 6.5, where a Phi(-a) is 2.6e-10, below half of fp16's smallest number.  No reciprocal, no
// select; a NaN stays one (`v_maximum3`).  One of the two transcendental instructions of the form above, which take four
// times an ordinary one, goes with them.
__device__ __forceinline__ float normal_tail_16bit(float a) {       // Phi(-a), 0 <= a <= 6.5
    float q = -8.44261482e-09f;
    q = q * a + 3.01195427e-07f;
    q = q * a - 4.53102646e-06f;
    q = q * a + 3.56483971e-05f;
    q = q * a - 0.000124659285f;
    q = q * a - 0.000360930182f;
    q = q * a + 0.00745342366f;
    q = q * a - 0.0528455773f;
    q = q * a - 0.459058428f;
    q = q * a - 1.15112928f;
    q = q * a - 0.999999368f;
    return __builtin_amdgcn_exp2f(q);
}
__device__ __forceinline__ float gelu_16bit(float v) {
    const float a = fminf(fabsf(v), 6.5f);
    return __builtin_elementwise_maximum(v, 0.f) - a * normal_tail_16bit(a);
}

// The GELU of a kernel whose results are stored as T.
template <typename T>
__device__ __forceinline__ float gelu_for(float v) {
    if constexpr (sizeof(T) == 2) return gelu_16bit(v);
    else return gelu_erf(v);
}

}  // namespace clusten
