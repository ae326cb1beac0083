// The exact (erf) GELU as the kernels of this library evaluate it.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace clusten {

// GELU(v) = v * Phi(v) with Phi(v) = erfc(-v / sqrt 2) / 2, and erfc(z) for z >= 0 as t * exp(-z^2 + P(t)), t = 1 / (1 + z/2),
// P a degree-9 polynomial: the classic Chebyshev fit whose fractional error stays below 1.2e-7 for every z.  No
// branches (eight of these interleave in the epilogue), and since it is erfc that is approximated to a relative
// bound the negative tail keeps its accuracy, which 0.5 * v * (1 + erf(v / sqrt 2)) loses to cancellation there:
// rounded to fp16 the result equals the exactly rounded GELU for all but a handful of the 63488 finite fp16 inputs
// (1 ulp), and differs from the erf formula only where that one is off (v < -2.5, by up to 6 ulp of values below
// 2e-4 in magnitude).  A bf16 result has fp32's range and is exactly rounded as far as fp32 reaches.  -inf gives NaN, as 0 * inf.
__device__ __forceinline__ float normal_cdf(float v) {       // Phi(v)
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
    return v < 0.f ? half_erfc : 1.f - half_erfc;
}
__device__ __forceinline__ float gelu_erf(float v) { return v * normal_cdf(v); }

// The same for fp16 results, in two thirds of the instructions: Phi(-a) = exp2(Q(a)) with Q a polynomial of degree 10 for
// log2 Phi(-a) on [0, 6.5] (minimax in log2, so the bound is relative: 1.3e-6 of Phi over the whole range, fp32 evaluation
// included; half a unit in the last place of fp16 is 4.9e-4), and GELU(v) = max(v, 0) - a Phi(-a) with a = |v|.  a stops at 6.5,
// where a Phi(-a) is 2.6e-10, below half of fp16's smallest number; bf16 goes on to 1e-38 and takes the form above.  A NaN stays one
// and -inf becomes one (0 * min(v, 0) is nothing else but for these two).  A recorded forward of 128 images: 4.89 ms, 5.00 with
// the form above.  What it is off by does not show: fc1 and GELU of the block kernels are 2.08e-4 from float64 at every width,
// 3.18e-4 as layers of their own, whose GELU reads a rounded argument.
__device__ __forceinline__ float gelu_f16(float v) {
    const float a = fminf(fabsf(v), 6.5f);
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
    return __builtin_elementwise_maximum(v, 0.f * __builtin_elementwise_minimum(v, 0.f)) - a * __builtin_amdgcn_exp2f(q);
}

// The GELU of results of type T.  For fp32 ones the fit's 1.2e-7 is more than what fp32 arithmetic leaves: over normal numbers of
// deviation 0.3 the root mean square error is 7.0e-8 of the result, 4.1e-8 with the erf formula, which costs nothing next to the fp32
// products (7.78 and 7.80 ms for a forward of 50 images).
template <typename T>
__device__ __forceinline__ float gelu_for(float v) {
    if constexpr (sizeof(T) == 4) return v * (0.5f + 0.5f * erff(0.70710678118654752440f * v));
    else if constexpr (std::is_same_v<T, f16_t>) return gelu_f16(v);
    else return gelu_erf(v);
}

// gelu(v) of results of type T, and gelu'(v) = Phi(v) + v phi(v).
template <typename T>
__device__ __forceinline__ float gelu_and_slope(float v, float& slope) {
    const float cdf = sizeof(T) == 2 ? normal_cdf(v) : 0.5f * erfcf(-0.70710678118654752440f * v);
    slope = cdf + v * 0.39894228040143267794f * __expf(-0.5f * v * v);
    return gelu_for<T>(v);
}

}  // namespace clusten
