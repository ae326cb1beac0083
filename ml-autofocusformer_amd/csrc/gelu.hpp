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
// 2e-4 in magnitude).  A bf16 result has fp32's range and is exactly rounded as far as fp32 reaches.  -inf gives NaN, as 0 * inf.
// Cheaper forms for 16-bit results end where fp16 does: exp2 of a polynomial of degree 10 clamped at |v| = 6.5 made a recorded
// forward of 128 images 2 % faster (4.89 against 5.00 ms) and returned -2.6e-10 for every bf16 number below -6.5.
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

// The GELU of results of type T.  For fp32 ones the fit's 1.2e-7 is more than what fp32 arithmetic leaves: over normal numbers of
// deviation 0.3 the root mean square error is 7.0e-8 of the result, 4.1e-8 with the erf formula, which costs nothing next to the fp32
// products (7.78 and 7.80 ms for a forward of 50 images).
template <typename T>
__device__ __forceinline__ float gelu_for(float v) {
    if constexpr (sizeof(T) == 2) return gelu_erf(v);
    else return v * (0.5f + 0.5f * erff(0.70710678118654752440f * v));
}

}  // namespace clusten
