// The table of merge weights in training, gelu(layer_norm(table W^T + b)): five columns in and four out for each of the relative positions
// (models/aff_transformer.py:343-350 before its lookup), and the gradients of its 32 parameters.
//
// Some 12 000 rows of a few operations each: bound by launches and a trip to memory.  As the framework's layers it was three launches
// forward and eight backward, among them a (4, rows) x (rows, 5) product whose library kernel takes one or two workgroups (91-117 us).
// Here a thread takes a row, the backward computes it anew, and one workgroup adds up all parameters' gradients in a fixed order: 37 us at
// 12 321 rows (fp16 operands 44), most of it the one compute unit's erfc and exp.  Kernel time of a step of AFF-Tiny at 64 images 14.93 -> 14.52 ms, launches
// 710 -> 668.
// The Linear layer's operands and result are rounded to T as under mixed precision; norm, GELU and all gradients are fp32.
#include "common.hpp"
#include "gelu.hpp"
#include "launch.hpp"

namespace clusten {
namespace {

constexpr int kIn = 5, kOut = 4, kParams = kOut * kIn + 3 * kOut;

struct Row {
    float t[kIn], h[kOut], rstd;     // operands, normalised results of the Linear layer
};

template <typename T>
__device__ __forceinline__ float rounded(float v) {
    return to_acc(from_acc<T>(v));
}

template <typename T>
__device__ __forceinline__ Row row_of(const MergeTable& a, const float (&w)[kOut][kIn], const float (&b)[kOut], int64_t row) {
    Row r;
    float y[kOut], mean = 0.f, var = 0.f;
#pragma unroll
    for (int j = 0; j < kIn; ++j) r.t[j] = rounded<T>(a.table[row * kIn + j]);
#pragma unroll
    for (int o = 0; o < kOut; ++o) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < kIn; ++j) s += r.t[j] * w[o][j];
        y[o] = rounded<T>(s + b[o]);
        mean += y[o];
    }
    mean *= 1.f / kOut;
#pragma unroll
    for (int o = 0; o < kOut; ++o) r.h[o] = y[o] - mean, var += r.h[o] * r.h[o];
    r.rstd = 1.f / sqrtf(var * (1.f / kOut) + a.eps);
#pragma unroll
    for (int o = 0; o < kOut; ++o) r.h[o] *= r.rstd;
    return r;
}

template <typename T>
__device__ __forceinline__ void parameters(const MergeTable& a, float (&w)[kOut][kIn], float (&b)[kOut]) {
#pragma unroll
    for (int o = 0; o < kOut; ++o) {
        b[o] = rounded<T>(a.bias[o]);
#pragma unroll
        for (int j = 0; j < kIn; ++j) w[o][j] = rounded<T>(a.weight[o * kIn + j]);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void merge_table_kernel(MergeTable a) {
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= a.rows) return;
    float w[kOut][kIn], b[kOut], y[kOut];
    parameters<T>(a, w, b);
    const Row r = row_of<T>(a, w, b, row);
#pragma unroll
    for (int o = 0; o < kOut; ++o) y[o] = gelu_for<float>(r.h[o] * a.norm_w[o] + a.norm_b[o]);
    *reinterpret_cast<float4*>(a.out + row * kOut) = make_float4(y[0], y[1], y[2], y[3]);
}

// d_params: d_weight (4, 5), d_bias (4), d_norm_w (4), d_norm_b (4).
template <typename T>
__global__ __launch_bounds__(1024) void merge_table_backward_kernel(MergeTable a) {
    __shared__ float sums[16][kParams];
    float w[kOut][kIn], b[kOut], nw[kOut], nb[kOut], s[kParams] = {};
    parameters<T>(a, w, b);
#pragma unroll
    for (int o = 0; o < kOut; ++o) nw[o] = a.norm_w[o], nb[o] = a.norm_b[o];
    for (int64_t row = threadIdx.x; row < a.rows; row += 1024) {
        const Row r = row_of<T>(a, w, b, row);
        const float4 d4 = *reinterpret_cast<const float4*>(a.d_out + row * kOut);
        const float d[kOut] = {d4.x, d4.y, d4.z, d4.w};
        float g[kOut], mean = 0.f, along = 0.f;
#pragma unroll
        for (int o = 0; o < kOut; ++o) {
            const float z = r.h[o] * nw[o] + nb[o];
            const float slope = 0.5f * erfcf(-0.70710678118654752440f * z) + z * 0.39894228040143267794f * expf(-0.5f * z * z);
            const float d_z = d[o] * slope;
            s[kOut * kIn + kOut + o] += d_z * r.h[o];
            s[kOut * kIn + 2 * kOut + o] += d_z;
            g[o] = d_z * nw[o];
            mean += g[o], along += g[o] * r.h[o];
        }
        mean *= 1.f / kOut, along *= 1.f / kOut;
#pragma unroll
        for (int o = 0; o < kOut; ++o) {
            const float d_y = r.rstd * (g[o] - mean - r.h[o] * along);
            s[kOut * kIn + o] += d_y;
#pragma unroll
            for (int j = 0; j < kIn; ++j) s[o * kIn + j] += d_y * r.t[j];
        }
    }
#pragma unroll
    for (int p = 0; p < kParams; ++p) {
        for (int o = 32; o > 0; o >>= 1) s[p] += __shfl_xor(s[p], o);
        if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6][p] = s[p];
    }
    __syncthreads();
    if (threadIdx.x < kParams) {
        float t = 0.f;
        for (int i = 0; i < 16; ++i) t += sums[i][threadIdx.x];
        a.d_params[threadIdx.x] = t;
    }
}

template <typename T>
int launch_typed(const MergeTable& a, bool backward, hipStream_t stream) {
    if (backward) hipLaunchKernelGGL((merge_table_backward_kernel<T>), dim3(1), dim3(1024), 0, stream, a);
    else hipLaunchKernelGGL((merge_table_kernel<T>), dim3((unsigned)((a.rows + 255) / 256)), dim3(256), 0, stream, a);
    return launch_status();
}

}  // namespace

int launch_merge_table(const MergeTable& a, bool backward, int dtype, hipStream_t stream) {
    switch (dtype) {
        case CLUSTEN_F32: return launch_typed<float>(a, backward, stream);
        case CLUSTEN_F16: return launch_typed<f16_t>(a, backward, stream);
        case CLUSTEN_BF16: return launch_typed<bf16_t>(a, backward, stream);
        default: return CLUSTEN_ERR_BAD_DTYPE;
    }
}

}  // namespace clusten
