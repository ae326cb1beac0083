// Backward of layer_norm for the norms that stand by themselves in training (patch embedding, merges, the end of the model:
// models/aff_transformer.py:362, 546, 663): d_x, d_weight and d_bias from the incoming gradient, the rows as they came in and the
// statistics the forward kept.
//
// Bound by its three streams.  A lane takes 8 consecutive channels a step (16-byte accesses), a row L lanes of V steps, so that both row
// sums are exchanges inside a wave; column sums stay in registers over all rows a lane takes and every workgroup leaves one partial row,
// added up in a fixed order.  At most 1024 workgroups, four a compute unit.  The framework ran a copy to fp32 and three kernels over fp32
// rows, one of them for the column sums alone.  Kernel time of a training step with this and the forward that keeps statistics, against
// the framework's: AFF-Tiny at 64 images, fp16 15.65 -> 14.93 ms (200 704 rows of 64 channels at the patch embedding, 50 176 of 256 and
// fewer, wider ones behind it), 24 images at 256 x 256 10.86 -> 10.43.
#include "common.hpp"
#include "launch.hpp"

namespace clusten {
namespace {

constexpr int kThreads = 256;

template <typename T>
__device__ __forceinline__ void load8(const T* p, float (&x)[8]) {
    constexpr int PER = 16 / (int)sizeof(T);
#pragma unroll
    for (int o = 0; o < 8; o += PER) {
        float v[PER];
        VecIO<T, PER>::unpack(*reinterpret_cast<const Piece*>(p + o), v);
#pragma unroll
        for (int e = 0; e < PER; ++e) x[o + e] = v[e];
    }
}
template <typename T>
__device__ __forceinline__ void store8(T* p, const float (&x)[8]) {
    constexpr int PER = 16 / (int)sizeof(T);
#pragma unroll
    for (int o = 0; o < 8; o += PER) {
        float v[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) v[e] = x[o + e];
        *reinterpret_cast<Piece*>(p + o) = VecIO<T, PER>::pack(v);
    }
}

// T: type of x and d_x, G: of the incoming gradient; C = 8 L V channels.
template <typename T, typename G, int L, int V>
__global__ __launch_bounds__(kThreads) void layer_norm_backward_kernel(const G* __restrict__ d_y, const T* __restrict__ x, const float2* __restrict__ stats,
                                                                       const float* __restrict__ weight, T* __restrict__ d_x,
                                                                       float* __restrict__ partial, int64_t rows) {
    constexpr int C = 8 * L * V, ROWS = kThreads / L;
    __shared__ float sums[ROWS * C];
    const int sub = threadIdx.x % L, slot = threadIdx.x / L;
    float w[V][8], dw[V][8] = {}, db[V][8] = {};
#pragma unroll
    for (int s = 0; s < V; ++s) load8(weight + 8 * (s * L + sub), w[s]);
    for (int64_t base = (int64_t)blockIdx.x * ROWS; base < rows; base += (int64_t)gridDim.x * ROWS) {
        const bool live = base + slot < rows;
        const int64_t row = live ? base + slot : rows - 1;      // every lane stays in the exchanges
        const float2 st = stats[row];
        float h[V][8], d[V][8], s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int s = 0; s < V; ++s) {
            load8(x + row * C + 8 * (s * L + sub), h[s]);
            load8(d_y + row * C + 8 * (s * L + sub), d[s]);
        }
#pragma unroll
        for (int s = 0; s < V; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                h[s][e] = (h[s][e] - st.x) * st.y;
                if (live) dw[s][e] += d[s][e] * h[s][e], db[s][e] += d[s][e];
                d[s][e] *= w[s][e];
                s1 += d[s][e];
                s2 += d[s][e] * h[s][e];
            }
        }
#pragma unroll
        for (int o = 1; o < L; o <<= 1) {
            s1 += __shfl_xor(s1, o);
            s2 += __shfl_xor(s2, o);
        }
        s1 *= 1.f / C, s2 *= 1.f / C;
        if (!live) continue;
#pragma unroll
        for (int s = 0; s < V; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) d[s][e] = st.y * (d[s][e] - s1 - h[s][e] * s2);
            store8(d_x + row * C + 8 * (s * L + sub), d[s]);
        }
    }
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        if (which) __syncthreads();
#pragma unroll
        for (int s = 0; s < V; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) sums[slot * C + 8 * (s * L + sub) + e] = which ? db[s][e] : dw[s][e];
        }
        __syncthreads();
        for (int c = threadIdx.x; c < C; c += kThreads) {
            float t = 0.f;
            for (int k = 0; k < ROWS; ++k) t += sums[k * C + c];
            partial[(int64_t)blockIdx.x * 2 * C + which * C + c] = t;
        }
    }
}

// Lanes a row and steps a lane.
struct Split {
    int lanes, steps;
};
Split split_of(int C) {
    switch (C) {
        case 64: return {8, 1};
        case 128: return {16, 1};
        case 256: return {32, 1};
        case 384: return {16, 3};
        case 512: return {64, 1};
        case 768: return {32, 3};
        case 1024: return {64, 2};
        default: return {0, 0};
    }
}
int groups_of(int64_t rows, int lanes) {
    const int64_t per = kThreads / lanes;
    return (int)min((rows + per - 1) / per, (int64_t)kRowSumGroups);
}

template <typename T, typename G>
int launch_typed(const void* d_y, const void* x, const float2* stats, const float* weight, void* d_x, float* partial, int64_t rows, int C,
                 hipStream_t stream) {
    const dim3 grid((unsigned)groups_of(rows, split_of(C).lanes));
#define CLUSTEN_LNB(L, V)                                                                                                                    \
    hipLaunchKernelGGL((layer_norm_backward_kernel<T, G, L, V>), grid, dim3(kThreads), 0, stream, static_cast<const G*>(d_y),                \
                       static_cast<const T*>(x), stats, weight, static_cast<T*>(d_x), partial, rows)
    switch (C) {
        case 64: CLUSTEN_LNB(8, 1); break;
        case 128: CLUSTEN_LNB(16, 1); break;
        case 256: CLUSTEN_LNB(32, 1); break;
        case 384: CLUSTEN_LNB(16, 3); break;
        case 512: CLUSTEN_LNB(64, 1); break;
        case 768: CLUSTEN_LNB(32, 3); break;
        case 1024: CLUSTEN_LNB(64, 2); break;
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
#undef CLUSTEN_LNB
    return launch_status();
}

}  // namespace

size_t layer_norm_backward_workspace_bytes(int64_t rows, int C) {
    const int lanes = split_of(C).lanes;
    return lanes && rows > 0 && rows < (int64_t)1 << 31 ? (size_t)groups_of(rows, lanes) * 2 * C * sizeof(float) : 0;
}

int launch_layer_norm_backward(const void* d_y, int dy_dtype, const void* x, int x_dtype, const float* stats_, const float* weight, void* d_x,
                               float* d_weight, float* d_bias, float* partial, int64_t rows, int C, hipStream_t stream) {
    const float2* stats = reinterpret_cast<const float2*>(stats_);
    int st = CLUSTEN_ERR_BAD_DTYPE;
    if (x_dtype == CLUSTEN_F32) {
        if (dy_dtype == CLUSTEN_F32) st = launch_typed<float, float>(d_y, x, stats, weight, d_x, partial, rows, C, stream);
        if (dy_dtype == CLUSTEN_F16) st = launch_typed<float, f16_t>(d_y, x, stats, weight, d_x, partial, rows, C, stream);
        if (dy_dtype == CLUSTEN_BF16) st = launch_typed<float, bf16_t>(d_y, x, stats, weight, d_x, partial, rows, C, stream);
    } else if (x_dtype == CLUSTEN_F16) {
        if (dy_dtype == CLUSTEN_F32) st = launch_typed<f16_t, float>(d_y, x, stats, weight, d_x, partial, rows, C, stream);
        if (dy_dtype == CLUSTEN_F16) st = launch_typed<f16_t, f16_t>(d_y, x, stats, weight, d_x, partial, rows, C, stream);
    } else if (x_dtype == CLUSTEN_BF16) {
        if (dy_dtype == CLUSTEN_F32) st = launch_typed<bf16_t, float>(d_y, x, stats, weight, d_x, partial, rows, C, stream);
        if (dy_dtype == CLUSTEN_BF16) st = launch_typed<bf16_t, bf16_t>(d_y, x, stats, weight, d_x, partial, rows, C, stream);
    }
    return st ? st : add_up(ColumnSums{partial, d_weight, d_bias, 1.f, groups_of(rows, split_of(C).lanes), C}, nullptr, stream);
}

}  // namespace clusten
