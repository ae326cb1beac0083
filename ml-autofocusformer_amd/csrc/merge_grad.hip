// Training passes of what a merge multiplies its neighbourhoods by (models/aff_transformer.py:340-358, 496-500 under autograd):
//
// merge_weights_backward, of  w[b,i,j,:] = table_w[pe_idx[b,i,j], :] * prob[b, nbhd_idx[b,i,j]] * mask[b,i,j]:  t = d_w prob mask laid out as
// (B,4,N',M), the form bias_table_grad sums into the table's rows, and d_prob by one fp32 addition per pair.  As recorded operations the
// lookup of four-value rows and its scatter went through (B N' M, 4) index tensors: 222 + 467 us a merge of AFF-Tiny at 64 images, of
// which this kernel and bias_table_grad leave some 60.
//
// row_score / row_score_backward: p = sigmoid(x w + b), one number a row, and d_z = d_p p (1 - p), d_x = d_z w, d_w = sum d_z x, d_b = sum d_z in
// one pass over the rows.  As library products the gradient of a (1, C) weight took 317 us at 200 704 rows, that of x 90 us, the bias 60.
// Bound by the rows: 2 streams forward and backward.  Neither has a counterpart in the reference's extension modules.
#include "launch.hpp"

namespace clusten {
namespace {

__global__ __launch_bounds__(256) void merge_weights_backward_kernel(const float* __restrict__ d_w, const float* __restrict__ table_w,
                                                                     const int64_t* __restrict__ pe_idx, const int64_t* __restrict__ nbhd_idx,
                                                                     const float* __restrict__ prob, const int64_t* __restrict__ mask,
                                                                     float* __restrict__ t, float* __restrict__ d_prob, int64_t pairs,
                                                                     int64_t per_image, int N, int64_t rows) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= pairs) return;
    const int64_t image = e / per_image, place = e - image * per_image;
    const float4 d = *reinterpret_cast<const float4*>(d_w + e * 4);
    const float m = mask ? (float)mask[e] : 1.f;
    float s = m;
    if (prob) {
        const int64_t nb = nbhd_idx[e];
        const bool inside = (uint64_t)nb < (uint64_t)N;      // a neighbour outside the image has no score: NaN, as in the forward
        const int64_t row = image * N + nb;
        s *= inside ? prob[row] : NAN;
        const int64_t at = pe_idx[e];
        float4 w = make_float4(NAN, NAN, NAN, NAN);          // a position outside the table
        if ((uint64_t)at < (uint64_t)rows) w = *reinterpret_cast<const float4*>(table_w + at * 4);
        if (inside && m != 0.f) unsafeAtomicAdd(d_prob + row, m * ((d.x * w.x + d.y * w.y) + (d.z * w.z + d.w * w.w)));
    }
    float* to = t + image * 4 * per_image + place;
    to[0] = d.x * s, to[per_image] = d.y * s, to[2 * per_image] = d.z * s, to[3 * per_image] = d.w * s;
}

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

// C / 8 lanes a row.
template <typename T, typename S, int C>
__global__ __launch_bounds__(kThreads) void row_score_kernel(RowScore a) {
    constexpr int LANES = C / 8, ROWS = kThreads / LANES;
    const int c = (threadIdx.x % LANES) * 8;
    const int64_t row = (int64_t)blockIdx.x * ROWS + threadIdx.x / LANES;
    float x[8], w[8], dot = 0.f;
    load8(static_cast<const S*>(a.x) + min(row, a.rows - 1) * C + c, x);
    load8(a.weight + c, w);
#pragma unroll
    for (int e = 0; e < 8; ++e) dot += to_acc(from_acc<T>(x[e])) * to_acc(from_acc<T>(w[e]));
#pragma unroll
    for (int o = 1; o < LANES; o <<= 1) dot += __shfl_xor(dot, o);
    if (row < a.rows && c == 0) {
        const float y = to_acc(from_acc<T>(dot + (a.bias ? to_acc(from_acc<T>(*a.bias)) : 0.f)));
        static_cast<T*>(a.score)[row] = from_acc<T>(1.f / (1.f + (sizeof(T) == 4 ? expf(-y) : __expf(-y))));
    }
}

template <typename T, typename S, int C>
__global__ __launch_bounds__(kThreads) void row_score_backward_kernel(RowScore a) {
    constexpr int LANES = C / 8, ROWS = kThreads / LANES;
    __shared__ float sums[kThreads * 8];
    __shared__ float totals[ROWS];
    const int c = (threadIdx.x % LANES) * 8;
    float w[8], dw[8] = {}, db = 0.f;
    load8(a.weight + c, w);
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = to_acc(from_acc<T>(w[e]));
    for (int64_t row = (int64_t)blockIdx.x * ROWS + threadIdx.x / LANES; row < a.rows; row += (int64_t)gridDim.x * ROWS) {
        float x[8], d[8];
        load8(static_cast<const S*>(a.x) + row * C + c, x);
        const float p = to_acc(static_cast<const T*>(a.score)[row]);
        const float dz = to_acc(static_cast<const T*>(a.d_score)[row]) * p * (1.f - p);
        db += dz;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            dw[e] += dz * to_acc(from_acc<T>(x[e]));
            d[e] = dz * w[e];
        }
        constexpr int PER = 16 / (int)sizeof(S);
#pragma unroll
        for (int o = 0; o < 8; o += PER) {
            float v[PER];
#pragma unroll
            for (int e = 0; e < PER; ++e) v[e] = d[o + e];
            *reinterpret_cast<Piece*>(static_cast<S*>(a.d_x) + row * C + c + o) = VecIO<S, PER>::pack(v);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) sums[threadIdx.x * 8 + e] = dw[e];
    if (c == 0) totals[threadIdx.x / LANES] = db;
    __syncthreads();
    float* partial = a.partial + (int64_t)blockIdx.x * 2 * C;
    for (int i = threadIdx.x; i < 2 * C; i += kThreads) {
        float s = 0.f;
        if (i < C) {
            for (int k = 0; k < ROWS; ++k) s += sums[k * C + i];
        } else if (i == C) {
            for (int k = 0; k < ROWS; ++k) s += totals[k];
        }
        partial[i] = s;
    }
}

template <typename T, typename S, int C>
int launch_width(const RowScore& a, hipStream_t stream) {
    const int64_t per = kThreads / (C / 8), groups = (a.rows + per - 1) / per;
    if (!a.d_x) {
        hipLaunchKernelGGL((row_score_kernel<T, S, C>), dim3((unsigned)groups), dim3(kThreads), 0, stream, a);
        return launch_status();
    }
    const int most = (int)min(groups, (int64_t)kRowSumGroups);
    hipLaunchKernelGGL((row_score_backward_kernel<T, S, C>), dim3(most), dim3(kThreads), 0, stream, a);
    if (int st = launch_status()) return st;
    return add_up(ColumnSums{a.partial, a.d_weight, a.d_bias, 1.f, most, C}, nullptr, stream);
}

template <typename T, typename S>
int launch_typed(const RowScore& a, int C, hipStream_t stream) {
    switch (C) {
        case 32: return launch_width<T, S, 32>(a, stream);
        case 64: return launch_width<T, S, 64>(a, stream);
        case 128: return launch_width<T, S, 128>(a, stream);
        case 256: return launch_width<T, S, 256>(a, stream);
        case 512: return launch_width<T, S, 512>(a, stream);
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
}

}  // namespace

int launch_merge_weights_backward(const float* d_w, const float* table_w, const int64_t* pe_idx, const int64_t* nbhd_idx, const float* prob,
                                  const int64_t* mask, float* t, float* d_prob, int B, int N, int Nout, int M, int64_t rows, hipStream_t stream) {
    const int64_t per = (int64_t)Nout * M, pairs = per * B;
    if (d_prob) {
        if (int st = launch_zero_f32(d_prob, (size_t)B * N, stream)) return st;
    }
    hipLaunchKernelGGL(merge_weights_backward_kernel, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, stream, d_w, table_w, pe_idx, nbhd_idx, prob,
                       mask, t, d_prob, pairs, per, N, rows);
    return launch_status();
}

int launch_row_score(const RowScore& a, int x_dtype, int C, int dtype, hipStream_t stream) {
    if (dtype == CLUSTEN_F32) return launch_typed<float, float>(a, C, stream);
    if (dtype == CLUSTEN_F16) return x_dtype == CLUSTEN_F32 ? launch_typed<f16_t, float>(a, C, stream) : launch_typed<f16_t, f16_t>(a, C, stream);
    return x_dtype == CLUSTEN_F32 ? launch_typed<bf16_t, float>(a, C, stream) : launch_typed<bf16_t, bf16_t>(a, C, stream);
}

}  // namespace clusten
