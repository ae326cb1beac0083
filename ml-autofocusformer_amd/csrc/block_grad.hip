// Row kernels of a transformer block's backward.  What a training step runs: the blank token's gradients (`blank_grad`) and the launch that
// adds up every kernel's partial sums (`grad_sums_kernel`).  The gradients of the GELU, of a layer norm with the residual addition ahead
// of it and of the position bias' Linear layer, and the order of the key and value gradients, are entry points that stand by themselves,
// for callers that take the products with the weights from elsewhere: a block's own backward has them inside the kernels of
// block_backward_impl.hpp, attention_train.hip and scatter_by_cluster.hip.
//
// All of them stream rows of C channels once and are bound by that.  A lane takes 8 consecutive channels (16 bytes of 16-bit
// data), C / 8 lanes a row, so that a wave holds 512 / C whole rows and row sums are a few lane exchanges; column sums stay in
// the lane's registers over all rows it takes, and every workgroup writes one partial row that `grad_sums_kernel` adds up in
// a fixed order.  No counterpart in the reference, which leaves all of it to autograd.
#include "common.hpp"
#include "gelu.hpp"
#include "launch.hpp"

namespace clusten {
namespace {

constexpr int kRowThreads = 256;

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

// g = gelu(h) and d_h = d_g gelu'(h), gelu'(v) = Phi(v) + v phi(v): the activation is made again rather than kept.
template <typename T>
__global__ __launch_bounds__(256) void gelu_backward_kernel(const T* __restrict__ h, const T* d_g, T* __restrict__ g, T* d_h, int64_t pieces) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    float v[8], d[8], y[8];
    load8(h + i * 8, v);
    load8(d_g + i * 8, d);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float slope;
        y[e] = gelu_and_slope<T>(v[e], slope);
        d[e] *= slope;
    }
    store8(g + i * 8, y);
    store8(d_h + i * 8, d);
}

// The partial sums of a workgroup's rows: lane groups that hold the same channels are added up in LDS.
template <int C>
__device__ __forceinline__ void store_partials(const float (&a)[8], const float (&b)[8], float* __restrict__ partial) {
    constexpr int LANES = C / 8, SLOTS = kRowThreads / LANES;
    __shared__ float sums[SLOTS * C];
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        if (which) __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; ++e) sums[threadIdx.x * 8 + e] = which ? b[e] : a[e];
        __syncthreads();
        for (int c = threadIdx.x; c < C; c += kRowThreads) {
            float s = 0.f;
            for (int k = 0; k < SLOTS; ++k) s += sums[k * C + c];
            partial[(int64_t)blockIdx.x * 2 * C + which * C + c] = s;
        }
    }
}

struct NormGrad {
    const void* d_y;          // (rows, C) of T: gradient of the norm's result
    const void* x;            // (rows, C) of S
    const float2* stats;      // mean, 1 / deviation
    const float* weight;
    const void* d_res;        // (rows, C) of S, or null
    void* d_x;                // (rows, C) of S
    void* branch;             // (rows, C) of T: d_x times the image's factor, or null
    const float* scale;       // (images), or null
    float* partial;           // (workgroups, 2 C)
    int64_t rows;
    int rows_per_image;
};

// d_x = d_res + rstd (g - mean(g) - xhat mean(g xhat)), g = d_y weight; sums of d_y xhat and d_y over the rows.
template <typename T, typename S, int C>
__global__ __launch_bounds__(kRowThreads) void norm_backward_kernel(NormGrad a) {
    constexpr int LANES = C / 8, ROWS = kRowThreads / LANES;
    const int c = (threadIdx.x % LANES) * 8;
    float w[8], dw[8] = {}, db[8] = {};
    load8(a.weight + c, w);
    const int64_t step = (int64_t)gridDim.x * ROWS;
    for (int64_t base = (int64_t)blockIdx.x * ROWS; base < a.rows; base += step) {
        const int64_t row = base + threadIdx.x / LANES;
        const bool live = row < a.rows;
        const int64_t at = min(row, a.rows - 1) * C + c;
        float x[8], d[8], r[8] = {};
        load8(static_cast<const S*>(a.x) + at, x);
        load8(static_cast<const T*>(a.d_y) + at, d);
        if (a.d_res) load8(static_cast<const S*>(a.d_res) + at, r);
        const float2 st = a.stats[min(row, a.rows - 1)];
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            x[e] = (x[e] - st.x) * st.y;
            if (live) dw[e] += d[e] * x[e], db[e] += d[e];
            d[e] *= w[e];
            s1 += d[e];
            s2 += d[e] * x[e];
        }
#pragma unroll
        for (int o = 1; o < LANES; o <<= 1) {
            s1 += __shfl_xor(s1, o);
            s2 += __shfl_xor(s2, o);
        }
        s1 *= 1.f / C, s2 *= 1.f / C;
#pragma unroll
        for (int e = 0; e < 8; ++e) r[e] += st.y * (d[e] - s1 - x[e] * s2);
        if (!live) continue;
        store8(static_cast<S*>(a.d_x) + at, r);
        if (a.branch) {
            const float f = a.scale ? a.scale[(uint32_t)row / (uint32_t)a.rows_per_image] : 1.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) r[e] = to_acc(from_acc<S>(r[e])) * f;
            store8(static_cast<T*>(a.branch) + at, r);
        }
    }
    store_partials<C>(dw, db, a.partial);
}

struct BlankGrad {
    const void* q;            // rows of C channels, q_stride apart
    const void* d_out;        // (rows, C)
    const float* d_logit;     // (B, H, N)
    const float* prob;        // (B, H, N)
    float* partial;
    int64_t rows;
    int q_stride, heads, tokens;
};

// Sums over the rows of d_logit q and prob d_out, each head's channels with its own factor.
template <typename T, int C>
__global__ __launch_bounds__(kRowThreads) void blank_grad_kernel(BlankGrad a) {
    constexpr int LANES = C / 8, ROWS = kRowThreads / LANES;
    const int c = (threadIdx.x % LANES) * 8, head = c / (C / a.heads);
    float dk[8] = {}, dv[8] = {};
    for (int64_t row = (int64_t)blockIdx.x * ROWS + threadIdx.x / LANES; row < a.rows; row += (int64_t)gridDim.x * ROWS) {
        const uint32_t image = (uint32_t)row / (uint32_t)a.tokens, token = (uint32_t)row - image * (uint32_t)a.tokens;
        const int64_t f = ((int64_t)image * a.heads + head) * a.tokens + token;
        const float fk = a.d_logit[f], fv = a.prob[f];
        float q[8], g[8];
        load8(static_cast<const T*>(a.q) + row * a.q_stride + c, q);
        load8(static_cast<const T*>(a.d_out) + row * C + c, g);
#pragma unroll
        for (int e = 0; e < 8; ++e) dk[e] += fk * q[e], dv[e] += fv * g[e];
    }
    store_partials<C>(dk, dv, a.partial);
}

// The sums of partial rows: 16 threads a column, 64 columns a workgroup, then a workgroup per head of a position bias layer.  Bound by the
// trips to memory of a few workgroups, 5 us however few they are: a block's backward adds its four kinds up in one launch
// at its end.  A step of AFF-Tiny at 64 images: 113 launches of 585 us, now 38 of 239 us, the
// norms that stand by themselves and the merges' scores among them.
constexpr int kPositionSums = 6;
__global__ __launch_bounds__(1024) void grad_sums_kernel(GradSums a) {
    __shared__ double shared[16 * 64 / 2];
    int at = blockIdx.x;
    for (int j = 0; j < a.columns; ++j) {
        const ColumnSums& job = a.column[j];
        const int blocks = job.C / 32;
        if (at >= blocks) {
            at -= blocks;
            continue;
        }
        float(*sums)[64] = reinterpret_cast<float(*)[64]>(shared);
        const int col = at * 64 + (threadIdx.x & 63), slice = threadIdx.x >> 6;
        float s = 0.f;
#pragma unroll 8
        for (int g = slice; g < job.groups; g += 16) s += job.partial[(int64_t)g * 2 * job.C + col];
        sums[slice][threadIdx.x & 63] = s;
        __syncthreads();
        if (slice == 0) {
            for (int k = 1; k < 16; ++k) s += sums[k][threadIdx.x];
            if (col < job.C) job.out0[col] = s * job.scale0;
            else job.out1[col - job.C] = s;
        }
        return;
    }
    const PositionSums& p = a.position;
    double s[kPositionSums] = {};
    for (int g = threadIdx.x; g < p.groups; g += 1024) {
#pragma unroll
        for (int j = 0; j < kPositionSums; ++j) s[j] += p.partial[((int64_t)g * p.heads + at) * kPositionSums + j];
    }
#pragma unroll
    for (int j = 0; j < kPositionSums; ++j) {
        for (int o = 32; o > 0; o >>= 1) s[j] += __shfl_xor(s[j], o);
        if ((threadIdx.x & 63) == 0) shared[(threadIdx.x >> 6) * kPositionSums + j] = s[j];
    }
    __syncthreads();
    if (threadIdx.x < kPositionSums) {
        double total = 0.;
        for (int w = 0; w < 16; ++w) total += shared[w * kPositionSums + threadIdx.x];
        if (threadIdx.x == kPositionSums - 1) p.d_b[at] = (float)total;
        else if ((int)threadIdx.x < p.k) p.d_w[at * p.k + threadIdx.x] = (float)total;
    }
}

// d_k and d_v (B, H, N, ch) into the key / value columns of d_qkv (B N, 3 H ch): per head ch of d_k times scale, ch of d_v.
template <typename T>
__global__ __launch_bounds__(256) void kv_columns_kernel(const T* __restrict__ d_k, const T* __restrict__ d_v, T* __restrict__ out, float scale,
                                                         int64_t pieces, int heads, int tokens, int ch) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;      // (row, head, k or v, piece of 8 channels)
    if (i >= pieces) return;
    const int per = ch / 8, p = (int)(i % per), is_v = (int)(i / per) & 1;
    const int64_t rest = i / (2 * per), row = rest / heads;
    const int head = (int)(rest % heads);
    const int64_t image = row / tokens, token = row % tokens;
    float v[8];
    load8((is_v ? d_v : d_k) + ((image * heads + head) * tokens + token) * ch + p * 8, v);
    if (!is_v) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= scale;
    }
    store8(out + row * 3 * heads * ch + heads * ch + (head * 2 + is_v) * ch + p * 8, v);
}

// d_weight (heads, k) = d^T x and d_bias (heads) for the few columns of a position bias layer: one workgroup a head.  The
// library's product for this form walks the 12 000 rows in one or two workgroups (90 us).
constexpr int kTableCols = 8;
template <typename T>
__global__ __launch_bounds__(1024) void table_linear_grad_kernel(const float* __restrict__ d, const T* __restrict__ x, float* __restrict__ d_w,
                                                                 float* __restrict__ d_b, int64_t rows, int heads, int k) {
    __shared__ float sums[16][kTableCols + 1];
    const int head = blockIdx.x;
    float s[kTableCols + 1] = {};
    for (int64_t r = threadIdx.x; r < rows; r += 1024) {
        const float g = d[r * heads + head];
#pragma unroll
        for (int j = 0; j < kTableCols; ++j) {
            if (j < k) s[j] += g * to_acc(x[r * k + j]);
        }
        s[kTableCols] += g;
    }
#pragma unroll
    for (int j = 0; j <= kTableCols; ++j) {
        for (int o = 32; o > 0; o >>= 1) s[j] += __shfl_xor(s[j], o);
        if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6][j] = s[j];
    }
    __syncthreads();
    if (threadIdx.x <= kTableCols) {
        float t = 0.f;
        for (int w = 0; w < 16; ++w) t += sums[w][threadIdx.x];
        if (threadIdx.x == kTableCols) d_b[head] = t;
        else if ((int)threadIdx.x < k) d_w[head * k + threadIdx.x] = t;
    }
}

// Workgroups for `rows` rows of C channels: four to six a compute unit are enough to keep the memory busy, and every one
// costs a partial row.
int row_groups(int64_t rows, int C) {
    const int64_t per = kRowThreads / (C / 8);
    return (int)min((rows + per - 1) / per, (int64_t)kRowSumGroups);
}

template <typename T, typename S>
int norm_backward_width(const NormGrad& a, int C, int groups, hipStream_t stream) {
    switch (C) {
        case 32: hipLaunchKernelGGL((norm_backward_kernel<T, S, 32>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 64: hipLaunchKernelGGL((norm_backward_kernel<T, S, 64>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 128: hipLaunchKernelGGL((norm_backward_kernel<T, S, 128>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 256: hipLaunchKernelGGL((norm_backward_kernel<T, S, 256>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 512: hipLaunchKernelGGL((norm_backward_kernel<T, S, 512>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
    return launch_status();
}

template <typename T>
int blank_grad_width(const BlankGrad& a, int C, int groups, hipStream_t stream) {
    switch (C) {
        case 32: hipLaunchKernelGGL((blank_grad_kernel<T, 32>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 64: hipLaunchKernelGGL((blank_grad_kernel<T, 64>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 128: hipLaunchKernelGGL((blank_grad_kernel<T, 128>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 256: hipLaunchKernelGGL((blank_grad_kernel<T, 256>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        case 512: hipLaunchKernelGGL((blank_grad_kernel<T, 512>), dim3(groups), dim3(kRowThreads), 0, stream, a); break;
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
    return launch_status();
}

}  // namespace

int launch_grad_sums(const GradSums& sums, hipStream_t stream) {
    int blocks = sums.position.heads;
    for (int j = 0; j < sums.columns; ++j) blocks += sums.column[j].C / 32;
    if (blocks == 0) return CLUSTEN_OK;
    hipLaunchKernelGGL(grad_sums_kernel, dim3((unsigned)blocks), dim3(1024), 0, stream, sums);
    return launch_status();
}

int add_up(const ColumnSums& sums, GradSums* later, hipStream_t stream) {
    GradSums now = {};
    GradSums& to = later ? *later : now;
    if (to.columns == 3) return CLUSTEN_ERR_BAD_DIMS;
    to.column[to.columns++] = sums;
    return later ? CLUSTEN_OK : launch_grad_sums(now, stream);
}

int add_up(const PositionSums& sums, GradSums* later, hipStream_t stream) {
    GradSums now = {};
    (later ? *later : now).position = sums;
    return later ? CLUSTEN_OK : launch_grad_sums(now, stream);
}

size_t row_sums_workspace_bytes(int64_t rows, int C) { return (size_t)row_groups(rows, C) * 2 * C * sizeof(float); }

int launch_gelu_backward(const void* h, const void* d_g, void* g, void* d_h, int64_t count, int dtype, hipStream_t stream) {
    const int64_t pieces = count / 8;
    const dim3 grid((unsigned)((pieces + 255) / 256));
    if (dtype == CLUSTEN_F16) {
        hipLaunchKernelGGL((gelu_backward_kernel<f16_t>), grid, dim3(256), 0, stream, static_cast<const f16_t*>(h), static_cast<const f16_t*>(d_g),
                           static_cast<f16_t*>(g), static_cast<f16_t*>(d_h), pieces);
    } else if (dtype == CLUSTEN_BF16) {
        hipLaunchKernelGGL((gelu_backward_kernel<bf16_t>), grid, dim3(256), 0, stream, static_cast<const bf16_t*>(h), static_cast<const bf16_t*>(d_g),
                           static_cast<bf16_t*>(g), static_cast<bf16_t*>(d_h), pieces);
    } else {
        hipLaunchKernelGGL((gelu_backward_kernel<float>), grid, dim3(256), 0, stream, static_cast<const float*>(h), static_cast<const float*>(d_g),
                           static_cast<float*>(g), static_cast<float*>(d_h), pieces);
    }
    return launch_status();
}

int launch_norm_backward(const void* d_y, const void* x, int x_dtype, const float* stats, const float* weight, const void* d_res, void* d_x,
                         void* branch, const float* scale, int rows_per_image, float* d_weight, float* d_bias, float* workspace, int64_t rows, int C,
                         int dtype, hipStream_t stream) {
    const NormGrad a = {d_y, x, reinterpret_cast<const float2*>(stats), weight, d_res, d_x, branch, scale, workspace, rows, rows_per_image};
    const int groups = row_groups(rows, C);
    int st;
    if (dtype == CLUSTEN_F32) st = norm_backward_width<float, float>(a, C, groups, stream);
    else if (dtype == CLUSTEN_F16) st = x_dtype == CLUSTEN_F32 ? norm_backward_width<f16_t, float>(a, C, groups, stream)
                                                                : norm_backward_width<f16_t, f16_t>(a, C, groups, stream);
    else st = x_dtype == CLUSTEN_F32 ? norm_backward_width<bf16_t, float>(a, C, groups, stream) : norm_backward_width<bf16_t, bf16_t>(a, C, groups, stream);
    return st ? st : add_up(ColumnSums{workspace, d_weight, d_bias, 1.f, groups, C}, nullptr, stream);
}

int launch_blank_grad(const void* q, int q_stride, const void* d_out, const float* d_logit, const float* prob, float scale, float* d_blank_k,
                      float* d_blank_v, float* workspace, GradSums* later, int B, int H, int N, int C, int dtype, hipStream_t stream) {
    const BlankGrad a = {q, d_out, d_logit, prob, workspace, (int64_t)B * N, q_stride, H, N};
    const int groups = row_groups(a.rows, C);
    const int st = dtype == CLUSTEN_F32 ? blank_grad_width<float>(a, C, groups, stream)
                   : dtype == CLUSTEN_F16 ? blank_grad_width<f16_t>(a, C, groups, stream) : blank_grad_width<bf16_t>(a, C, groups, stream);
    return st ? st : add_up(ColumnSums{workspace, d_blank_k, d_blank_v, scale, groups, C}, later, stream);
}

int launch_kv_columns(const void* d_k, const void* d_v, void* d_qkv, float scale, int B, int H, int N, int ch, int dtype, hipStream_t stream) {
    const int64_t pieces = (int64_t)B * N * H * 2 * (ch / 8);
    const dim3 grid((unsigned)((pieces + 255) / 256));
    if (dtype == CLUSTEN_F16) {
        hipLaunchKernelGGL((kv_columns_kernel<f16_t>), grid, dim3(256), 0, stream, static_cast<const f16_t*>(d_k), static_cast<const f16_t*>(d_v),
                           static_cast<f16_t*>(d_qkv), scale, pieces, H, N, ch);
    } else if (dtype == CLUSTEN_BF16) {
        hipLaunchKernelGGL((kv_columns_kernel<bf16_t>), grid, dim3(256), 0, stream, static_cast<const bf16_t*>(d_k), static_cast<const bf16_t*>(d_v),
                           static_cast<bf16_t*>(d_qkv), scale, pieces, H, N, ch);
    } else {
        hipLaunchKernelGGL((kv_columns_kernel<float>), grid, dim3(256), 0, stream, static_cast<const float*>(d_k), static_cast<const float*>(d_v),
                           static_cast<float*>(d_qkv), scale, pieces, H, N, ch);
    }
    return launch_status();
}

int launch_table_linear_grad(const float* d, const void* x, float* d_w, float* d_b, int64_t rows, int heads, int k, int dtype, hipStream_t stream) {
    if (dtype == CLUSTEN_F16) {
        hipLaunchKernelGGL((table_linear_grad_kernel<f16_t>), dim3(heads), dim3(1024), 0, stream, d, static_cast<const f16_t*>(x), d_w, d_b, rows, heads, k);
    } else if (dtype == CLUSTEN_BF16) {
        hipLaunchKernelGGL((table_linear_grad_kernel<bf16_t>), dim3(heads), dim3(1024), 0, stream, d, static_cast<const bf16_t*>(x), d_w, d_b, rows, heads, k);
    } else {
        hipLaunchKernelGGL((table_linear_grad_kernel<float>), dim3(heads), dim3(1024), 0, stream, d, static_cast<const float*>(x), d_w, d_b, rows, heads, k);
    }
    return launch_status();
}

}  // namespace clusten
