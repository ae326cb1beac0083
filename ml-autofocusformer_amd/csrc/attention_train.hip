// What the training pass of an attention layer needs beside its attention kernels: the position bias of every row of the
// relative-position table, the gradients of the small Linear layer that makes it, and the global attention of a short sequence
// (models/aff_transformer.py:108-155 with every token attending to every token) forward and backward.
//
// position_bias: bias (heads, rows) = W table^T + b for the (rows, k <= 8) table, W and b rounded to the layer's type as autocast rounds them, and
// the table's rows in that type padded to 8 values, a piece that position_grad gathers.  One launch; the casts and the product were four.
//
// position_grad: d_W (heads, k) = sum d_logit[b,h,i,j] table[pe_idx[b,i,j]], d_b = sum d_logit.  The gradient of the bias of every table row
// need not be formed (a scatter into 12 000 rows, then a product over them: 23 + 20 us a layer of AFF-Tiny at 64 images, now 14 + 5): a
// value meets its row of the table directly.  Every lane sums in double, so that nothing is lost where positive and negative values cancel;
// partial sums, doubles too, are added in a fixed order.  The same holds for these sums of global attention below.
//
// dense_attention_train / _backward: one workgroup per image and head, everything in LDS as fp32, fp32 arithmetic on the vector unit: 49
// tokens of 32 channels are 0.3 MFLOP a product, and the five products of a backward are bound by the reads of their operands from LDS.
// As library operations the layer took 25 launches a direction; 64 images of 49
// tokens and 16 heads fp16 now take 28 us forward and 71 us backward, 11 of them the sums over the images.  Probabilities are made again in the backward, as in the forward.
// None of it has a counterpart in the reference's extension modules.
#include "launch.hpp"

namespace clusten {
namespace {

constexpr int kTableCols = 8;

template <typename T>
__global__ __launch_bounds__(256) void position_bias_kernel(const float* __restrict__ table, const float* __restrict__ w,
                                                            const float* __restrict__ b, T* __restrict__ bias, T* __restrict__ padded, int rows,
                                                            int heads, int k) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * heads) return;
    const int head = i / rows, row = i - head * rows;
    float s = 0.f;
    for (int j = 0; j < k; ++j) s += to_acc(from_acc<T>(table[(int64_t)row * k + j])) * to_acc(from_acc<T>(w[head * k + j]));
    if (b) s += to_acc(from_acc<T>(b[head]));
    bias[(int64_t)head * rows + row] = from_acc<T>(s);
    if (padded && head == 0) {
        for (int j = 0; j < kTableCols; ++j) padded[(int64_t)row * kTableCols + j] = from_acc<T>(j < k ? table[(int64_t)row * k + j] : 0.f);
    }
}

template <typename T>
__device__ __forceinline__ void table_row(const T* __restrict__ padded, int64_t row, float (&t)[kTableCols]) {
    constexpr int PER = 16 / (int)sizeof(T);
#pragma unroll
    for (int o = 0; o < kTableCols; o += PER) {
        float v[PER];
        VecIO<T, PER>::unpack(*reinterpret_cast<const Piece*>(padded + row * kTableCols + o), v);
#pragma unroll
        for (int e = 0; e < PER; ++e) t[o + e] = v[e];
    }
}

constexpr int kGradHeads = 4;      // heads a workgroup of position_grad sums for
constexpr int kGradSums = 6;       // of a head: five columns and the bias

// Bound by the trips to memory of an index and its table row, and in a small launch by the exchanges at the end.  Mean of a layer of AFF-Tiny at 64
// images: 24.2 -> 14.0 us with the next indices requested ahead, fewer exchanges and four workgroups a compute unit instead of two.
// Workgroup (x, y): values x, x + gridDim.x, ... (in 256 quads) of heads 4 y ..; partial: (gridDim.x, heads, 6) doubles.
template <typename T>
__global__ __launch_bounds__(256) void position_grad_kernel(const T* __restrict__ d_logit, const int64_t* __restrict__ pe_idx,
                                                            const T* __restrict__ padded, double* __restrict__ partial, int heads, int64_t per_image,
                                                            int64_t total, int rows) {
    __shared__ double sums[4][kGradHeads * kGradSums];
    const int h0 = blockIdx.y * kGradHeads, here = min(kGradHeads, heads - h0);
    double acc[kGradHeads][kGradSums] = {};
    const int64_t quads = total / 4, step = (int64_t)gridDim.x * 256;
    int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x, row[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) row[e] = pe_idx[min(q, quads - 1) * 4 + e];
    for (; q < quads; q += step) {
        const int64_t at = q * 4, image = at / per_image, place = at - image * per_image;
        float t[4][kTableCols];
#pragma unroll
        for (int e = 0; e < 4; ++e) table_row(padded, min((uint64_t)row[e], (uint64_t)(rows - 1)), t[e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) row[e] = pe_idx[min(q + step, quads - 1) * 4 + e];      // the next quad's, while this one's rows travel
#pragma unroll
        for (int h = 0; h < kGradHeads; ++h) {
            if (h < here) {
                float d[4];
                Quad<T>::unpack(*reinterpret_cast<const typename Quad<T>::raw*>(d_logit + (image * heads + h0 + h) * per_image + place), d);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
#pragma unroll
                    for (int j = 0; j < kGradSums - 1; ++j) acc[h][j] += (double)d[e] * (double)t[e][j];
                    acc[h][kGradSums - 1] += (double)d[e];
                }
            }
        }
    }
    // sums over the wave: at each exchange a lane keeps half of its values and gives the other half away, value i ends in lanes 2 i and 2 i + 1
    // (32 exchanges of a double; 144 when every lane keeps all 24, which took longer than the values of a deep layer)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double v[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) v[j] = j < kGradHeads * kGradSums ? acc[j / kGradSums % kGradHeads][j % kGradSums] : 0.;
#pragma unroll
    for (int half = 16; half > 0; half >>= 1) {
        const bool upper = (lane & 2 * half) != 0;
#pragma unroll
        for (int j = 0; j < half; ++j) {
            const double kept = upper ? v[j + half] : v[j], given = upper ? v[j] : v[j + half];
            v[j] = kept + __shfl_xor(given, 2 * half);
        }
    }
    v[0] += __shfl_xor(v[0], 1);
    if ((lane & 1) == 0 && lane / 2 < kGradHeads * kGradSums) sums[wave][lane / 2] = v[0];
    __syncthreads();
    if ((int)threadIdx.x < here * kGradSums) {
        double s = 0.;
        for (int w = 0; w < 4; ++w) s += sums[w][threadIdx.x];
        partial[((int64_t)blockIdx.x * heads + h0) * kGradSums + threadIdx.x] = s;
    }
}

// ---- global attention of up to 64 tokens ----------------------------------------------------------------------------------

constexpr int kTokens = 64, kCh = 32, kPitch = kCh + 4, kSPitch = kTokens + 4;     // pitches in floats: 16-byte rows, spread over the banks
constexpr int kDenseThreads = 256;
constexpr int kDenseSums = 2 * kCh + kGradSums;      // partial sums of an image and head: blank key, blank value, position bias layer
constexpr int kDensePitch = 2 * kCh + 2 * kGradSums; // their floats: the last kind in double, from which an even place starts
static_assert(kCh % 2 == 0 && kDensePitch % 2 == 0, "doubles on 8-byte boundaries");

template <typename T>
__device__ __forceinline__ void rows_to_lds(const T* __restrict__ src, int64_t pitch, int n, float* dst) {
    constexpr int PER = 16 / (int)sizeof(T), PIECES = kCh / PER;
    for (int i = threadIdx.x; i < kTokens * PIECES; i += kDenseThreads) {
        const int row = i / PIECES, c = (i % PIECES) * PER;
        float v[PER] = {};
        if (row < n) VecIO<T, PER>::unpack(*reinterpret_cast<const Piece*>(src + row * pitch + c), v);
#pragma unroll
        for (int e = 0; e < PER; ++e) dst[row * kPitch + c + e] = v[e];
    }
}

// out[4][4] = rows 4 ty .. of a times rows 4 tx .. of b, over the channels.
__device__ __forceinline__ void row_products(const float* a, const float* b, int ty, int tx, float (&out)[4][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[i][j] = 0.f;
    }
#pragma unroll 2
    for (int c = 0; c < kCh; c += 4) {
        float4 x[4], y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const float4*>(a + (4 * ty + i) * kPitch + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = *reinterpret_cast<const float4*>(b + (tx + 16 * j) * kPitch + c);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) out[i][j] += x[i].x * y[j].x + x[i].y * y[j].y + x[i].z * y[j].z + x[i].w * y[j].w;
        }
    }
}

// out[2][4] = sum over k < n of m[k][2 ty ..] (transposed) or m[2 ty ..][k] times rows k, channels 4 tx .., of x.
template <bool TRANSPOSED>
__device__ __forceinline__ void weighted_rows(const float* m, const float* x, int n, int ty, int tx, float (&out)[2][4]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) out[i][e] = 0.f;
    }
#pragma unroll 4
    for (int k = 0; k < n; ++k) {
        const float4 v = *reinterpret_cast<const float4*>(x + k * kPitch + 4 * tx);
        float w[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) w[i] = TRANSPOSED ? m[k * kSPitch + 2 * ty + i] : m[(2 * ty + i) * kSPitch + k];
#pragma unroll
        for (int i = 0; i < 2; ++i) out[i][0] += w[i] * v.x, out[i][1] += w[i] * v.y, out[i][2] += w[i] * v.z, out[i][3] += w[i] * v.w;
    }
}

// exp for results of type T.  The short form rounds its argument times log2 e to fp32: 2e-6 of the result 50 below the maximum, which
// 16-bit results do not show and fp32 ones do.
template <typename T>
__device__ __forceinline__ float exponential(float x) {
    return sizeof(T) == 4 ? expf(x) : __expf(x);
}

// Probabilities of the rows and of the blank token (p, blank) from q, k in LDS.
template <typename T>
__device__ __forceinline__ void probabilities(const DenseTrain& a, int image, int head, const float* q, const float* k, float* p, float* blank) {
    const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
    float s[4][4];
    row_products(q, k, ty, tx, s);
    const T* bias = static_cast<const T*>(a.bias) + (int64_t)head * a.rows;
    const int64_t* pe = a.pe_idx + (int64_t)image * a.N * a.N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = 4 * ty + i, col = tx + 16 * j;
            float v = -INFINITY;
            if (row < a.N && col < a.N) v = s[i][j] * a.scale + to_acc(bias[min((uint64_t)pe[row * a.N + col], (uint64_t)(a.rows - 1))]);
            p[row * kSPitch + col] = v;
        }
    }
    __syncthreads();
    // four lanes a row
    const int row = threadIdx.x >> 2, part = threadIdx.x & 3;
    float z = 0.f;
#pragma unroll
    for (int c = 0; c < kCh / 4; ++c) z += q[row * kPitch + part * (kCh / 4) + c] * a.blank_k[head * kCh + part * (kCh / 4) + c];
    z += __shfl_xor(z, 1);
    z += __shfl_xor(z, 2);
    z *= a.scale;
    float top = z, v[kTokens / 4];
#pragma unroll
    for (int c = 0; c < kTokens / 4; ++c) v[c] = p[row * kSPitch + part + 4 * c], top = fmaxf(top, v[c]);
    top = fmaxf(top, __shfl_xor(top, 1));
    top = fmaxf(top, __shfl_xor(top, 2));
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < kTokens / 4; ++c) v[c] = exponential<T>(v[c] - top), sum += v[c];
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);
    z = exponential<T>(z - top);
    const float inv = 1.f / (sum + z);
#pragma unroll
    for (int c = 0; c < kTokens / 4; ++c) p[row * kSPitch + part + 4 * c] = v[c] * inv;
    if (part == 0) blank[row] = z * inv;
    __syncthreads();
}

template <typename T>
__global__ __launch_bounds__(kDenseThreads) void dense_train_kernel(DenseTrain a) {
    __shared__ __attribute__((aligned(16))) float q[kTokens * kPitch], k[kTokens * kPitch], v[kTokens * kPitch], p[kTokens * kSPitch], blank[kTokens];
    const int image = blockIdx.x / a.H, head = blockIdx.x - image * a.H, C = a.H * kCh;
    const T* rows = static_cast<const T*>(a.qkv) + (int64_t)image * a.N * 3 * C;
    rows_to_lds(rows + head * kCh, 3 * C, a.N, q);
    rows_to_lds(rows + C + head * 2 * kCh, 3 * C, a.N, k);
    rows_to_lds(rows + C + (head * 2 + 1) * kCh, 3 * C, a.N, v);
    __syncthreads();
    probabilities<T>(a, image, head, q, k, p, blank);
    const int ty = threadIdx.x >> 3, tx = threadIdx.x & 7;
    float o[2][4];
    weighted_rows<false>(p, v, a.N, ty, tx, o);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = 2 * ty + i;
        if (row < a.N) {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[i][e] += blank[row] * a.blank_v[head * kCh + 4 * tx + e];
            T* to = static_cast<T*>(a.out) + ((int64_t)image * a.N + row) * C + head * kCh + 4 * tx;
            *reinterpret_cast<typename Quad<T>::raw*>(to) = Quad<T>::pack(o[i]);
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kDenseThreads) void dense_train_backward_kernel(DenseTrain a) {
    __shared__ __attribute__((aligned(16))) float q[kTokens * kPitch], k[kTokens * kPitch], v[kTokens * kPitch], g[kTokens * kPitch];
    __shared__ __attribute__((aligned(16))) float p[kTokens * kSPitch], ds[kTokens * kSPitch], blank[kTokens], d_blank[kTokens];
    __shared__ double sums[4][kGradSums];
    const int image = blockIdx.x / a.H, head = blockIdx.x - image * a.H, C = a.H * kCh;
    const T* rows = static_cast<const T*>(a.qkv) + (int64_t)image * a.N * 3 * C;
    rows_to_lds(rows + head * kCh, 3 * C, a.N, q);
    rows_to_lds(rows + C + head * 2 * kCh, 3 * C, a.N, k);
    rows_to_lds(rows + C + (head * 2 + 1) * kCh, 3 * C, a.N, v);
    rows_to_lds(static_cast<const T*>(a.d_out) + (int64_t)image * a.N * C + head * kCh, C, a.N, g);
    __syncthreads();
    probabilities<T>(a, image, head, q, k, p, blank);
    {
        float d[4][4];
        const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
        row_products(g, v, ty, tx, d);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) ds[(4 * ty + i) * kSPitch + tx + 16 * j] = d[i][j];
        }
    }
    __syncthreads();
    double pos[kGradSums] = {};
    {
        // d_logit = p (d_p - sum p d_p), four lanes a row; the position bias layer's gradients on the way
        const int row = threadIdx.x >> 2, part = threadIdx.x & 3;
        float z = 0.f;
#pragma unroll
        for (int c = 0; c < kCh / 4; ++c) z += g[row * kPitch + part * (kCh / 4) + c] * a.blank_v[head * kCh + part * (kCh / 4) + c];
        z += __shfl_xor(z, 1);
        z += __shfl_xor(z, 2);
        float dot = 0.f;
#pragma unroll
        for (int c = 0; c < kTokens / 4; ++c) dot += p[row * kSPitch + part + 4 * c] * ds[row * kSPitch + part + 4 * c];
        dot += __shfl_xor(dot, 1);
        dot += __shfl_xor(dot, 2);
        dot += blank[row] * z;
        if (part == 0) d_blank[row] = blank[row] * (z - dot);
        const int64_t* pe = a.pe_idx + (int64_t)image * a.N * a.N;
#pragma unroll 4
        for (int c = 0; c < kTokens / 4; ++c) {
            const int col = part + 4 * c;
            const float d = p[row * kSPitch + col] * (ds[row * kSPitch + col] - dot);
            ds[row * kSPitch + col] = d;
            if (row < a.N && col < a.N) {
                float t[kTableCols];
                table_row(static_cast<const T*>(a.padded), (int64_t)min((uint64_t)pe[row * a.N + col], (uint64_t)(a.rows - 1)), t);
#pragma unroll
                for (int j = 0; j < kGradSums - 1; ++j) pos[j] += (double)d * (double)t[j];
                pos[kGradSums - 1] += (double)d;
            }
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < kGradSums; ++j) {
        for (int o = 32; o > 0; o >>= 1) pos[j] += __shfl_xor(pos[j], o);
        if (lane == 0) sums[wave][j] = pos[j];
    }
    __syncthreads();
    float* partial = a.partial + (int64_t)blockIdx.x * kDensePitch;
    const int ty = threadIdx.x >> 3, tx = threadIdx.x & 7;
    T* to = static_cast<T*>(a.d_qkv) + (int64_t)image * a.N * 3 * C;
    const auto store = [&](const float (&x)[2][4], int column, float scale) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = 2 * ty + i;
            if (row < a.N) {
                const float y[4] = {x[i][0] * scale, x[i][1] * scale, x[i][2] * scale, x[i][3] * scale};
                *reinterpret_cast<typename Quad<T>::raw*>(to + (int64_t)row * 3 * C + column + 4 * tx) = Quad<T>::pack(y);
            }
        }
    };
    float x[2][4];
    weighted_rows<false>(ds, k, a.N, ty, tx, x);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[i][e] += d_blank[2 * ty + i] * a.blank_k[head * kCh + 4 * tx + e];
    }
    store(x, head * kCh, a.scale);
    weighted_rows<true>(ds, q, a.N, ty, tx, x);
    store(x, C + head * 2 * kCh, a.scale);
    weighted_rows<true>(p, g, a.N, ty, tx, x);
    store(x, C + (head * 2 + 1) * kCh, 1.f);
    if (threadIdx.x < 2 * kCh) {
        const float* m = threadIdx.x < kCh ? q : g;
        const float* f = threadIdx.x < kCh ? d_blank : blank;
        float s = 0.f;
        for (int r = 0; r < a.N; ++r) s += f[r] * m[r * kPitch + (threadIdx.x & (kCh - 1))];
        partial[threadIdx.x] = threadIdx.x < kCh ? s * a.scale : s;
    } else if (threadIdx.x < kDenseSums) {
        const int j = threadIdx.x - 2 * kCh;
        reinterpret_cast<double*>(partial + 2 * kCh)[j] = (sums[0][j] + sums[1][j]) + (sums[2][j] + sums[3][j]);
    }
}

// One workgroup a head: the sums of its images' partial rows.
__global__ __launch_bounds__(256) void dense_sums_kernel(const float* __restrict__ partial, int images, int heads, int k, float* __restrict__ d_bk,
                                                         float* __restrict__ d_bv, float* __restrict__ d_w, float* __restrict__ d_b) {
    __shared__ double sums[2][128];
    const int head = blockIdx.x, col = threadIdx.x & 127, half = threadIdx.x >> 7;
    double s = 0.;
    if (col < kDenseSums) {
        for (int b = half; b < images; b += 2) {
            const float* row = partial + ((int64_t)b * heads + head) * kDensePitch;
            s += col < 2 * kCh ? (double)row[col] : reinterpret_cast<const double*>(row + 2 * kCh)[col - 2 * kCh];
        }
    }
    sums[half][col] = s;
    __syncthreads();
    if (half == 0 && col < kDenseSums) {
        const float t = (float)(sums[0][col] + sums[1][col]);
        if (col < kCh) d_bk[head * kCh + col] = t;
        else if (col < 2 * kCh) d_bv[head * kCh + col - kCh] = t;
        else if (col - 2 * kCh < k) d_w[head * k + col - 2 * kCh] = t;
        else if (col == kDenseSums - 1) d_b[head] = t;
    }
}

// Workgroups of position_grad: four fit a compute unit, and a thread takes at least two quads of values, else its last exchanges are the
// larger part.
int position_groups(int64_t total) { return (int)max((int64_t)1, min((total / 4 + 511) / 512, (int64_t)1024)); }

template <typename F>
int on_type(int dtype, F&& f) {
    switch (dtype) {
        case CLUSTEN_F32: f(float()); break;
        case CLUSTEN_F16: f(f16_t()); break;
        case CLUSTEN_BF16: f(bf16_t()); break;
        default: return CLUSTEN_ERR_BAD_DTYPE;
    }
    return launch_status();
}

}  // namespace

int launch_position_bias(const float* table, const float* w, const float* b, void* bias, void* padded, int rows, int heads, int k, int dtype,
                         hipStream_t stream) {
    return on_type(dtype, [&](auto t) {
        typedef decltype(t) T;
        hipLaunchKernelGGL((position_bias_kernel<T>), dim3((unsigned)(((int64_t)rows * heads + 255) / 256)), dim3(256), 0, stream, table, w, b,
                           static_cast<T*>(bias), static_cast<T*>(padded), rows, heads, k);
    });
}

size_t position_grad_workspace_bytes(int64_t total, int heads) { return (size_t)position_groups(total) * heads * kGradSums * sizeof(double); }

int launch_position_grad(const void* d_logit, const int64_t* pe_idx, const void* padded, float* d_w, float* d_b, void* workspace, GradSums* later, int B,
                         int H, int N, int M, int rows, int k, int dtype, hipStream_t stream) {
    const int64_t per_image = (int64_t)N * M, total = B * per_image;
    const int groups = position_groups(total);
    double* partial = static_cast<double*>(workspace);
    const int st = on_type(dtype, [&](auto t) {
        typedef decltype(t) T;
        hipLaunchKernelGGL((position_grad_kernel<T>), dim3(groups, (H + kGradHeads - 1) / kGradHeads), dim3(256), 0, stream,
                           static_cast<const T*>(d_logit), pe_idx, static_cast<const T*>(padded), partial, H, per_image, total, rows);
    });
    return st ? st : add_up(PositionSums{partial, d_w, d_b, groups, H, k}, later, stream);
}

size_t dense_train_workspace_bytes(int B, int H) { return (size_t)B * H * kDensePitch * sizeof(float); }

int launch_dense_train(const DenseTrain& a, int dtype, hipStream_t stream) {
    return on_type(dtype, [&](auto t) {
        hipLaunchKernelGGL((dense_train_kernel<decltype(t)>), dim3((unsigned)(a.B * a.H)), dim3(kDenseThreads), 0, stream, a);
    });
}

int launch_dense_train_backward(const DenseTrain& a, float* d_bk, float* d_bv, float* d_w, float* d_b, int dtype, hipStream_t stream) {
    const int st = on_type(dtype, [&](auto t) {
        hipLaunchKernelGGL((dense_train_backward_kernel<decltype(t)>), dim3((unsigned)(a.B * a.H)), dim3(kDenseThreads), 0, stream, a);
    });
    if (st) return st;
    hipLaunchKernelGGL(dense_sums_kernel, dim3(a.H), dim3(256), 0, stream, a.partial, a.B, a.H, a.k, d_bk, d_bv, d_w, d_b);
    return launch_status();
}

}  // namespace clusten
