// weight_grad: the parameter gradients of Linear layers, d_W = d_Y^T X and d_b = the column sums of d_Y, for up to eight
// layers over the same token rows in two launches.
//
// The products of the reference model's backward whose contraction runs over the tokens (models/aff_transformer.py:103-106,
// 157, 181-196 under autograd): a result of 64 x 64 to 2048 x 512 from up to 200 000 rows.  A library product takes tiles of
// the result as its unit of work - 12 workgroups for a 192 x 64 gradient on 256 compute units - and the bias is a reduction
// of its own over the same rows: 24 + 3.6 ms of a 76 ms training step of AFF-Tiny at batch 64.  Here every tile of the result is
// also cut along the rows, so that about two workgroups per compute unit run whatever the layer's size; their fp32 sums go
// to a workspace, and a second kernel adds them in a fixed order (no atomics: a gradient repeats bit for bit).  The bias
// falls out of the same pass: one more matrix instruction per d_Y fragment, against ones.
//
// A workgroup is four waves and stages rows x 64 (or 128) columns of both operands, row-major as they are in memory, by
// LDS-direct loads, the next stage on its way while this one is multiplied.  Both operands have the contraction along the
// rows, so the 16-bit fragments are read by `ds_read_b64_tr_b16`; a fragment's k slots are any eight rows as long as both
// operands agree, and the 32-byte blocks of a staged row are rotated by its number, which makes these reads conflict free.
// Layers whose sides are multiples of 128 take 128 x 128 tiles, a quarter per wave; others 64 x 64 tiles with the rows of a
// stage dealt to the waves (and their sums added in LDS at the end): a wave owns 64 x 64 either way, half a fragment read per
// matrix instruction.  200 704 rows, 192 x 64 fp16: 148 us + 20 us for the bias as library kernels.
// It has no counterpart in the reference's extension modules.
#include "launch.hpp"
#include "mfma.hpp"

namespace clusten {
namespace {

constexpr int kItems = 8;
constexpr int kThreads = 256;
constexpr int kStageBytes = 32 * 1024;
constexpr int kSegments = 2 * kItems;

struct Item {
    const void* dy;
    const void* x;
    int64_t ld_dy, ld_x;
    int64_t at, bias_at;       // offsets of the layer's sums within a split's block of the workspace; bias_at < 0: none
    int n, k, tiles_k, first_tile;
};
struct GradArgs {
    Item item[kItems];
    float* sums;
    int64_t per_split;
    int64_t rows;
    int64_t rows_per_split;    // a multiple of the rows of a stage
    int count, tiles, splits;
};

template <typename T, int TILE>
struct Stage {
    static constexpr int kElem = 16 / (int)sizeof(T);                 // elements of a piece
    static constexpr int kRowBytes = TILE * (int)sizeof(T);
    static constexpr int kRows = kStageBytes / (2 * kRowBytes);
    static constexpr int kPieces = kRowBytes / 16;                    // of a row
    static constexpr int kBlockBytes = 16 * (int)sizeof(T);           // 16 columns: what a fragment takes of a row
    static constexpr int kOperandBytes = kRows * kRowBytes;
    // rotation of a row's blocks: fragment reads of eight (16-bit) or four (fp32) rows then cover all banks once
    static __device__ __forceinline__ int turn(int row) {
        if (sizeof(T) == 4) return row & 3;
        return TILE == 64 ? (row >> 1) & 3 : row & 7;
    }
};

template <typename T, int TILE>
__device__ __forceinline__ void stage_operand(const T* base, int64_t ld, int64_t row0, int64_t last_row, int col0, int cols,
                                              char* lds, int wave, int lane) {
    typedef Stage<T, TILE> S;
    constexpr int ROWS_PER_LOAD = 64 / S::kPieces, LOADS = S::kRows / ROWS_PER_LOAD, BLOCK_PIECES = S::kBlockBytes / 16;
    const int p = lane % S::kPieces;
    const T* src = base + row0 * ld;
    const int last = (int)min(last_row - row0, (int64_t)S::kRows);
#pragma unroll
    for (int i = 0; i < LOADS / 4; ++i) {
        const int load = wave * (LOADS / 4) + i;
        const int row = load * ROWS_PER_LOAD + lane / S::kPieces;
        const int piece = ((p / BLOCK_PIECES) ^ S::turn(row)) * BLOCK_PIECES + p % BLOCK_PIECES;
        const int col = min(col0 + piece * S::kElem, cols - S::kElem);
        CLUSTEN_LDS_DMA16(src + (int64_t)min(row, last) * ld + col, lds + load * 1024);
    }
}

// 64 columns from 16 * block0 on as fragments of step `step`: lane (r16, kq) gets column r16 of block cb.
template <typename T, int TILE>
__device__ __forceinline__ void fragments(const char* lds, int step_row, int block0, int r16, int kq, Piece (&f)[4]) {
    typedef Stage<T, TILE> S;
    if constexpr (sizeof(T) == 2) {
        typedef short S4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) S4* LdsS4;
        const int row = 4 * kq + (r16 >> 2);
        const char* at = lds + (step_row + row) * S::kRowBytes + (r16 & 3) * 8;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const char* a = at + ((block0 + cb) ^ S::turn(row)) * S::kBlockBytes;
            const U32x2 lo = __builtin_bit_cast(U32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS4)a));
            const U32x2 hi = __builtin_bit_cast(U32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS4)(a + 16 * S::kRowBytes)));
            f[cb] = Piece{lo[0], lo[1], hi[0], hi[1]};
        }
    } else {
        // four steps of four rows: word e of the piece is row 4 e + kq
        const float* at = reinterpret_cast<const float*>(lds + (step_row + kq) * S::kRowBytes);
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const int col = ((block0 + cb) ^ S::turn(kq)) * 16 + r16;
#pragma unroll
            for (int e = 0; e < 4; ++e) f[cb][e] = __float_as_uint(at[4 * e * TILE + col]);
        }
    }
}

template <typename T>
__device__ __forceinline__ Piece ones() {
    const uint32_t w = storage_bits(from_acc<T>(1.f));
    const uint32_t both = sizeof(T) == 4 ? w : w | w << 16;
    return Piece{both, both, both, both};
}

template <typename T, int TILE>
__global__ __launch_bounds__(kThreads, 2) void weight_grad_kernel(GradArgs a) {
    typedef Stage<T, TILE> S;
    constexpr int WAVE_ROWS = TILE == 64 ? 4 : 1;              // waves that share the rows of a stage
    constexpr int STEP = sizeof(T) == 2 ? 32 : 16;             // rows of a fragment
    constexpr int STEPS = S::kRows / WAVE_ROWS / STEP;
    static_assert(STEPS >= 1, "a step per wave and stage");
    __shared__ __attribute__((aligned(1024))) char stage[2 * kStageBytes];

    const int unit = xcd_tile(blockIdx.x, a.tiles * a.splits);
    if (unit < 0) return;
    const int split = unit / a.tiles, tile = unit - split * a.tiles;     // tiles of one range of rows side by side: one XCD's L2
    int which = 0;
    while (which + 1 < a.count && tile >= a.item[which + 1].first_tile) ++which;
    const Item it = a.item[which];
    const int tn = (tile - it.first_tile) / it.tiles_k, tk = (tile - it.first_tile) % it.tiles_k;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int n0 = tn * TILE, k0 = tk * TILE;
    const int wn = TILE == 64 ? 0 : wave >> 1, wk = TILE == 64 ? 0 : wave & 1;      // the wave's 64 x 64 of the tile
    const int64_t first = (int64_t)split * a.rows_per_split, end = min(a.rows, first + a.rows_per_split);
    const bool with_bias = it.bias_at >= 0 && tk == 0 && wk == 0;
    const T* dy = static_cast<const T*>(it.dy);
    const T* x = static_cast<const T*>(it.x);

    F32x4 acc[4][4], acc_b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        acc_b[i] = F32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = F32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto fetch = [&](int64_t row, int slot) {
        char* to = stage + slot * kStageBytes;
        stage_operand<T, TILE>(dy, it.ld_dy, row, end - 1, n0, it.n, to, wave, lane);
        stage_operand<T, TILE>(x, it.ld_x, row, end - 1, k0, it.k, to + S::kOperandBytes, wave, lane);
    };
    auto barrier = [&]() {
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    if (first < end) fetch(first, 0);
    int slot = 0;
    for (int64_t row = first; row < end; row += S::kRows, slot ^= 1) {
        lds_sync_vm<0>();            // this wave's share of the stage is there, and it has read the stage before
        barrier();
        char* here = stage + slot * kStageBytes;
        if (row + S::kRows < end) fetch(row + S::kRows, slot ^ 1);
        const int valid = (int)min(end - row, (int64_t)S::kRows);
        if (valid < S::kRows) {      // the last stage: rows past the end count nothing
            for (int i = valid * S::kRowBytes + (int)threadIdx.x * 16; i < S::kOperandBytes; i += kThreads * 16) {
                *reinterpret_cast<Piece*>(here + i) = Piece{0, 0, 0, 0};
                *reinterpret_cast<Piece*>(here + S::kOperandBytes + i) = Piece{0, 0, 0, 0};
            }
            lds_sync();
            barrier();
        }
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int step_row = ((TILE == 64 ? wave * STEPS : 0) + s) * STEP;
            Piece fy[4], fx[4];
            fragments<T, TILE>(here, step_row, 4 * wn, r16, kq, fy);
            fragments<T, TILE>(here + S::kOperandBytes, step_row, 4 * wk, r16, kq, fx);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = tile_mfma<T>(fx[j], fy[i], acc[i][j]);
            }
            if (with_bias) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc_b[i] = tile_mfma<T>(ones<T>(), fy[i], acc_b[i]);
            }
        }
    }

    // lane: row n = 16 i + r16 of the wave's 64 x 64, columns k = 16 j + 4 kq .. + 3
    float* sums = a.sums + (int64_t)split * a.per_split;
    if constexpr (TILE == 64) {
        lds_sync();
        barrier();
        F32x4* part = reinterpret_cast<F32x4*>(stage);                       // [wave][i][j][lane]
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) part[((wave * 4 + i) * 4 + j) * 64 + lane] = acc[i][j];
        }
        lds_sync();
        barrier();
        // wave i adds the four shares of rows 16 i .. 16 i + 15
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            F32x4 v = part[(wave * 4 + j) * 64 + lane];
#pragma unroll
            for (int w = 1; w < 4; ++w) v += part[((w * 4 + wave) * 4 + j) * 64 + lane];
            const int n = n0 + 16 * wave + r16, k = k0 + 16 * j + 4 * kq;
            if (n < it.n && k < it.k) *reinterpret_cast<F32x4*>(sums + it.at + (int64_t)n * it.k + k) = v;
        }
        if (with_bias) {             // uniform over the workgroup here
            lds_sync();
            barrier();
            float* pb = reinterpret_cast<float*>(stage);
            if (kq == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) pb[wave * 64 + 16 * i + r16] = acc_b[i][0];
            }
            lds_sync();
            barrier();
            const int n = n0 + lane;
            if (wave == 0 && n < it.n) sums[it.bias_at + n] = (pb[lane] + pb[64 + lane]) + (pb[128 + lane] + pb[192 + lane]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + 64 * wn + 16 * i + r16;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = k0 + 64 * wk + 16 * j + 4 * kq;
                *reinterpret_cast<F32x4*>(sums + it.at + (int64_t)n * it.k + k) = acc[i][j];
            }
            if (with_bias && kq == 0) sums[it.bias_at + n] = acc_b[i][0];
        }
    }
}

// dst[i] = the sum of src[s * stride + i] over the splits, in a fixed order: 256 / GROUPS float4 columns per workgroup, GROUPS threads each.
struct Segment {
    float* dst;
    int64_t at, count;         // floats, multiples of 4
};
struct SumArgs {
    Segment segment[kSegments];
    const float* src;
    int64_t stride;
    int segments, splits;
};

template <int GROUPS>
__global__ __launch_bounds__(kThreads) void sum_splits_kernel(SumArgs a) {
    constexpr int COLUMNS = kThreads / GROUPS;
    const int col = threadIdx.x % COLUMNS, group = threadIdx.x / COLUMNS;
    int64_t at = ((int64_t)blockIdx.x * COLUMNS + col) * 4;
    int which = 0;
    while (which < a.segments && at >= a.segment[which].count) at -= a.segment[which++].count;
    F32x4 v = F32x4{0.f, 0.f, 0.f, 0.f};
    if (which < a.segments) {
        const float* src = a.src + a.segment[which].at + at;
#pragma unroll 8
        for (int s = group; s < a.splits; s += GROUPS) v += *reinterpret_cast<const F32x4*>(src + s * a.stride);
    }
    if constexpr (GROUPS > 1) {
        __shared__ F32x4 part[kThreads];
        part[threadIdx.x] = v;
        __syncthreads();
        if (group == 0) {
#pragma unroll
            for (int g = 1; g < GROUPS; ++g) v += part[g * COLUMNS + col];
        }
    }
    if (group == 0 && which < a.segments) *reinterpret_cast<F32x4*>(a.segment[which].dst + at) = v;
}

// Threads of a column: as many as leave each about a dozen splits, eight of which it requests together.  With 16 for any number of
// splits, the two of a block of 512 channels (12.6 MB each; 64 images of 49 tokens) left 14 of 16 threads without one: 44.2 -> 8.8 us; ten of
// 256 channels 14.1 -> 7.1 us.  Where there are more, the 42 of 128 channels take 9.2 us with four threads (9.1 with 16).
void launch_sum_splits(const SumArgs& a, int64_t columns, hipStream_t stream) {
    auto grid = [&](int per) { return dim3((unsigned)((columns + per - 1) / per)); };
    if (a.splits <= 12) hipLaunchKernelGGL((sum_splits_kernel<1>), grid(kThreads), dim3(kThreads), 0, stream, a);
    else if (a.splits <= 48) hipLaunchKernelGGL((sum_splits_kernel<4>), grid(kThreads / 4), dim3(kThreads), 0, stream, a);
    else hipLaunchKernelGGL((sum_splits_kernel<16>), grid(kThreads / 16), dim3(kThreads), 0, stream, a);
}

struct Split {
    int tile, tiles, splits;
    int64_t rows_per_split, per_split;
};

// Two workgroups of 64 KB of LDS fit a compute unit: as many splits as make 512 of them, no range of rows under four stages
// (a split costs its sums a trip to memory and back).
Split split_for(const clusten_weight_grad_item* items, int count, int64_t rows, int dtype) {
    Split s = {128, 0, 1, 0, 0};
    for (int i = 0; i < count; ++i) {
        if (items[i].n % 128 != 0 || items[i].k % 128 != 0) s.tile = 64;
    }
    for (int i = 0; i < count; ++i) {
        s.tiles += (items[i].n + s.tile - 1) / s.tile * ((items[i].k + s.tile - 1) / s.tile);
        s.per_split += (int64_t)items[i].n * items[i].k + (items[i].d_bias ? items[i].n : 0);
    }
    const int stage_rows = kStageBytes / (2 * s.tile * (int)dtype_size(dtype));
    const int64_t stages = (rows + stage_rows - 1) / stage_rows;
    const int64_t want = max((int64_t)1, min((int64_t)(512 / s.tiles), stages / 4));
    s.rows_per_split = (stages + want - 1) / want * stage_rows;
    s.splits = (int)((rows + s.rows_per_split - 1) / s.rows_per_split);
    return s;
}

template <typename T>
void launch_tiles(const GradArgs& g, int tile, hipStream_t stream) {
    const dim3 grid((unsigned)xcd_grid(g.tiles * g.splits));
    if (tile == 128) hipLaunchKernelGGL((weight_grad_kernel<T, 128>), grid, dim3(kThreads), 0, stream, g);
    else hipLaunchKernelGGL((weight_grad_kernel<T, 64>), grid, dim3(kThreads), 0, stream, g);
}

}  // namespace

size_t weight_grad_workspace_bytes(const clusten_weight_grad_item* items, int count, int64_t rows, int dtype) {
    const Split s = split_for(items, count, rows, dtype);
    return (size_t)s.splits * s.per_split * sizeof(float);
}

int launch_weight_grad(const clusten_weight_grad_item* items, int count, int64_t rows, float* workspace, int dtype,
                       hipStream_t stream) {
    const Split s = split_for(items, count, rows, dtype);
    GradArgs g = {};
    SumArgs sum = {};
    g.sums = workspace, g.per_split = s.per_split, g.rows = rows, g.rows_per_split = s.rows_per_split;
    g.count = count, g.splits = s.splits;
    sum.src = workspace, sum.stride = s.per_split, sum.splits = s.splits;
    int64_t at = 0;
    for (int i = 0; i < count; ++i) {
        const clusten_weight_grad_item& in = items[i];
        Item& it = g.item[i];
        it.dy = in.d_y, it.x = in.x, it.ld_dy = in.d_y_stride, it.ld_x = in.x_stride, it.n = in.n, it.k = in.k;
        it.tiles_k = (in.k + s.tile - 1) / s.tile, it.first_tile = g.tiles;
        g.tiles += (in.n + s.tile - 1) / s.tile * it.tiles_k;
        it.at = at, at += (int64_t)in.n * in.k, it.bias_at = -1;
        sum.segment[sum.segments++] = Segment{in.d_weight, it.at, (int64_t)in.n * in.k};
        if (in.d_bias) {
            it.bias_at = at, at += in.n;
            sum.segment[sum.segments++] = Segment{in.d_bias, it.bias_at, in.n};
        }
    }
    if (dtype == CLUSTEN_F16) launch_tiles<f16_t>(g, s.tile, stream);
    else if (dtype == CLUSTEN_BF16) launch_tiles<bf16_t>(g, s.tile, stream);
    else launch_tiles<float>(g, s.tile, stream);
    if (int st = launch_status()) return st;
    launch_sum_splits(sum, s.per_split / 4, stream);
    return launch_status();
}

}  // namespace clusten
