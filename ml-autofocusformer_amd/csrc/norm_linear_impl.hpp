// norm_linear: out = LayerNorm(x) W^T + bias over token rows of C channels, C a built width, N a multiple of C.
//
// The head of a transformer block of the reference model: `norm1` and the query and key / value projections
// (models/aff_transformer.py:219, 103-106).  As separate kernels the normalised rows travel through memory once each way
// and a product of (rows x C)(C x 3C) has its own launch; here the rows are normalised on their way into LDS and every
// output channel is computed from there.  What a call moves is x once, out once and the weights per workgroup from the L2.
// It has no counterpart in the reference's extension modules.
#pragma once

#include "token_block.hpp"

namespace clusten {

template <typename T, typename S, int C, int TR>
__global__ __launch_bounds__((64 * BlockCfg<T, C>::kWaves), 2) void norm_linear_kernel(NormLinearArgs a) {
    typedef BlockCfg<T, C> Cfg;
    constexpr int NB = Cfg::NB, KS = Cfg::kSteps, WAVES = Cfg::kWaves, E = Cfg::kElems, D = Cfg::ahead(TR);
    __shared__ __attribute__((aligned(16))) Piece act[KS * TR * Cfg::kParts * 64];
    __shared__ float red[2 * WAVES * TR * 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int64_t row0 = (int64_t)blockIdx.x * (16 * TR);
    const int ch0 = wave * NB * 16 + kq * E;

    float x[TR][Cfg::kFrags][E];
    {
        const S* rows[TR];
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            rows[t] = static_cast<const S*>(a.x) + min(row0 + 16 * t + r16, a.rows - 1) * C + ch0;
        }
        load_rows<T, S, C, TR>(rows, x);
    }
    // the workgroups of a row of the grid share the chunks of C output channels
    const int first = a.chunks * blockIdx.y / gridDim.y, last = a.chunks * (blockIdx.y + 1) / gridDim.y;
    constexpr size_t WEIGHTS = (size_t)KS * NB * 64 * Cfg::kRaw;       // of a wave's channels
    const Piece* w = static_cast<const Piece*>(a.w) + ((size_t)first * WAVES + wave) * WEIGHTS;
    Piece wb[D][NB][Cfg::kRaw];
    preload(w, lane * 16, wb);
    float mean[TR], rstd[TR];
    T* keep[TR];
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        const int64_t row = row0 + 16 * t + r16;
        keep[t] = a.normed && first == 0 && row < a.rows ? static_cast<T*>(a.normed) + row * C + ch0 : nullptr;
    }
    norm_to_fragments<T, C, TR>(a.norm_w, a.norm_b, a.eps, x, act, red, wave, lane, mean, rstd, keep);
    lds_barrier<WAVES>();
    if (a.stats && first == 0 && wave == 0 && kq == 0) {
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            if (row0 + 16 * t + r16 < a.rows) a.stats[row0 + 16 * t + r16] = float2{mean[t], rstd[t]};
        }
    }
    for (int chunk = first; chunk < last; ++chunk) {
        F32x4 acc[NB][TR];
        bias_acc<T, NB, TR>((chunk == 0 ? a.bias0 : a.bias1 + (size_t)(chunk - 1) * C) + wave * NB * 16, kq, acc);
        const Piece* next = w + (chunk + 1 < last ? WAVES * WEIGHTS : 0);
        gemm_pass<T, TR, NB, KS, D>(w, next, lane * 16, wb, act + lane, acc);
        w = next;
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            const int64_t row = row0 + 16 * t + r16;
            if (row < a.rows) {
                T* out = static_cast<T*>(a.out) + (row * a.chunks + chunk) * C + ch0;
#pragma unroll
                for (int f = 0; f < Cfg::kFrags; ++f) {
                    float v[E];
                    results<NB, TR, E>(acc, f, t, v);
                    store_values<T, E>(out + f * Cfg::kStep, v);
                }
            }
        }
    }
}

template <typename T, typename S, int C, int TR>
int launch_norm_linear_tiles(const NormLinearArgs& a, int split, hipStream_t stream) {
    const int64_t groups = (a.rows + 16 * TR - 1) / (16 * TR);
    hipLaunchKernelGGL((norm_linear_kernel<T, S, C, TR>), dim3((unsigned)groups, (unsigned)split), dim3(64 * BlockCfg<T, C>::kWaves), 0, stream,
                       a);
    return launch_status();
}

template <typename T, typename S, int C>
int launch_norm_linear_width(const NormLinearArgs& a, hipStream_t stream) {
    // Up to 64 channels two fp32 tiles (25 088 rows of 64: 11 us, 13 with four).  fp32 with three bf16 parts a value, against fp32
    // instructions: 9800 rows of 256 channels 51 -> 34 us, 39 200 of 128 48 -> 35, 156 800 of 64 58 -> 38, 2450 of 512 45 -> 31.
    constexpr int MOST = sizeof(T) == 4 ? (C > 256 || C <= 64 ? 2 : 4) : 4;
    const BlockSplit cut = block_split((int)sizeof(T), C, MOST, a.rows, a.chunks, true);
    if constexpr (MOST >= 4) {
        if (cut.tiles == 4) return launch_norm_linear_tiles<T, S, C, 4>(a, cut.split, stream);
    }
    if constexpr (MOST >= 3) {
        if (cut.tiles == 3) return launch_norm_linear_tiles<T, S, C, 3>(a, cut.split, stream);
    }
    if (cut.tiles == 2) return launch_norm_linear_tiles<T, S, C, 2>(a, cut.split, stream);
    return launch_norm_linear_tiles<T, S, C, 1>(a, cut.split, stream);
}

template <typename T, typename S>
int launch_norm_linear_typed(const NormLinearArgs& a, int C, hipStream_t stream) {
    switch (C) {
        case 32: return launch_norm_linear_width<T, S, 32>(a, stream);
        case 64: return launch_norm_linear_width<T, S, 64>(a, stream);
        case 128: return launch_norm_linear_width<T, S, 128>(a, stream);
        case 256: return launch_norm_linear_width<T, S, 256>(a, stream);
        case 512: return launch_norm_linear_width<T, S, 512>(a, stream);
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
}

}  // namespace clusten
