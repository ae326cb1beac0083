// block_tail: everything of a transformer block behind its attention, in one kernel over token rows of C channels:
//   x1 = x + s1 (attn Wp^T + bp)       out = x1 + s2 (gelu(LayerNorm(x1) W1^T + b1) W2^T + b2)
//
// The reference model's `proj`, residual, `norm2`, MLP and residual (models/aff_transformer.py:157-158, 230-232, 181-196; s1 and
// s2 are the per-sample factors of stochastic depth, 1 without it).  As separate kernels - three products, an addition with the
// norm, a GELU - the rows cross memory nine times and the hidden layer (2 to 3 C channels) four times; here a workgroup
// takes R rows from the attention's output to the block's output with the hidden layer in LDS, C channels of it at a time.  Every
// intermediate is rounded to the storage type where the separate kernels stored it, but for the hidden layer ahead of its GELU, which
// is rounded only where a backward pass keeps it.  It has no counterpart in the reference's extension modules.
#pragma once

#include "gelu.hpp"
#include "token_block.hpp"

namespace clusten {

// x + s * branch with the branch, its product with s and the sum rounded where separate kernels store them.
template <typename T, typename S, int E>
__device__ __forceinline__ void add_branch(float (&x)[E], const float (&branch)[E], bool scaled, float scale) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
        float v = to_acc(from_acc<T>(branch[e]));
        if (scaled) v = to_acc(from_acc<T>(v * scale));
        x[e] = to_acc(from_acc<S>(x[e] + v));
    }
}

template <typename T, typename S, int C, int TR>
__global__ __launch_bounds__((64 * BlockCfg<T, C>::kWaves), 2) void block_tail_kernel(BlockTailArgs a) {
    typedef BlockCfg<T, C> Cfg;
    constexpr int NB = Cfg::NB, KS = Cfg::kSteps, WAVES = Cfg::kWaves, E = Cfg::kElems, F = Cfg::kFrags, D = Cfg::ahead(TR);
    constexpr bool PARK = C > 64;
    constexpr int P = Cfg::kParts;
    __shared__ __attribute__((aligned(16))) Piece act[KS * TR * P * 64];
    __shared__ __attribute__((aligned(16))) Piece hid[KS * TR * P * 64];
    __shared__ float red[2 * WAVES * TR * 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int64_t row0 = (int64_t)blockIdx.x * (16 * TR);
    const int ch0 = wave * NB * 16 + kq * E;

    int64_t row[TR];       // this lane's rows, clamped into the matrix
#pragma unroll
    for (int t = 0; t < TR; ++t) row[t] = min(row0 + 16 * t + r16, a.rows - 1);
    for (int i = wave; i < KS * TR; i += WAVES) {
        const int s = i / TR, t = i % TR;
        const int64_t r = min(row0 + 16 * t + r16, a.rows - 1);
        const T* at = static_cast<const T*>(a.attn) + r * C + s * Cfg::kStep + kq * E;
        if constexpr (P == 1) {
            CLUSTEN_LDS_DMA16(at, act + (size_t)i * 64);
        } else {
            float v[E];
            load_values<T, E>(at, v);
            put_fragment<T>(act + (size_t)i * P * 64 + lane, v);
        }
    }
    const auto factors = [&](const float* of, float (&scale)[TR]) {
#pragma unroll
        for (int t = 0; t < TR; ++t) scale[t] = of ? to_acc(from_acc<T>(of[(uint32_t)row[t] / (uint32_t)a.rows_per_image])) : 1.f;
    };
    float x[TR][F][E];
    {
        const S* rows[TR];
#pragma unroll
        for (int t = 0; t < TR; ++t) rows[t] = static_cast<const S*>(a.x) + row[t] * C + ch0;
        load_rows<T, S, C, TR>(rows, x);
    }
    constexpr size_t WEIGHTS = (size_t)KS * NB * 64 * Cfg::kRaw;       // of a wave's channels and C inputs
    const Piece* wp = static_cast<const Piece*>(a.wp) + wave * WEIGHTS;
    const Piece* w1 = static_cast<const Piece*>(a.w1) + wave * WEIGHTS;
    const Piece* w2 = static_cast<const Piece*>(a.w2) + wave * a.chunks * WEIGHTS;
    Piece wb[D][NB][Cfg::kRaw];
    preload(wp, lane * 16, wb);
    float scale[TR];
    factors(a.scale, scale);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    lds_barrier<WAVES>();

    {
        F32x4 acc[NB][TR];
        bias_acc<T, NB, TR>(a.bp + wave * NB * 16, kq, acc);
        gemm_pass<T, TR, NB, KS, D>(wp, w1, lane * 16, wb, act + lane, acc);
        // Wide rows: x1 waits for the end in the output buffer (every lane reads back what it wrote itself), its registers
        // are worth more to the products between.  Up to 64 channels there are registers to spare and it is memory that counts.
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            const bool live = row0 + 16 * t + r16 < a.rows;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                float v[E];
                results<NB, TR, E>(acc, f, t, v);
                add_branch<T, S, E>(x[t][f], v, a.scale != nullptr, scale[t]);
                if (PARK && live) store_values<S, E>(static_cast<S*>(a.out) + row[t] * C + ch0 + f * Cfg::kStep, x[t][f]);
                if (live && a.x1) store_values<S, E>(static_cast<S*>(a.x1) + row[t] * C + ch0 + f * Cfg::kStep, x[t][f]);
            }
        }
    }
    float mean[TR], rstd[TR];
    float y[TR][F][E];
#pragma unroll
    for (int t = 0; t < TR; ++t) {
#pragma unroll
        for (int f = 0; f < F; ++f) {
#pragma unroll
            for (int e = 0; e < E; ++e) y[t][f][e] = x[t][f][e];
        }
    }
    T* keep[TR];
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        keep[t] = a.x1 && row0 + 16 * t + r16 < a.rows ? static_cast<T*>(a.normed) + row[t] * C + ch0 : nullptr;
    }
    norm_to_fragments<T, C, TR>(a.norm_w, a.norm_b, a.eps, y, act, red, wave, lane, mean, rstd, keep);
    lds_barrier<WAVES>();
    if (a.x1 && wave == 0 && kq == 0) {
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            if (row0 + 16 * t + r16 < a.rows) a.stats[row[t]] = float2{mean[t], rstd[t]};
        }
    }

    F32x4 acc2[NB][TR];
    bias_acc<T, NB, TR>(a.b2 + wave * NB * 16, kq, acc2);
    for (int chunk = 0; chunk < a.chunks; ++chunk) {
        F32x4 acc[NB][TR];
        bias_acc<T, NB, TR>(a.b1 + (size_t)chunk * C + wave * NB * 16, kq, acc);
        gemm_pass<T, TR, NB, KS, D>(w1, w2, lane * 16, wb, act + lane, acc);
        if (chunk > 0) lds_barrier<WAVES>();       // every wave is past its reads of the last chunk's hidden channels
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            const bool keep = a.hidden && row0 + 16 * t + r16 < a.rows;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                float v[E];
                results<NB, TR, E>(acc, f, t, v);
                if (keep) {
                    store_values<T, E>(static_cast<T*>(a.hidden) + (row[t] * a.chunks + chunk) * C + ch0 + f * Cfg::kStep, v);
                }
#pragma unroll
                for (int e = 0; e < E; ++e) v[e] = gelu_for<T>(v[e]);
                put_fragment<T>(hid + ((wave * F + f) * TR + t) * P * 64 + lane, v);
            }
        }
        lds_barrier<WAVES>();
        w1 += chunk + 1 < a.chunks ? WAVES * WEIGHTS : 0;
        gemm_pass<T, TR, NB, KS, D>(w2, w1, lane * 16, wb, hid + lane, acc2);
        w2 += WEIGHTS;
    }
    if (a.scale) factors(a.scale + a.rows / a.rows_per_image, scale);
    if constexpr (PARK) {
        const S* rows[TR];
#pragma unroll
        for (int t = 0; t < TR; ++t) rows[t] = static_cast<const S*>(a.out) + row[t] * C + ch0;
        load_rows<T, S, C, TR>(rows, x);
    }
#pragma unroll
    for (int t = 0; t < TR; ++t) {
#pragma unroll
        for (int f = 0; f < F; ++f) {
            float v[E];
            results<NB, TR, E>(acc2, f, t, v);
            add_branch<T, S, E>(x[t][f], v, a.scale != nullptr, scale[t]);
            if (row0 + 16 * t + r16 < a.rows) {
                store_values<S, E>(static_cast<S*>(a.out) + row[t] * C + ch0 + f * Cfg::kStep, x[t][f]);
            }
        }
    }
}

template <typename T, typename S, int C, int TR>
int launch_block_tail_tiles(const BlockTailArgs& a, hipStream_t stream) {
    const int64_t groups = (a.rows + 16 * TR - 1) / (16 * TR);
    hipLaunchKernelGGL((block_tail_kernel<T, S, C, TR>), dim3((unsigned)groups), dim3(64 * BlockCfg<T, C>::kWaves), 0, stream, a);
    return launch_status();
}

template <typename T, typename S, int C>
int launch_block_tail_width(const BlockTailArgs& a, hipStream_t stream) {
    // narrow rows are bound by memory and by their GELUs: more, smaller workgroups (16 bits, 2 tiles against 4: 98 against 110 us at
    // 401 408 rows of 64 channels, 62 against 67 at 100 352 of 128; fp32, 1 / 2 / 3 / 4 tiles: 98 / 84 / 87 / 105 at 156 800 rows of 64,
    // 10.8 / 12.4 / 17 / 20 at 25 088 of 32); one fp32 tile of 512 channels, three of 256 fill the LDS.
    // fp32 with three bf16 parts a value, against fp32 instructions: 9800 rows of 256 channels 111 -> 68 us, 39 200 of 128 115 -> 74,
    // 156 800 of 64 110 -> 86, 2450 of 512 136 -> 118, bound by the weights from the L2 (20 us of the 68) and the products (40).
    constexpr int MOST = sizeof(T) == 4 ? (C == 256 ? 3 : C == 64 || C == 128 ? 2 : 1) : (C > 128 ? 4 : 2);
    const int tiles = block_split((int)sizeof(T), C, MOST, a.rows, 1, false).tiles;
    if constexpr (MOST >= 4) {
        if (tiles == 4) return launch_block_tail_tiles<T, S, C, 4>(a, stream);
    }
    if constexpr (MOST >= 3) {
        if (tiles == 3) return launch_block_tail_tiles<T, S, C, 3>(a, stream);
    }
    if constexpr (MOST >= 2) {
        if (tiles == 2) return launch_block_tail_tiles<T, S, C, 2>(a, stream);
    }
    return launch_block_tail_tiles<T, S, C, 1>(a, stream);
}

template <typename T, typename S>
int launch_block_tail_typed(const BlockTailArgs& a, int C, hipStream_t stream) {
    switch (C) {
        case 32: return launch_block_tail_width<T, S, 32>(a, stream);
        case 64: return launch_block_tail_width<T, S, 64>(a, stream);
        case 128: return launch_block_tail_width<T, S, 128>(a, stream);
        case 256: return launch_block_tail_width<T, S, 256>(a, stream);
        case 512: return launch_block_tail_width<T, S, 512>(a, stream);
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
}

}  // namespace clusten
