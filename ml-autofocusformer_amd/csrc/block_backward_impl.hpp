// What a transformer block's backward pass does over its token rows, as two kernels:
//
// block_tail_backward, of  x1 = x + s1 (attn Wp^T + bp),  out = x1 + s2 (gelu(LayerNorm(x1) W1^T + b1) W2^T + b2):
//   d_f = s2 d_out,  d_h = (d_f W2) gelu'(h),  g = gelu(h),  d_x = d_out + norm'(d_h W1),  branch = s1 d_x,  d_attn = branch Wp
// norm_linear_backward, of  y = LayerNorm(x) W^T + b:   d_x = d_res + norm'(d_y W)
//
// (models/aff_transformer.py:103-106, 157-158, 181-196, 219, 230-232 under autograd.)  As library products with kernels between
// them the rows of d_f W2 and d_h W1 crossed memory twice each and a block took eight launches; here a workgroup takes its
// rows from the incoming gradient to the outgoing one with the machinery of token_block.hpp, the products' results in registers,
// and what it writes beside d_x is what the weights' gradients read: g, d_h, branch, d_f.  The norm's parameter gradients are
// sums over all rows: a workgroup walks tiles a grid apart, keeps its share in LDS and writes one partial row at the end.
// fp16, us, the products and kernels it replaces -> now: tail of 12 544 rows of 256 channels 86 -> 49, 200 704 rows of 64 some 330 ->
// 138 (bound by the four hidden-layer streams, 330 MB), 3136 rows of 512 some 110 -> 61 (the weights from the L2).
// Neither has a counterpart in the reference's extension modules.
#pragma once

#include "gelu.hpp"
#include "token_block.hpp"

namespace clusten {

// Sum over the 16 lanes of a row, in every lane.
__device__ __forceinline__ float row16_total(float x) {
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, true));
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, true));
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, true));
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, true));
    return x;
}

// d_x of a layer norm from the gradient of its result (`acc`, in the layout of a product's results): d_res + rstd (g - mean(g) - xhat
// mean(g xhat)), g = d_y weight.  Adds the rows' d_y xhat and d_y to `sums` (2 C floats of LDS; a channel has one owner).
template <typename T, typename S, int C, int TR>
__device__ __forceinline__ void norm_rows_backward(const F32x4 (&acc)[BlockCfg<T, C>::NB][TR], const S* x, const float2* stats,
                                                   const float* __restrict__ weight, const S* d_res, const int64_t (&row)[TR], const bool (&live)[TR],
                                                   float* red, float* sums, int wave, int lane,
                                                   float (&d_x)[TR][BlockCfg<T, C>::kFrags][BlockCfg<T, C>::kElems]) {
    typedef BlockCfg<T, C> Cfg;
    constexpr int E = Cfg::kElems, F = Cfg::kFrags, WAVES = Cfg::kWaves;
    const int ch0 = wave * Cfg::NB * 16 + (lane >> 4) * E;
    float xh[TR][F][E], s1[TR] = {}, s2[TR] = {}, rstd[TR];
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        const float2 st = stats[row[t]];
        rstd[t] = st.y;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            load_values<S, E>(x + row[t] * C + ch0 + f * Cfg::kStep, xh[t][f]);
#pragma unroll
            for (int e = 0; e < E; ++e) xh[t][f][e] = (xh[t][f][e] - st.x) * st.y;
        }
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        float w[E], dw[E] = {}, db[E] = {};
        load_values<float, E>(weight + ch0 + f * Cfg::kStep, w);
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            results<Cfg::NB, TR, E>(acc, f, t, d_x[t][f]);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (live[t]) dw[e] += d_x[t][f][e] * xh[t][f][e], db[e] += d_x[t][f][e];
                d_x[t][f][e] *= w[e];
                s1[t] += d_x[t][f][e];
                s2[t] += d_x[t][f][e] * xh[t][f][e];
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) dw[e] = row16_total(dw[e]), db[e] = row16_total(db[e]);
        if ((lane & 15) == 0) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                sums[ch0 + f * Cfg::kStep + e] += dw[e];
                sums[C + ch0 + f * Cfg::kStep + e] += db[e];
            }
        }
    }
    row_totals<WAVES, TR>(s1, red, wave, lane);
    row_totals<WAVES, TR>(s2, red + WAVES * TR * 16, wave, lane);
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        s1[t] *= 1.f / C, s2[t] *= 1.f / C;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            float r[E] = {};
            if (d_res) load_values<S, E>(d_res + row[t] * C + ch0 + f * Cfg::kStep, r);
#pragma unroll
            for (int e = 0; e < E; ++e) d_x[t][f][e] = r[e] + rstd[t] * (d_x[t][f][e] - s1[t] - xh[t][f][e] * s2[t]);
        }
    }
}

template <int NB, int TR>
__device__ __forceinline__ void zero_acc(F32x4 (&acc)[NB][TR]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int t = 0; t < TR; ++t) acc[nb][t] = F32x4{0.f, 0.f, 0.f, 0.f};
    }
}

template <typename T, typename S, int C, int TR>
__global__ __launch_bounds__((64 * BlockCfg<T, C>::kWaves), 2) void block_tail_backward_kernel(BlockTailGrad a) {
    typedef BlockCfg<T, C> Cfg;
    constexpr int NB = Cfg::NB, KS = Cfg::kSteps, WAVES = Cfg::kWaves, E = Cfg::kElems, F = Cfg::kFrags, D = Cfg::ahead(TR), P = Cfg::kParts;
    __shared__ __attribute__((aligned(16))) Piece act[KS * TR * P * 64];
    __shared__ __attribute__((aligned(16))) Piece hid[KS * TR * P * 64];
    __shared__ float red[2 * WAVES * TR * 16];
    __shared__ float sums[2 * C];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int ch0 = wave * NB * 16 + kq * E;
    constexpr size_t WEIGHTS = (size_t)KS * NB * 64 * Cfg::kRaw;       // of a wave's channels and C inputs
    const Piece* wp = static_cast<const Piece*>(a.wp) + wave * WEIGHTS;
    const Piece* w2_first = static_cast<const Piece*>(a.w2) + wave * WEIGHTS;
    const Piece* w1_first = static_cast<const Piece*>(a.w1) + wave * a.chunks * WEIGHTS;
    for (int i = threadIdx.x; i < 2 * C; i += 64 * WAVES) sums[i] = 0.f;
    Piece wb[D][NB][Cfg::kRaw];
    preload(w2_first, lane * 16, wb);
    for (int64_t row0 = (int64_t)blockIdx.x * (16 * TR); row0 < a.rows; row0 += (int64_t)gridDim.x * (16 * TR)) {
        int64_t row[TR];       // this lane's rows, clamped into the matrix
        bool live[TR];
        float scale[TR];
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            live[t] = row0 + 16 * t + r16 < a.rows;
            row[t] = min(row0 + 16 * t + r16, a.rows - 1);
            scale[t] = a.scale ? to_acc(from_acc<T>(a.scale[a.rows / a.rows_per_image + (uint32_t)row[t] / (uint32_t)a.rows_per_image])) : 1.f;
        }
        lds_barrier<WAVES>();                      // every wave is past its reads of act (and the sums are cleared)
#pragma unroll
        for (int t = 0; t < TR; ++t) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                float v[E];
                load_values<S, E>(static_cast<const S*>(a.d_out) + row[t] * C + ch0 + f * Cfg::kStep, v);
                if (a.scale) {
#pragma unroll
                    for (int e = 0; e < E; ++e) v[e] = to_acc(from_acc<T>(v[e])) * scale[t];
                }
                put_fragment<T>(act + ((wave * F + f) * TR + t) * P * 64 + lane, v);
                if (a.d_f && live[t]) store_values<T, E>(static_cast<T*>(a.d_f) + row[t] * C + ch0 + f * Cfg::kStep, v);
            }
        }
        lds_barrier<WAVES>();

        F32x4 acc2[NB][TR];
        zero_acc(acc2);
        const Piece* w2 = w2_first;
        const Piece* w1 = w1_first;
        for (int chunk = 0; chunk < a.chunks; ++chunk) {
            const int64_t at = (int64_t)chunk * C + ch0;
            Piece h[TR][F][Cfg::kRaw];
#pragma unroll
            for (int t = 0; t < TR; ++t) {
#pragma unroll
                for (int f = 0; f < F; ++f) {
#pragma unroll
                    for (int r = 0; r < Cfg::kRaw; ++r) {
                        h[t][f][r] = reinterpret_cast<const Piece*>(static_cast<const T*>(a.hidden) + row[t] * a.chunks * C + at + f * Cfg::kStep)[r];
                    }
                }
            }
            F32x4 acc[NB][TR];
            zero_acc(acc);
            gemm_pass<T, TR, NB, KS, D>(w2, w1, lane * 16, wb, act + lane, acc);
            if (chunk > 0) lds_barrier<WAVES>();       // every wave is past its reads of the last chunk's d_h
#pragma unroll
            for (int t = 0; t < TR; ++t) {
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    float d[E], x[E], g[E];
                    results<NB, TR, E>(acc, f, t, d);
#pragma unroll
                    for (int r = 0; r < Cfg::kRaw; ++r) {
                        float v[E / Cfg::kRaw];
                        VecIO<T, E / Cfg::kRaw>::unpack(h[t][f][r], v);
#pragma unroll
                        for (int e = 0; e < E / Cfg::kRaw; ++e) x[r * (E / Cfg::kRaw) + e] = v[e];
                    }
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        float slope;
                        g[e] = gelu_and_slope<T>(x[e], slope);
                        d[e] *= slope;
                    }
                    if (live[t]) {
                        const int64_t to = row[t] * a.chunks * C + at + f * Cfg::kStep;
                        store_values<T, E>(static_cast<T*>(a.g) + to, g);
                        store_values<T, E>(static_cast<T*>(a.d_h) + to, d);
                    }
                    put_fragment<T>(hid + ((wave * F + f) * TR + t) * P * 64 + lane, d);
                }
            }
            lds_barrier<WAVES>();
            w2 += chunk + 1 < a.chunks ? WAVES * WEIGHTS : 0;
            gemm_pass<T, TR, NB, KS, D>(w1, chunk + 1 < a.chunks ? w2 : wp, lane * 16, wb, hid + lane, acc2);
            w1 += WEIGHTS;
        }
        float d_x[TR][F][E];
        norm_rows_backward<T, S, C, TR>(acc2, static_cast<const S*>(a.x1), a.stats, a.norm_w, static_cast<const S*>(a.d_out), row, live, red, sums,
                                        wave, lane, d_x);
        // act has been read to the end: its last product lies ahead of the barriers of the hidden layer and the row totals
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            const float s = a.scale ? to_acc(from_acc<T>(a.scale[(uint32_t)row[t] / (uint32_t)a.rows_per_image])) : 1.f;     // as the forward rounds it
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const int64_t to = row[t] * C + ch0 + f * Cfg::kStep;
                if (live[t]) store_values<S, E>(static_cast<S*>(a.d_x) + to, d_x[t][f]);
#pragma unroll
                for (int e = 0; e < E; ++e) d_x[t][f][e] = to_acc(from_acc<S>(d_x[t][f][e])) * s;
                if (a.branch && live[t]) store_values<T, E>(static_cast<T*>(a.branch) + to, d_x[t][f]);
                put_fragment<T>(act + ((wave * F + f) * TR + t) * P * 64 + lane, d_x[t][f]);
            }
        }
        lds_barrier<WAVES>();
        F32x4 acc[NB][TR];
        zero_acc(acc);
        gemm_pass<T, TR, NB, KS, D>(wp, w2_first, lane * 16, wb, act + lane, acc);
#pragma unroll
        for (int t = 0; t < TR; ++t) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                float v[E];
                results<NB, TR, E>(acc, f, t, v);
                if (live[t]) store_values<T, E>(static_cast<T*>(a.d_attn) + row[t] * C + ch0 + f * Cfg::kStep, v);
            }
        }
    }
    lds_barrier<WAVES>();
    for (int i = threadIdx.x; i < 2 * C; i += 64 * WAVES) a.partial[(int64_t)blockIdx.x * 2 * C + i] = sums[i];
}

template <typename T, typename S, int C, int TR>
__global__ __launch_bounds__((64 * BlockCfg<T, C>::kWaves), 2) void norm_linear_backward_kernel(NormLinearGrad a) {
    typedef BlockCfg<T, C> Cfg;
    constexpr int NB = Cfg::NB, KS = Cfg::kSteps, WAVES = Cfg::kWaves, E = Cfg::kElems, F = Cfg::kFrags, D = Cfg::ahead(TR), P = Cfg::kParts;
    __shared__ __attribute__((aligned(16))) Piece act[2][KS * TR * P * 64];
    __shared__ float red[2 * WAVES * TR * 16];
    __shared__ float sums[2 * C];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int ch0 = wave * NB * 16 + kq * E;
    constexpr size_t WEIGHTS = (size_t)KS * NB * 64 * Cfg::kRaw;
    const Piece* w_first = static_cast<const Piece*>(a.w0) + wave * WEIGHTS;
    const Piece* w_rest = static_cast<const Piece*>(a.w1) + wave * (a.chunks - 1) * WEIGHTS;
    for (int i = threadIdx.x; i < 2 * C; i += 64 * WAVES) sums[i] = 0.f;
    Piece wb[D][NB][Cfg::kRaw];
    preload(w_first, lane * 16, wb);
    for (int64_t row0 = (int64_t)blockIdx.x * (16 * TR); row0 < a.rows; row0 += (int64_t)gridDim.x * (16 * TR)) {
        int64_t row[TR];
        bool live[TR];
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            live[t] = row0 + 16 * t + r16 < a.rows;
            row[t] = min(row0 + 16 * t + r16, a.rows - 1);
        }
        const auto bring = [&](int chunk) {        // C channels of the incoming gradient's rows as fragments
            for (int i = wave; i < KS * TR; i += WAVES) {
                const int s = i / TR, t = i % TR;
                const int64_t r = min(row0 + 16 * t + r16, a.rows - 1);
                const T* at = static_cast<const T*>(a.d_y) + (r * a.chunks + chunk) * C + s * Cfg::kStep + kq * E;
                if constexpr (P == 1) {
                    CLUSTEN_LDS_DMA16(at, act[chunk & 1] + (size_t)i * 64);
                } else {
                    float v[E];
                    load_values<T, E>(at, v);
                    put_fragment<T>(act[chunk & 1] + (size_t)i * P * 64 + lane, v);
                }
            }
        };
        lds_barrier<WAVES>();                      // every wave is past its reads of the buffers
        bring(0);
        F32x4 acc[NB][TR];
        zero_acc(acc);
        const Piece* w = w_first;
        for (int chunk = 0; chunk < a.chunks; ++chunk) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
            lds_barrier<WAVES>();                  // this chunk is there; every wave is past its reads of the last one
            if (chunk + 1 < a.chunks) bring(chunk + 1);
            const Piece* next = chunk + 1 < a.chunks ? w_rest + chunk * WEIGHTS : w_first;
            gemm_pass<T, TR, NB, KS, D>(w, next, lane * 16, wb, act[chunk & 1] + lane, acc);
            w = next;
        }
        float d_x[TR][F][E];
        norm_rows_backward<T, S, C, TR>(acc, static_cast<const S*>(a.x), a.stats, a.norm_w, static_cast<const S*>(a.d_res), row, live, red, sums,
                                        wave, lane, d_x);
#pragma unroll
        for (int t = 0; t < TR; ++t) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                if (live[t]) store_values<S, E>(static_cast<S*>(a.d_x) + row[t] * C + ch0 + f * Cfg::kStep, d_x[t][f]);
            }
        }
    }
    lds_barrier<WAVES>();
    for (int i = threadIdx.x; i < 2 * C; i += 64 * WAVES) a.partial[(int64_t)blockIdx.x * 2 * C + i] = sums[i];
}

template <typename T, typename S, int C, int TR, typename Args>
int launch_backward_tiles(const Args& a, hipStream_t stream) {
    const unsigned groups = (unsigned)min((a.rows + 16 * TR - 1) / (16 * TR), (int64_t)kRowSumGroups);
    const dim3 threads(64 * BlockCfg<T, C>::kWaves);
    if constexpr (std::is_same<Args, BlockTailGrad>::value) {
        hipLaunchKernelGGL((block_tail_backward_kernel<T, S, C, TR>), dim3(groups), threads, 0, stream, a);
    } else {
        hipLaunchKernelGGL((norm_linear_backward_kernel<T, S, C, TR>), dim3(groups), threads, 0, stream, a);
    }
    if (int st = launch_status()) return st;
    return add_up(ColumnSums{a.partial, a.d_norm_w, a.d_norm_b, 1.f, (int)groups, C}, a.later, stream);
}

template <typename T, typename S, int C, typename Args>
int launch_backward_width(const Args& a, hipStream_t stream) {
    // Two tiles at most: four 16-bit ones of 256 channels do not fit the registers, nor do two fp32 ones of 128 and 256 (37 and 10 spilled), which
    // are faster all the same where there are rows for them.  block_split's weights are the forward's, and its rounds
    // beyond the 1024 workgroups launched are turns of their loops.  us with 1 / 2 tiles, tail and
    // norm_linear, fp32: 784 rows of 256 channels 46 / 64 and 22 / 27, 6272 rows 91 / 71 and 43 / 32, 50 176 rows 575 / 484 and 258 / 207;
    // 50 176 rows of 128 195 / 174 and 76 / 59; 200 704 rows of 64 283 / 236 and 110 / 94.  fp16: 12 544 rows of 256 58 / 46 and 28 / 20, 6272 rows
    // of 512 96 / 66 and 42 / 29, 200 704 of 64 150 / 125 and 53 / 42.  Where workgroups of narrow rows share a unit the rule takes the second
    // tile too early: tails of 9800 to 16 384 rows of 64 channels 26 / 35 fp32 and 17 / 20 fp16, of 6272 rows of 128 fp32 35 / 39, 12 544
    // fp16 28 / 34.
    constexpr int MOST = sizeof(T) == 4 && (C == 32 || C == 512) ? 1 : 2;
    const int tiles = block_split((int)sizeof(T), C, MOST, a.rows, 1, false).tiles;
    if constexpr (MOST >= 2) {
        if (tiles == 2) return launch_backward_tiles<T, S, C, 2>(a, stream);
    }
    return launch_backward_tiles<T, S, C, 1>(a, stream);
}

template <typename T, typename S, typename Args>
int launch_backward_typed(const Args& a, int C, hipStream_t stream) {
    switch (C) {
        case 32: return launch_backward_width<T, S, 32>(a, stream);
        case 64: return launch_backward_width<T, S, 64>(a, stream);
        case 128: return launch_backward_width<T, S, 128>(a, stream);
        case 256: return launch_backward_width<T, S, 256>(a, stream);
        case 512: return launch_backward_width<T, S, 512>(a, stream);
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
}

}  // namespace clusten
