// Matrix products over token rows with the weights streamed from the L2 straight into the matrix instructions' registers:
// the pieces that norm_linear.hip and block_tail.hip are made of.
//
// A workgroup owns R = 16 * TR token rows and keeps their activations in LDS; its waves split the output channels, so that a
// weight is read by one wave of the workgroup only - from memory (the L2) into the A operand, with no LDS copy - while
// the activations, read by every wave, are the B operand.  All products are taken transposed (Y^T = W X^T): lane (r16, kq)
// of a wave then holds results of row r16, and with the weight rows dealt to the instruction's rows as `weight_channel`
// says, it holds 16 bytes of consecutive channels of that row - which is a store, and which is also what the same lane
// has to supply as B operand of the next product.  Results therefore go to the next product's activation buffer (or to
// memory) as they are, and both ends of the buffer are conflict free: it is kept in fragment order,
//   piece (s, t, lane) = channels s * kStep + kElems * kq .. of row 16 t + r16      (kStep = 64 bytes of a row).
#pragma once

#include <type_traits>

#include "launch.hpp"
#include "mfma.hpp"

namespace clusten {

// What a width of C channels is cut into.  A wave has NB blocks of 16 output channels: with 4 blocks and 4 row tiles an
// activation fragment read from LDS (1 KB) feeds 4 matrix instructions and a weight fragment another 4, half of the 128
// bytes a clock the LDS delivers; narrow layers have too few blocks for that and are bound by memory anyway.
template <typename T, int C>
struct BlockCfg {
    static constexpr int kElems = 16 / (int)sizeof(T);      // channels of a 16-byte piece
    static constexpr int kStep = 4 * kElems;                // channels of a fragment: one step of the contraction
    static constexpr int kPair = sizeof(T) == 2 ? 2 : 1;    // 16-channel blocks of a fragment
    static constexpr int NB = C >= 128 ? 4 : 2;             // blocks per wave
    static constexpr int kFrags = NB / kPair;               // fragments of a wave's output channels
    static constexpr int kWaves = C / 16 / NB;
    static constexpr int kSteps = C / kStep;
    static_assert(C % (16 * NB) == 0, "whole waves");
};

// Output channel (within a wave's group) that row i of the instruction stands for in block nb.
template <typename T>
__device__ __forceinline__ int weight_channel(int nb, int i) {
    if (sizeof(T) == 4) return 16 * nb + i;
    return 32 * (nb >> 1) + 8 * (i >> 2) + 4 * (nb & 1) + (i & 3);
}

// Barrier of the workgroup that orders LDS traffic only: vector-memory operations (weights on their way) stay in flight.
template <int WAVES>
__device__ __forceinline__ void lds_barrier() {
    lds_sync();
    if constexpr (WAVES > 1) {
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// A piece of the packed weights: uniform base, the lane's place in the fragment as a 32-bit offset.
__device__ __forceinline__ Piece weight_piece(const Piece* w, uint32_t lane16) {
    return *reinterpret_cast<const Piece*>(reinterpret_cast<const char*>(w) + lane16);
}

// acc[nb][t] += W X^T over KS steps.  `w` / `wnext`: this wave's weights, fragment (s, nb) at (s * NB + nb) * 64; wb holds
// the first D steps on entry and the first D steps of `wnext` on return, so that the weights of the next product travel
// while this one's results are worked on.  `act`: the activation buffer at this lane's piece, read one step ahead.  The
// scheduling barriers keep every load in the step that issues it: under register pressure the compiler otherwise moves the
// weight loads down to their use and waits for each (the first version of the C = 256 block tail: 62 us instead of 40).
template <typename T, int TR, int NB, int KS, int D>
__device__ __forceinline__ void gemm_pass(const Piece* __restrict__ w, const Piece* __restrict__ wnext, uint32_t lane16,
                                          Piece (&wb)[D][NB], const Piece* act, F32x4 (&acc)[NB][TR]) {
    constexpr int U = KS < 2 ? 1 : 2;      // steps per turn: the registers of wb and a are named statically
    static_assert(KS % U == 0 && U % D == 0, "whole turns of the weight registers");
    Piece a[2][TR];
#pragma unroll
    for (int t = 0; t < TR; ++t) a[0][t] = act[t * 64];
#pragma unroll 4
    for (int s0 = 0; s0 < KS; s0 += U) {
#pragma unroll
        for (int d = 0; d < U; ++d) {
            const int s = s0 + d;
            if (s + 1 < KS) {
#pragma unroll
                for (int t = 0; t < TR; ++t) a[(d + 1) & 1][t] = act[((s + 1) * TR + t) * 64];
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
                for (int t = 0; t < TR; ++t) acc[nb][t] = tile_mfma<T>(wb[d % D][nb], a[d & 1][t], acc[nb][t]);
            }
            const Piece* src = s + D < KS ? w + (size_t)(s + D) * NB * 64 : wnext + (size_t)(s + D - KS) * NB * 64;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) wb[d % D][nb] = weight_piece(src + nb * 64, lane16);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

template <int NB, int D>
__device__ __forceinline__ void preload(const Piece* __restrict__ w, uint32_t lane16, Piece (&wb)[D][NB]) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) wb[d][nb] = weight_piece(w + (d * NB + nb) * 64, lane16);
    }
    __builtin_amdgcn_sched_barrier(0);
}

// E consecutive values of storage type S between memory and fp32 registers (E * sizeof(S) is 16 or 32 bytes).
template <typename S, int E>
__device__ __forceinline__ void load_values(const S* p, float (&x)[E]) {
    constexpr int PER = 16 / (int)sizeof(S);
#pragma unroll
    for (int o = 0; o < E; o += PER) {
        const Piece r = *reinterpret_cast<const Piece*>(p + o);
        float v[PER];
        VecIO<S, PER>::unpack(r, v);
#pragma unroll
        for (int e = 0; e < PER; ++e) x[o + e] = v[e];
    }
}
template <typename S, int E>
__device__ __forceinline__ void store_values(S* p, const float (&x)[E]) {
    constexpr int PER = 16 / (int)sizeof(S);
#pragma unroll
    for (int o = 0; o < E; o += PER) {
        float v[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) v[e] = x[o + e];
        *reinterpret_cast<Piece*>(p + o) = VecIO<S, PER>::pack(v);
    }
}

// A wave's share of R rows of the token stream in the layout of its results, as fp32: fragment f of tile t.  rows[t]: the
// lane's first channel in row 16 t + r16, clamped into the matrix.
template <typename T, typename S, int C, int TR>
__device__ __forceinline__ void load_rows(const S* const (&rows)[TR], float (&x)[TR][BlockCfg<T, C>::kFrags][BlockCfg<T, C>::kElems]) {
    typedef BlockCfg<T, C> Cfg;
#pragma unroll
    for (int t = 0; t < TR; ++t) {
#pragma unroll
        for (int f = 0; f < Cfg::kFrags; ++f) load_values<S, Cfg::kElems>(rows[t] + f * Cfg::kStep, x[t][f]);
    }
}

// Sums over the channels of the R rows: `part[t]` is this lane's share of row 16 t + r16; on return it is the whole row's.
// `red`: WAVES * R floats of LDS that nothing else uses meanwhile.
template <int WAVES, int TR>
__device__ __forceinline__ void row_totals(float (&part)[TR], float* red, int wave, int lane) {
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        part[t] += __shfl_xor(part[t], 16);
        part[t] += __shfl_xor(part[t], 32);
    }
    if constexpr (WAVES > 1) {
        if (lane < 16) {
#pragma unroll
            for (int t = 0; t < TR; ++t) red[(wave * TR + t) * 16 + lane] = part[t];
        }
        lds_barrier<WAVES>();
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) s += red[(w * TR + t) * 16 + (lane & 15)];
            part[t] = s;
        }
    } else {
        lds_sync();
    }
}

// Layer norm of the R rows held in `x` (mean, then centred squares, all fp32), written as fragments of T into `act`; x is
// used up.  Every wave is past its reads of `act` when the first row total is complete.  mean / rstd: of the lane's rows.
template <typename T, int C, int TR>
__device__ __forceinline__ void norm_to_fragments(const float* __restrict__ weight, const float* __restrict__ bias, float eps,
                                                  float (&x)[TR][BlockCfg<T, C>::kFrags][BlockCfg<T, C>::kElems],
                                                  Piece* act, float* red, int wave, int lane, float (&mean)[TR],
                                                  float (&rstd)[TR]) {
    typedef BlockCfg<T, C> Cfg;
    constexpr int E = Cfg::kElems;
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        mean[t] = 0.f;
#pragma unroll
        for (int f = 0; f < Cfg::kFrags; ++f) {
#pragma unroll
            for (int e = 0; e < E; e += 4) mean[t] += (x[t][f][e] + x[t][f][e + 1]) + (x[t][f][e + 2] + x[t][f][e + 3]);
        }
    }
    row_totals<Cfg::kWaves, TR>(mean, red, wave, lane);
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        mean[t] *= 1.f / C;
        rstd[t] = 0.f;
#pragma unroll
        for (int f = 0; f < Cfg::kFrags; ++f) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                x[t][f][e] -= mean[t];
                rstd[t] += x[t][f][e] * x[t][f][e];
            }
        }
    }
    row_totals<Cfg::kWaves, TR>(rstd, red + Cfg::kWaves * TR * 16, wave, lane);
#pragma unroll
    for (int t = 0; t < TR; ++t) rstd[t] = rsqrtf(rstd[t] * (1.f / C) + eps);
    const int ch0 = wave * Cfg::NB * 16 + (lane >> 4) * E;
#pragma unroll
    for (int f = 0; f < Cfg::kFrags; ++f) {
        float g[E], b[E];
        load_values<float, E>(weight + ch0 + f * Cfg::kStep, g);
        load_values<float, E>(bias + ch0 + f * Cfg::kStep, b);
        const int s = wave * Cfg::kFrags + f;
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            float v[E];
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = x[t][f][e] * rstd[t] * g[e] + b[e];
            act[(s * TR + t) * 64 + lane] = VecIO<T, E>::pack(v);
        }
    }
}

// Starts a product's sums at the bias of the output channels, as the storage type T holds it.  `bias`: the wave's first channel.
template <typename T, int NB, int TR>
__device__ __forceinline__ void bias_acc(const float* __restrict__ bias, int kq, F32x4 (&acc)[NB][TR]) {
    constexpr int E = 16 / (int)sizeof(T), P = E / 4;
#pragma unroll
    for (int f = 0; f < NB / P; ++f) {
        float b[E];
        load_values<float, E>(bias + f * 4 * E + kq * E, b);
#pragma unroll
        for (int p = 0; p < P; ++p) {
            F32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = to_acc(from_acc<T>(b[4 * p + e]));
#pragma unroll
            for (int t = 0; t < TR; ++t) acc[f * P + p][t] = v;
        }
    }
}

// The lane's E results of fragment f, tile t.
template <int NB, int TR, int E>
__device__ __forceinline__ void results(const F32x4 (&acc)[NB][TR], int f, int t, float (&v)[E]) {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = acc[f * (E / 4) + (e >> 2)][t][e & 3];
}

}  // namespace clusten
