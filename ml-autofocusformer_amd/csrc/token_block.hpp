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
//   piece (s, t, lane) = channels s * kStep + kElems * kq .. of row 16 t + r16      (kStep = 32 channels).
//
// fp32 products run on the bf16 matrix instructions, every operand as the sum of three bf16 numbers (`split`): 24 bits, so that
// nothing of an operand of ordinary size is lost.  The six products of parts that reach above 2^-24 of a term are summed in fp32, what is left out is
// below 2^-25 of it.  The instructions round a sum down, by up to 2^-26 of it: six to a step on running sums shifted the mean of 33 000
// rows' results by 3e-6 of their deviation.  The six of a step therefore start from zero, smallest first, and their sum is
// added by a fp32 addition, which rounds to nearest; and every other step is summed negated and subtracted, so that what is left of
// the shift cancels (1e-8 of a result's deviation without: invisible in a row, but not in sums over all rows).  Six instructions of 16 clocks then stand for eight fp32 ones of 32.  Activations are split once, on their way
// into LDS (6 bytes a channel); weights stay fp32 in memory and are split by the one wave that reads them, next to the matrix
// instructions of all its row tiles, in their shadow.  Against float64 the results are nearer than the fp32 instructions' (relative
// 2-norm, norm_linear / block_tail, fp32 instructions -> parts): 1.56 / 1.69 -> 0.77 / 0.72e-7 at 64 channels, 2.14 / 2.34 ->
// 0.83 / 0.79e-7 at 128, 2.93 / 3.30 -> 0.92 / 0.93e-7 at 256, 4.12 / 4.63 -> 1.07 / 1.13e-7 at 512.
// Where it ends: an operand that is infinite, or finite above 3.38e38 (bf16's largest number), makes its results NaN where fp32 arithmetic
// may give infinity; of one below 2^-103 the last part falls among bf16's subnormals, below 2^-110 beneath them, so that fewer than 24
// bits are held, what is lost being some 2^-126 at most.
#pragma once

#include <type_traits>

#include "launch.hpp"
#include "mfma.hpp"

namespace clusten {

// Output channels of a wave: what the weights of a width are grouped by.
constexpr int block_group(int elem_size, int C) { return elem_size == 4 ? (C >= 512 ? 64 : 32) : (C >= 128 ? 64 : 32); }

// What a width of C channels is cut into.  A wave has NB blocks of 16 output channels: with 4 blocks and 4 row tiles an
// activation fragment read from LDS (1 KB) feeds 4 matrix instructions and a weight fragment another 4, half of the 128
// bytes a clock the LDS delivers; narrow layers have too few blocks for that and are bound by memory anyway.  In fp32 an activation
// fragment of 3 KB feeds 6 instructions a block: 2 blocks are enough, and twice the waves split twice the weights at a time.
template <typename T, int C>
struct BlockCfg {
    static constexpr int kElems = 8;                        // channels of a piece: what a lane brings to a matrix instruction
    static constexpr int kStep = 4 * kElems;                // channels of a fragment: one step of the contraction
    static constexpr int NB = block_group(sizeof(T), C) / 16;   // blocks per wave
    static constexpr int kFrags = NB / 2;                   // fragments of a wave's output channels
    static constexpr int kWaves = C / 16 / NB;
    static constexpr int kSteps = C / kStep;
    // Steps of weights on their way: as many as the registers of TR row tiles leave room for, up to four in fp32 (784 rows of 256
    // channels, tail: 43 us with two, 33 with four).
    static constexpr int ahead(int tr) { return kSteps < 2 ? 1 : sizeof(T) == 4 && NB == 2 && tr < 3 && kSteps >= 4 ? 4 : 2; }
    static constexpr int kParts = sizeof(T) == 2 ? 1 : 3;   // pieces of an activation fragment a lane has
    static constexpr int kRaw = (int)sizeof(T) / 2;         // pieces of a weight fragment a lane reads
    static_assert(C % (16 * NB) == 0, "whole waves");
};

// Output channel (within a wave's group) that row i of the instruction stands for in block nb.
__device__ __forceinline__ int weight_channel(int nb, int i) { return 32 * (nb >> 1) + 8 * (i >> 2) + 4 * (nb & 1) + (i & 3); }

// x = part[0] + part[1] + part[2] in bf16, each the rounding of what the ones before it leave.  Of x as rounded to fp32: without the
// pragma the product that x may come from is fused into the first subtraction.
__device__ __forceinline__ void split(const float (&x)[8], Piece (&part)[3]) {
#pragma clang fp contract(off)
    float left[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) left[e] = x[e];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        part[p] = VecIO<bf16_t, 8>::pack(left);
        if (p < 2) {
#pragma unroll
            for (int e = 0; e < 8; ++e) left[e] -= piece_get<bf16_t>(part[p], e);
        }
    }
}

__device__ __forceinline__ void split_piece(const Piece (&raw)[2], Piece (&part)[3], bool minus) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = minus ? -__uint_as_float(raw[e >> 2][e & 3]) : __uint_as_float(raw[e >> 2][e & 3]);
    split(v, part);
}

// A lane's 8 channels into the activation buffer (`at`: its place in the fragment's first piece).
template <typename T>
__device__ __forceinline__ void put_fragment(Piece* at, const float (&v)[8]) {
    if constexpr (sizeof(T) == 2) {
        *at = VecIO<T, 8>::pack(v);
    } else {
        Piece part[3];
        split(v, part);
#pragma unroll
        for (int p = 0; p < 3; ++p) at[p * 64] = part[p];
    }
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

// acc[nb][t] += W X^T over KS steps.  `w` / `wnext`: this wave's weights, fragment (s, nb) at (s * NB + nb) * 64 * kRaw; wb holds
// the first D steps on entry and the first D steps of `wnext` on return, so that the weights of the next product travel
// while this one's results are worked on.  `act`: the activation buffer at this lane's piece, read one step ahead.  The
// scheduling barriers keep every load in the step that issues it: under register pressure the compiler otherwise moves the
// weight loads down to their use and waits for each (the first version of the C = 256 block tail: 62 us instead of 40).
template <typename T, int TR, int NB, int KS, int D, int RAW = (int)sizeof(T) / 2>
__device__ __forceinline__ void gemm_pass(const Piece* __restrict__ w, const Piece* __restrict__ wnext, uint32_t lane16,
                                          Piece (&wb)[D][NB][RAW], const Piece* act, F32x4 (&acc)[NB][TR]) {
    constexpr int U = KS < 2 ? 1 : D > 2 ? D : 2;      // steps per turn: the registers of wb and a are named statically
    constexpr int P = sizeof(T) == 2 ? 1 : 3;
    static_assert(KS % U == 0 && U % D == 0, "whole turns of the weight registers");
    Piece a[2][TR][P];
#pragma unroll
    for (int t = 0; t < TR; ++t) {
#pragma unroll
        for (int p = 0; p < P; ++p) a[0][t][p] = act[(t * P + p) * 64];
    }
    Piece part[2][3];                      // fp32: of the weight fragment at hand and of the next
    if constexpr (P == 3) split_piece(wb[0][0], part[0], false);
#pragma unroll sizeof(T) == 2 ? 4 : 1
    for (int s0 = 0; s0 < KS; s0 += U) {
#pragma unroll
        for (int d = 0; d < U; ++d) {
            const int s = s0 + d;
            if (s + 1 < KS) {
#pragma unroll
                for (int t = 0; t < TR; ++t) {
#pragma unroll
                    for (int p = 0; p < P; ++p) a[(d + 1) & 1][t][p] = act[(((s + 1) * TR + t) * P + p) * 64];
                }
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if constexpr (P == 1) {
#pragma unroll
                    for (int t = 0; t < TR; ++t) acc[nb][t] = tile_mfma<T>(wb[d % D][nb][0], a[d & 1][t][0], acc[nb][t]);
                } else {
                    constexpr int last = NB - 1;
                    const int at = (d * NB + nb) & 1;
                    split_piece(wb[(d + (nb == last)) % D][nb == last ? 0 : nb + 1], part[at ^ 1], (d + (nb == last)) % U & 1);
                    // every other step sums the negated products and is subtracted; a lone step is taken in two halves
#pragma unroll
                    for (int half = 0; half < (KS == 1 ? 2 : 1); ++half) {
                        Piece here[3];
#pragma unroll
                        for (int p = 0; p < 3; ++p) {
                            here[p] = part[at][p];
                            if (KS == 1) {
                                const uint32_t keep = ((threadIdx.x >> 5) & 1) == half ? ~0u : 0u, minus = half ? 0x80008000u : 0u;
#pragma unroll
                                for (int e = 0; e < 4; ++e) here[p][e] = (here[p][e] & keep) ^ minus;
                            }
                        }
                        F32x4 sum[TR];
#pragma unroll
                        for (int t = 0; t < TR; ++t) sum[t] = F32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int order = 2; order >= 0; --order) {       // the smallest products first
#pragma unroll
                            for (int p = order; p >= 0; --p) {
#pragma unroll
                                for (int t = 0; t < TR; ++t) sum[t] = tile_mfma<bf16_t>(here[p], a[d & 1][t][order - p], sum[t]);
                            }
                        }
#pragma unroll
                        for (int t = 0; t < TR; ++t) {
                            if ((d + half) & 1) acc[nb][t] -= sum[t];
                            else acc[nb][t] += sum[t];
                        }
                    }
                    // the next fragment is split in the shadow of this one's products
#pragma unroll
                    for (int i = 0; i < 6 * TR; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, (44 + 6 * TR - 1) / (6 * TR), 0);
                    }
                }
            }
            const Piece* src = s + D < KS ? w + (size_t)(s + D) * NB * 64 * RAW : wnext + (size_t)(s + D - KS) * NB * 64 * RAW;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
                for (int r = 0; r < RAW; ++r) wb[d % D][nb][r] = weight_piece(src + (nb * RAW + r) * 64, lane16);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

template <int NB, int D, int RAW>
__device__ __forceinline__ void preload(const Piece* __restrict__ w, uint32_t lane16, Piece (&wb)[D][NB][RAW]) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
            for (int r = 0; r < RAW; ++r) wb[d][nb][r] = weight_piece(w + ((d * NB + nb) * RAW + r) * 64, lane16);
        }
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
// used up.  Every wave is past its reads of `act` when the first row total is complete.  mean / rstd: of the lane's rows.  keep:
// where the lane's rows of the result go in memory as well (from the lane's first channel on), or null.
template <typename T, int C, int TR>
__device__ __forceinline__ void norm_to_fragments(const float* __restrict__ weight, const float* __restrict__ bias, float eps,
                                                  float (&x)[TR][BlockCfg<T, C>::kFrags][BlockCfg<T, C>::kElems],
                                                  Piece* act, float* red, int wave, int lane, float (&mean)[TR],
                                                  float (&rstd)[TR], T* const (&keep)[TR]) {
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
            put_fragment<T>(act + (s * TR + t) * Cfg::kParts * 64 + lane, v);
            if (keep[t]) store_values<T, E>(keep[t] + f * Cfg::kStep, v);
        }
    }
}

// Starts a product's sums at the bias of the output channels, as the storage type T holds it.  `bias`: the wave's first channel.
template <typename T, int NB, int TR>
__device__ __forceinline__ void bias_acc(const float* __restrict__ bias, int kq, F32x4 (&acc)[NB][TR]) {
    constexpr int E = 8, P = E / 4;
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
