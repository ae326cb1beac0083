// scatter_by_cluster: the scatter of the attention backward passes, turned into a gather (no atomics).
//
//   y[b,h, idx[b,i,j], :] += p[b,h,i,j] * x[b,h,i,:]          (d_key with p = d_attn, x = query;
//                                                              d_value with p = attn, x = d_out:
//                                                              clusten/src/clustenqk_cuda_kernel.cu:96-133,
//                                                              clustenav_cuda_kernel.cu:96-131)
//
// for neighbour lists made of whole clusters: idx[b,i,8r+t] = 8 c(b,i,r) + t, the lists the reference model
// builds (models/aff_transformer.py:476-480).  Then the 8 rows of cluster g receive
//
//   y[b,h, 8g + t, :] = sum over the pairs (i, r) with c(b,i,r) = g of  p[b,h,i,8r+t] * x[b,h,i,:]
//
// and, with the pairs of every cluster listed once (cluster_pairs.hip: a counting sort of the cluster numbers on the
// device, shared by the heads), each cluster is an independent small matrix product
// Y_g (8 x C) = P_g^T (8 x pairs) X_g (pairs x C): one wave per cluster walks the heads, the x rows and the 8-element
// pieces of p of 32 pairs at a time travel to LDS by LDS-direct loads, and the product runs on
// `v_mfma_f32_16x16x4_f32` (16-bit data is widened when the operands are read from LDS; rows 8-15 of the instruction
// are idle).  Every row of y is written exactly once, from fp32 sums over all its pairs: no atomics, no zero-fill, no
// fp32 workspace for 16-bit data, and the sums do not depend on the order in which workgroups run.
// A sequence whose length is not a multiple of 8 ends in a short cluster, and the lists that name it hold row 0 in
// the slots past its rows (models/point_utils.py pads member lists with index 0): those slots add to row 0, so
// such a pair is listed a second time, flagged, under cluster 0, where the sum of its pad slots feeds row 0.
// It has no counterpart in the reference's extension modules.
#include <type_traits>

#include "launch.hpp"
#include "mfma.hpp"

namespace clusten {
namespace {

constexpr int kPass = 32;        // pairs per pass
constexpr int kListMax = 256;    // pairs of a cluster held in LDS at a time
constexpr int kPadEntry = 1 << 30;   // list entry flag: the pair names the short last cluster; here, for its pad slots
constexpr int kEntryMask = kPadEntry - 1;

// A launch takes one scatter, whose y is contiguous, or two over the same lists (d_key and d_value: PAIR): y += scale * ..., the rows of y
// strided.  A workgroup of one wave is short enough for what it does ahead of its first load to show: 128 images of 3136 tokens, 2 heads, fp32
// took 124.7 us with the pair's arguments and the heads' split worked out by a division, 122.9 with its own and the split as an argument.
struct Scatter {
    const void* p;
    const void* x;
    void* y;
    clusten_strides xs;
};
struct StridedScatter : Scatter {
    clusten_strides ys;
    float scale;
};
struct Pair {
    StridedScatter job[2];
};

// Jobs: Scatter or Pair; `heads` of a wave.
template <typename T, int C, typename Jobs, int WAVES>
__global__ __launch_bounds__(kWave * WAVES) void scatter_by_cluster_kernel(Jobs jobs, const int32_t* __restrict__ starts,
                                                                   const int32_t* __restrict__ ends,
                                                                   const int32_t* __restrict__ pairs,
                                                                   const int32_t* __restrict__ not_whole,
                                                                   int H, int heads, int N, int M, int clusters_per_image,
                                                                   int total_clusters) {
    constexpr bool PAIR = std::is_same<Jobs, Pair>::value;
    const auto& job = [&]() -> const auto& {
        if constexpr (PAIR) return jobs.job[blockIdx.z];
        else return jobs;
    }();
    const T* __restrict__ p = static_cast<const T*>(job.p);
    const T* __restrict__ x = static_cast<const T*>(job.x);
    T* __restrict__ y = static_cast<T*>(job.y);
    const clusten_strides xs = job.xs;
    // the waves of a workgroup and the workgroups of a column of the grid share the heads; no wave reads another's LDS
    const int wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int h_first = WAVES == 1 ? 0 : min(H, (int)(blockIdx.y * WAVES + wave) * heads), h_last = WAVES == 1 ? H : min(H, h_first + heads);
    constexpr int EB = (int)sizeof(T);
    constexpr int ROW_B = C * EB;                    // bytes of an x row
    constexpr int PIECE_B = 8 * EB;                  // bytes of the 8 elements of p a pair contributes
    constexpr int X_BYTES = kPass * ROW_B;
    constexpr int X_DMA = X_BYTES / 1024;            // LDS-direct loads per pass for the x rows
    constexpr int ROWS_PER_DMA = 1024 / ROW_B;
    constexpr int LANES_PER_ROW = ROW_B / 16;
    constexpr int CB = C / 16;                       // 16-channel blocks of a row
    constexpr int X_BASE = 0;
    constexpr int P_BASE = X_BASE + X_BYTES;
    constexpr int O_BASE = P_BASE + 1024;
    constexpr int L_BASE = O_BASE + 8 * C * 4;
    constexpr int LDS_BYTES = (L_BASE + kListMax * 4 + 1023) / 1024 * 1024;
    static_assert(X_BYTES % 1024 == 0 && 1024 % ROW_B == 0, "whole LDS-direct loads, whole rows per load");
    __shared__ __attribute__((aligned(1024))) char stages[WAVES * LDS_BYTES];
    char* const stage = stages + wave * LDS_BYTES;

    const int unit = xcd_tile(blockIdx.x, total_clusters);
    if (unit < 0) return;
    // the flag and the bounds of the cluster's list are requested together (one trip to memory, not two); the bounds
    // mean nothing when the flag is set, and are not used then
    const int flagged = not_whole != nullptr ? *not_whole : 0;
    const int first = starts[unit];
    const int last = ends[unit];
    const int b = unit / clusters_per_image;
    const int g = unit - b * clusters_per_image;
    const int lane = threadIdx.x % kWave;
    if (flagged != 0) {         // not lists of whole clusters
        if constexpr (PAIR) {   // nothing else writes these rows: NaN, so that it shows
            const float v[4] = {NAN, NAN, NAN, NAN};
            const int quads = min(8, N - 8 * g) * (C / 4);
            for (int i = h_first * quads + lane; i < h_last * quads; i += kWave) {
                const int h = i / quads, q = i - h * quads;
                T* row = y + (int64_t)b * job.ys.b + (int64_t)h * job.ys.h + (int64_t)(g * 8 + q / (C / 4)) * job.ys.n;
                *reinterpret_cast<typename Quad<T>::raw*>(row + q % (C / 4) * 4) = Quad<T>::pack(v);
            }
        }
        return;                 // a single scatter: the atomic kernels run instead
    }
    const int r16 = lane & 15, kq = lane >> 4;
    const int count = last - first;
    int* list = reinterpret_cast<int*>(stage + L_BASE);
    const int rows_here = min(8, N - 8 * g);   // the last cluster of a sequence may be short
    const int pad_from = N & 7;                // ... and the lists that name it hold row 0 in slots pad_from .. 7

    // a cluster listed by more than kListMax pairs is taken in segments, every head walking all of them before it
    // writes its rows; the usual cluster's list is read once for all heads
    const bool one_segment = count <= kListMax;
    if (one_segment) {
        for (int e = lane; e < count; e += kWave) list[e] = pairs[first + e];
    }
    for (int h = h_first; h < h_last; ++h) {
        const char* x_bh = reinterpret_cast<const char*>(x + (int64_t)b * xs.b + (int64_t)h * xs.h);
        const char* p_bh = reinterpret_cast<const char*>(p + ((int64_t)b * H + h) * N * M);
        F32x4 acc[CB];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[cb] = F32x4{0.f, 0.f, 0.f, 0.f};
        for (int seg = 0; seg < count; seg += kListMax) {
            const int n = min(kListMax, count - seg);
            if (!one_segment) {
                lds_sync();
                for (int e = lane; e < n; e += kWave) list[e] = pairs[first + seg + e];
            }
            for (int base = 0; base < n; base += kPass) {
                const int here = min(kPass, n - base);
                lds_sync();  // the previous pass has been read (and the list is in place)
#pragma unroll
                for (int a = 0; a < X_DMA; ++a) {
                    const int e = list[base + min(ROWS_PER_DMA * a + lane / LANES_PER_ROW, here - 1)] & kEntryMask;
                    CLUSTEN_LDS_DMA16(x_bh + lane_offset((uint32_t)(e >> kPairRunBits) * (uint32_t)xs.n * EB +
                                                         (uint32_t)(lane % LANES_PER_ROW) * 16),
                                      stage + X_BASE + a * 1024);
                }
                {
                    // 32 pieces of PIECE_B bytes: 16 bytes per lane
                    constexpr int LANES_PER_PIECE = PIECE_B / 16;
                    if (lane < kPass * LANES_PER_PIECE) {
                        const int e = list[base + min(lane / LANES_PER_PIECE, here - 1)] & kEntryMask;
                        CLUSTEN_LDS_DMA16(p_bh + lane_offset(((uint32_t)(e >> kPairRunBits) * (uint32_t)M + (uint32_t)(e & kPairRunMask) * 8) * EB +
                                                             (uint32_t)(lane % LANES_PER_PIECE) * 16),
                                          stage + P_BASE);
                    }
                }
                lds_sync_vm<0>();
#pragma unroll
                for (int s = 0; s < kPass / 4; ++s) {
                    if (4 * s < here) {
                        const int pr = 4 * s + kq;
                        const T* pp = reinterpret_cast<const T*>(stage + P_BASE + pr * PIECE_B);
                        float a = 0.f;
                        if (pr < here) {
                            if ((list[base + pr] & kPadEntry) == 0) {
                                if (r16 < rows_here) a = to_acc(pp[r16]);
                            } else if (r16 == 0) {
                                // a pair that names the short last cluster: its pad slots hold row 0, this cluster's first
                                for (int t = pad_from; t < 8; ++t) a += to_acc(pp[t]);
                            }
                        }
                        const T* xp = reinterpret_cast<const T*>(stage + X_BASE + pr * ROW_B) + r16;
#pragma unroll
                        for (int cb = 0; cb < CB; ++cb) {
                            acc[cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, to_acc(xp[16 * cb]), acc[cb], 0, 0, 0);
                        }
                    }
                }
            }
        }
        // rows 4*kq + j of the result (kq < 2: the cluster's 8 rows), channels 16*cb + r16
        T* y_rows;
        if constexpr (PAIR) y_rows = y + (int64_t)b * job.ys.b + (int64_t)h * job.ys.h + (int64_t)g * 8 * job.ys.n;
        else y_rows = y + (((int64_t)b * H + h) * N + (int64_t)g * 8) * C;
        lds_sync();
        if (kq < 2) {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    reinterpret_cast<float*>(stage + O_BASE)[(4 * kq + j) * C + 16 * cb + r16] = acc[cb][j];
                }
            }
        }
        lds_sync();
        // 8 rows x C channels, four consecutive channels per lane: 8*C/4 quads
#pragma unroll
        for (int q0 = 0; q0 < 8 * C / 4; q0 += kWave) {
            const int q = q0 + lane;
            if (q < 8 * C / 4 && q / (C / 4) < rows_here) {
                const F32x4 o = *reinterpret_cast<const F32x4*>(stage + O_BASE + q * 16);
                if constexpr (PAIR) {
                    const float v[4] = {o[0] * job.scale, o[1] * job.scale, o[2] * job.scale, o[3] * job.scale};
                    *reinterpret_cast<typename Quad<T>::raw*>(y_rows + (int64_t)(q / (C / 4)) * job.ys.n + q % (C / 4) * 4) = Quad<T>::pack(v);
                } else {
                    const float v[4] = {o[0], o[1], o[2], o[3]};
                    *reinterpret_cast<typename Quad<T>::raw*>(y_rows + q * 4) = Quad<T>::pack(v);
                }
            }
        }
    }
}

// Waves that share the heads of a cluster: a wave walks its heads one after the other, each a chain of loads, products and stores, so a
// launch is given enough waves to hide them, the list of a cluster being read again by each.  Two of them make a workgroup: where the lists
// are not whole clusters all of them leave, at 0.2 us a thousand workgroups.  us before the heads were shared / with as many one-wave
// workgroups / now, and the same where they leave: 50 images of 777 tokens, 4 heads, fp16 47.1 / 41.8 / 38.4 (four waves), lists of any rows, with
// the atomic kernels that take them 106.4 / 108.6 / 107.7; 2 of 1024, 8 heads, fp16 44.9 / 13.7 / 13.7; 8 of 777, 4 heads, fp32, any rows
// 144.7 / 145.6 / 145.1.  d_key and d_value of a layer of AFF-Tiny at 64 images, mean of 25 layers: 2 x 43.6 us in two launches of one wave
// a cluster, 47.8 us in one.
inline int head_shares(int64_t waves, int H) { return (int)min((int64_t)H, max((int64_t)1, (int64_t)16384 / waves)); }

template <typename T, int C, typename Jobs>
int launch_jobs_of(const Jobs& jobs, const int32_t* starts, const int32_t* ends, const int32_t* pairs, const int32_t* not_whole,
                   const clusten_attn_shape& s, hipStream_t stream) {
    constexpr bool PAIR = std::is_same<Jobs, Pair>::value;
    const int per_image = (s.N + 7) / 8;
    const int64_t total = (int64_t)s.B * per_image;
    if (total >= ((int64_t)1 << 30)) return CLUSTEN_ERR_BAD_DIMS;
    const int shares = head_shares(total * (PAIR ? 2 : 1), s.H), whole = shares == 1 ? 1 : min(s.H, (shares + 1) / 2 * 2);    // of two waves
    const int heads = (s.H + whole - 1) / whole;
    if (shares == 1) {
        hipLaunchKernelGGL((scatter_by_cluster_kernel<T, C, Jobs, 1>), dim3(xcd_grid((int)total), 1, PAIR ? 2 : 1), dim3(kWave), 0, stream, jobs,
                           starts, ends, pairs, not_whole, s.H, heads, s.N, s.M, per_image, (int)total);
    } else {
        const int waves = (s.H + heads - 1) / heads;
        hipLaunchKernelGGL((scatter_by_cluster_kernel<T, C, Jobs, 2>), dim3(xcd_grid((int)total), (waves + 1) / 2, PAIR ? 2 : 1), dim3(2 * kWave), 0,
                           stream, jobs, starts, ends, pairs, not_whole, s.H, heads, s.N, s.M, per_image, (int)total);
    }
    return launch_status();
}

template <typename T, typename Jobs>
int launch_typed(const Jobs& jobs, const int32_t* starts, const int32_t* ends, const int32_t* pairs, const int32_t* not_whole,
                 const clusten_attn_shape& s, hipStream_t stream) {
    switch (s.C) {
        case 16: return launch_jobs_of<T, 16>(jobs, starts, ends, pairs, not_whole, s, stream);
        case 32: return launch_jobs_of<T, 32>(jobs, starts, ends, pairs, not_whole, s, stream);
        case 64: return launch_jobs_of<T, 64>(jobs, starts, ends, pairs, not_whole, s, stream);
        default: return CLUSTEN_ERR_BAD_DIMS;
    }
}

template <typename Jobs>
int launch_jobs(const Jobs& jobs, const int32_t* starts, const int32_t* ends, const int32_t* pairs, const int32_t* not_whole,
                const clusten_attn_shape& s, int dtype, hipStream_t stream) {
    switch (dtype) {
        case CLUSTEN_F32: return launch_typed<float>(jobs, starts, ends, pairs, not_whole, s, stream);
        case CLUSTEN_F16: return launch_typed<f16_t>(jobs, starts, ends, pairs, not_whole, s, stream);
        case CLUSTEN_BF16: return launch_typed<bf16_t>(jobs, starts, ends, pairs, not_whole, s, stream);
        default: return CLUSTEN_ERR_BAD_DTYPE;
    }
}

}  // namespace

bool scatter_by_cluster_supported(const void* p, const void* x, clusten_strides xs, const void* y,
                                  const clusten_attn_shape& s, int dtype) {
    if (dtype != CLUSTEN_F32 && dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return false;
    if ((s.C != 16 && s.C != 32 && s.C != 64) || s.N < 8 || s.M % 8 != 0 || s.M > kPairMaxSlots || s.M <= 0) return false;
    const size_t eb = dtype_size(dtype);
    return rows_aligned16(x, xs, (int)eb) && aligned16(p) && aligned16(y) && slice_fits_int32(xs, s.H, s.N, s.C) &&
           (int64_t)s.N * s.M * (int64_t)eb < ((int64_t)1 << 31);
}

int launch_scatter_by_cluster(const void* p, const void* x, clusten_strides xs, const int32_t* starts, const int32_t* ends,
                              const int32_t* pairs, const int32_t* not_whole, void* y, clusten_attn_shape s, int dtype,
                              hipStream_t stream) {
    if ((s.C != 16 && s.C != 32 && s.C != 64) || s.N < 8 || s.M % 8 != 0 || s.M > kPairMaxSlots || s.M == 0) return CLUSTEN_ERR_BAD_DIMS;
    if (!scatter_by_cluster_supported(p, x, xs, y, s, dtype)) return CLUSTEN_ERR_UNALIGNED;
    return launch_jobs(Scatter{p, x, y, xs}, starts, ends, pairs, not_whole, s, dtype, stream);
}

bool scatter_pair_supported(const clusten_attn_shape& s, int dtype) {
    clusten_strides rows = {};
    rows.b = (int64_t)s.N * 3 * s.H * s.C, rows.n = 3 * s.H * s.C, rows.h = 2 * s.C;
    return scatter_by_cluster_supported(nullptr, nullptr, rows, nullptr, s, dtype) && cluster_pairs_supported(s.B, s.N, s.M, s.N);
}

int launch_scatter_pair(const void* d_logit, const void* query, clusten_strides qs, void* d_key, const void* probs, const void* d_out,
                        clusten_strides gs, void* d_value, clusten_strides ys, float scale, const void* pair_lists, clusten_attn_shape s,
                        int dtype, hipStream_t stream) {
    const size_t eb = dtype_size(dtype);
    if (!scatter_by_cluster_supported(d_logit, query, qs, d_key, s, dtype) || !scatter_by_cluster_supported(probs, d_out, gs, d_value, s, dtype) ||
        !rows_aligned16(d_key, ys, eb) || !rows_aligned16(d_value, ys, eb)) {
        return CLUSTEN_ERR_UNALIGNED;
    }
    const ClusterPairsLayout l = cluster_pairs_layout(s.B, s.N, s.M, s.N);
    const char* ws = static_cast<const char*>(pair_lists);
    const Pair jobs = {{{{d_logit, query, d_key, qs}, ys, scale}, {{probs, d_out, d_value, gs}, ys, 1.f}}};
    return launch_jobs(jobs, reinterpret_cast<const int32_t*>(ws + l.starts), reinterpret_cast<const int32_t*>(ws + l.ends),
                       reinterpret_cast<const int32_t*>(ws + l.pairs), reinterpret_cast<const int32_t*>(ws + l.flag), s, dtype, stream);
}

}  // namespace clusten
