// Weights of the block kernels (token_block.hpp) in the order their waves read them, and the choice of a kernel.
#include "token_block.hpp"

namespace clusten {

int launch_norm_linear_f16(const NormLinearArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_norm_linear_bf16(const NormLinearArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_norm_linear_f32(const NormLinearArgs& a, int C, hipStream_t stream);
int launch_block_tail_f16(const BlockTailArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_block_tail_bf16(const BlockTailArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_block_tail_f32(const BlockTailArgs& a, int C, hipStream_t stream);

namespace {

// matrices of a launch, 32 bytes of arguments each: the fp32 weights of a stage of 18 blocks are two launches in every forward
constexpr int kPackItems = 64;
struct PackItems {
    clusten_pack_item item[kPackItems];
};

// One thread per 16-byte piece: piece (group, s, nb, lane) holds channels k = kStep s + kElems (lane / 16) .. of the output
// channel that row lane % 16 of block nb stands for.
template <typename T>
__global__ __launch_bounds__(256) void block_pack_kernel(PackItems items, int NB) {
    constexpr int E = 16 / (int)sizeof(T), STEP = 4 * E;
    const clusten_pack_item it = items.item[blockIdx.y];
    const int64_t pieces = (int64_t)it.n * it.k / E;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    const int lane = (int)(i & 63), nb = (int)((i >> 6) % NB);
    const int64_t rest = (i >> 6) / NB;
    const int steps = it.k / STEP, s = (int)(rest % steps);
    const int64_t group = rest / steps;
    const int64_t n = group * 16 * NB + weight_channel<T>(nb, lane & 15);
    const int64_t k = (int64_t)s * STEP + E * (lane >> 4);
    float v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = it.transposed ? it.src[(k + e) * it.n + n] : it.src[n * it.k + k + e];
    static_cast<Piece*>(it.dst)[i] = VecIO<T, E>::pack(v);
}

}  // namespace

bool block_width_supported(int C) { return C == 32 || C == 64 || C == 128 || C == 256 || C == 512; }

int block_group_channels(int C) { return C >= 128 ? 64 : 32; }

// 16-bit products are bound by the weights every workgroup streams from the L2 (0.9 MB at C = 256, H = 768): as many rows as
// `most` allows, as long as half of the 256 compute units have a workgroup (tail, us with 4 / 2 / 1 tiles: 25 088 rows of 256
// channels 44 / 54 / -, 9216 rows of 512 48 / 68 / 76, 6272 rows of 512 60 / 48 / 67, 1003 rows of 256 21 / 15 / 13).  fp32
// products take sixteen times as long per weight and are bound by the compute unit that gets the most row tiles (9800 rows of
// 256 channels: 129 us with 2 tiles, 307 workgroups, two of them on some units; 104 us with 1, 613, three on most).
int block_row_tiles(int elem_size, int most, int64_t rows) {
    int best = 1;
    int64_t cost = 0;
    for (int tiles = most; tiles >= 1; tiles /= 2) {
        const int64_t groups = (rows + 16 * tiles - 1) / (16 * tiles);
        if (elem_size == 2) {
            if (groups >= 128 || tiles == 1) return tiles;
        } else {
            const int64_t here = (groups + 255) / 256 * tiles;
            if (cost == 0 || here < cost) cost = here, best = tiles;
        }
    }
    return best;
}

int launch_block_pack(const clusten_pack_item* items, int count, int C, int dtype, hipStream_t stream) {
    const int NB = block_group_channels(C) / 16;
    for (int at = 0; at < count; at += kPackItems) {
        PackItems p;
        const int here = min(kPackItems, count - at);
        int64_t most = 0;
        for (int i = 0; i < here; ++i) {
            p.item[i] = items[at + i];
            most = max(most, (int64_t)items[at + i].n * items[at + i].k);
        }
        const int64_t per = dtype == CLUSTEN_F32 ? 4 : 8;
        const dim3 grid((unsigned)((most / per + 255) / 256), (unsigned)here);
        if (dtype == CLUSTEN_F16) hipLaunchKernelGGL((block_pack_kernel<f16_t>), grid, dim3(256), 0, stream, p, NB);
        else if (dtype == CLUSTEN_BF16) hipLaunchKernelGGL((block_pack_kernel<bf16_t>), grid, dim3(256), 0, stream, p, NB);
        else if (dtype == CLUSTEN_F32) hipLaunchKernelGGL((block_pack_kernel<float>), grid, dim3(256), 0, stream, p, NB);
        else return CLUSTEN_ERR_BAD_DTYPE;
        if (int st = launch_status()) return st;
    }
    return CLUSTEN_OK;
}

int launch_norm_linear(const NormLinearArgs& a, int x_dtype, int C, int dtype, hipStream_t stream) {
    if (dtype == CLUSTEN_F16) return launch_norm_linear_f16(a, x_dtype, C, stream);
    if (dtype == CLUSTEN_BF16) return launch_norm_linear_bf16(a, x_dtype, C, stream);
    return launch_norm_linear_f32(a, C, stream);
}

int launch_block_tail(const BlockTailArgs& a, int x_dtype, int C, int dtype, hipStream_t stream) {
    if (dtype == CLUSTEN_F16) return launch_block_tail_f16(a, x_dtype, C, stream);
    if (dtype == CLUSTEN_BF16) return launch_block_tail_bf16(a, x_dtype, C, stream);
    return launch_block_tail_f32(a, C, stream);
}

}  // namespace clusten
