// Weights of the block kernels (token_block.hpp) in the order their waves read them, and the choice of a kernel.
#include "token_block.hpp"

namespace clusten {

int launch_norm_linear_f16(const NormLinearArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_norm_linear_bf16(const NormLinearArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_norm_linear_f32(const NormLinearArgs& a, int C, hipStream_t stream);
int launch_block_tail_f16(const BlockTailArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_block_tail_bf16(const BlockTailArgs& a, int x_dtype, int C, hipStream_t stream);
int launch_block_tail_f32(const BlockTailArgs& a, int C, hipStream_t stream);
int launch_block_tail_backward_f16(const BlockTailGrad& a, int x_dtype, int C, hipStream_t stream);
int launch_block_tail_backward_bf16(const BlockTailGrad& a, int x_dtype, int C, hipStream_t stream);
int launch_block_tail_backward_f32(const BlockTailGrad& a, int C, hipStream_t stream);
int launch_norm_linear_backward_f16(const NormLinearGrad& a, int x_dtype, int C, hipStream_t stream);
int launch_norm_linear_backward_bf16(const NormLinearGrad& a, int x_dtype, int C, hipStream_t stream);
int launch_norm_linear_backward_f32(const NormLinearGrad& a, int C, hipStream_t stream);

namespace {

// matrices of a launch, 32 bytes of arguments each: the fp32 weights of a stage of 18 blocks are two launches in every forward
constexpr int kPackItems = 64;
struct PackItems {
    clusten_pack_item item[kPackItems];
};

// One thread per 16-byte piece: piece (group, s, nb, part, lane) holds channels k = 32 s + 8 (lane / 16) + E part .. of the
// output channel that row lane % 16 of block nb stands for; fp32 pieces are two parts of four channels.
template <typename T>
__global__ __launch_bounds__(256) void block_pack_kernel(PackItems items, int NB) {
    constexpr int E = 16 / (int)sizeof(T), PARTS = 8 / E;
    const clusten_pack_item it = items.item[blockIdx.y];
    const int64_t pieces = (int64_t)it.n * it.k / E;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    const int lane = (int)(i & 63), part = (int)((i >> 6) % PARTS), nb = (int)((i >> 6) / PARTS % NB);
    const int64_t rest = (i >> 6) / (PARTS * NB);
    const int steps = it.k / 32, s = (int)(rest % steps);
    const int64_t group = rest / steps;
    const int64_t n = group * 16 * NB + weight_channel(nb, lane & 15);
    const int64_t k = (int64_t)s * 32 + 8 * (lane >> 4) + E * part;
    float v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = it.transposed ? it.src[(k + e) * it.n + n] : it.src[n * it.k + k + e];
    static_cast<Piece*>(it.dst)[i] = VecIO<T, E>::pack(v);
}

}  // namespace

bool block_width_supported(int C) { return C == 32 || C == 64 || C == 128 || C == 256 || C == 512; }

// 16-bit products are bound by the weights every workgroup streams from the L2 (0.9 MB at C = 256, H = 768): as many rows as
// `most` allows, as long as half of the 256 compute units have a workgroup (tail, us with 4 / 2 / 1 tiles: 25 088 rows of 256
// channels 44 / 54 / -, 9216 rows of 512 48 / 68 / 76, 6272 rows of 512 60 / 48 / 67, 1003 rows of 256 21 / 15 / 13).
int block_row_tiles(int most, int64_t rows) {
    int tiles = most;
    while (tiles > 1 && (rows + 16 * tiles - 1) / (16 * tiles) < 128) tiles /= 2;
    return tiles;
}

// fp32 weights are twice the bytes and are split next to the products: a workgroup's time is some w for the weights of a chunk of C
// outputs and m a row tile for its products, w : m = 5 : 3 (784 rows of 256 channels: tail 33 / 44 / 57 us with 1 / 2 / 3 tiles,
// norm_linear 16 / 20 / 24 / 30 with 1 .. 4), and a round of 256 workgroups, one a compute unit, takes as long as one.  What gives
// the fewest rounds' time is taken.  Tail, us with 1 / 2 / 3 tiles: 9800 rows of 256 channels 99 / 93 / 61, 3136 rows 34 / 44 / 57;
// norm_linear at 9800 rows 41 / 39 / 28 / 33 unsplit, 45 / 38 / 39 / 33 in three; 3136 rows 17 / 21 / 25 / 30 and 19 / 19 / 14 / 16;
// 2450 rows of 512 50 / 64 / 88 and 42 / 30 / 39.
BlockSplit block_split_f32(int most, int64_t rows, int chunks, bool may_split) {
    BlockSplit best = {1, 1};
    int64_t cost = 0;
    for (int tiles = 1; tiles <= most; ++tiles) {
        const int64_t groups = (rows + 16 * tiles - 1) / (16 * tiles);
        for (int split = 1; split <= (may_split && groups <= 256 ? chunks : 1); ++split) {
            // the norm ahead of the products is about as long as the weights of a chunk
            const int64_t here = (groups * split + 255) / 256 * ((chunks + split - 1) / split * (5 + 3 * tiles) + 5);
            if (cost == 0 || here < cost) cost = here, best = {tiles, split};
        }
    }
    return best;
}

int launch_block_pack(const clusten_pack_item* items, int count, int C, int dtype, hipStream_t stream) {
    const int NB = block_group(dtype == CLUSTEN_F32 ? 4 : 2, C) / 16;
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

size_t block_backward_workspace_bytes(int64_t rows, int C) {
    return (size_t)min((rows + 15) / 16, (int64_t)kRowSumGroups) * 2 * C * sizeof(float);
}

int launch_block_tail_backward(const BlockTailGrad& a, int x_dtype, int C, int dtype, hipStream_t stream) {
    if (dtype == CLUSTEN_F16) return launch_block_tail_backward_f16(a, x_dtype, C, stream);
    if (dtype == CLUSTEN_BF16) return launch_block_tail_backward_bf16(a, x_dtype, C, stream);
    return launch_block_tail_backward_f32(a, C, stream);
}

int launch_norm_linear_backward(const NormLinearGrad& a, int x_dtype, int C, int dtype, hipStream_t stream) {
    if (dtype == CLUSTEN_F16) return launch_norm_linear_backward_f16(a, x_dtype, C, stream);
    if (dtype == CLUSTEN_BF16) return launch_norm_linear_backward_bf16(a, x_dtype, C, stream);
    return launch_norm_linear_backward_f32(a, C, stream);
}

}  // namespace clusten
