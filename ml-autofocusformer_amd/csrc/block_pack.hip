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

// A workgroup's time is some w for a chunk of C outputs, whose weights every workgroup streams from the L2, m for its products of each
// row tile and n for what lies ahead of the chunks; the compute unit with the most workgroups decides, and with weights on their
// way and products going on in all of them at once it takes as long as they do one by one.  What gives the least is taken.
// w : m : n = 5 : 3 : 5 in fp32 (784 rows of 256 channels: tail 33 / 44 / 57 us with 1 / 2 / 3 tiles, norm_linear 16 / 20 / 24 / 30 with
// 1 .. 4), 5 : 3 : 8 in 16 bits, 9 : 2 : 12 with 512 channels (49 rows: tail 34 / 40 / 46 / 54, norm_linear 16 / 19 / 21 / 23).
// fp32, us with 1 / 2 / 3 tiles: tail 9800 rows of 256 channels 99 / 93 / 61, 3136 rows 34 / 44 / 57; norm_linear 9800 rows 41 / 39 / 28 / 33
// unsplit, 45 / 38 / 39 / 33 in three, 2450 rows of 512 50 / 64 and 42 / 30.
// fp16, us with 1 / 2 / 3 / 4 tiles: tail 25 088 rows of 256 channels 68 / 54 / 56 / 44, 36 864 89 / 65 / 60 / 70, 9216 of 512 105 / 94 / 55 / 64,
// 6272 66 / 47 / 52 / 61; norm_linear 9216 rows of 512 47 / 38 / 27 / 31 unsplit, 44 / 32 / 36 / 30 in three, 49 rows 16 and 10.
BlockSplit block_split(int elem_size, int C, int most, int64_t rows, int chunks, bool may_split) {
    const bool wide = elem_size == 2 && C == 512;
    const int w = wide ? 9 : 5, m = wide ? 2 : 3, n = wide ? 12 : elem_size == 2 ? 8 : 5;
    BlockSplit best = {1, 1};
    int64_t cost = 0;
    for (int tiles = 1; tiles <= most; ++tiles) {
        const int64_t groups = (rows + 16 * tiles - 1) / (16 * tiles);
        for (int split = 1; split <= (may_split && groups <= 256 ? chunks : 1); ++split) {
            const int64_t here = (groups * split + 255) / 256 * ((chunks + split - 1) / split * (w + m * tiles) + (may_split ? n : 0));
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
