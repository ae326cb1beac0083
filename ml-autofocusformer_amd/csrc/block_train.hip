// The training pass of a transformer block by one call a direction: the host side of clusten_block_train_forward and _backward.
//
// A block's forward is five launches, its backward some fifteen; issued one by one from Python, with the allocations, checks and
// autograd nodes between them, they took longer than their kernels.  One block of memory holds what the forward keeps, another
// what the backward passes from kernel to kernel; both are laid out here (256-byte pieces) and are the caller's.
// No kernels of its own.
#include <algorithm>

#include "launch.hpp"

namespace clusten {
namespace {

struct Layout {
    size_t bytes = 0;
    size_t take(size_t n) {
        const size_t at = bytes;
        bytes += (n + 255) / 256 * 256;
        return at;
    }
};

struct Sizes {
    int64_t rows;
    int C, H, heads, table_rows;
    size_t e, s;        // bytes of a value of the products' and of the stream's type
    clusten_attn_shape shape;
    bool local;
};

Sizes sizes_of(const clusten_block_train& a) {
    Sizes z;
    z.rows = (int64_t)a.shape.B * a.shape.N, z.C = a.shape.H * a.shape.C, z.H = a.hidden, z.heads = a.shape.H, z.table_rows = a.table_rows;
    z.e = dtype_size(a.dtype), z.s = dtype_size(a.x_dtype), z.shape = a.shape, z.local = a.plan != nullptr;
    return z;
}

// What the forward keeps.
struct Kept {
    size_t packed, bias, padded, qkv, normed1, stats1, attn, lse, x1, normed2, hidden, stats2, bytes;
};
Kept kept_layout(const Sizes& z) {
    Layout l;
    Kept k;
    const size_t row = (size_t)z.rows * z.C;
    k.packed = l.take(2 * ((size_t)4 * z.C * z.C + (size_t)2 * z.C * z.H) * z.e);
    k.bias = l.take((size_t)z.table_rows * z.heads * z.e);
    k.padded = l.take((size_t)z.table_rows * 8 * z.e);
    k.qkv = l.take(3 * row * z.e);
    k.normed1 = l.take(row * z.e);
    k.stats1 = l.take((size_t)z.rows * 8);
    k.attn = l.take(row * z.e);
    k.lse = l.take(z.local ? (size_t)z.rows * z.heads * 4 : 0);
    k.x1 = l.take(row * z.s);
    k.normed2 = l.take(row * z.e);
    k.hidden = l.take((size_t)z.rows * z.H * z.e);
    k.stats2 = l.take((size_t)z.rows * 8);
    k.bytes = l.bytes;
    return k;
}

// Elements ahead of matrix i (q, kv, proj, fc1, fc2) of either half of the packed weights.
size_t packed_at(const Sizes& z, int i) {
    const size_t cc = (size_t)z.C * z.C, ch = (size_t)z.C * z.H;
    const size_t at[6] = {0, cc, 3 * cc, 4 * cc, 4 * cc + ch, 4 * cc + 2 * ch};
    return at[i];
}

struct Scratch {
    size_t d_x1, branch, d_f, g, d_h, d_attn, d_qkv, probs, d_logit, blank_prob, d_blank, sums_tail, sums_blank, sums_attn, sums_head, weights, bytes;
    size_t weights_bytes;
};
Scratch scratch_layout(const clusten_block_train& a, const Sizes& z, const clusten_weight_grad_item* items, int count) {
    Layout l;
    Scratch s;
    const size_t row = (size_t)z.rows * z.C, pairs = z.local ? (size_t)z.rows * z.heads * z.shape.M : 0;
    const bool separate = a.factors != nullptr || a.x_dtype != a.dtype;
    s.d_x1 = l.take(row * z.s);
    s.branch = l.take(separate ? row * z.e : 0);
    s.d_f = l.take(separate ? row * z.e : 0);
    s.g = l.take((size_t)z.rows * z.H * z.e);
    s.d_h = l.take((size_t)z.rows * z.H * z.e);
    s.d_attn = l.take(row * z.e);
    s.d_qkv = l.take(3 * row * z.e);
    s.probs = l.take(pairs * z.e);
    s.d_logit = l.take(pairs * z.e);
    s.blank_prob = l.take(z.local ? (size_t)z.rows * z.heads * 4 : 0);
    s.d_blank = l.take(z.local ? (size_t)z.rows * z.heads * 4 : 0);
    // partial sums, all of them added up at the end
    s.sums_tail = l.take(block_backward_workspace_bytes(z.rows, z.C));
    s.sums_blank = l.take(z.local ? row_sums_workspace_bytes(z.rows, z.C) : 0);
    s.sums_attn = l.take(z.local ? position_grad_workspace_bytes((int64_t)z.rows * z.shape.M, z.heads) : dense_train_workspace_bytes(z.shape.B, z.heads));
    s.sums_head = l.take(block_backward_workspace_bytes(z.rows, z.C));
    s.weights_bytes = count ? weight_grad_workspace_bytes(items, count, z.rows, a.dtype) : 0;
    s.weights = l.take(s.weights_bytes);
    s.bytes = l.bytes;
    return s;
}

int check(const clusten_block_train& a) {
    if (a.dtype != CLUSTEN_F32 && a.dtype != CLUSTEN_F16 && a.dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (a.x_dtype != a.dtype && a.x_dtype != CLUSTEN_F32) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(a.shape)) return st;
    const int C = a.shape.H * a.shape.C;
    if (a.shape.C != 32 || !block_width_supported(C) || a.hidden <= 0 || a.hidden % C != 0 || a.table_rows <= 0 || a.table_cols <= 0 ||
        a.table_cols > 5 || (int64_t)a.table_rows * a.shape.H >= (int64_t)1 << 31 || (int64_t)a.shape.B * a.shape.N >= (int64_t)1 << 31) {
        return CLUSTEN_ERR_BAD_DIMS;
    }
    if (a.plan ? a.shape.M != 48 || !scatter_pair_supported(a.shape, a.dtype) : a.shape.N > 64) return CLUSTEN_ERR_BAD_DIMS;
    for (int i = 0; i < 18; ++i) {
        if (!a.param[i]) return CLUSTEN_ERR_NULL_POINTER;
        if (!aligned16(a.param[i]) || !aligned16(a.grad[i])) return CLUSTEN_ERR_UNALIGNED;
    }
    if (!a.x || !a.table || !a.pe_idx || !a.kept) return CLUSTEN_ERR_NULL_POINTER;
    if (!aligned16(a.x) || !aligned16(a.kept) || !aligned16(a.plan) || !aligned16(a.pair_lists)) return CLUSTEN_ERR_UNALIGNED;
    return CLUSTEN_OK;
}

enum Param { kNorm1W, kNorm1B, kNorm2W, kNorm2B, kBq, kBkv, kBproj, kB1, kB2, kBlankK, kBlankV, kWq, kWkv, kWproj, kW1, kW2, kPeW, kPeB };

// q, k and v inside the rows of the projections' output, and rows of C channels by head.
void strides_of(const Sizes& z, clusten_strides& q, clusten_strides& kv, clusten_strides& rows) {
    q.b = (int64_t)z.shape.N * 3 * z.C, q.n = 3 * z.C, q.h = 32;
    kv = q, kv.h = 64;
    rows.b = (int64_t)z.shape.N * z.C, rows.n = z.C, rows.h = 32;
}

DenseTrain dense_args(const clusten_block_train& a, const Sizes& z, const char* kept, const Kept& k) {
    DenseTrain d = {};
    d.qkv = kept + k.qkv, d.bias = kept + k.bias, d.padded = kept + k.padded, d.pe_idx = a.pe_idx, d.blank_k = a.param[kBlankK];
    d.blank_v = a.param[kBlankV], d.scale = a.attn_scale, d.B = z.shape.B, d.H = z.heads, d.N = z.shape.N, d.rows = z.table_rows, d.k = a.table_cols;
    return d;
}

// Layers whose parameter gradients are wanted.
int grad_items(const clusten_block_train& a, const Sizes& z, const char* kept, const Kept& k, const char* branch, const char* d_f, char* work,
               const Scratch& s, clusten_weight_grad_item (&items)[5]) {
    const struct {
        int w, b, n, k;
        const char *d_y, *x;
        int64_t ld;
    } layers[5] = {{kWq, kBq, z.C, z.C, work + s.d_qkv, kept + k.normed1, 3 * z.C},
                   {kWkv, kBkv, 2 * z.C, z.C, work + s.d_qkv + (size_t)z.C * z.e, kept + k.normed1, 3 * z.C},
                   {kWproj, kBproj, z.C, z.C, branch, kept + k.attn, z.C},
                   {kW1, kB1, z.H, z.C, work + s.d_h, kept + k.normed2, z.H},
                   {kW2, kB2, z.C, z.H, d_f, work + s.g, z.C}};
    int count = 0;
    for (const auto& l : layers) {
        if (!a.grad[l.w]) continue;
        clusten_weight_grad_item& it = items[count++];
        it = {};
        it.d_y = l.d_y, it.x = l.x, it.d_weight = a.grad[l.w], it.d_bias = a.grad[l.b], it.d_y_stride = l.ld, it.x_stride = l.k;
        it.n = l.n, it.k = l.k;
    }
    return count;
}

}  // namespace
}  // namespace clusten

using namespace clusten;

extern "C" {

size_t clusten_block_train_kept_bytes(const clusten_block_train* a) { return a ? kept_layout(sizes_of(*a)).bytes : 0; }

size_t clusten_block_train_workspace_bytes(const clusten_block_train* a) {
    if (!a) return 0;
    const Sizes z = sizes_of(*a);
    clusten_weight_grad_item items[5];
    static char none[1];
    const int count = grad_items(*a, z, none, Kept{}, none, none, none, Scratch{}, items);
    return scratch_layout(*a, z, items, count).bytes;
}

int clusten_block_train_forward(const clusten_block_train* args, void* out, clusten_stream stream_) {
    if (!args || !out) return CLUSTEN_ERR_NULL_POINTER;
    const clusten_block_train& a = *args;
    if (int st = check(a)) return st;
    if (!aligned16(out)) return CLUSTEN_ERR_UNALIGNED;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const Sizes z = sizes_of(a);
    if (a.factors && z.rows % a.shape.N != 0) return CLUSTEN_ERR_BAD_DIMS;
    const Kept k = kept_layout(z);
    if (a.kept_bytes < k.bytes) return CLUSTEN_ERR_WORKSPACE;
    char* kept = static_cast<char*>(a.kept);
    clusten_pack_item items[10] = {};
    const int mats[5] = {kWq, kWkv, kWproj, kW1, kW2}, ns[5] = {z.C, 2 * z.C, z.C, z.H, z.C}, ks[5] = {z.C, z.C, z.C, z.C, z.H};
    char* packed = kept + k.packed;
    const size_t half = packed_at(z, 5);
    for (int i = 0; i < 5; ++i) {
        items[i].src = items[5 + i].src = a.param[mats[i]];
        items[i].dst = packed + packed_at(z, i) * z.e, items[i].n = ns[i], items[i].k = ks[i];
        items[5 + i].dst = packed + (half + packed_at(z, i)) * z.e, items[5 + i].n = ks[i], items[5 + i].k = ns[i], items[5 + i].transposed = 1;
    }
    if (int st = launch_block_pack(items, 10, z.C, a.dtype, stream)) return st;
    if (int st = launch_position_bias(a.table, a.param[kPeW], a.param[kPeB], kept + k.bias, kept + k.padded, z.table_rows, z.heads, a.table_cols,
                                      a.dtype, stream)) {
        return st;
    }
    NormLinearArgs head = {};
    head.x = a.x, head.norm_w = a.param[kNorm1W], head.norm_b = a.param[kNorm1B], head.w = packed, head.bias0 = a.param[kBq];
    head.bias1 = a.param[kBkv], head.out = kept + k.qkv, head.normed = kept + k.normed1, head.stats = reinterpret_cast<float2*>(kept + k.stats1);
    head.rows = z.rows, head.chunks = 3, head.eps = a.eps1;
    if (int st = launch_norm_linear(head, a.x_dtype, z.C, a.dtype, stream)) return st;
    if (z.local) {
        clusten_strides q, kv, rows;
        strides_of(z, q, kv, rows);
        const char* key = kept + k.qkv + (size_t)z.C * z.e;
        if (int st = launch_cluster_attention(kept + k.qkv, q, key, kv, key + 32 * z.e, kv, nullptr, table_by_heads(kept + k.bias, z.table_rows), nullptr, nullptr,
                                              a.param[kBlankK], a.param[kBlankV], kept + k.attn, rows, a.attn_scale, a.lists_shared != 0, a.plan,
                                              reinterpret_cast<float*>(kept + k.lse), z.shape, a.dtype, stream)) {
            return st;
        }
    } else {
        DenseTrain d = dense_args(a, z, kept, k);
        d.out = kept + k.attn;
        if (int st = launch_dense_train(d, a.dtype, stream)) return st;
    }
    BlockTailArgs tail = {};
    tail.attn = kept + k.attn, tail.x = a.x, tail.wp = packed + packed_at(z, 2) * z.e, tail.bp = a.param[kBproj], tail.norm_w = a.param[kNorm2W];
    tail.norm_b = a.param[kNorm2B], tail.w1 = packed + packed_at(z, 3) * z.e, tail.b1 = a.param[kB1], tail.w2 = packed + packed_at(z, 4) * z.e;
    tail.b2 = a.param[kB2], tail.out = out, tail.scale = a.factors, tail.rows_per_image = a.factors ? a.shape.N : 1, tail.chunks = z.H / z.C;
    tail.rows = z.rows, tail.eps = a.eps2, tail.x1 = kept + k.x1, tail.normed = kept + k.normed2, tail.hidden = kept + k.hidden;
    tail.stats = reinterpret_cast<float2*>(kept + k.stats2);
    return launch_block_tail(tail, a.x_dtype, z.C, a.dtype, stream);
}

int clusten_block_train_backward(const clusten_block_train* args, const void* d_out, void* d_x, void* workspace, size_t workspace_bytes,
                                 clusten_stream stream_) {
    if (!args || !d_out || !d_x || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    const clusten_block_train& a = *args;
    if (int st = check(a)) return st;
    if (!aligned16(d_out) || !aligned16(d_x) || !aligned16(workspace)) return CLUSTEN_ERR_UNALIGNED;
    // the norms', the blank token's and the position bias' gradients are by-products of what d_x takes
    for (int i : {kNorm1W, kNorm1B, kNorm2W, kNorm2B, kBlankK, kBlankV, kPeW, kPeB}) {
        if (!a.grad[i]) return CLUSTEN_ERR_NULL_POINTER;
    }
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const Sizes z = sizes_of(a);
    const Kept k = kept_layout(z);
    if (a.kept_bytes < k.bytes) return CLUSTEN_ERR_WORKSPACE;
    if (z.local && !a.pair_lists) return CLUSTEN_ERR_NULL_POINTER;
    const char* kept = static_cast<const char*>(a.kept);
    char* work = static_cast<char*>(workspace);
    clusten_weight_grad_item items[5];
    int count = grad_items(a, z, kept, k, kept, kept, work, Scratch{}, items);
    const Scratch s = scratch_layout(a, z, items, count);
    if (workspace_bytes < s.bytes) return CLUSTEN_ERR_WORKSPACE;
    const bool separate = a.factors != nullptr || a.x_dtype != a.dtype;
    const char* packed_t = kept + k.packed + packed_at(z, 5) * z.e;
    GradSums sums = {};
    auto partial = [&](size_t at) { return reinterpret_cast<float*>(work + at); };

    BlockTailGrad tail = {};
    tail.d_out = d_out, tail.x1 = kept + k.x1, tail.stats = reinterpret_cast<const float2*>(kept + k.stats2), tail.norm_w = a.param[kNorm2W];
    tail.hidden = kept + k.hidden, tail.wp = packed_t + packed_at(z, 2) * z.e, tail.w1 = packed_t + packed_at(z, 3) * z.e;
    tail.w2 = packed_t + packed_at(z, 4) * z.e, tail.scale = a.factors, tail.d_x = work + s.d_x1, tail.branch = separate ? work + s.branch : nullptr;
    tail.d_f = separate ? work + s.d_f : nullptr, tail.g = work + s.g, tail.d_h = work + s.d_h, tail.d_attn = work + s.d_attn;
    tail.d_norm_w = a.grad[kNorm2W], tail.d_norm_b = a.grad[kNorm2B], tail.partial = partial(s.sums_tail), tail.later = &sums, tail.rows = z.rows;
    tail.rows_per_image = a.factors ? a.shape.N : 1, tail.chunks = z.H / z.C;
    if (int st = launch_block_tail_backward(tail, a.x_dtype, z.C, a.dtype, stream)) return st;

    if (z.local) {
        clusten_strides q, kv, rows;
        strides_of(z, q, kv, rows);
        const char* query = kept + k.qkv;
        const char* key = query + (size_t)z.C * z.e;
        char* d_key = work + s.d_qkv + (size_t)z.C * z.e;
        if (int st = launch_cluster_attention_backward(query, q, key, kv, key + 32 * z.e, kv, work + s.d_attn, rows, kept + k.attn, rows,
                                                       reinterpret_cast<const float*>(kept + k.lse), nullptr, table_by_heads(kept + k.bias, z.table_rows), nullptr, nullptr,
                                                       a.param[kBlankK], a.param[kBlankV], work + s.d_qkv, q, work + s.probs, work + s.d_logit,
                                                       reinterpret_cast<float*>(work + s.blank_prob), reinterpret_cast<float*>(work + s.d_blank),
                                                       a.attn_scale, a.lists_shared != 0, a.plan, z.shape, a.dtype, stream)) {
            return st;
        }
        if (int st = launch_scatter_pair(work + s.d_logit, query, q, d_key, work + s.probs, work + s.d_attn, rows, d_key + 32 * z.e, kv, a.attn_scale,
                                         a.pair_lists, z.shape, a.dtype, stream)) {
            return st;
        }
        if (int st = launch_blank_grad(query, 3 * z.C, work + s.d_attn, reinterpret_cast<const float*>(work + s.d_blank),
                                       reinterpret_cast<const float*>(work + s.blank_prob), a.attn_scale, a.grad[kBlankK], a.grad[kBlankV],
                                       partial(s.sums_blank), &sums, z.shape.B, z.heads, z.shape.N, z.C, a.dtype, stream)) {
            return st;
        }
        if (int st = launch_position_grad(work + s.d_logit, a.pe_idx, kept + k.padded, a.grad[kPeW], a.grad[kPeB], work + s.sums_attn,
                                          &sums, z.shape.B, z.heads, z.shape.N, z.shape.M, z.table_rows, a.table_cols, a.dtype, stream)) {
            return st;
        }
    } else {
        DenseTrain d = dense_args(a, z, kept, k);
        d.d_out = work + s.d_attn, d.d_qkv = work + s.d_qkv, d.partial = partial(s.sums_attn);
        if (int st = launch_dense_train_backward(d, a.grad[kBlankK], a.grad[kBlankV], a.grad[kPeW], a.grad[kPeB], a.dtype, stream)) return st;
    }

    NormLinearGrad head = {};
    head.d_y = work + s.d_qkv, head.x = a.x, head.stats = reinterpret_cast<const float2*>(kept + k.stats1), head.norm_w = a.param[kNorm1W];
    head.w0 = packed_t, head.w1 = packed_t + packed_at(z, 1) * z.e, head.d_res = work + s.d_x1, head.d_x = d_x, head.d_norm_w = a.grad[kNorm1W];
    head.d_norm_b = a.grad[kNorm1B], head.partial = partial(s.sums_head), head.later = &sums, head.rows = z.rows, head.chunks = 3;
    if (int st = launch_norm_linear_backward(head, a.x_dtype, z.C, a.dtype, stream)) return st;
    if (int st = launch_grad_sums(sums, stream)) return st;

    const char* branch = separate ? work + s.branch : work + s.d_x1;
    const char* d_f = separate ? work + s.d_f : static_cast<const char*>(d_out);
    count = grad_items(a, z, kept, k, branch, d_f, work, s, items);
    return count ? launch_weight_grad(items, count, z.rows, reinterpret_cast<float*>(work + s.weights), a.dtype, stream) : CLUSTEN_OK;
}

}  // extern "C"
