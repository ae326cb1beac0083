// Internal launch functions behind the C ABI.  Each one validates nothing: the extern "C" layer
// has already checked pointers, sizes and strides.  All return a clusten_status.
#pragma once

#include "common.hpp"

namespace clusten {

// An entry of a pair list (cluster_pairs.hip) names run r of token i of its image as i << kPairRunBits | r: lists of
// up to 256 slots, i.e. 32 runs of 8.  Bit 30 flags the second listing of a pair that names a short last cluster.
constexpr int kPairRunBits = 5;
constexpr int kPairRunMask = (1 << kPairRunBits) - 1;
constexpr int kPairMaxSlots = 8 << kPairRunBits;


// out[b,h,i,j] = sum_c a[b,h,i,c] * rows[b,h,idx[b,i,j],c]      (QK forward; AV's d_attn)
//   a, rows : strided (B,H,N,C);  out : contiguous (B,H,N,M)
int launch_gather_dot(const void* a, clusten_strides a_strides, const void* rows, clusten_strides rows_strides,
                      const int64_t* idx, void* out, clusten_attn_shape s, int dtype, hipStream_t stream);

// The same with the lists given as cluster numbers: cluster_idx (B,N,M/8) int32, slot j of a token = row
// 8*g + j%8 of its cluster number j/8 (row 0 where that is >= N).  F32/F16/BF16, C in {16,32,64}, M % 8 == 0, M <= 64.
int launch_gather_dot_clusters(const void* a, clusten_strides a_strides, const void* rows, clusten_strides rows_strides,
                               const int32_t* cluster_idx, void* out, clusten_attn_shape s, int dtype,
                               hipStream_t stream);

// out[b,h,i,c] = sum_j p[b,h,i,j] * rows[b,h,idx[b,i,j],c]      (AV forward; QK's d_query)
//   p : contiguous (B,H,N,M);  rows, out : strided (B,H,N,C)
int launch_gather_sum(const void* p, const void* rows, clusten_strides rows_strides, const int64_t* idx, void* out,
                      clusten_strides out_strides, clusten_attn_shape s, int dtype, hipStream_t stream);

// The same for fp32 p and out over rows of rows_dtype = F16 / BF16, read in place (equal to a cast of the rows first).
int launch_gather_sum_mixed(const void* p, const void* rows, clusten_strides rows_strides, const int64_t* idx, void* out,
                            clusten_strides out_strides, clusten_attn_shape s, int rows_dtype, hipStream_t stream);

// Cluster size the cluster-number forms read a list of M slots in: 8 up to 64 slots, then the run length of the kernels
// for long runs (24, 32 or 16; gather_runs_impl.hpp), 0 when M is neither.
int cluster_size_for(int M);
// The same with the lists given as cluster numbers (see launch_gather_dot_clusters).
int launch_gather_sum_clusters(const void* p, const void* rows, clusten_strides rows_strides, const int32_t* cluster_idx,
                               void* out, clusten_strides out_strides, clusten_attn_shape s, int dtype,
                               hipStream_t stream);

// out[b,h,idx[b,i,j],c] += p[b,h,i,j] * x[b,h,i,c]               (QK's d_key; AV's d_value)
//   p : contiguous (B,H,N,M);  x : strided (B,H,N,C);  out : contiguous (B,H,N,C), zeroed here.
//   Lists made of whole clusters (found out on the device) go through pair lists in `workspace` and a gather without
//   atomics; for any other list the sum is built with fp32 atomics (for F16/BF16 in `workspace`, rounded once).
//   `pair_lists` (may be null): the block launch_cluster_pairs filled for these lists (layout cluster_pairs_layout(B,
//   N, M, N)); the pair lists are then not rebuilt in the workspace.
size_t scatter_rows_workspace_bytes(clusten_attn_shape s, int dtype);
int launch_scatter_rows(const void* p, const void* x, clusten_strides x_strides, const int64_t* idx, void* out,
                        void* workspace, clusten_attn_shape s, int dtype, hipStream_t stream,
                        const void* pair_lists = nullptr);

// out[b,i,ic,c] = sum_j w[b,i,j,ic] * feat[b,idx[b,i,j],c]      (WF forward)
int launch_wf_forward(const void* w, const void* feat, const int64_t* idx, void* out, clusten_wf_shape s, int dtype,
                      hipStream_t stream);

// The same for fp32 w and out over feat of feat_dtype = F16 / BF16, read in place (equal to a cast of feat first).
int launch_wf_forward_mixed(const void* w, const void* feat, const int64_t* idx, void* out, clusten_wf_shape s,
                            int feat_dtype, hipStream_t stream);

// d_w[b,i,j,ic] = sum_c feat[b,idx[b,i,j],c] * d_out[b,i,ic,c]  (WF backward, weights)
int launch_wf_dweights(const void* d_out, const void* feat, const int64_t* idx, void* d_w, clusten_wf_shape s,
                       int dtype, hipStream_t stream);

// d_feat[b,idx[b,i,j],c] += sum_ic d_out[b,i,ic,c] * w[b,i,j,ic]  (WF backward, features; zeroed here)
size_t wf_dfeat_workspace_bytes(clusten_wf_shape s, int dtype);
int launch_wf_dfeat(const void* d_out, const void* w, const int64_t* idx, void* d_feat, void* workspace,
                    clusten_wf_shape s, int dtype, hipStream_t stream);

// probs[b,h,i,:M], blank_prob[b,h,i] = softmax over j <= M of
//   attn[b,h,i,j] + table[pe_idx[b,i,j], h] - 100 * (1 - mask[b,i,j])  (j < M)  and  blank[b,h,i]  (j = M)
//   attn, table : T;  pe_idx, mask (may be null) : int64 (B,N,M);  blank, probs, blank_prob : fp32.  M <= 64, M % 4 == 0.
//   With q (strided (B,H,N,C), T) and blank_k ((H,C), fp32) given, blank[b,h,i] is computed here as their dot product.
int launch_attn_softmax(const void* attn, const void* table, const int64_t* pe_idx, const int64_t* mask,
                        const float* blank, const void* q, clusten_strides qs, const float* blank_k, float* probs,
                        float* blank_prob, clusten_attn_shape s, int dtype, hipStream_t stream);

// Position bias of (row of the relative-position table, head): element row * per_row + head * per_head.  Neighbours of a token are
// neighbouring rows of the table: by heads, the bias of a run of eight neighbours lies in a line or two, by rows in eight.
struct BiasTable {
    const void* cells;
    int32_t per_row, per_head;
};
inline BiasTable table_by_rows(const void* cells, int heads) { return {cells, heads, 1}; }     // (rows, heads)
inline BiasTable table_by_heads(const void* cells, int rows) { return {cells, 1, rows}; }      // (heads, rows)


// Local attention of a cluster-ordered sequence in one kernel (QK, position bias, mask, blank token, softmax, AV,
// blank value): see cluster_attention.hip.  q, k, v, out : strided (B,H,N,C) of T in {F16, BF16, F32}, C = 32;
//   cluster_idx (B,N,6) int32; table (rows,H) of T; pe_idx, mask (may be null) : int64 (B,N,M) — or (1,N,.) each
//   when lists_shared; M = 48 (clusters of 8) or, for 16-bit data, 144 (clusters of 24);
//   blank_k, blank_v : fp32 (H,C);  lse (may be null): fp32 (B,H,N), the logarithm of each softmax's denominator.
int launch_cluster_attention(const void* q, clusten_strides qs, const void* k, clusten_strides ks, const void* v,
                             clusten_strides vs, const int32_t* cluster_idx, BiasTable table, const int64_t* pe_idx,
                             const int64_t* mask, const float* blank_k, const float* blank_v, void* out,
                             clusten_strides os, float scale, int lists_shared, const void* plan, float* lse,
                             clusten_attn_shape s, int dtype, hipStream_t stream);
// The query-side half of that kernel's backward (16-bit data): d_q, the recomputed probabilities and the logit
// gradients as (B,H,N,48) tensors of T, the blank token's probability and logit gradient as fp32 (B,H,N): see
// cluster_attention_bwd.hip.  d_out, out: strided (B,H,N,C) like q; lse: what the forward wrote.
int launch_cluster_attention_backward(const void* q, clusten_strides qs, const void* k, clusten_strides ks, const void* v,
                                      clusten_strides vs, const void* d_out, clusten_strides gs, const void* out,
                                      clusten_strides os, const float* lse, const int32_t* cluster_idx, BiasTable table,
                                      const int64_t* pe_idx, const int64_t* mask, const float* blank_k,
                                      const float* blank_v, void* d_q, clusten_strides dqs, void* probs, void* d_logit,
                                      float* p_blank, float* ds_blank, float scale, int lists_shared, const void* plan,
                                      clusten_attn_shape s, int dtype, hipStream_t stream);
// The per-tile plan the kernel above reads instead of cluster_idx, pe_idx and mask when it is given one (what it
// would work out from them before its first head): B = batch elements of the index tensors, M = 48 or 144.
size_t cluster_attention_plan_bytes(int B, int N, int M);
int launch_cluster_attention_plan(const int32_t* cluster_idx, const int64_t* pe_idx, const int64_t* mask, void* plan,
                                  int B, int N, int M, hipStream_t stream);

// The pair lists of lists made of whole clusters (cluster_pairs.hip), built on the device: for `rows` list rows per
//   image of M slots that point into a sequence of D rows (K = ceil(D/8) clusters), pairs[starts[b*K+g] .. ends[b*K+g])
//   holds the entries i*8 + r whose run r of list row i is cluster g of image b, ascending; *not_whole becomes 1 when
//   some run is not a whole cluster (then the other outputs mean nothing), else 0.  `keys` and `wg_bad` are scratch.
//   Sizes as cluster_pairs_layout() gives them (byte offsets into one 16-byte aligned block, `bytes` in all).
struct ClusterPairsLayout {
    size_t flag, wg_bad, keys, pairs, starts, ends, bytes;
};
bool cluster_pairs_supported(int B, int rows, int M, int D);
ClusterPairsLayout cluster_pairs_layout(int B, int rows, int M, int D);
// `numbers` != nullptr: the lists as (B,rows,M/8) int32 cluster numbers instead of `idx` (not read then); a number
//   outside [0, ceil(D/8)) raises *not_whole.
int launch_cluster_pairs(const int64_t* idx, int32_t* keys, int32_t* wg_bad, int32_t* not_whole, int32_t* pairs,
                         int32_t* starts, int32_t* ends, int B, int rows, int M, int D, hipStream_t stream,
                         const int32_t* numbers = nullptr);
// The entries (i, j) of a list tensor (B, rows, M) by the row of the D-row sequence they name, built on the device
//   (cluster_pairs.hip): entries[starts[b*D+n] .. ends[b*D+n]) holds e = i*M + j for every idx[b,i,j] = n, ascending.
//   `only_if` (may be null): device flag; nothing is done when it points to zero.  Sizes as row_entries_layout() gives
//   them (byte offsets into one 16-byte aligned block).
struct RowEntriesLayout {
    size_t entries, starts, ends, bytes;
};
bool row_entries_supported(int B, int rows, int M, int D);
RowEntriesLayout row_entries_layout(int B, int rows, int M, int D);
int launch_row_entries(const int64_t* idx, const int32_t* only_if, int32_t* entries, int32_t* starts, int32_t* ends, int B,
                       int rows, int M, int D, hipStream_t stream);
// d_feat[b,n,:] = sum over the entries (i,j) of row (b,n) of sum_ic w[b,i,j,ic] * d_out[b,i,ic,:]: see wf_dfeat_rows.hip.
bool wf_dfeat_rows_supported(const void* d_out, const void* d_feat, const clusten_wf_shape& s, int dtype);
int launch_wf_dfeat_rows(const void* d_out, const void* w, const int32_t* starts, const int32_t* ends,
                         const int32_t* entries, const int32_t* only_if, void* d_feat, clusten_wf_shape s, int dtype,
                         hipStream_t stream);

// y[b,h,8g+t,:] = sum over the listed pairs (i,r) of cluster (b,g) of p[b,h,i,8r+t] * x[b,h,i,:]: see scatter_by_cluster.hip.
//   C in {16,32,64}.  `not_whole` (may be null): device flag; the kernel does nothing when it points to non-zero.
bool scatter_by_cluster_supported(const void* p, const void* x, clusten_strides xs, const void* y,
                                  const clusten_attn_shape& s, int dtype);
int launch_scatter_by_cluster(const void* p, const void* x, clusten_strides xs, const int32_t* starts, const int32_t* ends,
                              const int32_t* pairs, const int32_t* not_whole, void* y, clusten_attn_shape s, int dtype,
                              hipStream_t stream);
// d_feat[b,8g+t,:] = sum over the listed pairs (i,r) of cluster (b,g) of sum_ic w[b,i,8r+t,ic] * d_out[b,i,ic,:]: see
//   wf_dfeat_by_cluster.hip.  IC = 4, C % 32 == 0.  `not_whole` as above.
bool wf_dfeat_by_cluster_supported(const void* d_out, const void* w, const void* d_feat, const clusten_wf_shape& s,
                                   int dtype);
int launch_wf_dfeat_by_cluster(const void* d_out, const void* w, const int32_t* starts, const int32_t* ends,
                               const int32_t* pairs, const int32_t* not_whole, void* d_feat, clusten_wf_shape s, int dtype,
                               hipStream_t stream);

// Attention of every token over every token (N <= 64) in one kernel: see dense_attention.hip.  q, k, v, out : strided
//   (B,H,N,C) of T in {F16, BF16}, C = 32; table (rows,H) of T; pe_idx int64 (B,N,N); blank_k, blank_v : fp32 (H,C).
int launch_dense_attention(const void* q, clusten_strides qs, const void* k, clusten_strides ks, const void* v,
                           clusten_strides vs, const void* table, const int64_t* pe_idx, const float* blank_k,
                           const float* blank_v, void* out, clusten_strides os, float scale, clusten_attn_shape s,
                           int dtype, hipStream_t stream);

// y = act(x W^T + b) for tall x and small W (see skinny_linear.hip): x (M,K) of T with row stride ldx elements,
//   w (NOUT,K), bias (NOUT) or null, y (M,NOUT), all of T in {F16, BF16}; act 0 = identity, 1 = exact GELU.
bool skinny_linear_supported(int K, int NOUT, int act);
int launch_skinny_linear(const void* x, int64_t ldx, const void* w, const void* bias, void* y, int64_t M, int K, int NOUT,
                         int act, int dtype, hipStream_t stream);

// out[r,:] = (x[r,:] - mean) * rsqrt(var + eps) * weight + bias for `rows` rows of C channels
//   (C in {64,128,256,384,512,768,1024}); x and out of dtype F32, F16 or BF16 each, arithmetic in fp32.
int launch_layer_norm(const void* x, int in_dtype, const float* weight, const float* bias, void* out, float* stats, int64_t rows, int C,
                      float eps, int out_dtype, hipStream_t stream);
// Its backward (layer_norm_grad.hip); stats (rows, 2) as the forward left them, partial of the bytes below (0: not supported).
size_t layer_norm_backward_workspace_bytes(int64_t rows, int C);
int launch_layer_norm_backward(const void* d_y, int dy_dtype, const void* x, int x_dtype, const float* stats, const float* weight, void* d_x,
                               float* d_weight, float* d_bias, float* partial, int64_t rows, int C, hipStream_t stream);

// layer norm of rows read in a given order (order may be null) with a per-channel bias (may be null) added first.
int launch_layer_norm_rows(const void* x, int in_dtype, const int64_t* order, int group, const void* pre_bias,
                           const float* weight, const float* bias, void* out, int64_t rows, int C, float eps,
                           int out_dtype, hipStream_t stream);

// y = GELU(x * scale[c] + shift[c]) over (B,C,HW) of T in {F16, BF16}; HW % 8 == 0.
int launch_channel_affine_gelu(const void* x, const float* scale, const float* shift, void* y, int64_t B, int C, int HW,
                               int dtype, hipStream_t stream);

// sum_out = x + branch (x's type), out = layer norm of sum_out (branch's 16-bit type); x of F32 or branch's type.
int launch_add_layer_norm(const void* x, int x_dtype, const void* branch, int branch_dtype, void* sum_out,
                          const float* weight, const float* bias, void* out, int64_t rows, int C, float eps,
                          hipStream_t stream);

// member_idx, mask (may be null), pe_idx (B,N,nnc*m) int64 and cluster_idx (B,N,nnc) int32 (may be null) from
//   nearest (B,N,nnc) int64 and pos (B,N,2) fp32: see neighbour_lists.hip.
int launch_neighbour_lists(const float* pos, const int64_t* nearest, int64_t* member_idx, int64_t* mask, int64_t* pe_idx,
                           int32_t* cluster_idx, int B, int N, int nnc, int m, int radius, int table_width,
                           hipStream_t stream);

// score[r] = sigmoid(<x[r] (+ branch[r]), w> + b) with the sum written to sum_out: see row_score.hip.
int launch_add_row_score(const void* x, int x_dtype, const void* branch, void* sum_out, const void* w, const void* b,
                         void* score, int64_t rows, int C, int dtype, hipStream_t stream);

// d_logit = probs * (d_probs - s), d_blank_logit = blank_prob * (d_blank_prob - s), s the row's sum of p * dp.
int launch_attn_softmax_backward(const float* probs, const float* blank_prob, const float* d_probs,
                                 const float* d_blank_prob, void* d_logit, float* d_blank_logit, int64_t rows, int M,
                                 int dtype, hipStream_t stream);

// d_table[pe_idx[b,i,j], h] += d_logit[b,h,i,j]; d_table (rows,H) fp32 zeroed by the caller.
int launch_bias_table_grad(const void* d_logit, const int64_t* pe_idx, float* d_table, int B, int H, int N, int M, int rows,
                           int dtype, hipStream_t stream);

// w[b,i,j,:4] = table_w[pe_idx[b,i,j], :4] * prob[b, nbhd_idx[b,i,j]] * mask[b,i,j]   (prob, mask may be null)
//   table_w (rows,4), prob (B,N), w (B,Nout,M,4): fp32;  pe_idx, nbhd_idx, mask: int64 (B,Nout,M).
int launch_merge_weights(const float* table_w, const int64_t* pe_idx, const int64_t* nbhd_idx, const float* prob,
                         const int64_t* mask, float* out, int B, int N, int Nout, int M, int64_t rows, hipStream_t stream);

// ranking[b,:] = the order of the tokens of image b along the scan-line walk over a rows x cols anchor grid with
//   cells of cell_w x cell_h (see scanline_rank.hip).  pos (B,N,2) fp32 as (x, y); ranking (B,N) int64; N <= scanline_rank_max_tokens()
//   (the sort of an image runs in the LDS of one compute unit: 16384 tokens on an MI355X),
//   rows * cols >= 2; workspace of scanline_rank_workspace_bytes(B, N) bytes.
size_t scanline_rank_workspace_bytes(int B, int N);
int scanline_rank_max_tokens();   // the longest sequence the LDS of the current device sorts (a power of two)

// pos_sorted[b,i] = pos[b, ranking[b,i]] (may be null) and centres[b,g] = mean of the positions of tokens
//   ranking[b, g*m .. g*m+m-1] (the last cluster may be short): pos, pos_sorted (B,N,2), centres (B,ceil(N/m),2) fp32.
int launch_cluster_centres(const float* pos, const int64_t* ranking, float* pos_sorted, float* centres, int B, int N, int m,
                           hipStream_t stream);

// out[b,i,:] = x[b, order[b,i], :] for rows of row_bytes bytes (a multiple of 16); order (B,N) int64, or (N) for
//   every b when order_shared.
int launch_gather_rows(const void* x, const int64_t* order, void* out, int64_t B, int N, int row_bytes, int order_shared,
                       hipStream_t stream);
// centre[b, :] = the tokens the adaptive down-sampling keeps (models/aff_transformer.py:296-334): the sample_num tokens
//   of highest score = grid prior + prob * alpha [- 100 on the reserved grid], ascending index among those above the
//   sample_num-th score, then those equal to it; then, with reserve_on, the reserve_num reserved tokens by ascending
//   index.  pos (B,N,2) fp32; min_dist (B,N) fp32 distance to the nearest other token, or null for the regular grid of
//   `stride`; prob (B,N) of prob_dtype or null; centre (B, sample_num [+ reserve_num]) int64.
int merge_centres_max_tokens();
int launch_merge_centres(const float* pos, const float* min_dist, const void* prob, int prob_dtype, int64_t* centre, int B,
                         int N, int sample_num, int reserve_num, int reserve_on, float alpha, int stride,
                         hipStream_t stream);
// dst[t][b,i,:] = src[t][b, centre[b,i], :] for t < count <= 4 tensors (B,N,.) with rows of row_bytes[t] bytes
//   (multiples of 8); centre (B,n_out) int64.
int launch_merge_rows(const void* const* src, void* const* dst, const int* row_bytes, int count, const int64_t* centre,
                      int64_t B, int N, int n_out, hipStream_t stream);
int launch_scanline_rank(const float* pos, int64_t* ranking, void* workspace, int B, int N, int rows, int cols,
                         float cell_w, float cell_h, hipStream_t stream);

// idx[b,q,:K], dist[b,q,:K] = the K (1..8, K <= N) database points of batch element b nearest to query q,
//   ascending Euclidean distance, equal distances by index.  query (B,Nq,2), database (B,N,2): fp32;
//   idx int64; dist fp32 or null.
int launch_knn2d(const float* query, const float* database, int64_t* idx, float* dist, int B, int Nq, int N, int K,
                 hipStream_t stream);

// ---- transformer blocks over token rows (token_block.hpp) -----------------------------------------------------------

// out = LayerNorm(x) W^T + bias (norm_linear_impl.hpp) and the block behind its attention (block_tail_impl.hpp).
//   T: the dtype of the call (weights as packed, results); S: the token stream's, fp32 or T.  C in {32,64,128,256,512}.
struct NormLinearArgs {
    const void* x;
    const float* norm_w;
    const float* norm_b;
    const void* w;         // packed for width C
    const float* bias0;    // first C output channels
    const float* bias1;    // the others
    void* out;             // (rows, N)
    void* normed;          // (rows, C) of T, or null
    float2* stats;         // (rows) mean and 1 / deviation, or null
    int64_t rows;
    int chunks;            // N / C
    float eps;
};
struct BlockTailArgs {
    const void* attn;      // (rows, C) of T
    const void* x;         // (rows, C) of S
    const void* wp;
    const float* bp;
    const float* norm_w;
    const float* norm_b;
    const void* w1;        // (H, C), packed for width C
    const float* b1;
    const void* w2;        // (C, H), packed for width C
    const float* b2;
    void* out;             // (rows, C) of S
    const float* scale;    // (2, images): each image's factor of the attention's branch, then of the MLP's, or null
    int rows_per_image;
    int chunks;            // H / C
    int64_t rows;
    float eps;
    // what a backward pass wants to keep, each may be null
    void* x1;              // (rows, C) of S
    void* normed;          // (rows, C) of T
    void* hidden;          // (rows, H) of T, ahead of the GELU
    float2* stats;         // (rows)
};
bool block_width_supported(int C);
// Tiles of 16 rows a workgroup takes (1 .. most), and, when they may be shared, over how many workgroups the chunks of C outputs are.
struct BlockSplit {
    int tiles, split;
};
BlockSplit block_split(int elem_size, int C, int most, int64_t rows, int chunks, bool may_split);
// dst = a weight matrix of fp32 in the order the block kernels of width C read it in, as dtype.  src is (n,k), or (k,n)
//   when transposed (dst is then that of its transpose); n and k multiples of C.
int launch_block_pack(const clusten_pack_item* items, int count, int C, int dtype, hipStream_t stream);
int launch_norm_linear(const NormLinearArgs& a, int x_dtype, int C, int dtype, hipStream_t stream);
int launch_block_tail(const BlockTailArgs& a, int x_dtype, int C, int dtype, hipStream_t stream);

// Backward of the two (block_backward_impl.hpp); the weights are packed transposes.
// Partial rows that kernels left, added up in one launch: up to three of 2 C columns (the first C times scale0 to out0, the others to out1) and
// a position bias layer's.  Kernels that are given one leave their sums to it, and launch them themselves otherwise.
struct ColumnSums {
    const float* partial;      // (groups, 2 C)
    float* out0;
    float* out1;
    float scale0;
    int groups, C;
};
struct PositionSums {
    const double* partial;     // (groups, heads, 6): five columns and the bias
    float* d_w;                // (heads, k)
    float* d_b;
    int groups, heads, k;
};
struct GradSums {
    ColumnSums column[3];
    PositionSums position;     // heads 0: none
    int columns;
};
int launch_grad_sums(const GradSums& sums, hipStream_t stream);
int add_up(const ColumnSums& sums, GradSums* later, hipStream_t stream);
int add_up(const PositionSums& sums, GradSums* later, hipStream_t stream);

struct BlockTailGrad {
    const void* d_out;     // (rows, C) of S
    const void* x1;        // (rows, C) of S
    const float2* stats;
    const float* norm_w;
    const void* hidden;    // (rows, H) of T
    const void* wp;        // Wp^T (C, C)
    const void* w1;        // W1^T (C, H)
    const void* w2;        // W2^T (H, C)
    const float* scale;    // as in BlockTailArgs
    void* d_x;             // (rows, C) of S
    void* branch;          // (rows, C) of T: d_x times the image's first factor, or null
    void* d_f;             // (rows, C) of T: d_out times the image's second factor, or null
    void* g;               // (rows, H) of T
    void* d_h;             // (rows, H) of T
    void* d_attn;          // (rows, C) of T
    float* d_norm_w;
    float* d_norm_b;
    float* partial;
    GradSums* later;       // or null
    int64_t rows;
    int rows_per_image, chunks;
};
struct NormLinearGrad {
    const void* d_y;       // (rows, N) of T
    const void* x;         // (rows, C) of S
    const float2* stats;
    const float* norm_w;
    const void* w0;        // W^T of the first C outputs (C, C)
    const void* w1;        // W^T of the others (C, N - C)
    const void* d_res;     // (rows, C) of S, or null
    void* d_x;             // (rows, C) of S
    float* d_norm_w;
    float* d_norm_b;
    float* partial;
    GradSums* later;       // or null
    int64_t rows;
    int chunks;
};
constexpr int kRowSumGroups = 1024;     // partial rows of a sum over all rows, at most
size_t block_backward_workspace_bytes(int64_t rows, int C);
int launch_block_tail_backward(const BlockTailGrad& a, int x_dtype, int C, int dtype, hipStream_t stream);
int launch_norm_linear_backward(const NormLinearGrad& a, int x_dtype, int C, int dtype, hipStream_t stream);

// Training pass of an attention layer beside its attention kernels (attention_train.hip).
int launch_position_bias(const float* table, const float* w, const float* b, void* bias, void* padded, int rows, int heads, int k, int dtype,
                         hipStream_t stream);
size_t position_grad_workspace_bytes(int64_t total, int heads);
int launch_position_grad(const void* d_logit, const int64_t* pe_idx, const void* padded, float* d_w, float* d_b, void* workspace, GradSums* later, int B,
                         int H, int N, int M, int rows, int k, int dtype, hipStream_t stream);
// The table of merge weights in training and its 32 parameters' gradients (merge_table.hip).
struct MergeTable {
    const float* table;    // (rows, 5)
    const float* weight;   // (4, 5)
    const float* bias;
    const float* norm_w;
    const float* norm_b;
    const float* d_out;    // (rows, 4)
    float* out;            // (rows, 4)
    float* d_params;       // (32): weight, bias, norm_w, norm_b
    int64_t rows;
    float eps;
};
int launch_merge_table(const MergeTable& a, bool backward, int dtype, hipStream_t stream);
struct DenseTrain {
    const void* qkv;       // (B, N, 3 C): [q | head 0: k v | head 1: k v ...]
    const void* bias;      // (H, rows)
    const void* padded;    // (rows, 8)
    const int64_t* pe_idx; // (B, N, N)
    const float* blank_k;
    const float* blank_v;
    const void* d_out;     // (B, N, C)
    void* out;             // (B, N, C)
    void* d_qkv;           // (B, N, 3 C)
    float* partial;
    float scale;
    int B, H, N, rows, k;
};
size_t dense_train_workspace_bytes(int B, int H);
int launch_dense_train(const DenseTrain& a, int dtype, hipStream_t stream);
int launch_dense_train_backward(const DenseTrain& a, float* d_bk, float* d_bv, float* d_w, float* d_b, int dtype, hipStream_t stream);
// d_key and d_value of a local attention from its pair lists in one launch: scale * scatter(d_logit, query) and scatter(probs, d_out)
//   into strided rows (scatter_by_cluster.hip).
bool scatter_pair_supported(const clusten_attn_shape& s, int dtype);
int launch_scatter_pair(const void* d_logit, const void* query, clusten_strides qs, void* d_key, const void* probs, const void* d_out,
                        clusten_strides gs, void* d_value, clusten_strides ys, float scale, const void* pair_lists, clusten_attn_shape s,
                        int dtype, hipStream_t stream);

// Training passes of a merge's weights and of the importance score (merge_grad.hip).
int launch_merge_weights_backward(const float* d_w, const float* table_w, const int64_t* pe_idx, const int64_t* nbhd_idx, const float* prob,
                                  const int64_t* mask, float* t, float* d_prob, int B, int N, int Nout, int M, int64_t rows, hipStream_t stream);
struct RowScore {
    const void* x;         // (rows, C) of S
    const float* weight;   // (C)
    const float* bias;     // (1), or null
    void* score;           // (rows) of T
    const void* d_score;   // (rows) of T
    void* d_x;             // (rows, C) of S: the backward; null: the forward
    float* d_weight;       // (C)
    float* d_bias;         // (C): the first value
    float* partial;
    int64_t rows;
};
int launch_row_score(const RowScore& a, int x_dtype, int C, int dtype, hipStream_t stream);

// Parameter gradients of Linear layers over the same rows (weight_grad.hip).
size_t weight_grad_workspace_bytes(const clusten_weight_grad_item* items, int count, int64_t rows, int dtype);
int launch_weight_grad(const clusten_weight_grad_item* items, int count, int64_t rows, float* workspace, int dtype, hipStream_t stream);

// Backward of a block between its products (block_grad.hip); arguments as in the C entry points.
size_t row_sums_workspace_bytes(int64_t rows, int C);
int launch_gelu_backward(const void* h, const void* d_g, void* g, void* d_h, int64_t count, int dtype, hipStream_t stream);
int launch_norm_backward(const void* d_y, const void* x, int x_dtype, const float* stats, const float* weight, const void* d_res, void* d_x,
                         void* branch, const float* scale, int rows_per_image, float* d_weight, float* d_bias, float* workspace, int64_t rows, int C,
                         int dtype, hipStream_t stream);
int launch_blank_grad(const void* q, int q_stride, const void* d_out, const float* d_logit, const float* prob, float scale, float* d_blank_k,
                      float* d_blank_v, float* workspace, GradSums* later, int B, int H, int N, int C, int dtype, hipStream_t stream);
int launch_kv_columns(const void* d_k, const void* d_v, void* d_qkv, float scale, int B, int H, int N, int ch, int dtype, hipStream_t stream);
int launch_table_linear_grad(const float* d, const void* x, float* d_w, float* d_b, int64_t rows, int heads, int k, int dtype, hipStream_t stream);

// Fill `count` fp32 / fp64 words with zero (a kernel, so that callers may capture it in a HIP graph).
//   `only_if` (may be null): a device flag; the kernel does nothing when it points to zero.
int launch_zero_f32(float* dst, size_t count, hipStream_t stream, const int32_t* only_if = nullptr);
int launch_zero_f64(double* dst, size_t count, hipStream_t stream);

// dst[i] = round(src[i]) for i < count, T in {F16, BF16}.  `only_if` as above.
int launch_round_from_f32(const float* src, void* dst, size_t count, int dtype, hipStream_t stream,
                          const int32_t* only_if = nullptr);

}  // namespace clusten
