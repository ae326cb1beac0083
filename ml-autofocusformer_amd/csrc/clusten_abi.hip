// extern "C" surface of libclusten_hip.so (declared in include/clusten_hip.h): argument checks,
// then the internal launch functions.  Nothing here allocates, frees or synchronises.
#include "launch.hpp"

using namespace clusten;

namespace {

inline hipStream_t as_stream(clusten_stream s) { return static_cast<hipStream_t>(s); }

inline int check_attn_call(const clusten_attn_shape& s, int dtype) {
    if (!dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    return check_attn_shape(s);
}

inline bool block_dtype_ok(int dtype) { return dtype == CLUSTEN_F32 || dtype == CLUSTEN_F16 || dtype == CLUSTEN_BF16; }

inline clusten_strides contiguous_strides(const clusten_attn_shape& s) {
    clusten_strides r;
    r.n = s.C;
    r.h = (int64_t)s.N * s.C;
    r.b = (int64_t)s.H * s.N * s.C;
    return r;
}

}  // namespace

extern "C" {

int clusten_abi_version(void) { return CLUSTEN_ABI_VERSION; }

const char* clusten_status_string(int status) {
    switch (status) {
        case CLUSTEN_OK: return "ok";
        case CLUSTEN_ERR_NULL_POINTER: return "a required pointer is NULL";
        case CLUSTEN_ERR_BAD_DTYPE: return "unknown dtype code";
        case CLUSTEN_ERR_BAD_DIMS: return "a size is not positive or exceeds the 32-bit indexing limits";
        case CLUSTEN_ERR_BAD_STRIDE: return "a stride is negative or rows overlap";
        case CLUSTEN_ERR_WORKSPACE: return "workspace missing or too small";
        case CLUSTEN_ERR_LAUNCH: return "kernel launch failed";
        case CLUSTEN_ERR_UNALIGNED: return "pointer or stride is not aligned";
        case CLUSTEN_ERR_TOO_LARGE: return "problem exceeds the fixed scratch of the allocation-free entry point";
        default: return "unknown status";
    }
}

int clusten_qk_forward(const void* query, clusten_strides query_strides, const void* key, clusten_strides key_strides,
                       const int64_t* nbhd_idx, void* attn, clusten_attn_shape shape, int dtype,
                       clusten_stream stream) {
    if (!query || !key || !nbhd_idx || !attn) return CLUSTEN_ERR_NULL_POINTER;
    if (int st = check_attn_call(shape, dtype)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    return launch_gather_dot(query, query_strides, key, key_strides, nbhd_idx, attn, shape, dtype, as_stream(stream));
}

size_t clusten_qk_backward_workspace_bytes(clusten_attn_shape shape, int dtype) {
    if (!dtype_ok(dtype) || check_attn_shape(shape) != CLUSTEN_OK) return 0;
    return scatter_rows_workspace_bytes(shape, dtype);
}

int clusten_qk_backward(const void* d_attn, const void* query, clusten_strides query_strides, const void* key,
                        clusten_strides key_strides, const int64_t* nbhd_idx, void* d_query, void* d_key,
                        void* workspace, size_t workspace_bytes, clusten_attn_shape shape, int dtype,
                        clusten_stream stream) {
    if (!d_attn || !query || !key || !nbhd_idx || !d_query || !d_key) return CLUSTEN_ERR_NULL_POINTER;
    if (int st = check_attn_call(shape, dtype)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    const size_t need = scatter_rows_workspace_bytes(shape, dtype);
    if (need && (!workspace || workspace_bytes < need)) return CLUSTEN_ERR_WORKSPACE;
    // d_query = gather_sum(d_attn, key)
    int st = launch_gather_sum(d_attn, key, key_strides, nbhd_idx, d_query, contiguous_strides(shape), shape, dtype,
                               as_stream(stream));
    if (st != CLUSTEN_OK) return st;
    // d_key = scatter_rows(d_attn, query)
    return launch_scatter_rows(d_attn, query, query_strides, nbhd_idx, d_key, workspace, shape, dtype,
                               as_stream(stream));
}

int clusten_av_forward(const void* attn, const void* value, clusten_strides value_strides, const int64_t* nbhd_idx,
                       void* feat, clusten_strides feat_strides, clusten_attn_shape shape, int dtype,
                       clusten_stream stream) {
    if (!attn || !value || !nbhd_idx || !feat) return CLUSTEN_ERR_NULL_POINTER;
    if (int st = check_attn_call(shape, dtype)) return st;
    if (!strides_ok(value_strides, shape.C) || !strides_ok(feat_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    return launch_gather_sum(attn, value, value_strides, nbhd_idx, feat, feat_strides, shape, dtype,
                             as_stream(stream));
}

int clusten_av_forward_mixed(const void* attn, const void* value, clusten_strides value_strides, int value_dtype,
                             const int64_t* nbhd_idx, void* feat, clusten_strides feat_strides, clusten_attn_shape shape,
                             clusten_stream stream) {
    if (!attn || !value || !nbhd_idx || !feat) return CLUSTEN_ERR_NULL_POINTER;
    if (value_dtype != CLUSTEN_F16 && value_dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(value_strides, shape.C) || !strides_ok(feat_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    return launch_gather_sum_mixed(attn, value, value_strides, nbhd_idx, feat, feat_strides, shape, value_dtype,
                                   as_stream(stream));
}

size_t clusten_av_backward_workspace_bytes(clusten_attn_shape shape, int dtype) {
    if (!dtype_ok(dtype) || check_attn_shape(shape) != CLUSTEN_OK) return 0;
    return scatter_rows_workspace_bytes(shape, dtype);
}

int clusten_av_backward(const void* d_feat, clusten_strides d_feat_strides, const void* attn, const void* value,
                        clusten_strides value_strides, const int64_t* nbhd_idx, void* d_attn, void* d_value,
                        void* workspace, size_t workspace_bytes, clusten_attn_shape shape, int dtype,
                        clusten_stream stream) {
    if (!d_feat || !attn || !value || !nbhd_idx || !d_attn || !d_value) return CLUSTEN_ERR_NULL_POINTER;
    if (int st = check_attn_call(shape, dtype)) return st;
    if (!strides_ok(d_feat_strides, shape.C) || !strides_ok(value_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    const size_t need = scatter_rows_workspace_bytes(shape, dtype);
    if (need && (!workspace || workspace_bytes < need)) return CLUSTEN_ERR_WORKSPACE;
    // d_attn = gather_dot(d_feat, value)
    int st = launch_gather_dot(d_feat, d_feat_strides, value, value_strides, nbhd_idx, d_attn, shape, dtype,
                               as_stream(stream));
    if (st != CLUSTEN_OK) return st;
    // d_value = scatter_rows(attn, d_feat)
    return launch_scatter_rows(attn, d_feat, d_feat_strides, nbhd_idx, d_value, workspace, shape, dtype,
                               as_stream(stream));
}

int clusten_wf_forward(const void* weights, const void* feat, const int64_t* nbhd_idx, void* feat_new,
                       clusten_wf_shape shape, int dtype, clusten_stream stream) {
    if (!weights || !feat || !nbhd_idx || !feat_new) return CLUSTEN_ERR_NULL_POINTER;
    if (!dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_wf_shape(shape)) return st;
    return launch_wf_forward(weights, feat, nbhd_idx, feat_new, shape, dtype, as_stream(stream));
}

int clusten_wf_forward_mixed(const void* weights, const void* feat, int feat_dtype, const int64_t* nbhd_idx, void* feat_new,
                             clusten_wf_shape shape, clusten_stream stream) {
    if (!weights || !feat || !nbhd_idx || !feat_new) return CLUSTEN_ERR_NULL_POINTER;
    if (feat_dtype != CLUSTEN_F16 && feat_dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_wf_shape(shape)) return st;
    return launch_wf_forward_mixed(weights, feat, nbhd_idx, feat_new, shape, feat_dtype, as_stream(stream));
}

size_t clusten_wf_backward_workspace_bytes(clusten_wf_shape shape, int dtype) {
    if (!dtype_ok(dtype) || check_wf_shape(shape) != CLUSTEN_OK) return 0;
    return wf_dfeat_workspace_bytes(shape, dtype);
}

int clusten_wf_backward(const void* d_feat_new, const void* weights, const void* feat, const int64_t* nbhd_idx,
                        void* d_weights, void* d_feat, void* workspace, size_t workspace_bytes, clusten_wf_shape shape,
                        int dtype, clusten_stream stream) {
    if (!d_feat_new || !weights || !feat || !nbhd_idx || !d_weights || !d_feat) return CLUSTEN_ERR_NULL_POINTER;
    if (!dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_wf_shape(shape)) return st;
    const size_t need = wf_dfeat_workspace_bytes(shape, dtype);
    if (need && (!workspace || workspace_bytes < need)) return CLUSTEN_ERR_WORKSPACE;
    int st = launch_wf_dweights(d_feat_new, feat, nbhd_idx, d_weights, shape, dtype, as_stream(stream));
    if (st != CLUSTEN_OK) return st;
    return launch_wf_dfeat(d_feat_new, weights, nbhd_idx, d_feat, workspace, shape, dtype, as_stream(stream));
}

int clusten_cluster_size_for(int M) { return cluster_size_for(M); }

int clusten_qk_forward_clusters(const void* query, clusten_strides query_strides, const void* key,
                                clusten_strides key_strides, const int32_t* cluster_idx, void* attn,
                                clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!query || !key || !cluster_idx || !attn) return CLUSTEN_ERR_NULL_POINTER;
    if (int st = check_attn_call(shape, dtype)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    return launch_gather_dot_clusters(query, query_strides, key, key_strides, cluster_idx, attn, shape, dtype,
                                      as_stream(stream));
}

int clusten_av_forward_clusters(const void* attn, const void* value, clusten_strides value_strides,
                                const int32_t* cluster_idx, void* feat, clusten_strides feat_strides,
                                clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!attn || !value || !cluster_idx || !feat) return CLUSTEN_ERR_NULL_POINTER;
    if (int st = check_attn_call(shape, dtype)) return st;
    if (!strides_ok(value_strides, shape.C) || !strides_ok(feat_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    return launch_gather_sum_clusters(attn, value, value_strides, cluster_idx, feat, feat_strides, shape, dtype,
                                      as_stream(stream));
}

int clusten_attn_softmax_forward(const void* attn, const void* bias_table, const int64_t* pe_idx, const int64_t* mask,
                                 const float* blank_logit, const void* query, clusten_strides query_strides,
                                 const float* blank_key, float* probs, float* blank_prob, clusten_attn_shape shape,
                                 int dtype, clusten_stream stream) {
    if (!attn || !bias_table || !pe_idx || !probs || !blank_prob) return CLUSTEN_ERR_NULL_POINTER;
    if (!blank_logit && !(query && blank_key)) return CLUSTEN_ERR_NULL_POINTER;
    if (query && !strides_ok(query_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    if (dtype != CLUSTEN_F32 && dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (shape.M > 256 || shape.M % 4 != 0) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(attn) || !aligned16(probs)) return CLUSTEN_ERR_UNALIGNED;
    return launch_attn_softmax(attn, bias_table, pe_idx, mask, blank_logit, blank_logit ? nullptr : query, query_strides,
                               blank_key, probs, blank_prob, shape, dtype, as_stream(stream));
}

int clusten_cluster_attention_forward(const void* query, clusten_strides query_strides, const void* key,
                                      clusten_strides key_strides, const void* value, clusten_strides value_strides,
                                      const int32_t* cluster_idx, const void* bias_table, const int64_t* pe_idx,
                                      const int64_t* mask, int lists_shared, const float* blank_key,
                                      const float* blank_value, void* out, clusten_strides out_strides, float scale,
                                      clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!query || !key || !value || !cluster_idx || !bias_table || !pe_idx || !blank_key || !blank_value || !out) {
        return CLUSTEN_ERR_NULL_POINTER;
    }
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16 && dtype != CLUSTEN_F32) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C) || !strides_ok(value_strides, shape.C) ||
        !strides_ok(out_strides, shape.C)) {
        return CLUSTEN_ERR_BAD_STRIDE;
    }
    return launch_cluster_attention(query, query_strides, key, key_strides, value, value_strides, cluster_idx, table_by_rows(bias_table, shape.H),
                                    pe_idx, mask, blank_key, blank_value, out, out_strides, scale, lists_shared != 0, nullptr,
                                    nullptr, shape, dtype, as_stream(stream));
}

size_t clusten_cluster_attention_plan_bytes(int B, int N, int M) {
    if (B <= 0 || N <= 0) return 0;
    return cluster_attention_plan_bytes(B, N, M);
}

int clusten_cluster_attention_plan(const int32_t* cluster_idx, const int64_t* pe_idx, const int64_t* mask, void* plan,
                                   size_t plan_bytes, int B, int N, int M, clusten_stream stream) {
    if (!cluster_idx || !pe_idx || !plan) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || N <= 0 || cluster_attention_plan_bytes(1, 8, M) == 0) return CLUSTEN_ERR_BAD_DIMS;
    if (plan_bytes < cluster_attention_plan_bytes(B, N, M)) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(plan)) return CLUSTEN_ERR_UNALIGNED;
    return launch_cluster_attention_plan(cluster_idx, pe_idx, mask, plan, B, N, M, as_stream(stream));
}

int clusten_cluster_attention_forward_planned(const void* query, clusten_strides query_strides, const void* key,
                                              clusten_strides key_strides, const void* value,
                                              clusten_strides value_strides, const void* plan, const void* bias_table,
                                              int lists_shared, const float* blank_key, const float* blank_value, void* out,
                                              clusten_strides out_strides, float scale, clusten_attn_shape shape, int dtype,
                                              clusten_stream stream) {
    if (!query || !key || !value || !plan || !bias_table || !blank_key || !blank_value || !out) {
        return CLUSTEN_ERR_NULL_POINTER;
    }
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16 && dtype != CLUSTEN_F32) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C) || !strides_ok(value_strides, shape.C) ||
        !strides_ok(out_strides, shape.C)) {
        return CLUSTEN_ERR_BAD_STRIDE;
    }
    if (!aligned16(plan)) return CLUSTEN_ERR_UNALIGNED;
    return launch_cluster_attention(query, query_strides, key, key_strides, value, value_strides, nullptr, table_by_rows(bias_table, shape.H),
                                    nullptr, nullptr, blank_key, blank_value, out, out_strides, scale, lists_shared != 0, plan,
                                    nullptr, shape, dtype, as_stream(stream));
}

int clusten_cluster_attention_forward_train(const void* query, clusten_strides query_strides, const void* key,
                                            clusten_strides key_strides, const void* value, clusten_strides value_strides,
                                            const void* plan, const void* bias_table, int lists_shared,
                                            const float* blank_key, const float* blank_value, void* out,
                                            clusten_strides out_strides, float* lse, float scale, clusten_attn_shape shape,
                                            int dtype, clusten_stream stream) {
    if (!query || !key || !value || !plan || !bias_table || !blank_key || !blank_value || !out || !lse) {
        return CLUSTEN_ERR_NULL_POINTER;
    }
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16 && dtype != CLUSTEN_F32) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C) || !strides_ok(value_strides, shape.C) ||
        !strides_ok(out_strides, shape.C)) {
        return CLUSTEN_ERR_BAD_STRIDE;
    }
    if (!aligned16(plan)) return CLUSTEN_ERR_UNALIGNED;
    return launch_cluster_attention(query, query_strides, key, key_strides, value, value_strides, nullptr, table_by_rows(bias_table, shape.H),
                                    nullptr, nullptr, blank_key, blank_value, out, out_strides, scale, lists_shared != 0, plan,
                                    lse, shape, dtype, as_stream(stream));
}

int clusten_cluster_attention_backward(const void* query, clusten_strides query_strides, const void* key,
                                       clusten_strides key_strides, const void* value, clusten_strides value_strides,
                                       const void* d_out, clusten_strides d_out_strides, const void* out,
                                       clusten_strides out_strides, const float* lse, const void* plan,
                                       const void* bias_table, int lists_shared, const float* blank_key,
                                       const float* blank_value, void* d_query, clusten_strides d_query_strides,
                                       void* probs, void* d_logit, float* blank_prob, float* d_blank_logit, float scale,
                                       clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!query || !key || !value || !d_out || !out || !lse || !plan || !bias_table || !blank_key || !blank_value ||
        !d_query || !probs || !d_logit || !blank_prob || !d_blank_logit) {
        return CLUSTEN_ERR_NULL_POINTER;
    }
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16 && dtype != CLUSTEN_F32) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C) || !strides_ok(value_strides, shape.C) ||
        !strides_ok(d_out_strides, shape.C) || !strides_ok(out_strides, shape.C) || !strides_ok(d_query_strides, shape.C)) {
        return CLUSTEN_ERR_BAD_STRIDE;
    }
    if (!aligned16(plan)) return CLUSTEN_ERR_UNALIGNED;
    return launch_cluster_attention_backward(query, query_strides, key, key_strides, value, value_strides, d_out,
                                             d_out_strides, out, out_strides, lse, nullptr, table_by_rows(bias_table, shape.H), nullptr, nullptr,
                                             blank_key, blank_value, d_query, d_query_strides, probs, d_logit, blank_prob,
                                             d_blank_logit, scale, lists_shared != 0, plan, shape, dtype, as_stream(stream));
}

size_t clusten_cluster_pairs_bytes(int B, int rows, int M, int n_rows) {
    if (!cluster_pairs_supported(B, rows, M, n_rows)) return 0;
    return cluster_pairs_layout(B, rows, M, n_rows).bytes;
}

int clusten_cluster_pairs(const int64_t* nbhd_idx, void* pair_lists, size_t pair_lists_bytes, int B, int rows, int M,
                          int n_rows, clusten_stream stream) {
    if (!nbhd_idx || !pair_lists) return CLUSTEN_ERR_NULL_POINTER;
    if (!cluster_pairs_supported(B, rows, M, n_rows)) return CLUSTEN_ERR_BAD_DIMS;
    const ClusterPairsLayout l = cluster_pairs_layout(B, rows, M, n_rows);
    if (pair_lists_bytes < l.bytes) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(pair_lists)) return CLUSTEN_ERR_UNALIGNED;
    char* ws = static_cast<char*>(pair_lists);
    return launch_cluster_pairs(nbhd_idx, reinterpret_cast<int32_t*>(ws + l.keys), reinterpret_cast<int32_t*>(ws + l.wg_bad),
                                reinterpret_cast<int32_t*>(ws + l.flag),
                                reinterpret_cast<int32_t*>(ws + l.pairs), reinterpret_cast<int32_t*>(ws + l.starts),
                                reinterpret_cast<int32_t*>(ws + l.ends), B, rows, M, n_rows, as_stream(stream));
}

int clusten_cluster_pairs_from_numbers(const int32_t* cluster_idx, void* pair_lists, size_t pair_lists_bytes, int B, int rows,
                                       int nnc, int n_rows, clusten_stream stream) {
    if (!cluster_idx || !pair_lists) return CLUSTEN_ERR_NULL_POINTER;
    if (nnc <= 0 || nnc > kPairMaxSlots / 8) return CLUSTEN_ERR_BAD_DIMS;
    const int M = 8 * nnc;
    if (!cluster_pairs_supported(B, rows, M, n_rows)) return CLUSTEN_ERR_BAD_DIMS;
    const ClusterPairsLayout l = cluster_pairs_layout(B, rows, M, n_rows);
    if (pair_lists_bytes < l.bytes) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(pair_lists)) return CLUSTEN_ERR_UNALIGNED;
    char* ws = static_cast<char*>(pair_lists);
    return launch_cluster_pairs(nullptr, reinterpret_cast<int32_t*>(ws + l.keys), reinterpret_cast<int32_t*>(ws + l.wg_bad),
                                reinterpret_cast<int32_t*>(ws + l.flag), reinterpret_cast<int32_t*>(ws + l.pairs),
                                reinterpret_cast<int32_t*>(ws + l.starts), reinterpret_cast<int32_t*>(ws + l.ends), B, rows, M,
                                n_rows, as_stream(stream), cluster_idx);
}

int clusten_wf_backward_by_cluster(const void* d_feat_new, const void* weights, const void* feat, const int64_t* nbhd_idx,
                                   const void* pair_lists, void* d_weights, void* d_feat, clusten_wf_shape shape, int dtype,
                                   clusten_stream stream) {
    if (!d_feat_new || !weights || !feat || !nbhd_idx || !pair_lists || !d_weights || !d_feat) {
        return CLUSTEN_ERR_NULL_POINTER;
    }
    if (dtype != CLUSTEN_F32 && dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_wf_shape(shape)) return st;
    if (!cluster_pairs_supported(shape.B, shape.Nout, shape.M, shape.N)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(pair_lists)) return CLUSTEN_ERR_UNALIGNED;
    int st = launch_wf_dweights(d_feat_new, feat, nbhd_idx, d_weights, shape, dtype, as_stream(stream));
    if (st != CLUSTEN_OK) return st;
    const ClusterPairsLayout l = cluster_pairs_layout(shape.B, shape.Nout, shape.M, shape.N);
    const char* ws = static_cast<const char*>(pair_lists);
    return launch_wf_dfeat_by_cluster(d_feat_new, weights, reinterpret_cast<const int32_t*>(ws + l.starts),
                                      reinterpret_cast<const int32_t*>(ws + l.ends),
                                      reinterpret_cast<const int32_t*>(ws + l.pairs),
                                      reinterpret_cast<const int32_t*>(ws + l.flag), d_feat, shape, dtype, as_stream(stream));
}

int clusten_scatter_rows_by_cluster(const void* p, const void* x, clusten_strides x_strides, const void* pair_lists, void* y,
                                    clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!p || !x || !pair_lists || !y) return CLUSTEN_ERR_NULL_POINTER;
    if (dtype != CLUSTEN_F32 && dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(x_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    if (!cluster_pairs_supported(shape.B, shape.N, shape.M, shape.N)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(pair_lists)) return CLUSTEN_ERR_UNALIGNED;
    const ClusterPairsLayout l = cluster_pairs_layout(shape.B, shape.N, shape.M, shape.N);
    const char* ws = static_cast<const char*>(pair_lists);
    return launch_scatter_by_cluster(p, x, x_strides, reinterpret_cast<const int32_t*>(ws + l.starts),
                                     reinterpret_cast<const int32_t*>(ws + l.ends),
                                     reinterpret_cast<const int32_t*>(ws + l.pairs),
                                     reinterpret_cast<const int32_t*>(ws + l.flag), y, shape, dtype, as_stream(stream));
}

size_t clusten_scatter_rows_workspace_bytes(clusten_attn_shape shape, int dtype) {
    if (!dtype_ok(dtype) || check_attn_shape(shape) != CLUSTEN_OK) return 0;
    return scatter_rows_workspace_bytes(shape, dtype);
}

int clusten_scatter_rows(const void* p, const void* x, clusten_strides x_strides, const int64_t* nbhd_idx,
                         const void* pair_lists, void* y, void* workspace, size_t workspace_bytes,
                         clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!p || !x || !nbhd_idx || !y) return CLUSTEN_ERR_NULL_POINTER;
    if (int st = check_attn_call(shape, dtype)) return st;
    if (!strides_ok(x_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    const size_t need = scatter_rows_workspace_bytes(shape, dtype);
    if (need && (!workspace || workspace_bytes < need)) return CLUSTEN_ERR_WORKSPACE;
    if (pair_lists) {
        if (!cluster_pairs_supported(shape.B, shape.N, shape.M, shape.N)) return CLUSTEN_ERR_BAD_DIMS;
        if (!aligned16(pair_lists)) return CLUSTEN_ERR_UNALIGNED;
    }
    return launch_scatter_rows(p, x, x_strides, nbhd_idx, y, workspace, shape, dtype, as_stream(stream), pair_lists);
}

int clusten_dense_attention_forward(const void* query, clusten_strides query_strides, const void* key,
                                    clusten_strides key_strides, const void* value, clusten_strides value_strides,
                                    const void* bias_table, const int64_t* pe_idx, const float* blank_key,
                                    const float* blank_value, void* out, clusten_strides out_strides, float scale,
                                    clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!query || !key || !value || !bias_table || !pe_idx || !blank_key || !blank_value || !out) {
        return CLUSTEN_ERR_NULL_POINTER;
    }
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(key_strides, shape.C) || !strides_ok(value_strides, shape.C) ||
        !strides_ok(out_strides, shape.C)) {
        return CLUSTEN_ERR_BAD_STRIDE;
    }
    return launch_dense_attention(query, query_strides, key, key_strides, value, value_strides, bias_table, pe_idx,
                                  blank_key, blank_value, out, out_strides, scale, shape, dtype, as_stream(stream));
}

int clusten_linear_supported(int K, int Nout, int act) { return skinny_linear_supported(K, Nout, act) ? 1 : 0; }

int clusten_linear_forward(const void* x, int64_t x_row_stride, const void* weight, const void* bias, void* out,
                           int64_t rows, int K, int Nout, int act, int dtype, clusten_stream stream) {
    if (!x || !weight || !out) return CLUSTEN_ERR_NULL_POINTER;
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || !skinny_linear_supported(K, Nout, act)) return CLUSTEN_ERR_BAD_DIMS;
    if (x_row_stride < K || 16 * x_row_stride * 2 >= ((int64_t)1 << 32)) return CLUSTEN_ERR_BAD_STRIDE;
    if (!aligned16(x) || !aligned16(weight) || !aligned16(out) || (x_row_stride & 7) != 0) return CLUSTEN_ERR_UNALIGNED;
    if (bias && !aligned16(bias)) return CLUSTEN_ERR_UNALIGNED;
    return launch_skinny_linear(x, x_row_stride, weight, bias, out, rows, K, Nout, act, dtype, as_stream(stream));
}

static int layer_norm_call(const void* x, int in_dtype, const float* weight, const float* bias, void* out, float* stats, int64_t rows, int C,
                           float eps, int out_dtype, clusten_stream stream) {
    if (!x || !weight || !bias || !out) return CLUSTEN_ERR_NULL_POINTER;
    if (out_dtype != CLUSTEN_F32 && out_dtype != CLUSTEN_F16 && out_dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (in_dtype != CLUSTEN_F32 && in_dtype != CLUSTEN_F16 && in_dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || C <= 0 || (rows + 3) / 4 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(x) || !aligned16(weight) || !aligned16(bias) || !aligned16(out) || !aligned16(stats)) return CLUSTEN_ERR_UNALIGNED;
    return launch_layer_norm(x, in_dtype, weight, bias, out, stats, rows, C, eps, out_dtype, as_stream(stream));
}

int clusten_layer_norm_forward(const void* x, int in_dtype, const float* weight, const float* bias, void* out,
                               int64_t rows, int C, float eps, int out_dtype, clusten_stream stream) {
    return layer_norm_call(x, in_dtype, weight, bias, out, nullptr, rows, C, eps, out_dtype, stream);
}

int clusten_layer_norm_forward_train(const void* x, int in_dtype, const float* weight, const float* bias, void* out, float* stats,
                                     int64_t rows, int C, float eps, int out_dtype, clusten_stream stream) {
    if (!stats) return CLUSTEN_ERR_NULL_POINTER;
    return layer_norm_call(x, in_dtype, weight, bias, out, stats, rows, C, eps, out_dtype, stream);
}

size_t clusten_layer_norm_backward_workspace_bytes(int64_t rows, int C) { return layer_norm_backward_workspace_bytes(rows, C); }

int clusten_layer_norm_backward(const void* d_y, int dy_dtype, const void* x, int x_dtype, const float* stats, const float* weight, void* d_x,
                                float* d_weight, float* d_bias, void* workspace, size_t workspace_bytes, int64_t rows, int C,
                                clusten_stream stream) {
    if (!d_y || !x || !stats || !weight || !d_x || !d_weight || !d_bias || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    const size_t need = layer_norm_backward_workspace_bytes(rows, C);
    if (need == 0) return CLUSTEN_ERR_BAD_DIMS;
    if (workspace_bytes < need) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(d_y) || !aligned16(x) || !aligned16(stats) || !aligned16(weight) || !aligned16(d_x) || !aligned16(workspace)) {
        return CLUSTEN_ERR_UNALIGNED;
    }
    return launch_layer_norm_backward(d_y, dy_dtype, x, x_dtype, stats, weight, d_x, d_weight, d_bias, static_cast<float*>(workspace), rows, C,
                                      as_stream(stream));
}

int clusten_layer_norm_rows_forward(const void* x, int in_dtype, const int64_t* order, int group, const void* pre_bias,
                                    const float* weight, const float* bias, void* out, int64_t rows, int C, float eps,
                                    int out_dtype, clusten_stream stream) {
    if (!x || !weight || !bias || !out) return CLUSTEN_ERR_NULL_POINTER;
    if (out_dtype != CLUSTEN_F32 && out_dtype != CLUSTEN_F16 && out_dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (in_dtype != CLUSTEN_F32 && in_dtype != CLUSTEN_F16 && in_dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || C <= 0 || (rows + 3) / 4 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (order && (group <= 0 || rows % group != 0)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(x) || !aligned16(weight) || !aligned16(bias) || !aligned16(out) || (pre_bias && !aligned16(pre_bias))) {
        return CLUSTEN_ERR_UNALIGNED;
    }
    return launch_layer_norm_rows(x, in_dtype, order, order ? group : 1, pre_bias, weight, bias, out, rows, C, eps,
                                  out_dtype, as_stream(stream));
}

int clusten_channel_affine_gelu_forward(const void* x, const float* scale, const float* shift, void* y, int64_t B, int C,
                                        int HW, int dtype, clusten_stream stream) {
    if (!x || !scale || !shift || !y) return CLUSTEN_ERR_NULL_POINTER;
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (B <= 0 || C <= 0 || HW <= 0 || HW % 8 != 0) return CLUSTEN_ERR_BAD_DIMS;
    if (B * C >= 65536) return CLUSTEN_ERR_BAD_DIMS;  // one grid row per (image, channel) plane
    if (!aligned16(x) || !aligned16(y)) return CLUSTEN_ERR_UNALIGNED;
    return launch_channel_affine_gelu(x, scale, shift, y, B, C, HW, dtype, as_stream(stream));
}

int clusten_add_layer_norm_forward(const void* x, int x_dtype, const void* branch, int branch_dtype, void* sum_out,
                                   const float* weight, const float* bias, void* out, int64_t rows, int C, float eps,
                                   clusten_stream stream) {
    if (!x || !branch || !sum_out || !weight || !bias || !out) return CLUSTEN_ERR_NULL_POINTER;
    if (branch_dtype != CLUSTEN_F16 && branch_dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (x_dtype != CLUSTEN_F32 && x_dtype != branch_dtype) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || C <= 0 || (rows + 3) / 4 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(x) || !aligned16(branch) || !aligned16(sum_out) || !aligned16(weight) || !aligned16(bias) ||
        !aligned16(out)) {
        return CLUSTEN_ERR_UNALIGNED;
    }
    return launch_add_layer_norm(x, x_dtype, branch, branch_dtype, sum_out, weight, bias, out, rows, C, eps,
                                 as_stream(stream));
}

int clusten_neighbour_lists(const float* pos, const int64_t* nearest, int64_t* member_idx, int64_t* mask,
                            int64_t* pe_idx, int32_t* cluster_idx, int B, int N, int nnc, int m, int radius,
                            int table_width, clusten_stream stream) {
    if (!pos || !nearest || !member_idx || !pe_idx) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || N <= 0 || nnc <= 0 || m <= 0 || table_width <= 0) return CLUSTEN_ERR_BAD_DIMS;
    if (((int64_t)B * N * nnc * m + 255) / 256 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if ((reinterpret_cast<uintptr_t>(pos) & 7) != 0) return CLUSTEN_ERR_UNALIGNED;
    return launch_neighbour_lists(pos, nearest, member_idx, mask, pe_idx, cluster_idx, B, N, nnc, m, radius, table_width,
                                  as_stream(stream));
}

int clusten_add_row_score_forward(const void* x, int x_dtype, const void* branch, void* sum_out, const void* weight,
                                  const void* bias, void* score, int64_t rows, int C, int dtype,
                                  clusten_stream stream) {
    if (!x || !weight || !score || (branch && !sum_out)) return CLUSTEN_ERR_NULL_POINTER;
    if (dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (x_dtype != CLUSTEN_F32 && x_dtype != dtype) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || (rows + 3) / 4 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(x) || !aligned16(weight) || (branch && (!aligned16(branch) || !aligned16(sum_out)))) {
        return CLUSTEN_ERR_UNALIGNED;
    }
    return launch_add_row_score(x, x_dtype, branch, sum_out, weight, bias, score, rows, C, dtype, as_stream(stream));
}

int clusten_attn_softmax_backward(const float* probs, const float* blank_prob, const float* d_probs,
                                  const float* d_blank_prob, void* d_logit, float* d_blank_logit, int64_t rows, int M,
                                  int dtype, clusten_stream stream) {
    if (!probs || !blank_prob || !d_probs || !d_blank_prob || !d_logit || !d_blank_logit) return CLUSTEN_ERR_NULL_POINTER;
    if (dtype != CLUSTEN_F32 && dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || M <= 0 || M > 256 || M % 4 != 0 || (rows + 3) / 4 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(probs) || !aligned16(d_probs) || !aligned16(d_logit)) return CLUSTEN_ERR_UNALIGNED;
    return launch_attn_softmax_backward(probs, blank_prob, d_probs, d_blank_prob, d_logit, d_blank_logit, rows, M, dtype,
                                        as_stream(stream));
}

int clusten_bias_table_grad(const void* d_logit, const int64_t* pe_idx, float* d_table, int B, int H, int N, int M,
                            int rows, int dtype, clusten_stream stream) {
    if (!d_logit || !pe_idx || !d_table) return CLUSTEN_ERR_NULL_POINTER;
    if (dtype != CLUSTEN_F32 && dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (B <= 0 || H <= 0 || H > 65535 || N <= 0 || M <= 0 || rows <= 0) return CLUSTEN_ERR_BAD_DIMS;
    return launch_bias_table_grad(d_logit, pe_idx, d_table, B, H, N, M, rows, dtype, as_stream(stream));
}

int clusten_merge_weights_forward_rows(const float* table_weights, int64_t rows, const int64_t* pe_idx, const int64_t* nbhd_idx,
                                       const float* prob, const int64_t* mask, float* weights, int B, int N, int Nout, int M,
                                       int IC, clusten_stream stream) {
    if (!table_weights || !pe_idx || !weights) return CLUSTEN_ERR_NULL_POINTER;
    if (prob && !nbhd_idx) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || N <= 0 || Nout <= 0 || M <= 0 || IC != 4 || rows <= 0) return CLUSTEN_ERR_BAD_DIMS;
    if (((int64_t)B * Nout * M + 255) / 256 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(table_weights) || !aligned16(weights)) return CLUSTEN_ERR_UNALIGNED;
    return launch_merge_weights(table_weights, pe_idx, nbhd_idx, prob, mask, weights, B, N, Nout, M, rows, as_stream(stream));
}

int clusten_merge_weights_forward(const float* table_weights, const int64_t* pe_idx, const int64_t* nbhd_idx,
                                  const float* prob, const int64_t* mask, float* weights, int B, int N, int Nout, int M,
                                  int IC, clusten_stream stream) {
    return clusten_merge_weights_forward_rows(table_weights, INT64_MAX, pe_idx, nbhd_idx, prob, mask, weights, B, N, Nout, M, IC, stream);
}

size_t clusten_scanline_rank_workspace_bytes(int B, int N) {
    if (B <= 0 || N <= 0) return 0;
    return scanline_rank_workspace_bytes(B, N);
}

int clusten_scanline_rank(const float* pos, int64_t* ranking, void* workspace, size_t workspace_bytes, int B, int N,
                          int rows, int cols, float cell_w, float cell_h, clusten_stream stream) {
    if (!pos || !ranking || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || N <= 0 || N > scanline_rank_max_tokens() || rows <= 0 || cols <= 0 || (int64_t)rows * cols < 2 ||
        (int64_t)rows * cols >= ((int64_t)1 << 24) || !(cell_w > 0.f) || !(cell_h > 0.f)) {
        return CLUSTEN_ERR_BAD_DIMS;
    }
    if (workspace_bytes < scanline_rank_workspace_bytes(B, N)) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(workspace) || (reinterpret_cast<uintptr_t>(pos) & 7u) != 0) return CLUSTEN_ERR_UNALIGNED;
    return launch_scanline_rank(pos, ranking, workspace, B, N, rows, cols, cell_w, cell_h, as_stream(stream));
}

int clusten_scanline_rank_max_tokens(void) { return scanline_rank_max_tokens(); }

int clusten_cluster_centres(const float* pos, const int64_t* ranking, float* pos_sorted, float* centres, int B, int N, int m,
                            clusten_stream stream) {
    if (!pos || !ranking || !centres) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || N <= 0 || m <= 0 || (int64_t)B * ((N + m - 1) / m) >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if ((reinterpret_cast<uintptr_t>(pos) & 7u) != 0 || (reinterpret_cast<uintptr_t>(centres) & 7u) != 0 ||
        (reinterpret_cast<uintptr_t>(pos_sorted) & 7u) != 0) {
        return CLUSTEN_ERR_UNALIGNED;
    }
    return launch_cluster_centres(pos, ranking, pos_sorted, centres, B, N, m, as_stream(stream));
}

int clusten_gather_rows(const void* x, const int64_t* order, void* out, int64_t B, int N, int row_bytes, int order_shared,
                        clusten_stream stream) {
    if (!x || !order || !out) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || N <= 0 || row_bytes <= 0 || row_bytes % 16 != 0) return CLUSTEN_ERR_BAD_DIMS;
    if ((B * N * (row_bytes / 16) + 255) / 256 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(x) || !aligned16(out)) return CLUSTEN_ERR_UNALIGNED;
    return launch_gather_rows(x, order, out, B, N, row_bytes, order_shared, as_stream(stream));
}

int clusten_merge_centres_max_tokens(void) { return merge_centres_max_tokens(); }

int clusten_merge_centres(const float* pos, const float* min_dist, const void* learned_prob, int prob_dtype,
                          int64_t* centre, int B, int N, int sample_num, int reserve_num, int reserve_on, float alpha,
                          int stride, clusten_stream stream) {
    if (!pos || !centre) return CLUSTEN_ERR_NULL_POINTER;
    if (learned_prob && prob_dtype != CLUSTEN_F32 && prob_dtype != CLUSTEN_F16 && prob_dtype != CLUSTEN_BF16)
        return CLUSTEN_ERR_BAD_DTYPE;
    if (!(reinterpret_cast<uintptr_t>(pos) % 8 == 0)) return CLUSTEN_ERR_UNALIGNED;
    return launch_merge_centres(pos, min_dist, learned_prob, learned_prob ? prob_dtype : CLUSTEN_F32, centre, B, N,
                                sample_num, reserve_num, reserve_on, alpha, stride, as_stream(stream));
}

int clusten_merge_rows(const void* const* src, void* const* dst, const int* row_bytes, int count, const int64_t* centre,
                       int64_t B, int N, int n_out, clusten_stream stream) {
    if (!src || !dst || !row_bytes || !centre) return CLUSTEN_ERR_NULL_POINTER;
    if (count < 1 || count > 4 || B <= 0 || N <= 0 || n_out <= 0) return CLUSTEN_ERR_BAD_DIMS;
    int64_t words = 0;
    for (int t = 0; t < count; ++t) words += row_bytes[t] / 8;
    if ((B * n_out * words + 255) / 256 >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    return launch_merge_rows(src, dst, row_bytes, count, centre, B, N, n_out, as_stream(stream));
}

int clusten_knn2d(const float* query, const float* database, int64_t* idx, float* dist, int B, int Nq, int N, int K,
                  clusten_stream stream) {
    if (!query || !database || !idx) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || Nq <= 0 || N <= 0 || K < 1 || K > 8 || K > N) return CLUSTEN_ERR_BAD_DIMS;
    if ((int64_t)B * ((Nq + 255) / 256) >= ((int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    return launch_knn2d(query, database, idx, dist, B, Nq, N, K, as_stream(stream));
}

int clusten_block_pack(const clusten_pack_item* items, int count, int C, int dtype, clusten_stream stream) {
    if (!items) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (count <= 0 || !block_width_supported(C)) return CLUSTEN_ERR_BAD_DIMS;
    for (int i = 0; i < count; ++i) {
        const clusten_pack_item& it = items[i];
        if (!it.src || !it.dst) return CLUSTEN_ERR_NULL_POINTER;
        if (it.n <= 0 || it.k <= 0 || it.n % C != 0 || it.k % C != 0) return CLUSTEN_ERR_BAD_DIMS;
        if (!aligned16(it.dst)) return CLUSTEN_ERR_UNALIGNED;
    }
    return launch_block_pack(items, count, C, dtype, as_stream(stream));
}

int clusten_norm_linear_forward(const void* x, int x_dtype, const float* norm_w, const float* norm_b, float eps,
                                const void* w, const float* bias0, const float* bias1, void* out, void* normed,
                                float* stats, int64_t rows, int C, int N, int dtype, clusten_stream stream) {
    if (!x || !norm_w || !norm_b || !w || !bias0 || !out || (N > C && !bias1)) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype) || (x_dtype != dtype && x_dtype != CLUSTEN_F32)) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || rows >= (int64_t)1 << 31 || !block_width_supported(C) || N <= 0 || N % C != 0) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(x) || !aligned16(norm_w) || !aligned16(norm_b) || !aligned16(w) || !aligned16(bias0) || !aligned16(bias1) ||
        !aligned16(out) || !aligned16(normed) || (reinterpret_cast<uintptr_t>(stats) & 7)) {
        return CLUSTEN_ERR_UNALIGNED;
    }
    NormLinearArgs a = {};
    a.x = x, a.norm_w = norm_w, a.norm_b = norm_b, a.w = w, a.bias0 = bias0, a.bias1 = bias1, a.out = out, a.normed = normed;
    a.stats = reinterpret_cast<float2*>(stats), a.rows = rows, a.chunks = N / C, a.eps = eps;
    return launch_norm_linear(a, x_dtype, C, dtype, as_stream(stream));
}

int clusten_block_tail_forward(const void* attn, const void* x, int x_dtype, const void* wp, const float* bp,
                               const float* norm_w, const float* norm_b, float eps, const void* w1, const float* b1,
                               const void* w2, const float* b2, void* out, const float* scale, int rows_per_image,
                               void* x1, void* normed, void* hidden, float* stats, int64_t rows, int C, int H, int dtype,
                               clusten_stream stream) {
    if (!attn || !x || !wp || !bp || !norm_w || !norm_b || !w1 || !b1 || !w2 || !b2 || !out) return CLUSTEN_ERR_NULL_POINTER;
    const int kept = (x1 != nullptr) + (normed != nullptr) + (hidden != nullptr) + (stats != nullptr);
    if (kept != 0 && kept != 4) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype) || (x_dtype != dtype && x_dtype != CLUSTEN_F32)) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || rows >= (int64_t)1 << 31 || !block_width_supported(C) || H <= 0 || H % C != 0) return CLUSTEN_ERR_BAD_DIMS;
    if (scale && (rows_per_image <= 0 || rows % rows_per_image != 0)) return CLUSTEN_ERR_BAD_DIMS;
    const void* all[] = {attn, x, wp, bp, norm_w, norm_b, w1, b1, w2, b2, out, x1, normed, hidden};
    for (const void* p : all) {
        if (!aligned16(p)) return CLUSTEN_ERR_UNALIGNED;
    }
    if (reinterpret_cast<uintptr_t>(stats) & 7) return CLUSTEN_ERR_UNALIGNED;
    BlockTailArgs a = {};
    a.attn = attn, a.x = x, a.wp = wp, a.bp = bp, a.norm_w = norm_w, a.norm_b = norm_b, a.w1 = w1, a.b1 = b1, a.w2 = w2;
    a.b2 = b2, a.out = out, a.scale = scale, a.rows_per_image = scale ? rows_per_image : 1, a.chunks = H / C, a.rows = rows;
    a.eps = eps, a.x1 = x1, a.normed = normed, a.hidden = hidden, a.stats = reinterpret_cast<float2*>(stats);
    return launch_block_tail(a, x_dtype, C, dtype, as_stream(stream));
}

int clusten_blocks_forward(const clusten_block* blocks, int count, const void* x, int x_dtype, void* out, void* qkv, void* attn,
                           const void* plan, int lists_shared, const int64_t* pe_idx, clusten_attn_shape shape, int hidden,
                           float scale, int dtype, clusten_stream stream) {
    return clusten_blocks_forward_tables(blocks, count, x, x_dtype, out, qkv, attn, plan, lists_shared, pe_idx, 0, shape, hidden, scale, dtype,
                                         stream);
}

int clusten_blocks_forward_tables(const clusten_block* blocks, int count, const void* x, int x_dtype, void* out, void* qkv, void* attn,
                                  const void* plan, int lists_shared, const int64_t* pe_idx, int table_rows, clusten_attn_shape shape,
                                  int hidden, float scale, int dtype, clusten_stream stream) {
    // attention over all tokens: 16-bit data by matrix instructions with (rows, heads) tables, fp32 by the training pass' forward kernel,
    // which takes them by heads.  A forward of 50 images in fp32, five such layers of 49 tokens and 16 heads: 6334 us with an
    // fp32 layer's library products, gather, copies and softmax (20 launches between norm_linear and block_tail), 5690 with the kernel.
    const bool by_heads = plan ? table_rows > 0 : dtype == CLUSTEN_F32;
    if (table_rows < 0 || (!plan && by_heads != (table_rows > 0))) return CLUSTEN_ERR_BAD_DIMS;
    if (!plan && by_heads && (shape.C != 32 || shape.N > 64 || (int64_t)shape.B * shape.H >= (int64_t)1 << 31)) return CLUSTEN_ERR_BAD_DIMS;
    if (plan && !aligned16(plan)) return CLUSTEN_ERR_UNALIGNED;
    if (!blocks || !x || !out || !qkv || !attn || (!plan && !pe_idx)) return CLUSTEN_ERR_NULL_POINTER;
    if (count <= 0) return CLUSTEN_ERR_BAD_DIMS;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    const int C = shape.H * shape.C;
    const int64_t rows = (int64_t)shape.B * shape.N;
    const size_t elem = dtype_size(dtype);
    // q, k and v inside the rows of the projections' output: [q | head 0: k v | head 1: k v ...]
    clusten_strides qs, kv, os;
    qs.b = (int64_t)shape.N * 3 * C, qs.n = 3 * C, qs.h = shape.C;
    kv = qs, kv.h = 2 * shape.C;
    os.b = (int64_t)shape.N * C, os.n = C, os.h = shape.C;
    char* q = static_cast<char*>(qkv);
    char* k = q + (size_t)C * elem;
    char* v = k + (size_t)shape.C * elem;
    for (int i = 0; i < count; ++i) {
        const clusten_block& b = blocks[i];
        const void* in = i == 0 ? x : out;
        if (int st = clusten_norm_linear_forward(in, x_dtype, b.norm1_w, b.norm1_b, b.eps1, b.w_qkv, b.b_q, b.b_kv, qkv, nullptr,
                                                 nullptr, rows, C, 3 * C, dtype, stream)) {
            return st;
        }
        if (!b.bias_table || !b.blank_k || !b.blank_v) return CLUSTEN_ERR_NULL_POINTER;
        int st;
        if (plan) {
            st = launch_cluster_attention(q, qs, k, kv, v, kv, nullptr,
                                          by_heads ? table_by_heads(b.bias_table, table_rows) : table_by_rows(b.bias_table, shape.H), nullptr,
                                          nullptr, b.blank_k, b.blank_v, attn, os, scale, lists_shared != 0, plan, nullptr, shape, dtype,
                                          as_stream(stream));
        } else if (by_heads) {
            st = clusten_dense_attention_train_forward(qkv, b.bias_table, pe_idx, b.blank_k, b.blank_v, attn, scale, shape.B, shape.H, shape.N,
                                                       table_rows, dtype, stream);
        } else {
            st = clusten_dense_attention_forward(q, qs, k, kv, v, kv, b.bias_table, pe_idx, b.blank_k, b.blank_v, attn, os, scale, shape, dtype,
                                                 stream);
        }
        if (st) return st;
        // a workgroup of the tail reads its own rows only, all of them before it writes the first: in place from block 1 on
        if (int st2 = clusten_block_tail_forward(attn, in, x_dtype, b.w_proj, b.b_proj, b.norm2_w, b.norm2_b, b.eps2, b.w1, b.b1,
                                                 b.w2, b.b2, out, nullptr, 1, nullptr, nullptr, nullptr, nullptr, rows, C, hidden,
                                                 dtype, stream)) {
            return st2;
        }
    }
    return CLUSTEN_OK;
}

size_t clusten_block_backward_workspace_bytes(int64_t rows, int C) {
    return rows > 0 && rows < (int64_t)1 << 31 && block_width_supported(C) ? block_backward_workspace_bytes(rows, C) : 0;
}

int clusten_block_tail_backward(const void* d_out, const void* x1, int x_dtype, const float* stats, const float* norm_w, const void* hidden,
                                const void* wp_t, const void* w1_t, const void* w2_t, const float* scale, int rows_per_image, void* d_x,
                                void* branch, void* d_f, void* g, void* d_h, void* d_attn, float* d_norm_w, float* d_norm_b, void* workspace,
                                size_t workspace_bytes, int64_t rows, int C, int H, int dtype, clusten_stream stream) {
    if (!d_out || !x1 || !stats || !norm_w || !hidden || !wp_t || !w1_t || !w2_t || !d_x || !g || !d_h || !d_attn || !d_norm_w || !d_norm_b ||
        !workspace) {
        return CLUSTEN_ERR_NULL_POINTER;
    }
    if (!block_dtype_ok(dtype) || (x_dtype != dtype && x_dtype != CLUSTEN_F32)) return CLUSTEN_ERR_BAD_DTYPE;
    const size_t need = clusten_block_backward_workspace_bytes(rows, C);
    if (need == 0 || H <= 0 || H % C != 0) return CLUSTEN_ERR_BAD_DIMS;
    if (scale && (rows_per_image <= 0 || rows % rows_per_image != 0)) return CLUSTEN_ERR_BAD_DIMS;
    if (workspace_bytes < need) return CLUSTEN_ERR_WORKSPACE;
    const void* all[] = {d_out, x1, norm_w, hidden, wp_t, w1_t, w2_t, d_x, branch, d_f, g, d_h, d_attn, workspace};
    for (const void* p : all) {
        if (!aligned16(p)) return CLUSTEN_ERR_UNALIGNED;
    }
    if (reinterpret_cast<uintptr_t>(stats) & 7) return CLUSTEN_ERR_UNALIGNED;
    BlockTailGrad a = {};
    a.d_out = d_out, a.x1 = x1, a.stats = reinterpret_cast<const float2*>(stats), a.norm_w = norm_w, a.hidden = hidden, a.wp = wp_t, a.w1 = w1_t;
    a.w2 = w2_t, a.scale = scale, a.d_x = d_x, a.branch = branch, a.d_f = d_f, a.g = g, a.d_h = d_h, a.d_attn = d_attn, a.d_norm_w = d_norm_w;
    a.d_norm_b = d_norm_b, a.partial = static_cast<float*>(workspace), a.rows = rows, a.rows_per_image = scale ? rows_per_image : 1;
    a.chunks = H / C;
    return launch_block_tail_backward(a, x_dtype, C, dtype, as_stream(stream));
}

int clusten_norm_linear_backward(const void* d_y, const void* x, int x_dtype, const float* stats, const float* norm_w, const void* w0_t,
                                 const void* w1_t, const void* d_res, void* d_x, float* d_norm_w, float* d_norm_b, void* workspace, size_t workspace_bytes,
                                 int64_t rows, int C, int N, int dtype, clusten_stream stream) {
    if (!d_y || !x || !stats || !norm_w || !w0_t || (N > C && !w1_t) || !d_x || !d_norm_w || !d_norm_b || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype) || (x_dtype != dtype && x_dtype != CLUSTEN_F32)) return CLUSTEN_ERR_BAD_DTYPE;
    const size_t need = clusten_block_backward_workspace_bytes(rows, C);
    if (need == 0 || N <= 0 || N % C != 0) return CLUSTEN_ERR_BAD_DIMS;
    if (workspace_bytes < need) return CLUSTEN_ERR_WORKSPACE;
    const void* all[] = {d_y, x, norm_w, w0_t, w1_t, d_res, d_x, workspace};
    for (const void* p : all) {
        if (!aligned16(p)) return CLUSTEN_ERR_UNALIGNED;
    }
    if (reinterpret_cast<uintptr_t>(stats) & 7) return CLUSTEN_ERR_UNALIGNED;
    NormLinearGrad a = {};
    a.d_y = d_y, a.x = x, a.stats = reinterpret_cast<const float2*>(stats), a.norm_w = norm_w, a.w0 = w0_t, a.w1 = w1_t, a.d_res = d_res;
    a.d_x = d_x, a.d_norm_w = d_norm_w, a.d_norm_b = d_norm_b, a.partial = static_cast<float*>(workspace), a.rows = rows, a.chunks = N / C;
    return launch_norm_linear_backward(a, x_dtype, C, dtype, as_stream(stream));
}

size_t clusten_row_sums_workspace_bytes(int64_t rows, int C) {
    return rows > 0 && rows < (int64_t)1 << 31 && block_width_supported(C) ? row_sums_workspace_bytes(rows, C) : 0;
}

int clusten_gelu_backward(const void* h, const void* d_g, void* g, void* d_h, int64_t count, int dtype, clusten_stream stream) {
    if (!h || !d_g || !g || !d_h) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (count <= 0 || count % 8 != 0 || count >= (int64_t)1 << 40) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(h) || !aligned16(d_g) || !aligned16(g) || !aligned16(d_h)) return CLUSTEN_ERR_UNALIGNED;
    return launch_gelu_backward(h, d_g, g, d_h, count, dtype, as_stream(stream));
}

int clusten_norm_backward(const void* d_y, const void* x, int x_dtype, const float* stats, const float* weight, const void* d_res,
                          void* d_x, void* branch, const float* scale, int rows_per_image, float* d_weight, float* d_bias,
                          void* workspace, size_t workspace_bytes, int64_t rows, int C, int dtype, clusten_stream stream) {
    if (!d_y || !x || !stats || !weight || !d_x || !d_weight || !d_bias || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype) || (x_dtype != dtype && x_dtype != CLUSTEN_F32)) return CLUSTEN_ERR_BAD_DTYPE;
    const size_t need = clusten_row_sums_workspace_bytes(rows, C);
    if (need == 0 || (scale && (rows_per_image <= 0 || rows % rows_per_image != 0))) return CLUSTEN_ERR_BAD_DIMS;
    if (workspace_bytes < need) return CLUSTEN_ERR_TOO_LARGE;
    const void* all[] = {d_y, x, weight, d_res, d_x, branch, workspace};
    for (const void* p : all) {
        if (!aligned16(p)) return CLUSTEN_ERR_UNALIGNED;
    }
    if (reinterpret_cast<uintptr_t>(stats) & 7) return CLUSTEN_ERR_UNALIGNED;
    return launch_norm_backward(d_y, x, x_dtype, stats, weight, d_res, d_x, branch, scale, scale ? rows_per_image : 1, d_weight, d_bias,
                                static_cast<float*>(workspace), rows, C, dtype, as_stream(stream));
}

int clusten_blank_grad(const void* q, int q_stride, const void* d_out, const float* d_logit, const float* prob, float scale,
                       float* d_blank_k, float* d_blank_v, void* workspace, size_t workspace_bytes, int B, int H, int N, int C,
                       int dtype, clusten_stream stream) {
    if (!q || !d_out || !d_logit || !prob || !d_blank_k || !d_blank_v || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (B <= 0 || N <= 0 || H <= 0 || C <= 0 || C % H != 0 || C / H % 8 != 0 || q_stride < C || q_stride % 8 != 0) return CLUSTEN_ERR_BAD_DIMS;
    const size_t need = clusten_row_sums_workspace_bytes((int64_t)B * N, C);
    if (need == 0) return CLUSTEN_ERR_BAD_DIMS;
    if (workspace_bytes < need) return CLUSTEN_ERR_TOO_LARGE;
    if (!aligned16(q) || !aligned16(d_out) || !aligned16(workspace)) return CLUSTEN_ERR_UNALIGNED;
    return launch_blank_grad(q, q_stride, d_out, d_logit, prob, scale, d_blank_k, d_blank_v, static_cast<float*>(workspace), nullptr, B, H, N, C,
                             dtype, as_stream(stream));
}

int clusten_kv_columns(const void* d_k, const void* d_v, void* d_qkv, float scale, int B, int H, int N, int ch, int dtype,
                       clusten_stream stream) {
    if (!d_k || !d_v || !d_qkv) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (B <= 0 || H <= 0 || N <= 0 || ch <= 0 || ch % 8 != 0 || (int64_t)B * N >= (int64_t)1 << 31 || (int64_t)H * ch > 1 << 16) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(d_k) || !aligned16(d_v) || !aligned16(d_qkv)) return CLUSTEN_ERR_UNALIGNED;
    return launch_kv_columns(d_k, d_v, d_qkv, scale, B, H, N, ch, dtype, as_stream(stream));
}

int clusten_table_linear_grad(const float* d, const void* x, float* d_weight, float* d_bias, int64_t rows, int n, int k, int dtype,
                              clusten_stream stream) {
    if (!d || !x || !d_weight || !d_bias) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || n <= 0 || n > 1024 || k <= 0 || k > 8) return CLUSTEN_ERR_BAD_DIMS;
    return launch_table_linear_grad(d, x, d_weight, d_bias, rows, n, k, dtype, as_stream(stream));
}

int clusten_position_bias(const float* table, const float* weight, const float* bias_param, void* bias, void* padded, int rows, int n, int k,
                          int dtype, clusten_stream stream) {
    if (!table || !weight || !bias) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || n <= 0 || k <= 0 || k > 8 || (int64_t)rows * n >= (int64_t)1 << 31) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(bias) || !aligned16(padded)) return CLUSTEN_ERR_UNALIGNED;
    return launch_position_bias(table, weight, bias_param, bias, padded, rows, n, k, dtype, as_stream(stream));
}

size_t clusten_position_grad_workspace_bytes(int B, int H, int N, int M) {
    return B > 0 && H > 0 && N > 0 && M > 0 ? position_grad_workspace_bytes((int64_t)B * N * M, H) : 0;
}

int clusten_position_grad(const void* d_logit, const int64_t* pe_idx, const void* padded, float* d_weight, float* d_bias, void* workspace,
                          size_t workspace_bytes, int B, int H, int N, int M, int rows, int k, int dtype, clusten_stream stream) {
    if (!d_logit || !pe_idx || !padded || !d_weight || !d_bias || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (B <= 0 || H <= 0 || H > 65535 || N <= 0 || M <= 0 || M % 4 != 0 || rows <= 0 || k <= 0 || k > 5) return CLUSTEN_ERR_BAD_DIMS;
    if (workspace_bytes < clusten_position_grad_workspace_bytes(B, H, N, M)) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(d_logit) || !aligned16(padded) || !aligned16(workspace)) return CLUSTEN_ERR_UNALIGNED;
    return launch_position_grad(d_logit, pe_idx, padded, d_weight, d_bias, workspace, nullptr, B, H, N, M, rows, k, dtype, as_stream(stream));
}

static int dense_train_args(DenseTrain& a, const void* qkv, const void* bias, const int64_t* pe_idx, const float* blank_k, const float* blank_v,
                            float scale, int B, int H, int N, int rows, int dtype) {
    if (!qkv || !bias || !pe_idx || !blank_k || !blank_v) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (B <= 0 || H <= 0 || N <= 0 || N > 64 || rows <= 0 || (int64_t)B * H >= (int64_t)1 << 31 || H > 1 << 16) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(qkv)) return CLUSTEN_ERR_UNALIGNED;
    a = {};
    a.qkv = qkv, a.bias = bias, a.pe_idx = pe_idx, a.blank_k = blank_k, a.blank_v = blank_v, a.scale = scale, a.B = B, a.H = H, a.N = N;
    a.rows = rows;
    return CLUSTEN_OK;
}

int clusten_dense_attention_train_forward(const void* qkv, const void* bias, const int64_t* pe_idx, const float* blank_k, const float* blank_v,
                                          void* out, float scale, int B, int H, int N, int rows, int dtype, clusten_stream stream) {
    DenseTrain a;
    if (int st = dense_train_args(a, qkv, bias, pe_idx, blank_k, blank_v, scale, B, H, N, rows, dtype)) return st;
    if (!out) return CLUSTEN_ERR_NULL_POINTER;
    if (!aligned16(out)) return CLUSTEN_ERR_UNALIGNED;
    a.out = out;
    return launch_dense_train(a, dtype, as_stream(stream));
}

size_t clusten_dense_attention_train_workspace_bytes(int B, int H) { return B > 0 && H > 0 ? dense_train_workspace_bytes(B, H) : 0; }

int clusten_dense_attention_train_backward(const void* qkv, const void* bias, const void* padded, const int64_t* pe_idx, const float* blank_k,
                                           const float* blank_v, const void* d_out, void* d_qkv, float* d_blank_k, float* d_blank_v,
                                           float* d_weight, float* d_bias, void* workspace, size_t workspace_bytes, float scale, int B, int H,
                                           int N, int rows, int k, int dtype, clusten_stream stream) {
    DenseTrain a;
    if (int st = dense_train_args(a, qkv, bias, pe_idx, blank_k, blank_v, scale, B, H, N, rows, dtype)) return st;
    if (!padded || !d_out || !d_qkv || !d_blank_k || !d_blank_v || !d_weight || !d_bias || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    if (k <= 0 || k > 5) return CLUSTEN_ERR_BAD_DIMS;
    if (workspace_bytes < clusten_dense_attention_train_workspace_bytes(B, H)) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(padded) || !aligned16(d_out) || !aligned16(d_qkv) || !aligned16(workspace)) return CLUSTEN_ERR_UNALIGNED;
    a.padded = padded, a.d_out = d_out, a.d_qkv = d_qkv, a.partial = static_cast<float*>(workspace), a.k = k;
    return launch_dense_train_backward(a, d_blank_k, d_blank_v, d_weight, d_bias, dtype, as_stream(stream));
}

int clusten_scatter_attention_pair(const void* d_logit, const void* query, clusten_strides query_strides, void* d_key, const void* probs,
                                   const void* d_out, clusten_strides d_out_strides, void* d_value, clusten_strides out_strides, float scale,
                                   const void* pair_lists, clusten_attn_shape shape, int dtype, clusten_stream stream) {
    if (!d_logit || !query || !d_key || !probs || !d_out || !d_value || !pair_lists) return CLUSTEN_ERR_NULL_POINTER;
    if (dtype != CLUSTEN_F32 && dtype != CLUSTEN_F16 && dtype != CLUSTEN_BF16) return CLUSTEN_ERR_BAD_DTYPE;
    if (int st = check_attn_shape(shape)) return st;
    if (!strides_ok(query_strides, shape.C) || !strides_ok(d_out_strides, shape.C) || !strides_ok(out_strides, shape.C)) return CLUSTEN_ERR_BAD_STRIDE;
    if (!cluster_pairs_supported(shape.B, shape.N, shape.M, shape.N)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(pair_lists)) return CLUSTEN_ERR_UNALIGNED;
    return launch_scatter_pair(d_logit, query, query_strides, d_key, probs, d_out, d_out_strides, d_value, out_strides, scale, pair_lists, shape,
                               dtype, as_stream(stream));
}

static int merge_table_call(MergeTable a, bool backward, int dtype, clusten_stream stream) {
    if (!a.table || !a.weight || !a.bias || !a.norm_w || !a.norm_b || (backward ? !a.d_out || !a.d_params : !a.out)) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (a.rows <= 0 || a.rows >= (int64_t)1 << 31) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(a.d_out) || !aligned16(a.out)) return CLUSTEN_ERR_UNALIGNED;
    return launch_merge_table(a, backward, dtype, as_stream(stream));
}

int clusten_merge_table_forward(const float* table, const float* weight, const float* bias, const float* norm_w, const float* norm_b, float eps,
                                float* out, int64_t rows, int dtype, clusten_stream stream) {
    return merge_table_call(MergeTable{table, weight, bias, norm_w, norm_b, nullptr, out, nullptr, rows, eps}, false, dtype, stream);
}

int clusten_merge_table_backward(const float* d_out, const float* table, const float* weight, const float* bias, const float* norm_w,
                                 const float* norm_b, float eps, float* d_params, int64_t rows, int dtype, clusten_stream stream) {
    return merge_table_call(MergeTable{table, weight, bias, norm_w, norm_b, d_out, nullptr, d_params, rows, eps}, true, dtype, stream);
}

int clusten_merge_weights_backward_rows(const float* d_weights, const float* table_weights, int64_t rows, const int64_t* pe_idx,
                                        const int64_t* nbhd_idx, const float* prob, const int64_t* mask, float* d_rows, float* d_prob,
                                        int B, int N, int Nout, int M, clusten_stream stream) {
    if (!d_weights || !pe_idx || !d_rows || (prob && (!table_weights || !nbhd_idx || !d_prob))) return CLUSTEN_ERR_NULL_POINTER;
    if (B <= 0 || N <= 0 || Nout <= 0 || M <= 0 || rows <= 0 || ((int64_t)B * Nout * M + 255) / 256 >= (int64_t)1 << 31) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(d_weights) || !aligned16(table_weights) || !aligned16(d_prob)) return CLUSTEN_ERR_UNALIGNED;
    return launch_merge_weights_backward(d_weights, table_weights, pe_idx, nbhd_idx, prob, mask, d_rows, prob ? d_prob : nullptr, B, N, Nout, M,
                                         rows, as_stream(stream));
}

int clusten_merge_weights_backward(const float* d_weights, const float* table_weights, const int64_t* pe_idx, const int64_t* nbhd_idx,
                                   const float* prob, const int64_t* mask, float* d_rows, float* d_prob, int B, int N, int Nout, int M,
                                   clusten_stream stream) {
    return clusten_merge_weights_backward_rows(d_weights, table_weights, INT64_MAX, pe_idx, nbhd_idx, prob, mask, d_rows, d_prob, B, N, Nout, M,
                                               stream);
}

static int row_score_args(RowScore& a, const void* x, int x_dtype, const float* weight, void* score, int64_t rows, int C, int dtype) {
    if (!x || !weight || !score) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype) || (x_dtype != dtype && x_dtype != CLUSTEN_F32)) return CLUSTEN_ERR_BAD_DTYPE;
    if (rows <= 0 || rows >= (int64_t)1 << 31 || !block_width_supported(C)) return CLUSTEN_ERR_BAD_DIMS;
    if (!aligned16(x) || !aligned16(weight)) return CLUSTEN_ERR_UNALIGNED;
    a = {};
    a.x = x, a.weight = weight, a.score = score, a.rows = rows;
    return CLUSTEN_OK;
}

int clusten_row_score_forward(const void* x, int x_dtype, const float* weight, const float* bias, void* score, int64_t rows, int C, int dtype,
                              clusten_stream stream) {
    RowScore a;
    if (int st = row_score_args(a, x, x_dtype, weight, score, rows, C, dtype)) return st;
    a.bias = bias;
    return launch_row_score(a, x_dtype, C, dtype, as_stream(stream));
}

int clusten_row_score_backward(const void* x, int x_dtype, const float* weight, const void* score, const void* d_score, void* d_x,
                               float* d_weight, float* d_bias, void* workspace, size_t workspace_bytes, int64_t rows, int C, int dtype,
                               clusten_stream stream) {
    RowScore a;
    if (int st = row_score_args(a, x, x_dtype, weight, const_cast<void*>(score), rows, C, dtype)) return st;
    if (!d_score || !d_x || !d_weight || !d_bias || !workspace) return CLUSTEN_ERR_NULL_POINTER;
    if (workspace_bytes < row_sums_workspace_bytes(rows, C)) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(d_x) || !aligned16(workspace)) return CLUSTEN_ERR_UNALIGNED;
    a.d_score = d_score, a.d_x = d_x, a.d_weight = d_weight, a.d_bias = d_bias, a.partial = static_cast<float*>(workspace);
    return launch_row_score(a, x_dtype, C, dtype, as_stream(stream));
}

static int check_weight_grad(const clusten_weight_grad_item* items, int count, int64_t rows, int dtype) {
    if (!items) return CLUSTEN_ERR_NULL_POINTER;
    if (!block_dtype_ok(dtype)) return CLUSTEN_ERR_BAD_DTYPE;
    if (count < 1 || count > 8 || rows <= 0 || rows >= (int64_t)1 << 31) return CLUSTEN_ERR_BAD_DIMS;
    for (int i = 0; i < count; ++i) {
        const clusten_weight_grad_item& it = items[i];
        if (it.n <= 0 || it.k <= 0 || it.n % 8 != 0 || it.k % 8 != 0 || (int64_t)it.n * it.k >= (int64_t)1 << 26 ||
            it.d_y_stride < it.n || it.x_stride < it.k || it.d_y_stride >= (int64_t)1 << 24 || it.x_stride >= (int64_t)1 << 24) {
            return CLUSTEN_ERR_BAD_DIMS;
        }
    }
    return CLUSTEN_OK;
}

size_t clusten_weight_grad_workspace_bytes(const clusten_weight_grad_item* items, int count, int64_t rows, int dtype) {
    return check_weight_grad(items, count, rows, dtype) == CLUSTEN_OK ? weight_grad_workspace_bytes(items, count, rows, dtype) : 0;
}

int clusten_weight_grad(const clusten_weight_grad_item* items, int count, int64_t rows, void* workspace, size_t workspace_bytes,
                        int dtype, clusten_stream stream) {
    if (int st = check_weight_grad(items, count, rows, dtype)) return st;
    const int64_t elem = (int64_t)dtype_size(dtype);
    for (int i = 0; i < count; ++i) {
        const clusten_weight_grad_item& it = items[i];
        if (!it.d_y || !it.x || !it.d_weight) return CLUSTEN_ERR_NULL_POINTER;
        if (!aligned16(it.d_y) || !aligned16(it.x) || !aligned16(it.d_weight) || !aligned16(it.d_bias) ||
            it.d_y_stride * elem % 16 != 0 || it.x_stride * elem % 16 != 0) {
            return CLUSTEN_ERR_UNALIGNED;
        }
    }
    if (!workspace || workspace_bytes < weight_grad_workspace_bytes(items, count, rows, dtype)) return CLUSTEN_ERR_WORKSPACE;
    if (!aligned16(workspace)) return CLUSTEN_ERR_UNALIGNED;
    return launch_weight_grad(items, count, rows, static_cast<float*>(workspace), dtype, as_stream(stream));
}

}  // extern "C"
