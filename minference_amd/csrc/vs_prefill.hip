// The vertical-slash layer in one call: estimation, top-k, index build and attention on one stream and one workspace.
// Host code only.  On short prompts the host sets the pace: with an allocation for each of the dozen tensors between the
// stages and a call from Python for each stage, enqueueing a layer took longer than its kernels.  One head, 1000 to 4096
// tokens 80 -> 58 .. 68 us, a first pass on new tensors 165 -> 121; where the kernels take longer, as before.
#include "minf_common.h"
#include "vs_stages.h"

namespace {

constexpr size_t PART_ALIGN = 256;

// the parts of the workspace, in bytes from its start
struct PrefillParts {
    size_t v_idx, s_idx, block_count, block_offset, column_count, column_index, shared;   // what lives on until the attention is done
    size_t slash, estimate, tables;              // inside `shared`, until the index is built (the vertical scores first)
    size_t estimate_bytes, table_bytes, split_bytes, total;
};

PrefillParts prefill_parts(const minf_qkvo *t, int nnz_v, int nnz_s) {
    PrefillParts w;
    const size_t heads = (size_t)t->batch * t->heads_q, rows = ((size_t)t->n + 63) / 64;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + PART_ALIGN - 1) / PART_ALIGN * PART_ALIGN;
        return here;
    };
    w.v_idx = take(4 * heads * nnz_v);
    w.s_idx = take(4 * heads * nnz_s);
    w.block_count = take(4 * heads * rows);
    w.block_offset = take(4 * heads * rows * nnz_s);
    w.column_count = take(4 * heads * rows);
    w.column_index = take(4 * heads * rows * nnz_v);
    // one stretch for what the stages need for themselves: scores, their partial sums and the index builder's tables, then
    // the split walks' sums
    w.shared = at;
    w.estimate_bytes = minf_vs_estimate_workspace_bytes(t->batch, t->heads_q, t->n);
    w.table_bytes = minf_vs_index_workspace_bytes(t->batch, t->heads_q, nnz_s, (int)rows);
    w.split_bytes = minf_attn_workspace_bytes(t, MINF_OP_VERTICAL_SLASH, nnz_v, nnz_s, 0);
    take(4 * heads * t->n);
    w.slash = take(4 * heads * t->n);
    w.estimate = take(w.estimate_bytes);
    w.tables = take(w.table_bytes);              // (tables are made while other heads' scores are still selected)
    const size_t tables_end = at;
    at = w.shared;
    take(w.split_bytes);
    w.total = at > tables_end ? at : tables_end;
    return w;
}

int check(const minf_qkvo *t, int nnz_v, int nnz_s) {
    if (!t || t->batch <= 0 || t->heads_q <= 0 || t->heads_kv <= 0 || t->n <= 0) return MINF_ERR_INVALID_ARG;
    if (nnz_v < 1 || nnz_v > t->n || nnz_s < 1 || nnz_s > t->n) return MINF_ERR_INVALID_ARG;
    if (t->seqlens || t->head_list) return MINF_ERR_INVALID_ARG;
    if (t->dtype != MINF_BF16 && t->dtype != MINF_F16) return MINF_ERR_UNSUPPORTED;
    return MINF_OK;
}

}  // namespace

extern "C" size_t minf_vs_prefill_workspace_bytes(const minf_qkvo *t, int nnz_v, int nnz_s) {
    return check(t, nnz_v, nnz_s) == MINF_OK ? prefill_parts(t, nnz_v, nnz_s).total : 0;
}

extern "C" int minf_vs_prefill(const minf_qkvo *t, int nnz_v, int nnz_s, int last_q, int force_vertical, int force_slash,
                               int rounding, void *workspace, size_t workspace_bytes, void *stream) {
    int st = check(t, nnz_v, nnz_s);
    if (st != MINF_OK) return st;
    const PrefillParts w = prefill_parts(t, nnz_v, nnz_s);
    if (!workspace || workspace_bytes < w.total) return MINF_ERR_WORKSPACE;
    if ((uintptr_t)workspace & 15) return MINF_ERR_ALIGNMENT;
    char *const ws = (char *)workspace, *const shared = ws + w.shared;
    auto ints = [&](size_t at) { return (int32_t *)(ws + at); };
    float *const vertical = (float *)shared, *const slash = (float *)(ws + w.slash);
    const int heads = t->batch * t->heads_q, rows = (t->n + 63) / 64;
    if (vs_select_takes(heads, t->n)) {
        EstWindows e;
        st = vs_estimate_windows(t, last_q, force_vertical, force_slash, rounding, vertical, ws + w.estimate, w.estimate_bytes, &e, stream);
        if (st != MINF_OK) return st;
        st = vs_select(e, heads, t->n, nnz_v, ints(w.v_idx), nnz_s, ints(w.s_idx), ints(w.tables), (hipStream_t)stream);
        if (st != MINF_OK) return st;
        st = vs_index_rows(ints(w.v_idx), ints(w.s_idx), ints(w.block_count), ints(w.block_offset), ints(w.column_count),
                           ints(w.column_index), t->batch, t->heads_q, rows, nnz_v, nnz_s, ints(w.tables), (hipStream_t)stream);
    } else {
        st = minf_vs_estimate(t->q, t->k, t->q_stride, t->k_stride, t->batch, t->heads_q, t->heads_kv, t->n, t->head_dim, t->dtype,
                              t->sm_scale, last_q, force_vertical, force_slash, rounding, vertical, slash, ws + w.estimate,
                              w.estimate_bytes, stream);
        if (st != MINF_OK) return st;
        st = minf_topk_indices_pair(vertical, nnz_v, ints(w.v_idx), nnz_v, -1, slash, nnz_s, ints(w.s_idx), nnz_s, t->n - 1, heads,
                                    t->n, t->n, stream);
        if (st != MINF_OK) return st;
        st = minf_vs_index_build_full_ws(ints(w.v_idx), ints(w.s_idx), ints(w.block_count), ints(w.block_offset), ints(w.column_count),
                                         ints(w.column_index), t->batch, t->heads_q, rows, nnz_v, nnz_s, 0, nullptr,
                                         ints(w.tables), w.table_bytes, stream);
    }
    if (st != MINF_OK) return st;
    minf_qkvo a = *t;
    a.workspace = w.split_bytes ? shared : nullptr;
    a.workspace_bytes = w.split_bytes;
    return minf_vs_attn_fwd(&a, ints(w.block_count), ints(w.block_offset), ints(w.column_count), ints(w.column_index), rows,
                            nnz_s, nnz_v, stream);
}
