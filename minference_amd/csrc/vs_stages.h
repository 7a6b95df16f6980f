// What the stages of the vertical-slash layer hand to each other inside the library (vs_prefill.hip).
#pragma once
#include "minf_common.h"

// The estimation's sums before its last kernel: vertical sums without their forced entries, the diagonal sums as windows
// of nchunks chunks of kc keys (a power of two) and EST_WINDOW_TAIL more positions each
constexpr int EST_WINDOW_TAIL = 64;
struct EstWindows {
    const float *vertical;       // [batch * heads, n]
    const float *windows;        // [batch * heads, nchunks, kc + EST_WINDOW_TAIL]
    int kc_log2, nchunks, force_v, force_s;
};
// entry i of a head's diagonal sums: position i % kc of its chunk, and where the chunk before it reaches that far (keys
// of that chunk seen by later rows), position kc + i % kc of that one, which is added first
__device__ __forceinline__ float est_slash(const float *windows, int kc_log2, int i) {
    const int kc = 1 << kc_log2, width = kc + EST_WINDOW_TAIL, c = i >> kc_log2, off = i & (kc - 1);
    const bool two = c > 0 && off < EST_WINDOW_TAIL;
    const float *here = windows + (long long)c * width + off;
    const float v = *here, before = *(two ? here - width + kc : here);       // (no branch between the loads of several entries)
    return two ? before + v : v;
}

// minf_vs_estimate but for its last kernel
int vs_estimate_windows(const minf_qkvo *t, int last_q, int force_vertical, int force_slash, int rounding, float *vertical,
                        void *workspace, size_t workspace_bytes, EstWindows *out, void *stream);
// whether vs_select takes the selections of `heads` rows of n scores
bool vs_select_takes(int heads, int n);
// last kernel of the estimation, both selections and the index builder's tables
int vs_select(const EstWindows &e, int heads, int n, int nnz_v, int32_t *v_idx, int nnz_s, int32_t *s_idx, int32_t *tables, hipStream_t stream);
// minf_vs_index_build_full_ws without zero fill, the tables already there
int vs_index_rows(const int32_t *v_idx, const int32_t *s_idx, int32_t *block_count, int32_t *block_offset, int32_t *column_count,
                  int32_t *column_index, int batch, int heads, int rows, int nnz_v, int nnz_s, int32_t *tables, hipStream_t stream);
