// Sorting the index rows a caller hands to the vertical-slash operator: vertical positions ascending,
// slash offsets descending (reference minference/ops/pit_sparse_flash_attention_v2.py:224-225 sorts
// both with torch after a conversion to int32).
//
// One workgroup of 16 wavefronts sorts one row in LDS, both lists in one launch: a least significant
// digit radix sort on the values alone, eight bits a pass, with the passes skipped in which all values of
// the row agree (key positions below 65536 take two).  Bound by latency (a few hundred kilobytes are
// read and written in all): each wavefront owns a contiguous stretch of the row in registers and ranks it
// 64 values at a time -- eight ballots find the lanes with the same digit, one LDS word per digit and
// wavefront counts them -- so that nothing is contended and the order of equal digits is kept.
// A pass has three barriers; the scan reads a digit's counts of all wavefronts before it stores any (a load behind
// each store was a round trip to LDS each).  Pairs of 500 + 700 int64 values, one row: 7.5 -> 4.9 us; 1000 + 6096,
// 32 rows: 17.2 -> 13.7.
// Before this kernel the conversions, the two sorts and the copies around them were ten launches and 50 us of GPU
// time (1000 + 2048 values, 4 heads).  The operator on such indices: fp32 tensors of 8192 tokens 309 -> 265 us, rows of
// 100 + 750 values, 2 x 16 heads of 597 tokens 119 -> 78.
#include "minf_common.h"
#include "vs_index_tables.h"
#include "vs_stages.h"

namespace {

constexpr int SORT_WAVES = 16, SORT_THREADS = SORT_WAVES * MINF_WAVE;
constexpr int SORT_DIGITS = 256;

struct SortProblem {
    const void *in;
    int32_t *out;
    int n;              // values per row
    int is64;           // int64 input (truncated to 32 bits, as the conversion it replaces)
    unsigned flip;      // key = value ^ flip: ascending 0x80000000, descending 0x7fffffff
};

// E: 64-value groups per wavefront (rows of up to 1024 E values).  Row `row` of p, sorted to p.out and, as values, to
// keys[0 .. n) (each thread its own i % SORT_THREADS: no barrier behind).
template <int E>
__device__ __forceinline__ void sort_row(const SortProblem &p, const long long row, unsigned (&keys)[E * SORT_THREADS]) {
    __shared__ unsigned hist[SORT_WAVES][SORT_DIGITS];     // values of a digit in the wavefronts before (after the scan)
    __shared__ unsigned first[SORT_DIGITS];                // place of a digit's first value behind those of its 64 digits
    __shared__ unsigned wsum[SORT_DIGITS / MINF_WAVE], differ;     // values of 64 digits; bytes in which values differ
    const int tid = (int)threadIdx.x, lane = minf_lane();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int groups = (p.n + SORT_THREADS - 1) / SORT_THREADS;          // <= E
    const int base = wave * groups * MINF_WAVE + lane;
    const uint64_t lt = minf_lanemask_lt();

    // padding sorts last whatever passes run: all ones in every digit, behind equal values of the row
    unsigned key[E];
    auto load = [&](int i) -> unsigned {
        const long long at = row * p.n + i;
        return (unsigned)(p.is64 ? (int32_t)reinterpret_cast<const int64_t *>(p.in)[at] : reinterpret_cast<const int32_t *>(p.in)[at]) ^ p.flip;
    };
    // (each wavefront alone uses its row of hist between the scans: no barrier around the zeros)
    auto clear_own = [&]() {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < SORT_DIGITS; i += MINF_WAVE) hist[wave][i + lane] = 0;
    };
    clear_own();
    if (tid == 0) differ = 0;
    __syncthreads();
    const unsigned key0 = load(0);
    unsigned diff = 0;
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int i = base + r * MINF_WAVE;
        key[r] = 0xffffffffu;
        if (r < groups && i < p.n) {
            key[r] = load(i);
            diff |= key[r] ^ key0;
        }
    }
    unsigned bytes = 0;                                    // bit b: values of this wavefront differ in byte b
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if (__ballot(((diff >> (8 * b)) & 0xffu) != 0)) bytes |= 1u << b;
    if (lane == 0 && bytes) atomicOr(&differ, bytes);
#pragma unroll
    for (int r = 0; r < E; ++r)
        if (r < groups) keys[base + r * MINF_WAVE] = key[r];
    __syncthreads();
    const unsigned differing = differ;

    for (int shift = 0; shift < 32; shift += 8) {
        if (((differing >> (shift / 8)) & 1u) == 0) continue;             // (uniform)
        unsigned rank[E];
#pragma unroll
        for (int r = 0; r < E; ++r) {
            if (r >= groups) continue;                                    // (uniform)
            const unsigned d = (key[r] >> shift) & 0xffu;
            uint64_t same = ~0ull;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const bool bit = (d >> b) & 1u;
                const uint64_t has = __ballot(bit);
                same &= bit ? has : ~has;
            }
            const unsigned before = hist[wave][d];                        // (this wavefront's own row: no race)
            const unsigned in_group = __builtin_popcountll(same & lt);
            rank[r] = before + in_group;
            __builtin_amdgcn_wave_barrier();
            if (in_group == 0) hist[wave][d] = before + __builtin_popcountll(same);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        if (tid < SORT_DIGITS) {
            unsigned c[SORT_WAVES], total = 0;                            // (read at once, not each behind a store)
#pragma unroll
            for (int w = 0; w < SORT_WAVES; ++w) c[w] = hist[w][tid];
#pragma unroll
            for (int w = 0; w < SORT_WAVES; ++w) {
                hist[w][tid] = total;
                total += c[w];
            }
            unsigned incl = total;
#pragma unroll
            for (int s = 1; s < MINF_WAVE; s <<= 1) {
                const unsigned up = __shfl_up(incl, s);
                if (lane >= s) incl += up;
            }
            if (lane == MINF_WAVE - 1) wsum[wave] = incl;
            first[tid] = incl - total;
        }
        __syncthreads();
        const unsigned below1 = wsum[0], below2 = below1 + wsum[1], below3 = below2 + wsum[2];
#pragma unroll
        for (int r = 0; r < E; ++r)
            if (r < groups) {
                const unsigned d = (key[r] >> shift) & 0xffu;
                const unsigned below = d < 128 ? (d < 64 ? 0 : below1) : (d < 192 ? below2 : below3);
                keys[below + first[d] + hist[wave][d] + rank[r]] = key[r];
            }
        clear_own();
        __syncthreads();
#pragma unroll
        for (int r = 0; r < E; ++r)
            if (r < groups) key[r] = keys[base + r * MINF_WAVE];
    }
    for (int i = tid; i < p.n; i += SORT_THREADS) p.out[row * p.n + i] = (int32_t)(keys[i] ^= p.flip);
}

template <int E>
__global__ __launch_bounds__(SORT_THREADS) void index_sort_kernel(const SortProblem pa, const SortProblem pb, int rows) {
    __shared__ unsigned keys[E * SORT_THREADS];
    const bool second = (int)blockIdx.x >= rows;           // (workgroup-uniform)
    sort_row<E>(second ? pb : pa, (long long)blockIdx.x - (second ? rows : 0), keys);
}

// Both lists sorted as above (the slashes are pa's), and behind a head's slashes, where they lie in LDS, the index builder's tables.
// As two launches, each a chain of latency on a workgroup or two per head, 4 heads, 1000 and 2048 int64 values 7.4 + 8.2 us, now
// 13.5 and a gap less.  Operator on unsorted lists, us: 4 heads 600 tokens 56.8 -> 49.4, one head 4096 tokens 61.3 -> 53.5
// (paced by the host, one call and one launch less), 4 heads 8192 tokens 130.1 -> 126.7, fp32 157.8 -> 156.5.
template <int E>
__global__ __launch_bounds__(SORT_THREADS) void index_sort_tables_kernel(const SortProblem pa, const SortProblem pb, int rows,
                                                                         int32_t *__restrict__ tables, int blocks, int bm_words) {
    __shared__ unsigned keys[E * SORT_THREADS];
    extern __shared__ uint64_t prep_lds[];                 // (see prep_tables)
    if ((int)blockIdx.x >= rows) {                         // (workgroup-uniform)
        sort_row<E>(pb, (long long)blockIdx.x - rows, keys);
        return;
    }
    sort_row<E>(pa, (long long)blockIdx.x, keys);
    __syncthreads();
    prep_tables(reinterpret_cast<const int32_t *>(keys), tables + (long long)blockIdx.x * idx_tab_ints(pa.n, blocks), pa.n, blocks, bm_words, prep_lds);
}

// the bitmap of the longest context that fits LDS beside 16384 slashes
constexpr long long SORT_BITMAP_BYTES = 65536;

}  // namespace

extern "C" int minf_index_sort_pair(const void *vertical, int vertical_is64, int nnz_v, int32_t *vertical_out,
                                    const void *slash, int slash_is64, int nnz_s, int32_t *slash_out, int rows,
                                    void *stream) {
    if (rows < 0 || nnz_v < 0 || nnz_s < 0) return MINF_ERR_INVALID_ARG;
    if (rows == 0 || (nnz_v == 0 && nnz_s == 0)) return MINF_OK;
    if ((nnz_v && (!vertical || !vertical_out)) || (nnz_s && (!slash || !slash_out))) return MINF_ERR_INVALID_ARG;
    if (nnz_v > MINF_INDEX_SORT_MAX || nnz_s > MINF_INDEX_SORT_MAX || rows > (1 << 29)) return MINF_ERR_UNSUPPORTED;
    const SortProblem v{vertical, vertical_out, nnz_v, vertical_is64 != 0, 0x80000000u};
    const SortProblem s{slash, slash_out, nnz_s, slash_is64 != 0, 0x7fffffffu};
    // an empty list has no workgroups; the longer list's rows are handed out first
    const bool v_first = nnz_v > nnz_s;
    const SortProblem &a = v_first ? v : s, &b = v_first ? s : v;
    const dim3 grid((unsigned)(b.n ? 2 * rows : rows)), block(SORT_THREADS);
    hipStream_t st = (hipStream_t)stream;
    if (a.n <= 1024) hipLaunchKernelGGL((index_sort_kernel<1>), grid, block, 0, st, a, b, rows);
    else if (a.n <= 2048) hipLaunchKernelGGL((index_sort_kernel<2>), grid, block, 0, st, a, b, rows);
    else if (a.n <= 4096) hipLaunchKernelGGL((index_sort_kernel<4>), grid, block, 0, st, a, b, rows);
    else if (a.n <= 8192) hipLaunchKernelGGL((index_sort_kernel<8>), grid, block, 0, st, a, b, rows);
    else hipLaunchKernelGGL((index_sort_kernel<16>), grid, block, 0, st, a, b, rows);
    return minf_launch_status();
}

extern "C" int minf_vs_index_from_lists(const void *vertical, int vertical_is64, int nnz_v, int32_t *vertical_out,
                                        const void *slash, int slash_is64, int nnz_s, int32_t *slash_out,
                                        int32_t *block_count, int32_t *block_offset, int32_t *column_count,
                                        int32_t *column_index, int batch, int heads, int rows, void *workspace,
                                        size_t workspace_bytes, void *stream) {
    if (!vertical || !vertical_out || !slash || !slash_out || !block_count || !block_offset || !column_count || !column_index)
        return MINF_ERR_INVALID_ARG;
    if (batch < 0 || heads < 0 || rows < 0 || nnz_v < 1 || nnz_s < 1) return MINF_ERR_INVALID_ARG;
    const long long lists = (long long)batch * heads;
    if (lists * rows == 0) return MINF_OK;
    if (nnz_v > MINF_INDEX_SORT_MAX || nnz_s > MINF_INDEX_SORT_MAX || lists > 65535) return MINF_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < minf_vs_index_workspace_bytes(batch, heads, nnz_s, rows) || ((uintptr_t)workspace & 3))
        return MINF_ERR_WORKSPACE;
    const long long bm_words = idx_bm_words(rows);
    if (bm_words * 4 > SORT_BITMAP_BYTES) {
        const int st = minf_index_sort_pair(vertical, vertical_is64, nnz_v, vertical_out, slash, slash_is64, nnz_s, slash_out, (int)lists, stream);
        return st ? st : minf_vs_index_build_full_ws(vertical_out, slash_out, block_count, block_offset, column_count, column_index,
                                                     batch, heads, rows, nnz_v, nnz_s, 0, nullptr, workspace, workspace_bytes, stream);
    }
    const SortProblem v{vertical, vertical_out, nnz_v, vertical_is64 != 0, 0x80000000u};
    const SortProblem s{slash, slash_out, nnz_s, slash_is64 != 0, 0x7fffffffu};
    const int most = nnz_v > nnz_s ? nnz_v : nnz_s;
    const size_t marks = 16 * (size_t)((nnz_s + MINF_WAVE - 1) / MINF_WAVE), bitmap = (size_t)bm_words * 4;
    const size_t lds = marks > bitmap ? marks : bitmap;
    const dim3 grid((unsigned)(2 * lists)), block(SORT_THREADS);
    hipStream_t st = (hipStream_t)stream;
    int32_t *const tables = (int32_t *)workspace;
    auto *const kernel = most <= 1024 ? index_sort_tables_kernel<1> : most <= 2048 ? index_sort_tables_kernel<2> :
                         most <= 4096 ? index_sort_tables_kernel<4> : most <= 8192 ? index_sort_tables_kernel<8> : index_sort_tables_kernel<16>;
    hipLaunchKernelGGL(kernel, grid, block, lds, st, s, v, (int)lists, tables, rows, (int)bm_words);
    const int status = minf_launch_status();
    if (status != MINF_OK) return status;
    return vs_index_rows(vertical_out, slash_out, block_count, block_offset, column_count, column_index, batch, heads, rows,
                         nnz_v, nnz_s, tables, st);
}
