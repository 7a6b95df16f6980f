// Vertical/slash index conversion for gfx950: one 64-lane wavefront per
// (batch, head, 64-row block).  Produces the same four tensors as the
// reference's one-thread-per-row kernel (csrc/vertical_slash_index.cu:27-99),
// bit for bit, but walks the slash list 64 entries at a time:
//
//   * each valid slash offset o maps to a column end t = max(end_m - o, 64)
//     (ascending in list order);
//   * inside one merged range starting at `a`, the running range end after
//     consuming t is the closed form  e(t) = a + 64*ceil((t - a)/64), so all
//     64 lanes evaluate it at once; a new range starts exactly where
//     t > e(previous t) + 64, found with a ballot, and lanes past the break
//     switch to the new start.  A block [e-64, e) is emitted wherever e
//     changes, at a position given by a wave prefix count;
//   * a vertical index x lands in the output iff, with i the first slash
//     entry whose t exceeds x,  x < a_i  and  x >= e_{i-1}  (it lies in the
//     gap before entry i's range); verticals at or past the last t are never
//     emitted.  Verticals are consumed 64 at a time against the current
//     chunk's (t, a, e) triples kept in LDS.
//
// Writes: payload by prefix-compacted 4-byte stores, zero tails by 16-byte
// stores; all row offsets are 64-bit.
#include "minf_common.h"
#include "vs_index_tables.h"
#include "vs_stages.h"
#include <limits.h>
#include <atomic>

#define IDX_WAVES 4

__device__ __forceinline__ void zero_range(int32_t *p, int from, int to, int lane) {
    int n = to - from;
    if (n <= 0) return;
    int32_t *q = p + from;
    int head = (int)(((16u - (unsigned)((uintptr_t)q & 15u)) & 15u) >> 2);
    if (head > n) head = n;
    if (lane < head) q[lane] = 0;
    q += head;
    n -= head;
    int n4 = n >> 2;
    int4 z = make_int4(0, 0, 0, 0);
    for (int i = lane; i < n4; i += MINF_WAVE) reinterpret_cast<int4 *>(q)[i] = z;
    int tail = n & 3;
    if (lane < tail) q[n4 * 4 + lane] = 0;
}

// dst[i] = src[i] + shift for i < n with 16-byte stores: dst is brought to a 16-byte boundary with
// single stores first (src then sits at any 4-byte phase; its 16-byte loads need no alignment)
__device__ __forceinline__ void copy_shifted(int32_t *dst, const int32_t *src, int n, int shift, int lane) {
    if (n <= 0) return;
    int head = (int)(((16u - (unsigned)((uintptr_t)dst & 15u)) & 15u) >> 2);
    if (head > n) head = n;
    if (lane < head) dst[lane] = src[lane] + shift;
    dst += head;
    src += head;
    n -= head;
    const int n4 = n >> 2;
    for (int i = lane; i < n4; i += MINF_WAVE) {
        int4 v;
        __builtin_memcpy(&v, src + 4 * i, 16);
        v.x += shift; v.y += shift; v.z += shift; v.w += shift;
        reinterpret_cast<int4 *>(dst)[i] = v;
    }
    const int tail = n & 3;
    if (lane < tail) dst[n4 * 4 + lane] = src[n4 * 4 + lane] + shift;
}

__global__ __launch_bounds__(IDX_WAVES *MINF_WAVE) void vs_index_kernel(
    const int32_t *__restrict__ seqlens, const int32_t *__restrict__ vertical,
    const int32_t *__restrict__ slash, int32_t *__restrict__ block_count,
    int32_t *__restrict__ block_offset, int32_t *__restrict__ column_count,
    int32_t *__restrict__ column_index, int heads, int rows, int nnz_v, int nnz_s,
    int zero_fill, int32_t *error_flag, long long total_rows) {
    __shared__ int lds_t[IDX_WAVES][MINF_WAVE];
    __shared__ int lds_a[IDX_WAVES][MINF_WAVE];
    __shared__ int lds_e[IDX_WAVES][MINF_WAVE];

    const int lane = minf_lane();
    const int wave = (int)(threadIdx.x >> 6);
    const long long ro = (long long)blockIdx.x * IDX_WAVES + wave;   // (b*H + h)*rows + m
    if (ro >= total_rows) return;
    const int m = (int)(ro % rows);
    const long long bh = ro / rows;
    const int b = (int)(bh / heads);

    int32_t *bo_row = block_offset + ro * (long long)nnz_s;
    int32_t *ci_row = column_index + ro * (long long)nnz_v;
    const int32_t *vert = vertical + bh * (long long)nnz_v;
    const int32_t *sl = slash + bh * (long long)nnz_s;

    const int seqlen = seqlens ? seqlens[b] : INT_MAX;
    const int start_m = m * 64;
    const int end_m = start_m + 64;

    int nb = 0, ncol = 0;
    bool live = start_m < seqlen;

    // first list position whose offset is below end_m (list is descending)
    int s0 = nnz_s;
    if (live) {
        int lo = 0, hi = nnz_s;
        while (lo < hi) {
            int mid = (lo + hi) >> 1;
            if (sl[mid] >= end_m) lo = mid + 1; else hi = mid;
        }
        s0 = lo;
        if (s0 >= nnz_s) {           // the reference would read past the list here
            live = false;
            if (error_flag && lane == 0) *error_flag = 1;
        }
    }

    if (live) {
        const int n = nnz_s - s0;
        const int nchunks = (n + MINF_WAVE - 1) / MINF_WAVE;
        int vp = 0;
        int carried_e = 0, carried_t = 0, cur_a = 0;
        int ep0 = INT_MIN;           // e of the entry before the chunk's first
        for (int c = 0; c < nchunks; ++c) {
            const int base = s0 + c * MINF_WAVE;
            const int cnt = min(MINF_WAVE, nnz_s - base);
            const bool valid = lane < cnt;
            int t = valid ? max(end_m - sl[base + lane], 64) : 0;
            const int tlast = minf_readlane(t, cnt - 1);
            if (!valid) t = tlast;   // padding lanes repeat the last entry (no-ops)
            if (c == 0) {
                const int t0 = minf_readlane(t, 0);
                cur_a = t0 - 64;
                carried_e = t0 - 64;
                carried_t = t0;
            }
            uint64_t starts;
            const int a = chunk_ranges(t, lane, cur_a, carried_e, carried_t, starts);
            const int e = a + ((((t - a) + 63) >> 6) << 6);
            int eprev = lane_above(e);
            if (lane == 0) eprev = carried_e;
            const bool changed = valid && (e != eprev);
            const uint64_t cm = __ballot(changed);
            if (changed) bo_row[nb + __builtin_popcountll(cm & minf_lanemask_lt())] = e - 64;
            nb += __builtin_popcountll(cm);

            // verticals below this chunk's last t
            if (vp < nnz_v && vert[vp] < tlast) {
                lds_t[wave][lane] = t;
                lds_a[wave][lane] = a;
                lds_e[wave][lane] = e;
                __builtin_amdgcn_wave_barrier();
                while (vp < nnz_v) {
                    const int x = (vp + lane < nnz_v) ? vert[vp + lane] : INT_MAX;
                    const bool ok = x < tlast;
                    const uint64_t okm = __ballot(ok);
                    const int k = __builtin_popcountll(okm);
                    bool emit = false;
                    if (ok) {
                        int lo = 0, hi = MINF_WAVE - 1;      // first i with t[i] > x (exists)
                        while (lo < hi) {
                            int mid = (lo + hi) >> 1;
                            if (lds_t[wave][mid] > x) hi = mid; else lo = mid + 1;
                        }
                        const int ai = lds_a[wave][lo];
                        const int ep = lo == 0 ? ep0 : lds_e[wave][lo - 1];
                        emit = (x < ai) && (x >= ep);
                    }
                    const uint64_t em = __ballot(emit);
                    if (emit) ci_row[ncol + __builtin_popcountll(em & minf_lanemask_lt())] = x;
                    ncol += __builtin_popcountll(em);
                    vp += k;
                    if (k < MINF_WAVE) break;
                }
                __builtin_amdgcn_wave_barrier();
            }
            carried_e = minf_readlane(e, cnt - 1);
            carried_t = tlast;
            cur_a = minf_readlane(a, cnt - 1);
            ep0 = carried_e;
        }
    }

    if (lane == 0) {                 // (rows past the sequence and rows without an entry: zero)
        block_count[ro] = nb;
        column_count[ro] = ncol;
    }
    if (zero_fill) {
        zero_range(bo_row, nb, nnz_s, lane);
        zero_range(ci_row, ncol, nnz_v, lane);
    }
}

__global__ __launch_bounds__(PREP_WAVES *MINF_WAVE) void vs_index_prep_kernel(const int32_t *__restrict__ slash,
                                                                              int32_t *__restrict__ tables, int nnz_s, int rows, int bm_words) {
    extern __shared__ uint64_t prep_lds[];           // sure and maybe marks of every chunk, later the bitmap
    const long long bh = blockIdx.x;
    prep_tables(slash + bh * (long long)nnz_s, tables + bh * idx_tab_ints(nnz_s, rows), nnz_s, rows, bm_words, prep_lds);
}

// The coverage bitmap where the table pass leaves it out: contexts whose bitmap does not fit its LDS (beyond 786304
// tokens), lists that one wavefront walks for being longer than the mark arrays (its atomics would lengthen that chain).
// One thread per 32-bit word: a binary search finds the first range that ends after the word's first position; ranges
// are at least 64 long, so at most two of them touch a word.
__global__ __launch_bounds__(256) void vs_index_bitmap_kernel(int32_t *__restrict__ tables, int nnz_s, int rows) {
    const long long bh = blockIdx.y;
    int32_t *hdr = tables + bh * idx_tab_ints(nnz_s, rows);
    const int32_t *run_a = hdr + IDX_TAB_HDR + 3ll * nnz_s, *run_e = run_a + nnz_s;
    uint32_t *bm = reinterpret_cast<uint32_t *>(hdr + IDX_TAB_HDR + 7ll * nnz_s);
    const long long w = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= idx_bm_words(rows) || !hdr[3]) return;
    const int nr = hdr[1];
    const long long p0 = 32 * w, p1 = p0 + 32;
    int lo = 0, hi = nr;                       // first range with run_e > p0
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (run_e[mid] > p0) hi = mid; else lo = mid + 1;
    }
    uint32_t bits = 0;
    for (int r = lo; r < nr; ++r) {
        const long long a = run_a[r], e = run_e[r];
        if (a >= p1) break;
        const int from = (int)(max(a, p0) - p0), to = (int)(min(e, p1) - p0);      // [from, to) inside the word
        if (to > from) bits |= (to - from >= 32 ? 0xffffffffu : ((1u << (to - from)) - 1u)) << from;
    }
    bm[w] = bits;
}

// Zero-filled rows of more than IDX_SHORT_ROW slashes (LONG) are bound by their stores: six workgroups per CU (see
// index_build_tables), held to 64 registers, which measures 3 % faster at 512K tokens.  Shorter ones are bound by
// their chains of dependent loads like the payload alone: every wave that 72 registers allow, no spills.  Us, as
// the long rows run and so: 32 heads, 262144 tokens, 30 columns and 800 slashes 187 -> 156, 500 and 700 275 -> 226, 3500
// and 100 637 -> 548; 131072 tokens, 1000 and 3000 295 -> 254; 4 heads 100000 tokens, 100 and 750 27.2 -> 23.5.
// The line: 32 heads, 131072 tokens, 1000 columns and, uniform, 4000 slashes 322 -> 293, 4500 338 -> 339, 5000 357 ->
// 363, 6096 411 -> 436; clustered ones as fast or faster up to 5600, 6096 410 -> 422.
constexpr int IDX_SHORT_ROW = 4096;
template <bool ZERO_FILL, bool LONG>
__global__ __launch_bounds__(IDX_WAVES *MINF_WAVE, ZERO_FILL ? (LONG ? 8 : 7) : 1) void vs_index_fast_kernel(
    const int32_t *__restrict__ seqlens, const int32_t *__restrict__ vertical,
    const int32_t *__restrict__ slash, const int32_t *__restrict__ tables,
    int32_t *__restrict__ block_count, int32_t *__restrict__ block_offset,
    int32_t *__restrict__ column_count, int32_t *__restrict__ column_index, int heads, int rows,
    int nnz_v, int nnz_s, int32_t *error_flag, long long total_rows) {
    constexpr int zero_fill = ZERO_FILL ? 1 : 0;
    __shared__ int lds_t[IDX_WAVES][MINF_WAVE];
    __shared__ int lds_a[IDX_WAVES][MINF_WAVE];
    __shared__ int lds_e[IDX_WAVES][MINF_WAVE];

    const int lane = minf_lane();
    const int wave = (int)(threadIdx.x >> 6);
    const long long ro = (long long)blockIdx.x * IDX_WAVES + wave;   // (b*H + h)*rows + m
    if (ro >= total_rows) return;
    const int m = (int)(ro % rows);
    const long long bh = ro / rows;
    const int b = (int)(bh / heads);

    int32_t *bo_row = block_offset + ro * (long long)nnz_s;
    int32_t *ci_row = column_index + ro * (long long)nnz_v;
    const int32_t *vert = vertical + bh * (long long)nnz_v;
    const int32_t *sl = slash + bh * (long long)nnz_s;
    const int32_t *hdr = tables + bh * idx_tab_ints(nnz_s, rows);
    const int32_t *cpos = hdr + IDX_TAB_HDR, *cpre = cpos + nnz_s, *crun = cpre + nnz_s;
    const int32_t *run_a = crun + nnz_s, *run_e = run_a + nnz_s, *cgaps = run_e + nnz_s, *glist = cgaps + nnz_s;
    const uint32_t *bm = reinterpret_cast<const uint32_t *>(glist + nnz_s);

    const int seqlen = seqlens ? seqlens[b] : INT_MAX;
    const int start_m = m * 64;
    const int end_m = start_m + 64;
    const uint64_t lt = minf_lanemask_lt();

    int nb = 0, ncol = 0;
    bool live = start_m < seqlen;

    // loads that do not depend on each other, issued together (the kernel is bound by chains of
    // dependent loads, not by bandwidth)
    const int o_first = sl[0], o_last = sl[nnz_s - 1];
    const int tab_blocks = hdr[0], tab_runs = hdr[1], tab_v = hdr[2], bm_ok = hdr[3], ngaps = hdr[4];
    const bool whole_list = o_first <= end_m - 64;      // nothing skipped, nothing clipped

    int s0 = nnz_s;
    if (live) {
        // first entry with an offset below end_m = number of entries >= end_m (descending list):
        // 64 samples one stride apart locate the segment, the lanes then count inside it -- two
        // rounds of independent loads instead of a 13-step chain of dependent ones
        s0 = 0;
        if (!whole_list) {
            const int stride = (nnz_s + MINF_WAVE - 1) / MINF_WAVE;
            const int si = min(lane * stride, nnz_s - 1);
            const bool above = lane * stride < nnz_s && sl[si] >= end_m;
            const int nseg = __builtin_popcountll(__ballot(above));       // samples 0..nseg-1 are >= end_m
            if (nseg > 0) {
                const int seg = (nseg - 1) * stride;                      // entries [0, seg] are >= end_m
                int cnt = 0;
                for (int i0 = 0; i0 < stride; i0 += MINF_WAVE) {        // same trip count in every lane
                    const int idx = seg + i0 + lane;
                    const bool ab = i0 + lane < stride && idx < nnz_s && sl[idx] >= end_m;
                    cnt += __builtin_popcountll(__ballot(ab));
                }
                s0 = seg + cnt;
            }
        }
        if (s0 >= nnz_s) {           // the reference would read past the list here
            live = false;
            if (error_flag && lane == 0) *error_flag = 1;
        }
    }

    if (live) {
        int vp = 0;
        int g = -1;                  // list entry from which the tables apply
        int e_lim = INT_MIN;         // end of the last explicitly built range
        if (whole_list) {
            g = 0;
        } else {
            int carried_e = 0, carried_t = 0, cur_a = 0;
            int ep0 = INT_MIN;
            bool first = true;
            for (int base = s0; base < nnz_s; base += MINF_WAVE) {
                int cnt = min(MINF_WAVE, nnz_s - base);
                const bool full = cnt == MINF_WAVE;
                bool valid = lane < cnt;
                int t = valid ? max(end_m - sl[base + lane], 64) : 0;
                int tlast = minf_readlane(t, cnt - 1);
                if (!valid) t = tlast;
                if (first) {
                    const int t0 = minf_readlane(t, 0);
                    cur_a = t0 - 64;
                    carried_e = t0 - 64;
                    carried_t = t0;
                    first = false;
                }
                uint64_t starts, gm;         // gm: entries of this chunk more than 64 above their predecessor
                int a = chunk_ranges(t, lane, cur_a, carried_e, carried_t, starts, &gm);
                const bool any_gap = gm != 0;
                // the first range start of this chunk that is also a tabulated range start
                const bool tab = ((starts >> lane) & 1ull) && cpre[base + lane] >= 0;
                const uint64_t tm = __ballot(tab);
                const int cut = tm ? __builtin_ctzll(tm) : -1;
                if (cut == 0) {          // nothing of this chunk belongs to the explicit part
                    g = base;
                    e_lim = carried_e;
                    break;
                }
                if (cut > 0) {           // entries [0, cut) only; later lanes repeat entry cut-1
                    cnt = cut;
                    valid = lane < cnt;
                    tlast = minf_readlane(t, cnt - 1);
                    const int alast = minf_readlane(a, cnt - 1);
                    if (!valid) { t = tlast; a = alast; }
                }
                const int e = a + ((((t - a) + 63) >> 6) << 6);
                int eprev = lane_above(e);
                if (lane == 0) eprev = carried_e;
                const bool changed = valid && (e != eprev);
                const uint64_t cm = __ballot(changed);
                if (changed) bo_row[nb + __builtin_popcountll(cm & lt)] = e - 64;
                nb += __builtin_popcountll(cm);

                if (vp < nnz_v && vert[vp] < tlast) {
                    lds_t[wave][lane] = t;
                    lds_a[wave][lane] = a;
                    lds_e[wave][lane] = e;
                    __builtin_amdgcn_wave_barrier();
                    while (vp < nnz_v) {
                        const int x = (vp + lane < nnz_v) ? vert[vp + lane] : INT_MAX;
                        const bool ok = x < tlast;
                        const uint64_t okm = __ballot(ok);
                        const int k = __builtin_popcountll(okm);
                        bool emit = false;
                        if (ok) {
                            int lo = 0, hi = MINF_WAVE - 1;      // first i with t[i] > x (exists)
                            while (lo < hi) {
                                int mid = (lo + hi) >> 1;
                                if (lds_t[wave][mid] > x) hi = mid; else lo = mid + 1;
                            }
                            const int ai = lds_a[wave][lo];
                            const int ep = lo == 0 ? ep0 : lds_e[wave][lo - 1];
                            emit = (x < ai) && (x >= ep);
                        }
                        const uint64_t em = __ballot(emit);
                        if (emit) ci_row[ncol + __builtin_popcountll(em & lt)] = x;
                        ncol += __builtin_popcountll(em);
                        vp += k;
                        if (k < MINF_WAVE) break;
                    }
                    __builtin_amdgcn_wave_barrier();
                }
                carried_e = minf_readlane(e, cnt - 1);
                carried_t = tlast;
                cur_a = minf_readlane(a, cnt - 1);
                ep0 = carried_e;
                if (cut > 0) {
                    g = base + cut;
                    e_lim = carried_e;
                    break;
                }
                // A whole chunk without a gap: a dense run.  No range can start before the next entry of
                // the gap list, so the entries up to there only extend the current range; their blocks
                // are written at once and the walk resumes at that entry.
                const int lo = base + MINF_WAVE;             // first entry not looked at yet
                if (full && !any_gap && lo < nnz_s) {
                    const int pos = __builtin_amdgcn_readfirstlane(cgaps[lo - 1]);   // gap entries below lo
                    const int X = pos < ngaps ? __builtin_amdgcn_readfirstlane(glist[pos]) : nnz_s;      // first one >= lo
                    if (X > lo) {
                        const int t_end = max(end_m - __builtin_amdgcn_readfirstlane(sl[X - 1]), 64);
                        const int e_end = cur_a + ((((t_end - cur_a) + 63) >> 6) << 6);
                        const int nnew = (e_end - carried_e) >> 6;
                        for (int j = lane; j < nnew; j += MINF_WAVE) bo_row[nb + j] = carried_e + 64 * j;
                        nb += nnew;
                        // the verticals below t_end lie inside the current range: none is emitted
                        while (vp < nnz_v) {
                            const int x = (vp + lane < nnz_v) ? vert[vp + lane] : INT_MAX;
                            const int k = __builtin_popcountll(__ballot(x < t_end));
                            vp += k;
                            if (k < MINF_WAVE) break;
                        }
                        carried_e = e_end;
                        carried_t = t_end;
                        ep0 = e_end;
                        base = X - MINF_WAVE;                // (the loop's increment makes it X)
                    }
                }
            }
        }
        if (g >= 0) {
            const int shift = end_m - tab_v;
            const int k0 = g == 0 ? 0 : cpre[g], r0 = g == 0 ? 0 : crun[g];   // entry 0 starts range 0
            const int nblk = tab_blocks - k0, nruns = tab_runs;
            copy_shifted(bo_row + nb, cpos + k0, nblk, shift, lane);
            nb += nblk;
            const int t_end = end_m - o_last;             // t of the last entry (not clipped here)
            const int first_a = run_a[r0];                // start of the first remaining range
            // four batches of 64 verticals per round: their loads and their coverage look-ups are
            // independent, only the ordered emit is sequential
            while (vp < nnz_v) {
                int x[4];
                bool emit[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) x[u] = (vp + u * MINF_WAVE + lane < nnz_v) ? vert[vp + u * MINF_WAVE + lane] : INT_MAX;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    emit[u] = false;
                    if (x[u] < t_end && x[u] >= e_lim) {
                        const int xv = x[u] - shift;
                        if (xv < first_a) {                   // below every remaining range
                            emit[u] = true;
                        } else if (bm_ok) {                   // xv < tab_v: inside the bitmap
                            emit[u] = !((bm[xv >> 5] >> (xv & 31)) & 1u);
                        } else {
                            int lo = r0, hi = nruns;          // first range >= r0 that ends after xv
                            while (lo < hi) {
                                int mid = (lo + hi) >> 1;
                                if (run_e[mid] > xv) hi = mid; else lo = mid + 1;
                            }
                            emit[u] = !(lo < nruns && run_a[lo] <= xv);
                        }
                    }
                }
                bool more = true;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint64_t em = __ballot(emit[u]);
                    if (emit[u]) ci_row[ncol + __builtin_popcountll(em & lt)] = x[u];
                    ncol += __builtin_popcountll(em);
                    more = more && __builtin_popcountll(__ballot(x[u] < t_end)) == MINF_WAVE;
                }
                vp += 4 * MINF_WAVE;
                if (!more) break;                             // verticals ascend: nothing further is below t_end
            }
        }
    }

    if (lane == 0) {                 // (rows past the sequence and rows without an entry: zero)
        block_count[ro] = nb;
        column_count[ro] = ncol;
    }
    if (zero_fill) {
        zero_range(bo_row, nb, nnz_s, lane);
        zero_range(ci_row, ncol, nnz_v, lane);
    }
}

extern "C" int minf_vs_index_build(const int32_t *seqlens, const int32_t *vertical_idx,
                                   const int32_t *slash_idx, int32_t *block_count,
                                   int32_t *block_offset, int32_t *column_count,
                                   int32_t *column_index, int batch, int heads, int rows,
                                   int nnz_v, int nnz_s, int zero_fill, int32_t *error_flag,
                                   void *stream) {
    if (!seqlens || !vertical_idx || !slash_idx || !block_count || !block_offset ||
        !column_count || !column_index)
        return MINF_ERR_INVALID_ARG;
    if (batch < 0 || heads < 0 || rows < 0 || nnz_v < 1 || nnz_s < 1) return MINF_ERR_INVALID_ARG;
    const long long total = (long long)batch * heads * rows;
    if (total == 0) return MINF_OK;
    const long long nblk = (total + IDX_WAVES - 1) / IDX_WAVES;
    if (nblk > 0x7fffffffLL) return MINF_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(vs_index_kernel, dim3((unsigned)nblk), dim3(IDX_WAVES * MINF_WAVE), 0,
                       (hipStream_t)stream, seqlens, vertical_idx, slash_idx, block_count,
                       block_offset, column_count, column_index, heads, rows, nnz_v, nnz_s,
                       zero_fill, error_flag, total);
    return minf_launch_status();
}


extern "C" size_t minf_vs_index_workspace_bytes(int batch, int heads, int nnz_s, int rows) {
    if (batch <= 0 || heads <= 0 || nnz_s <= 0 || rows < 0) return 0;
    return (size_t)batch * heads * (size_t)idx_tab_ints(nnz_s, rows) * sizeof(int32_t);
}

// launches of the table-driven builder on a workspace that is known to be large enough
static int index_build_tables(const int32_t *seqlens, const int32_t *vertical_idx, const int32_t *slash_idx,
                              int32_t *block_count, int32_t *block_offset, int32_t *column_count,
                              int32_t *column_index, int batch, int heads, int rows, int nnz_v, int nnz_s,
                              int zero_fill, int32_t *error_flag, int32_t *workspace, long long total,
                              hipStream_t stream, bool have_tables = false) {
    const long long nblk = (total + IDX_WAVES - 1) / IDX_WAVES;
    if (nblk > 0x7fffffffLL || (long long)batch * heads > 65535) return MINF_ERR_UNSUPPORTED;
    if (!have_tables) {
        const int nchunks = (nnz_s + MINF_WAVE - 1) / MINF_WAVE;
        const long long bm_words = idx_bm_words(rows);
        const bool bm_in_lds = bm_words * 4 <= PREP_LDS_MAX_BYTES && nchunks <= PREP_MAX_CHUNKS;
        size_t lds = nchunks <= PREP_MAX_CHUNKS ? 16 * (size_t)nchunks : 0;
        if (bm_in_lds && (size_t)bm_words * 4 > lds) lds = (size_t)bm_words * 4;
        hipLaunchKernelGGL(vs_index_prep_kernel, dim3((unsigned)(batch * heads)), dim3(PREP_WAVES * MINF_WAVE), lds,
                           stream, slash_idx, workspace, nnz_s, rows, bm_in_lds ? (int)bm_words : 0);
        const int status = minf_launch_status();
        if (status != MINF_OK) return status;
        if (!bm_in_lds) {
            hipLaunchKernelGGL(vs_index_bitmap_kernel, dim3((unsigned)((bm_words + 255) / 256), (unsigned)(batch * heads)),
                               dim3(256), 0, stream, workspace, nnz_s, rows);
            const int status = minf_launch_status();
            if (status != MINF_OK) return status;
        }
    }
    // Long zero-filled rows: 24 resident waves per CU write faster than 32 (6-9 % at 128K-512K tokens: fewer rows in
    // flight, better DRAM locality).  Unused dynamic LDS is the occupancy limiter: 3 KB static + 24000 B -> 6
    // workgroups per CU.
    const bool long_rows = zero_fill && nnz_s > IDX_SHORT_ROW;
    const unsigned occupancy_lds = long_rows ? 24000u : 0u;
    auto *const kernel = long_rows ? vs_index_fast_kernel<true, true> : zero_fill ? vs_index_fast_kernel<true, false> : vs_index_fast_kernel<false, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)nblk), dim3(IDX_WAVES * MINF_WAVE), occupancy_lds, stream, seqlens, vertical_idx,
                       slash_idx, (const int32_t *)workspace, block_count, block_offset, column_count, column_index, heads,
                       rows, nnz_v, nnz_s, error_flag, total);
    return minf_launch_status();
}

// (seqlens NULL: every sequence fills the context)
static int index_build_ws(const int32_t *seqlens, const int32_t *vertical_idx, const int32_t *slash_idx, int32_t *block_count,
                          int32_t *block_offset, int32_t *column_count, int32_t *column_index, int batch, int heads, int rows,
                          int nnz_v, int nnz_s, int zero_fill, int32_t *error_flag,
                          void *workspace, size_t workspace_bytes, void *stream) {
    if (!vertical_idx || !slash_idx || !block_count || !block_offset ||
        !column_count || !column_index)
        return MINF_ERR_INVALID_ARG;
    if (batch < 0 || heads < 0 || rows < 0 || nnz_v < 1 || nnz_s < 1) return MINF_ERR_INVALID_ARG;
    const long long total = (long long)batch * heads * rows;
    if (total == 0) return MINF_OK;
    if (!workspace || workspace_bytes < minf_vs_index_workspace_bytes(batch, heads, nnz_s, rows) ||
        ((uintptr_t)workspace & 3))
        return MINF_ERR_WORKSPACE;
    return index_build_tables(seqlens, vertical_idx, slash_idx, block_count, block_offset, column_count,
                              column_index, batch, heads, rows, nnz_v, nnz_s, zero_fill, error_flag,
                              (int32_t *)workspace, total, (hipStream_t)stream);
}

extern "C" int minf_vs_index_build_ws(const int32_t *seqlens, const int32_t *vertical_idx,
                                      const int32_t *slash_idx, int32_t *block_count,
                                      int32_t *block_offset, int32_t *column_count,
                                      int32_t *column_index, int batch, int heads, int rows,
                                      int nnz_v, int nnz_s, int zero_fill, int32_t *error_flag,
                                      void *workspace, size_t workspace_bytes, void *stream) {
    if (!seqlens) return MINF_ERR_INVALID_ARG;
    return index_build_ws(seqlens, vertical_idx, slash_idx, block_count, block_offset, column_count, column_index, batch, heads,
                          rows, nnz_v, nnz_s, zero_fill, error_flag, workspace, workspace_bytes, stream);
}

extern "C" int minf_vs_index_build_full_ws(const int32_t *vertical_idx, const int32_t *slash_idx, int32_t *block_count,
                                           int32_t *block_offset, int32_t *column_count, int32_t *column_index, int batch,
                                           int heads, int rows, int nnz_v, int nnz_s, int zero_fill, int32_t *error_flag,
                                           void *workspace, size_t workspace_bytes, void *stream) {
    return index_build_ws(nullptr, vertical_idx, slash_idx, block_count, block_offset, column_count, column_index, batch, heads,
                          rows, nnz_v, nnz_s, zero_fill, error_flag, workspace, workspace_bytes, stream);
}

int vs_index_rows(const int32_t *v_idx, const int32_t *s_idx, int32_t *block_count, int32_t *block_offset, int32_t *column_count,
                  int32_t *column_index, int batch, int heads, int rows, int nnz_v, int nnz_s, int32_t *tables, hipStream_t stream) {
    return index_build_tables(nullptr, v_idx, s_idx, block_count, block_offset, column_count, column_index, batch, heads, rows,
                              nnz_v, nnz_s, 0, nullptr, tables, (long long)batch * heads * rows, stream, true);
}

// ---- the entry point that allocates nothing ---------------------------------------------------
// The tables and bitmaps of minf_vs_index_build_ws live in this array instead of a caller-owned
// workspace.  Every GPU holds its own copy at its own address; host code only ever uses the address
// hipGetSymbolAddress returned for the current device, never the array's name.  Nothing in it has
// to start at zero: the table pass and the bitmap pass write every word the row-block pass reads.
static __device__ __align__(256) int32_t scratch[MINF_VS_INDEX_STATIC_BYTES / sizeof(int32_t)];

#define IDX_MAX_DEVICES 64
static std::atomic<int32_t *> scratch_ptr[IDX_MAX_DEVICES];

static int scratch_for_current_device(int32_t **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return minf_hip_status(e);
    if (dev < 0 || dev >= IDX_MAX_DEVICES) return MINF_ERR_UNSUPPORTED;
    int32_t *ptr = scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        // first call on this device; two threads racing here get the same address
        e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return minf_hip_status(e);
        if (!ptr) return MINF_ERR_HIP_BASE;
        scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return MINF_OK;
}

extern "C" int minf_vs_index_build_static(const int32_t *seqlens, const int32_t *vertical_idx,
                                          const int32_t *slash_idx, int32_t *block_count,
                                          int32_t *block_offset, int32_t *column_count,
                                          int32_t *column_index, int batch, int heads, int rows,
                                          int nnz_v, int nnz_s, int zero_fill, int32_t *error_flag,
                                          void *stream) {
    if (!seqlens || !vertical_idx || !slash_idx || !block_count || !block_offset ||
        !column_count || !column_index)
        return MINF_ERR_INVALID_ARG;
    if (batch < 0 || heads < 0 || rows < 0 || nnz_v < 1 || nnz_s < 1) return MINF_ERR_INVALID_ARG;
    const long long total = (long long)batch * heads * rows;
    if (total == 0) return MINF_OK;
    // sizes beyond the array are refused before any HIP call
    if (minf_vs_index_workspace_bytes(batch, heads, nnz_s, rows) > (size_t)MINF_VS_INDEX_STATIC_BYTES)
        return MINF_ERR_WORKSPACE;
    int32_t *ws = nullptr;
    const int st = scratch_for_current_device(&ws);
    if (st != MINF_OK) return st;
    return index_build_tables(seqlens, vertical_idx, slash_idx, block_count, block_offset, column_count,
                              column_index, batch, heads, rows, nnz_v, nnz_s, zero_fill, error_flag,
                              ws, total, (hipStream_t)stream);
}
