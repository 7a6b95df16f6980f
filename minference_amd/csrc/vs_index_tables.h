// The table pass of the index builder (see vs_index.hip): device code of vs_index_prep_kernel and of the kernels that make
// the tables right behind a selection (topk.hip) or a sort (index_sort.hip).
#pragma once
#include "minf_common.h"

// value of the lane below (lane 0 gets 0): one data-parallel-primitive move, where the general
// shuffle goes through the LDS crossbar -- the table pass is one wave walking a chain of chunks and
// pays every cycle of it
__device__ __forceinline__ int lane_above(int x) {
    return __builtin_amdgcn_update_dpp(0, x, 0x138 /* wave_shr:1 */, 0xf, 0xf, true);
}

// Range starts of one chunk of 64 entries.  `t` ascends along the lanes (padding lanes repeat the
// last entry); the state carried in from the previous chunk is the current range start `cur_a`,
// the running range end `carried_e` and the previous entry `carried_t`.  Entry i starts a new
// range iff t_i > e_{i-1} + 64, and t_{i-1} <= e_{i-1} < t_{i-1} + 64, so
//   t_i >  t_{i-1} + 127  is always a start,      (decided for all lanes with one ballot)
//   t_i <= t_{i-1} + 64   never is,
// and only the lanes in between depend on the 64-phase of their range; those are resolved one by
// one in lane order with scalar arithmetic.  Returns this lane's range start; `starts` gets the
// mask of lanes that start a range.
__device__ __forceinline__ int chunk_ranges(int t, int lane, int cur_a, int carried_e, int carried_t,
                                            uint64_t &starts, uint64_t *gaps = nullptr) {
    int tprev = lane_above(t);
    if (lane == 0) tprev = carried_t;
    const bool sure = lane == 0 ? (t > carried_e + 64) : (t > tprev + 127);
    const bool maybe = lane != 0 && !sure && (t > tprev + 64);
    uint64_t sm = __ballot(sure);
    uint64_t mm = __ballot(maybe);
    // entries more than 64 above their predecessor (lane 0: above the last entry of the previous chunk)
    if (gaps) *gaps = ((sm | mm) & ~1ull) | (minf_readlane(t, 0) > carried_t + 64 ? 1ull : 0ull);
    const uint64_t le = minf_lanemask_lt() | (1ull << lane);
    const uint64_t below = sm & le;
    const int j0 = below ? 63 - __builtin_clzll(below) : 0;
    const int tj0 = sm ? __shfl(t, j0) : 0;        // (wave-uniform: no shuffle for a chunk without sure starts)
    int a = below ? tj0 - 64 : cur_a;
    while (mm) {
        const int j = __builtin_ctzll(mm);
        mm &= mm - 1;
        const int ap = minf_readlane(a, j - 1), tp = minf_readlane(t, j - 1), tj = minf_readlane(t, j);
        const int ep = ap + ((((tp - ap) + 63) >> 6) << 6);
        if (tj > ep + 64) {
            const uint64_t later = sm & ~((2ull << j) - 1ull);          // sure starts above lane j
            const int next = later ? __builtin_ctzll(later) : 64;
            if (lane >= j && lane < next) a = tj - 64;
            sm |= 1ull << j;
        }
    }
    starts = sm;
    return a;
}

// ---------------------------------------------------------------------------------------------
// Translation-invariant fast path.
//
// For an entry that is neither skipped (o >= end_m) nor clipped (end_m - o < 64), t = end_m - o,
// so the whole range logic depends on the row block only through a shift: once a range STARTS at
// list entry g, everything the reference does from g on (ranges, blocks) is the same for every row
// block, moved by end_m.  vs_index_prep_kernel therefore walks each head's slash list ONCE, as a
// virtual row whose end is V = slash[0] + 64 (nothing skipped, nothing clipped), and tabulates
//   cpos[k]   start of the k-th block,                     k < nblocks
//   cpre[i]   index of the first block of the range that starts at entry i, else -1
//   crun[i]   ordinal of that range, else -1
//   run_a[r], run_e[r]   [start, end) of range r
//   cgaps[i]  the number of entries j <= i with t_j > t_{j-1} + 64 ("gap entries": the only entries
//             at which a range can start, for any row block -- skipping and clipping only shrink gaps)
//   glist[j]  the gap entries, ascending, j < ngaps: the first gap entry at or after entry x is glist[cgaps[x - 1]]
// all in the virtual row's coordinates (real position = virtual + end_m - V).
// vs_index_fast_kernel then handles a row block as follows: entries from the first valid one are
// processed exactly like vs_index_kernel until a range starts at an entry that also starts a range
// of the table (at once when no entry is skipped or clipped; after a few entries otherwise: chains
// that start at different entries meet at the first gap both see); from there the remaining blocks
// are copied from cpos with a shift (coalesced), and each remaining vertical x is emitted iff it is
// not inside one of the remaining tabulated ranges, is not below the end of the last range of the
// explicit part, and is below the last entry's t - the reference's merge rule restated per element.
// Inside the explicit part, a chunk of 64 entries without any gap above 64 means a dense run of
// diagonals: the entries up to the next entry of glist cannot start a range, so they only extend
// the current one, to a + 64 ceil((t_last - a) / 64), and their blocks are an arithmetic progression
// written at once -- lists whose slashes cluster (the usual case near the diagonal) would otherwise
// walk thousands of entries, 64 at a time, before they meet a tabulated range start.
#define IDX_TAB_HDR 8
// per head: header, seven tables of nnz_s ints, then a coverage bitmap of the virtual row (one bit
// per key position, set inside the tabulated ranges) of bm_words 32-bit words
__host__ __device__ __forceinline__ long long idx_bm_words(int rows) { return ((long long)rows * 64 + 64 + 31) / 32 + 1; }
__host__ __device__ __forceinline__ long long idx_tab_ints(int nnz_s, int rows) {
    return IDX_TAB_HDR + 7ll * nnz_s + idx_bm_words(rows);
}

// Coverage bitmap of a head's virtual row: bit p is set iff position p lies inside one of the tabulated ranges.  A
// range is the union of its blocks (its end moves by 64 at a time), so every block sets its 64 bits; what lies past the
// bitmap (up to 63 positions behind the last entry) is never looked up.
__device__ __forceinline__ void mark_block(uint32_t *bm, int words, int p) {
    const unsigned w = (unsigned)(p >> 5), sh = (unsigned)p & 31u;
    if (w < (unsigned)words) atomicOr(&bm[w], ~0u << sh);
    if (w + 1 < (unsigned)words) atomicOr(&bm[w + 1], ~0u);
    if (sh && w + 2 < (unsigned)words) atomicOr(&bm[w + 2], (1u << sh) - 1u);
}

// The walk of a head's list over chunks of 64 entries by one wavefront: (cur_a, carried_e, carried_t) is what the
// entries before a chunk leave behind, (nb, nr, ng) the number of blocks, ranges and gap entries before it.
struct PrepState { int cur_a, carried_e, carried_t; };
struct PrepCount { int nb, nr, ng; };
struct PrepChunk {                                   // one chunk, taken through the range logic
    int t, a, e, eprev;                              // this lane's entry, its range's start and end, the end one entry before
    uint64_t starts, gaps, changed;                  // entries that start a range, that follow a gap, that end a new block
    int base, cnt;
};
__device__ __forceinline__ void prep_chunk(PrepChunk &k, PrepState &st) {
    const int lane = minf_lane();
    if (k.base == 0) {
        const int t0 = minf_readlane(k.t, 0);
        st.cur_a = st.carried_e = t0 - 64;
        st.carried_t = t0;
    }
    k.a = chunk_ranges(k.t, lane, st.cur_a, st.carried_e, st.carried_t, k.starts, &k.gaps);
    const uint64_t valid = k.cnt == MINF_WAVE ? ~0ull : (1ull << k.cnt) - 1ull;
    if (k.base == 0) k.starts |= 1ull;
    k.starts &= valid;
    k.e = k.a + ((((k.t - k.a) + 63) >> 6) << 6);
    k.eprev = lane_above(k.e);
    if (lane == 0) k.eprev = st.carried_e;
    k.changed = __ballot(lane < k.cnt && k.e != k.eprev);
    st.carried_e = minf_readlane(k.e, k.cnt - 1);
    st.carried_t = minf_readlane(k.t, k.cnt - 1);
    st.cur_a = minf_readlane(k.a, k.cnt - 1);
}
// the counts behind a chunk
__device__ __forceinline__ void prep_count(const PrepChunk &k, PrepCount &n) {
    n.nb += __builtin_popcountll(k.changed);
    n.nr += __builtin_popcountll(k.starts);
    n.ng += __builtin_popcountll(k.gaps);            // (padding lanes repeat the last entry: never a gap)
}
// writes a chunk's entries of the tables; n: the counts before the chunk
__device__ __forceinline__ void prep_write(const PrepChunk &k, const PrepCount &n, int32_t *hdr, int nnz_s, uint32_t *bm, int bm_words) {
    const int lane = minf_lane();
    int32_t *cpos = hdr + IDX_TAB_HDR, *cpre = cpos + nnz_s, *crun = cpre + nnz_s;
    int32_t *run_a = crun + nnz_s, *run_e = run_a + nnz_s, *cgaps = run_e + nnz_s, *glist = cgaps + nnz_s;
    const uint64_t lt = minf_lanemask_lt();
    const bool valid = lane < k.cnt, is_start = (k.starts >> lane) & 1ull;
    const int kpos = n.nb + __builtin_popcountll(k.changed & lt);
    if ((k.changed >> lane) & 1ull) {
        cpos[kpos] = k.e - 64;
        if (bm) mark_block(bm, bm_words, k.e - 64);
    }
    if (valid) {
        const int r = n.nr + __builtin_popcountll(k.starts & lt), gapno = n.ng + __builtin_popcountll(k.gaps & lt);
        const bool gap = (k.gaps >> lane) & 1ull;
        cgaps[k.base + lane] = gapno + (gap ? 1 : 0);
        if (gap) glist[gapno] = k.base + lane;
        cpre[k.base + lane] = is_start ? kpos : -1;
        crun[k.base + lane] = is_start ? r : -1;
        if (is_start) {
            run_a[r] = k.a;
            if (r > 0) run_e[r - 1] = k.eprev;
        }
    }
}
__device__ __forceinline__ int prep_entry(const int32_t *__restrict__ sl, int nnz_s, int c) {      // this lane's entry of chunk c
    return sl[min(c * MINF_WAVE + minf_lane(), nnz_s - 1)];          // (padding lanes repeat the last entry)
}
__device__ __forceinline__ PrepChunk prep_place(int entry, int nnz_s, int V, int c) {
    PrepChunk k;
    k.base = c * MINF_WAVE;
    k.cnt = min(MINF_WAVE, nnz_s - k.base);
    k.t = max(V - entry, 64);
    return k;
}
__device__ __forceinline__ PrepChunk prep_load(const int32_t *__restrict__ sl, int nnz_s, int V, int c) {
    return prep_place(prep_entry(sl, nnz_s, c), nnz_s, V, c);
}
// f(chunk) for chunks [c0, c1) in turn.  What f does is one chain over the chunks, so the entries of the next two are
// on their way meanwhile (60000 slashes, 8 heads, builder with payload only: 174 -> 170 us against each chunk loaded
// where it is used; in the walk of one wavefront 140000 slashes 1443 -> 1116).
template <typename F> __device__ __forceinline__ void prep_each(const int32_t *__restrict__ sl, int nnz_s, int V, int c0, int c1, F f) {
    int next = prep_entry(sl, nnz_s, c0), next2 = prep_entry(sl, nnz_s, c0 + 1);
    for (int c = c0; c < c1; ++c) {
        PrepChunk k = prep_place(next, nnz_s, V, c);
        next = next2;
        next2 = prep_entry(sl, nnz_s, c + 2);
        f(k);
    }
}

__device__ __forceinline__ void prep_header(int32_t *hdr, int nnz_s, int rows, int V, const PrepState &st, const PrepCount &n) {
    int32_t *run_e = hdr + IDX_TAB_HDR + 4ll * nnz_s;
    run_e[n.nr - 1] = st.carried_e;
    hdr[0] = n.nb;
    hdr[1] = n.nr;
    hdr[2] = V;
    // the bitmap covers positions [0, 32 * bm_words); a list whose largest offset lies far
    // outside the context does not fit and the row blocks fall back to searching the ranges
    hdr[3] = (long long)V <= 32 * (idx_bm_words(rows) - 1) ? 1 : 0;
    hdr[4] = n.ng;
}

// The table pass: one workgroup of PREP_WAVES wavefronts per head.  The walk over the list is a chain
// (which range an entry belongs to depends on where the ranges before it started), but an entry more
// than 127 above its predecessor starts a range whatever came before ("sure" start) and only entries
// 65..127 above their predecessor ("maybe") depend on the 64-phase of the current range.  So every
// wavefront takes a contiguous share of the chunks; all of them first mark the sure and maybe entries
// of their chunks (independent work); a wavefront then finds the state at the head of its share by
// going back to the last sure start before it and replaying only the maybe entries in between (none
// inside a dense run, a handful when the offsets are scattered); it takes its share through the range logic,
// the counts of blocks, ranges and gap entries are summed over the wavefronts before it, and it writes the tables.
// A share of at most PREP_KEEP chunks stays in registers from the marks to the tables (one round of loads in flight
// together); longer ones are loaded and walked once to count and again to write.  Lists of at most two chunks, or of
// more chunks than LDS holds marks for, are walked by one wavefront alone: 500000 slashes, one head, take 3365 us (no
// bitmap atomics in that chain; with them 4895), 393216, the most that are shared, 625 (a limit of 131072: 3652).
// The coverage bitmap is built in LDS beside the tables (where it fits: `bm_words` > 0) and copied out at the end.
// Latency-bound, one workgroup per head.  With a bitmap kernel behind it that searched the ranges, and a share's state
// found by reading the marks one chunk at a time, the two took (us, now in one kernel): 6096 slashes, clustered, 16001
// tokens 29 + 5 -> 16, 131072 tokens 25 + 5 -> 15; uniform, 262144 tokens 39 + 7 -> 28; 2048 slashes, 8192 tokens,
// 4 heads 12 + 5 -> 9.
#define PREP_WAVES 16
#define PREP_KEEP 8
#define PREP_LDS_MAX_BYTES 98304
#define PREP_MAX_CHUNKS (PREP_LDS_MAX_BYTES / 16)          // 393216 entries
// One workgroup: the tables of one head at `hdr` from its list `sl` of nnz_s offsets (in global memory or in LDS).
// prep_lds: 16 bytes per chunk of 64 entries up to PREP_MAX_CHUNKS, or bm_words 32-bit words if that is more.
__device__ __forceinline__ void prep_tables(const int32_t *__restrict__ sl, int32_t *hdr, int nnz_s, int rows, int bm_words, uint64_t *prep_lds) {
    __shared__ int cnt_b[PREP_WAVES], cnt_r[PREP_WAVES], cnt_g[PREP_WAVES];
    const int lane = minf_lane();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int V = sl[0] + 64;
    const int nchunks = (nnz_s + MINF_WAVE - 1) / MINF_WAVE;
    uint32_t *bm = bm_words > 0 ? reinterpret_cast<uint32_t *>(prep_lds) : nullptr;
    auto clear_bitmap = [&]() {
        for (int i = (int)threadIdx.x; i < bm_words; i += PREP_WAVES * MINF_WAVE) bm[i] = 0u;
        __syncthreads();
    };

    if (nchunks <= 2 || nchunks > PREP_MAX_CHUNKS) {        // (workgroup-uniform)
        clear_bitmap();
        if (wave == 0) {
            PrepState st{0, 0, 0};
            PrepCount n{0, 0, 0};
            prep_each(sl, nnz_s, V, 0, nchunks, [&](PrepChunk &k) {
                prep_chunk(k, st);
                prep_write(k, n, hdr, nnz_s, bm, bm_words);
                prep_count(k, n);
            });
            if (lane == 0) prep_header(hdr, nnz_s, rows, V, st, n);
        }
    } else {
        uint64_t *sure_m = prep_lds, *maybe_m = prep_lds + nchunks;
        const int per = (nchunks + PREP_WAVES - 1) / PREP_WAVES;
        const int c0 = min(wave * per, nchunks), c1 = min(c0 + per, nchunks);
        const bool keep = per <= PREP_KEEP;
        PrepChunk held[PREP_KEEP];
        // ---- marks: entry i is a sure start when t_i > t_{i-1} + 127, a maybe when t_i > t_{i-1} + 64
        // (entry 0 starts the first range)
        auto mark = [&](const PrepChunk &k, int before) {
            const int i = k.base + lane;
            int tp = lane_above(k.t);
            if (lane == 0) tp = before;
            const bool valid = lane < k.cnt;
            const bool sure = valid && (i == 0 || k.t > tp + 127);
            const bool maybe = valid && !sure && k.t > tp + 64;
            const uint64_t sm = __ballot(sure), mm = __ballot(maybe);
            if (lane == 0) { sure_m[k.base / MINF_WAVE] = sm; maybe_m[k.base / MINF_WAVE] = mm; }
        };
        const int t_before = c0 > 0 ? max(V - sl[c0 * MINF_WAVE - 1], 64) : 0;      // the entry before the share
        if (keep) {
#pragma unroll
            for (int j = 0; j < PREP_KEEP; ++j)
                if (c0 + j < c1) held[j] = prep_load(sl, nnz_s, V, c0 + j);
#pragma unroll
            for (int j = 0; j < PREP_KEEP; ++j)
                if (c0 + j < c1) mark(held[j], j ? minf_readlane(held[j ? j - 1 : 0].t, 63) : t_before);
        } else {
            for (int c = c0; c < c1; ++c)
                mark(prep_load(sl, nnz_s, V, c), c > 0 ? max(V - sl[c * MINF_WAVE - 1], 64) : 0);
        }
        __syncthreads();
        // ---- the state at the head of this wavefront's share (wave-uniform scalar work)
        PrepState st{0, 0, 0};
        if (c0 > 0 && c0 < nchunks) {
            // (64 chunks' marks per step, one a lane: a dense run has none over a hundred chunks)
            int cs = c0 - 1;
            uint64_t smask = 0, some;
            for (;;) {                                           // (chunk 0 holds entry 0, a sure start)
                const uint64_t mine = sure_m[max(cs - lane, 0)];
                some = __ballot(mine != 0 && lane <= cs);
                if (some) break;
                cs -= 64;
            }
            cs -= __builtin_ctzll(some);
            smask = sure_m[cs];
            const int js = cs * MINF_WAVE + (63 - __builtin_clzll(smask));     // the last sure start before the share
            int a = max(V - sl[js], 64) - 64;
            for (int cb = cs; cb < c0; cb += 64) {
                uint64_t mine = cb + lane < c0 ? maybe_m[cb + lane] : 0;
                if (cb + lane == cs) mine &= ~((2ull << (js - cs * MINF_WAVE)) - 1ull);      // maybes above the sure start only
                for (uint64_t left = __ballot(mine != 0); left; left &= left - 1) {
                    const int c = __builtin_ctzll(left);
                    uint64_t mm = ((uint64_t)(unsigned)minf_readlane((int)(mine >> 32), c) << 32) | (unsigned)minf_readlane((int)mine, c);
                    while (mm) {
                        const int j = (cb + c) * MINF_WAVE + __builtin_ctzll(mm);
                        mm &= mm - 1;
                        const int tj = max(V - sl[j], 64), tp = max(V - sl[j - 1], 64);
                        const int ep = a + ((((tp - a) + 63) >> 6) << 6);
                        if (tj > ep + 64) a = tj - 64;
                    }
                }
            }
            st.cur_a = a;
            st.carried_t = t_before;
            st.carried_e = a + ((((t_before - a) + 63) >> 6) << 6);
        }
        // ---- count, sum over the wavefronts before this one, write
        const PrepState head = st;
        PrepCount n{0, 0, 0};
        if (keep) {
#pragma unroll
            for (int j = 0; j < PREP_KEEP; ++j)
                if (c0 + j < c1) {
                    prep_chunk(held[j], st);
                    prep_count(held[j], n);
                }
        } else {
            prep_each(sl, nnz_s, V, c0, c1, [&](PrepChunk &k) {
                prep_chunk(k, st);
                prep_count(k, n);
            });
        }
        if (lane == 0) { cnt_b[wave] = n.nb; cnt_r[wave] = n.nr; cnt_g[wave] = n.ng; }
        __syncthreads();
        PrepCount at{0, 0, 0}, all{0, 0, 0};
#pragma unroll
        for (int w = 0; w < PREP_WAVES; ++w) {
            const int b = cnt_b[w], r = cnt_r[w], g = cnt_g[w];
            if (w < wave) { at.nb += b; at.nr += r; at.ng += g; }
            all.nb += b; all.nr += r; all.ng += g;
        }
        clear_bitmap();                                          // (everyone is done with the marks)
        if (keep) {
#pragma unroll
            for (int j = 0; j < PREP_KEEP; ++j)
                if (c0 + j < c1) {
                    prep_write(held[j], at, hdr, nnz_s, bm, bm_words);
                    prep_count(held[j], at);
                }
        } else {
            st = head;
            prep_each(sl, nnz_s, V, c0, c1, [&](PrepChunk &k) {
                prep_chunk(k, st);
                prep_write(k, at, hdr, nnz_s, bm, bm_words);
                prep_count(k, at);
            });
        }
        if (c0 < nchunks && c1 == nchunks && lane == 0) prep_header(hdr, nnz_s, rows, V, st, all);
    }
    if (bm) {
        __syncthreads();                                         // every block is marked
        uint32_t *dst = reinterpret_cast<uint32_t *>(hdr + IDX_TAB_HDR + 7ll * nnz_s);
        for (int i = (int)threadIdx.x; i < bm_words; i += PREP_WAVES * MINF_WAVE) dst[i] = bm[i];
    }
}
