// Sparse flash-attention forward for gfx950: one 64x64 tile engine, four tile
// sources (vertical-slash block+column lists, block-sparse lists, analytic
// A-shape ranges, dense causal).
//
// Work split: one workgroup of 4 wavefronts per (batch, query head, PAIR of neighbouring 64-row
// blocks); each wavefront owns 32 query rows.  The two row blocks walk their tile lists in lockstep:
// a tile that is on both lists is copied into LDS once for 128 query rows, a tile that only one of
// them visits is copied by that half into buffers of its own while the other half does the same
// with a tile of its list.  For dense causal and A-shape / tri-shape the lists are analytic and
// differ by at most their ends; vertical-slash and block-sparse lists are split into common and
// leftover entries once, in LDS, before the tile loop.  Besides halving the
// copies of shared tiles, the lockstep is what keeps long scattered lists fast: row block m+1's
// list is row block m's shifted by 64 keys, so what one half fetches now the other fetched a step
// ago and finds in L2 (measured +23..38 % on lists of several hundred blocks, +1 % on the
// cache-friendly benchmark layer, against an earlier form of this kernel with one 2-wave workgroup
// per row block).
// Everything is computed in the TRANSPOSED orientation so that softmax statistics are per lane:
//
//   S^T[token][qrow] = K_tile . Q^T      v_mfma_f32_32x32x16 (A = K from LDS, B = Q in VGPRs)
//   O^T[d][qrow]    += V_tile^T . P^T    (A = V^T via ds_read_b64_tr_b16, B = P straight from
//                                          the S^T accumulators, converted to bf16/f16)
//
// In the 32x32 accumulator layout lane l holds column n = l%32 (one query row)
// and rows 8*(r/4) + 4*(l/32) + r%4, so the running max / sum / rescale factor
// of a query row live in lanes l and l^32 and never need a row broadcast, and
// the probabilities of a lane are exactly the B operand of the second MFMA once
// the contraction (token) index is permuted the same way on the V side.
//
// LDS: one K and one V tile per workgroup (two of each for the list walks: the second pair serves
// row block B in split steps; a second K tile's room in every form: the epilogue's 128 output rows
// lie there), [64 tokens][128] 16-bit, 256-byte rows whose 16-byte
// chunks are XOR-permuted (K: chunk ^ row%16, V: chunk ^ 4*(row%4)) so that the ds_read_b128 of 32
// K rows and the 4-row transpose reads of V hit distinct banks.  Tiles are copied global -> LDS
// directly (no staging registers, no LDS store instructions); the permutation is applied on the
// global-address side.  Contiguous tiles use buffer_load_dwordx4 ... lds with a scalar descriptor of
// the 64 tile rows, a scalar row offset and one of five loop-invariant per-lane offsets: no vector
// instruction per copy and 8 cycles less issue time per copy than the 64-bit-address form, which
// remains for gathered and clamped rows (global_load_lds_dwordx4).  At head_dim 128 48 KB of LDS (68 for
// lists, which also hold the split ones) and <= 256 registers keep two waves per SIMD resident (two
// 4-wave workgroups per CU); at 64 24 (36) KB and three of them, at 256 96 KB and one.
//
// One iteration of a wave (two workgroup barriers per tile, single buffers):
//   wait own K(it) copies; barrier (all of K(it) visible, everyone done with V(it-1))
//   issue V(it) copy; S^T = K.Q^T with the K fragments read two k-steps ahead of their MFMAs
//   wait own V(it) copies; barrier (all of V(it) visible, everyone done with K(it))
//   issue K(it+1) copy; read all V^T fragments; row max where it is needed; exponentials of keys 0..15
//   O^T += V^T.P^T with the exponentials of key group s+1 (16 keys) placed behind the MFMAs of
//   group s
// The compiler's own schedule read every fragment right before its MFMA (full LDS latency exposed
// sixteen times per tile); the order above is pinned with sched_barrier / sched_group_barrier.
//
// Other choices that measure faster on MI355X:
//  * index entries (block offsets, column counts) are wave-uniform and read through the constant
//    address space, i.e. scalar loads that do not queue behind the vector memory traffic; gathered
//    column ids are fetched one per lane an iteration ahead and distributed with wave shuffles;
//  * the running max is only raised when a tile exceeds it by more than 2^20 (bf16; 2^8 for f16
//    operands, whose probabilities must stay inside the f16 range), so nearly all tiles skip the
//    O^T rescale; for bf16 the row maximum is not even computed in most tiles (see sm_pv_block);
//  * the cross-half max uses v_permlane32_swap, the row sums v_dot2 on the rounded probabilities
//    (the same values the second MFMA consumes);
//  * s_setprio raises the wave while it issues MFMAs;
//  * the epilogue transposes O^T through LDS so each global store is 16 B of one 256-byte row.
#include "minf_common.h"
#include <math.h>
#include <string.h>
#include <type_traits>

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short short4_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
// native vectors, not HIP's u32x4_t/u32x2_t structs: arrays of those are not promoted to registers
typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u32x2_t;

enum { MODE_VS = MINF_OP_VERTICAL_SLASH, MODE_BS = MINF_OP_BLOCK_SPARSE, MODE_ASHAPE = MINF_OP_ASHAPE, MODE_DENSE = MINF_OP_DENSE };

constexpr int BM = 64;        // query rows per workgroup
constexpr int BN = 64;        // keys per tile
// head_dim (template parameter HD of the kernel): 64, 128 or, for dense / A-shape / tri-shape only, 256
constexpr int NTHREADS = 128; // 2 wavefronts per 64-row block, two row blocks per workgroup
// Scheduling constants (measured on MI355X): K fragments are read QK_AHEAD k-steps ahead of their
// MFMAs; VALU_PER_MFMA softmax instructions (five, or six with the row sums among them) are placed behind each of the first
// twelve PV MFMAs.
constexpr int QK_AHEAD = 2;
#ifndef MAX_PERIOD
#define MAX_PERIOD 8      // (a power of two) the row maximum is recomputed at least every MAX_PERIOD tiles
#endif
#ifndef LAZY_MAX_BF16
#define LAZY_MAX_BF16 20.0f
#endif
constexpr int VALU_MASK = 0x402;             // sched_group_barrier classes: VALU | transcendental

struct AttnParams {
    const char *q, *k, *v;
    char *o;
    long long qs[3], ks[3], vs[3], os[3];   // element strides: batch, head, token
    int batch, hq, hk, n;
    const int *seqlens;
    float scale_log2;
    float scale_log2_dense;  // tri-shape: scale of the rows >= dense_from (the reference scales them by the unpadded head_dim)
    int rows;
    // vertical-slash
    const int *bc, *bo, *cc, *ci;
    int nnz_s, nnz_v;
    // block-sparse
    const int *bidx;
    int max_blocks, bidx_rows;
    // a-shape; query rows >= dense_from attend to every earlier key (tri-shape), INT_MAX = none
    int n_init, n_local, dense_from;
    int descending;          // row blocks are handed out from the last one down
    int chunk, turn;         // units per deal; an XCD takes another place every 2^turn rounds of deals, 31: never (see plan_launch)
    FastDiv by_deal, by_group, by_groups, by_heads;   // workgroups of a deal; hq / hk; batch x kv groups; kv heads, or chunks of the head list
    // optional head selection: head_list[i], i < index_heads, are the query heads to process and i is
    // the head's position in the index tensors (which then have index_heads heads); without a list
    // every head is processed and index_heads = hq
    const int *head_list;
    int index_heads;
    // split walks (see SplitPlan): the row-block pairs >= split_first are walked by up to nseg workgroups,
    // one segment of the walk each, which leave their share of the sums in `part`
    int split_first, nseg, seg_len;
    char *part;
    int dtype;               // MINF_BF16, MINF_F16 or MINF_16BIT_SELECT
    const int *select;       // not null: this launch is one of two, and only the one for dtype *select does anything
    // CHOSEN launches only.  Behind the rest: every workgroup starts with a chain of reads of these arguments, and with two of
    // them in front the others' lay across one more cache line (A-shape, window 64, fp32 tensors, 32 / 8 heads, 65536 tokens 1185 : 1203 us)
    FastDiv by_set, by_chunks;      // groups of a set; deals of a group
    int far_turn;            // turn where most of four heads keep more than an eighth of the blocks, 0: no such turn
};

// Split walks.  A launch whose row-block pairs cannot fill the chip, or whose longest walks would outlast
// everything else, cuts the walks of its pairs >= `first` into segments of about `len` steps (at most
// `nseg` of them).  One workgroup walks one segment and writes its unnormalised sums -- O^T in fp32 in
// accumulator layout, row maximum and row sum -- to a slot of the caller's workspace; attn_merge_kernel
// folds the segments of a pair in ascending order and writes the output rows.
struct SplitPlan { int first, nseg, len; };
template <int HD> struct SplitSlot {
    static constexpr int ACC = 4 * HD * 32 * 4;              // four waves x [HD/32][4][64 lanes] x 16 bytes
    static constexpr int BYTES = ACC + 4 * 64 * 8;           // ... and (maximum, sum) per lane
};

typedef const __attribute__((address_space(4))) int *cint_ptr;
__device__ __forceinline__ cint_ptr as_const(const int *p) { return (cint_ptr)(unsigned long long)p; }
template <typename T> struct Mma;
template <> struct Mma<__bf16> {
    typedef bf16x8_t vec;
    static __device__ __forceinline__ f32x16_t mfma(vec a, vec b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mma<_Float16> {
    typedef f16x8_t vec;
    static __device__ __forceinline__ f32x16_t mfma(vec a, vec b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

union Frag {
    u32x4_t u;
    bf16x8_t b;
    f16x8_t h;
    short4_t s4[2];
};

template <typename T> __device__ __forceinline__ typename Mma<T>::vec frag_as(const Frag &f);
template <> __device__ __forceinline__ bf16x8_t frag_as<__bf16>(const Frag &f) { return f.b; }
template <> __device__ __forceinline__ f16x8_t frag_as<_Float16>(const Frag &f) { return f.h; }

template <typename T> __device__ __forceinline__ void cvt8(const float *x, Frag &f);
template <> __device__ __forceinline__ void cvt8<__bf16>(const float *x, Frag &f) {
#pragma unroll
    for (int j = 0; j < 8; ++j) f.b[j] = (__bf16)x[j];
}
template <> __device__ __forceinline__ void cvt8<_Float16>(const float *x, Frag &f) {
#pragma unroll
    for (int j = 0; j < 8; ++j) f.h[j] = (_Float16)x[j];
}

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 f16x2_t;
template <typename T> __device__ __forceinline__ float pair_sum(const Frag &f, float acc);
template <> __device__ __forceinline__ float pair_sum<__bf16>(const Frag &f, float acc) {
    const bf16x2_t one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
    for (int j = 0; j < 4; ++j) { bf16x2_t pr = {f.b[2 * j], f.b[2 * j + 1]}; acc = __builtin_amdgcn_fdot2_f32_bf16(pr, one, acc, false); }
    return acc;
}
template <> __device__ __forceinline__ float pair_sum<_Float16>(const Frag &f, float acc) {
    const f16x2_t one = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
    for (int j = 0; j < 4; ++j) { f16x2_t pr = {f.h[2 * j], f.h[2 * j + 1]}; acc = __builtin_amdgcn_fdot2(pr, one, acc, false); }
    return acc;
}
// One tile of keys: either 64 consecutive tokens from `start`, or 64 gathered
// token ids read from `gather` (entries >= nvalid are padding).
struct Tile {
    int start;          // first token (contiguous) / first list position (gathered)
    int gathered;       // 0/1
    int nvalid;         // gathered: number of valid list entries in this tile
    int on_a, on_b;     // paired walks: is the tile on the list of row block A / B
    int split;          // paired list walks: each row block has a tile of its own in this step
};
// (the longest block list the paired kernel splits in LDS is what a K tile holds twice: 2048 entries
// at head_dim 128, 1024 at 64)
constexpr int VS_ONLY_MAX = 512;   // ... and the most entries of one list that the other one lacks

// One workgroup of 4 waves covers the row blocks mA = 2*mp and mB = mA + 1.  It
// walks the union of their two tile lists once, so every K/V tile is copied into LDS once for 128
// query rows; a half skips the tiles that are not on its own list.  For dense causal and A-shape /
// tri-shape the lists are analytic and differ by at most the ends (the three helpers below); for
// block-sparse the two lists are merged on the fly inside the kernel.
template <int MODE>
__device__ __forceinline__ int pair_tile_count(const AttnParams &p, int mA, int mB, int &nblk) {
    if (MODE == MODE_DENSE || mB * BM + BM - 1 >= p.dense_from) {
        nblk = mB + 1;
        return nblk;
    }
    int lo_key = mA * BM - p.n_local + 1;
    int t_lo = lo_key > 0 ? (lo_key >> 6) : 0;
    int sink_tiles = (p.n_init + BN - 1) >> 6;
    nblk = min(sink_tiles, t_lo);
    return nblk + (mB - t_lo + 1);
}
template <int MODE>
__device__ __forceinline__ int pair_tile_start(const AttnParams &p, int mA, int mB, int nblk, int it) {
    if (MODE == MODE_DENSE || mB * BM + BM - 1 >= p.dense_from) return it * BN;
    int lo_key = mA * BM - p.n_local + 1;
    int t_lo = lo_key > 0 ? (lo_key >> 6) : 0;
    return (it < nblk ? it : t_lo + (it - nblk)) * BN;
}
// is the tile that starts at key `start` on the list of row block m ?
template <int MODE>
__device__ __forceinline__ bool tile_on_list(const AttnParams &p, int m, int start) {
    const int ti = start >> 6;
    if (ti > m) return false;
    if (MODE == MODE_DENSE || m * BM + BM - 1 >= p.dense_from) return true;
    int lo_key = m * BM - p.n_local + 1;
    int t_lo = lo_key > 0 ? (lo_key >> 6) : 0;
    return ti >= t_lo || ti < ((p.n_init + BN - 1) >> 6);
}

// LDS of one workgroup (declared by the kernel, see attn_fwd_kernel): separate objects, so that the
// compiler lets reads of one overtake copies into the other.
template <int MODE, int HD> struct AttnLds {
    static constexpr bool VSP = MODE == MODE_VS || MODE == MODE_BS;      // walks of two block lists
    static constexpr int TILE_BYTES = BN * HD * 2;
    static constexpr int NK = 2 * TILE_BYTES;                            // (the epilogue's 128 rows of O, too)
    static constexpr int NV = (VSP ? 2 : 1) * TILE_BYTES;
    static constexpr int NONLY = VSP ? 2 * VS_ONLY_MAX : 1;
};

// The whole walk of one workgroup (CUT: or one segment of it, see SplitPlan; a kernel of its own, because
// the bookkeeping costs the whole walk 2-3 % in scalar registers).  EVERY_MAX: the row maximum is computed for every tile; otherwise
// only where it is needed (see sm_pv_block), and the function returns true -- for the whole
// workgroup -- when a row sum left the safe range, i.e. when the walk has to be run again with
// EVERY_MAX (the output it wrote is then overwritten).
template <typename T, int MODE, int HD, bool EVERY_MAX, bool CUT>
__device__ __forceinline__ bool attn_walk(const AttnParams &p, const unsigned wg, char (&lds_k)[AttnLds<MODE, HD>::NK],
                                          char (&lds_v)[AttnLds<MODE, HD>::NV],
                                          int (&vs_only)[AttnLds<MODE, HD>::NONLY], int (&vs_wsum)[4], int (&vs_bad)[2],
                                          int &lds_redo) {
    static_assert(HD == 256 || HD == 128 || HD == 64, "head_dim 64, 128 or 256");
    static_assert(HD <= 128 || !(MODE == MODE_VS || MODE == MODE_BS), "the list walks are built for head_dim <= 128");
    constexpr int ROW_BYTES = HD * 2;                       // one token row of K / V / Q / O
    constexpr int KS = HD / 16;                             // k-steps of S^T = K.Q^T
    constexpr int NDB = HD / 32;                            // 32-row blocks of O^T
    constexpr int NCH = ROW_BYTES / 16;                     // 16-byte chunks per row
    constexpr int RPI = 64 / NCH;                           // tile rows one copy instruction fills (64 lanes x 16 B)
    // LDS chunk permutations (conflict-free ds_read_b128 of 32 K rows / transpose reads of 4 V rows):
    // 256-byte rows: K chunk ^ row%16, V chunk ^ 4*(row%4); 128-byte rows (two rows per bank sweep):
    // K chunk ^ (row/2)%8, V chunk ^ 4*((row/2)%2)
    auto swz_k = [](int row) { return HD >= 128 ? (row & 15) : ((row >> 1) & 7); };
    auto swz_v = [](int row) { return HD >= 128 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); };
    constexpr int NT = 2 * NTHREADS;                        // threads per workgroup
    constexpr int CROWS = 16;                               // tile rows copied by one wave (shared tile)
    // VSP: the paired walk of two block lists -- the vertical-slash block lists, or the block-sparse
    // lists (block numbers, i.e. key starts / 64; no columns)
    constexpr bool VSP = MODE == MODE_VS || MODE == MODE_BS;
    constexpr int LIST_SCALE = MODE == MODE_BS ? BN : 1;     // list entry -> first key of the block
    constexpr int TILE_BYTES = BN * ROW_BYTES;
    constexpr int VS_PAIR_MAX = TILE_BYTES / 8;             // both staged lists fit the second K tile
    // paired list walks (vertical-slash, block-sparse): a second K and V tile (row block B's buffers in the steps in which each
    // row block has a tile of its own); before that, the second K tile stages the two block lists and
    // the second V tile holds their merge
    char *const lds_k1 = lds_k + (VSP ? TILE_BYTES : 0);
    char *const lds_v1 = lds_v + (VSP ? TILE_BYTES : 0);

    // ---- which (batch, head, row block): XCD-aware remap --------------------
    // Consecutive workgroup ids go round-robin to the 8 XCDs.  Deal number 8 r + x of the launch, the workgroups
    // that share K/V and so an L2 (some neighbouring row-block pairs of the query heads of a kv group), is worked
    // through by one of them, consecutive deals by different ones (see plan_launch).
    // (32-bit arithmetic: the launcher refuses grids beyond 2^31 workgroups, and 64-bit divisions of
    // wave-uniform values cost a thousand scalar instructions per workgroup here)
    const int group = (int)p.by_group.d;
    unsigned rest = wg >> 3;
    auto next_digit = [&](const FastDiv &f) { const unsigned q = fast_quot(rest, f), r = rest - q * f.d; rest = q; return r; };
    const unsigned in_deal = next_digit(p.by_deal);
    rest = 8u * rest + ((wg + (rest >> p.turn)) & 7u);
    const unsigned gi = next_digit(p.by_groups);
    const unsigned first_unit = rest * (unsigned)p.chunk;
    rest = in_deal;
    const int hin = (int)next_digit(p.by_group);
    // Dense causal work grows with the row block, so the heavy (late) blocks go first.  The sparse
    // modes have near-constant work per row block once the context is long and then measure 1 %
    // faster in ascending order; up to 64K tokens their early row blocks are still growing and the
    // descending order wins for vertical-slash lists (+4 % at 16K, +1.7 % at 32K): the launcher picks.
    const int rows_wg = (p.rows + 1) >> 1;                           // row-block pairs per (batch, head)
    const int split_units = (rows_wg - p.split_first) * p.nseg;      // (no split: split_first == rows_wg)
    const unsigned units = (unsigned)(p.split_first + split_units);
    const int mi = (int)(first_unit + rest);
    rest = gi;
    if (mi >= (int)units) return false;              // padding of the last deal (workgroup-uniform)
    int mslot, seg = -1;                             // row-block pair, segment of its walk (-1: the whole walk)
    if (CUT && mi < split_units) {                    // the split pairs, longest walks first
        // first segments of all of them, then second segments, ...: a walk's own segments side by side, of
        // which only every nseg-th exists where walks are short, all went to the same shader engines
        // (workgroups are dealt to them in turn: dense, 12000 tokens, 16 heads of 64, two segments: 450 us)
        const int split_pairs = rows_wg - p.split_first;
        mslot = rows_wg - 1 - mi % split_pairs;
        seg = mi / split_pairs;
    } else {
        mslot = p.descending ? rows_wg - 1 - mi : mi - split_units;
        if (p.descending) mslot += split_units - (rows_wg - p.split_first);
    }
    int hkv, b, h, hs;                               // hs: head position in the index tensors
    if (p.head_list) {
        // the selected heads in chunks of `group` consecutive list entries take the place of the kv
        // groups: neighbours in the (ascending) list mostly share a kv head
        const int ch = (int)next_digit(p.by_heads);
        b = (int)rest;
        hs = ch * group + hin;
        if (hs >= p.index_heads) return false;       // padding of the last chunk (workgroup-uniform)
        h = as_const(p.head_list)[hs];
        hkv = (int)fast_quot((unsigned)h, p.by_group);
    } else {
        hkv = (int)next_digit(p.by_heads);
        b = (int)rest;
        h = hkv * group + hin;
        hs = h;
    }

    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wave_wg = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: keep it in an SGPR
    const int half = wave_wg >> 1;                                   // which row block of the pair
    const int wave = wave_wg & 1;                                    // wave inside the row block
    const int m = 2 * mslot + half;
    const int mA = 2 * mslot, mB = min(mA + 1, p.rows - 1);
    const int l32 = lane & 31;
    const int g = lane >> 5;

    const int seqlen = p.seqlens ? min(p.seqlens[b], p.n) : p.n;
    const int row0 = m * BM;
    const int qrow = row0 + wave * 32 + l32;          // this lane's query row
    char *o_base = p.o + ((long long)b * p.os[0] + (long long)h * p.os[1]) * 2;

    // row block past the sequence: zeros (16 B per lane-step); the other
    // half may still have work, so this half stays for the copies and barriers without tiles
    const bool have_rows = m < p.rows && row0 < seqlen;
    if (!have_rows) {
        if (m < p.rows && !(CUT && seg >= 0))         // (rows of a split pair are written by the merge)
            for (int i = tid & (NTHREADS - 1); i < BM * NCH; i += NTHREADS) {
                int r = row0 + i / NCH;
                if (r < p.n) *reinterpret_cast<u32x4_t *>(o_base + (long long)r * p.os[2] * 2 + (i % NCH) * 16) = u32x4_t{0u, 0u, 0u, 0u};
            }
        if (mA * BM >= seqlen) return false;            // (workgroup-uniform: both halves are past)
    }

    const char *q_base = p.q + ((long long)b * p.qs[0] + (long long)h * p.qs[1]) * 2;
    const char *k_base = p.k + ((long long)b * p.ks[0] + (long long)hkv * p.ks[1]) * 2;
    const char *v_base = p.v + ((long long)b * p.vs[0] + (long long)hkv * p.vs[1]) * 2;
    const long long k_row = p.ks[2] * 2, v_row = p.vs[2] * 2;
    const long long ridx = ((long long)b * p.index_heads + hs) * p.rows + min(m, p.rows - 1);

    // where the block lists live: [batch, heads, list_rows, list_w]
    [[maybe_unused]] const int *const list_base = MODE == MODE_BS ? p.bidx : p.bo;
    [[maybe_unused]] const int list_w = MODE == MODE_BS ? p.max_blocks : p.nnz_s;
    [[maybe_unused]] const int list_rows = MODE == MODE_BS ? p.bidx_rows : p.rows;
    [[maybe_unused]] int vs_na = 0, vs_nb = 0, vs_cca = 0, vs_ccb = 0, vs_nc = 0;
    [[maybe_unused]] bool vs_merged = false;
    [[maybe_unused]] long long vs_ra = 0, vs_rb = 0;
    [[maybe_unused]] const int *ga = nullptr, *gb = nullptr;
    [[maybe_unused]] int vs_head_a = 0, vs_head_b = 0;
    if constexpr (VSP) {
        const bool b_exists = 2 * mslot + 1 < p.rows && (2 * mslot + 1) * BM < seqlen;
        vs_ra = ((long long)b * p.index_heads + hs) * list_rows + mA;
        vs_rb = b_exists ? vs_ra + 1 : vs_ra;
        // the lists' first 256 entries are fetched beside their lengths, not after them (a list row has list_w
        // entries whatever its length)
        ga = list_base + vs_ra * list_w;
        gb = list_base + vs_rb * list_w;
        vs_head_a = ga[min(tid, list_w - 1)];
        vs_head_b = gb[min(tid, list_w - 1)];
        if constexpr (MODE == MODE_BS) {
            // row block m visits the first min(m + 1, max_blocks) entries of its row; no columns
            vs_na = min(mA + 1, p.max_blocks);
            vs_nb = b_exists ? min(mA + 2, p.max_blocks) : 0;
        } else {
            vs_na = max(0, min(as_const(p.bc)[vs_ra], p.nnz_s));
            vs_cca = max(0, min(as_const(p.cc)[vs_ra], p.nnz_v));
            vs_nb = b_exists ? max(0, min(as_const(p.bc)[vs_rb], p.nnz_s)) : 0;
            vs_ccb = b_exists ? max(0, min(as_const(p.cc)[vs_rb], p.nnz_v)) : 0;
        }
    }
    // steps of the walk (splitting the lists into common and leftover entries does not change their number)
    int nblk = 0, ntiles;
    if constexpr (VSP) ntiles = max(vs_na + ((vs_cca + BN - 1) >> 6), vs_nb + ((vs_ccb + BN - 1) >> 6));
    else ntiles = pair_tile_count<MODE>(p, mA, mB, nblk);
    // the part of the walk this workgroup makes: all of it, or one segment
    int it_begin = 0, it_end = ntiles;
    char *slot = nullptr;
    if (CUT && seg >= 0) {
        const int ns = max(1, min(p.nseg, (ntiles + p.seg_len - 1) / p.seg_len));
        const int len = (ntiles + ns - 1) / ns;
        it_begin = min(seg * len, ntiles);
        it_end = seg < ns ? min(it_begin + len, ntiles) : it_begin;
        const int heads = p.head_list ? p.index_heads : p.hq;
        slot = p.part + (((long long)(b * heads + hs) * (rows_wg - p.split_first) + (mslot - p.split_first)) * p.nseg + seg) * SplitSlot<HD>::BYTES;
        if (it_begin >= it_end) {                       // (workgroup-uniform) nothing to add: a row sum of zero says so, before any of the walk's set-up
            float2 *ml = reinterpret_cast<float2 *>(slot + SplitSlot<HD>::ACC) + tid;
            *ml = make_float2(-INFINITY, 0.f);
            return false;
        }
    }

    constexpr bool every_max = EVERY_MAX;
    // log2-domain scale of this lane's query row: one value per launch, except for the dense rows of a
    // tri-shape launch (the reference scales its A-shape rows by the padded head_dim and its last
    // rows by the unpadded one, streaming_kernel.py:575 against :826)
    float sc_l2 = p.scale_log2;
    if constexpr (MODE == MODE_ASHAPE) sc_l2 = qrow >= p.dense_from ? p.scale_log2_dense : p.scale_log2;
    // ---- Q fragments (B operand of S^T): row qrow, d = 16*ks + 8*g + 0..7 ----
    Frag qf[KS];
    {
        const bool ok = qrow < seqlen;
        const char *qp = q_base + (long long)(ok ? qrow : min(row0, seqlen - 1)) * p.qs[2] * 2 + g * 16;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            qf[ks].u = *reinterpret_cast<const u32x4_t *>(qp + ks * 32);
            if (!ok) qf[ks].u = u32x4_t{0u, 0u, 0u, 0u};
        }
    }

    // Paired list walks (vertical-slash block lists, block-sparse lists scaled to key starts): the
    // block lists of the two row blocks (ascending key starts; vertical-slash lists of
    // neighbouring row blocks are each other's translate by 64 keys wherever no entry is clipped, so
    // runs of blocks share all but their ends) are split ONCE, by all 256 threads, before the tile
    // loop: both lists are staged in LDS, every entry looks itself up in the other list by binary
    // search, and a workgroup prefix sum over the hits places it either in the list of COMMON
    // entries (tiles that both row blocks visit: copied once by four waves, one LDS word per step)
    // or in its row block's list of entries the other one lacks (run ends).  Each pair of waves looks up one
    // list, both at once; with a pass per list and a check before them a workgroup took 6.5 us to its first tile
    // copy (block-sparse, top-100; 2.9 of them chains of LDS reads and six barriers) where it takes 3.4 now:
    // vertical-slash, 16001 tokens, 32 / 8 heads 1531 -> 1519 us (runs of one side 0.5 % apart); on longer
    // walks nothing beyond noise.
    // The walk is then
    //   common tiles, both halves computing;
    //   split steps: every half visits its own leftover tiles -- the entries the other list lacks,
    //   then its gathered column tiles -- with the K/V buffers of its own half,
    // i.e. exactly max(tiles of A, tiles of B) steps, never more than the longer list alone.
    // Lists that are too long for LDS or not strictly ascending are not split: each half then walks
    // its whole list in split steps (still in lockstep with its neighbour, which is what keeps the
    // neighbour's tiles in L2 when the lists are long and scattered).
    if constexpr (VSP) {
        if (vs_na <= VS_PAIR_MAX && vs_nb <= VS_PAIR_MAX && vs_na > 0 && vs_nb > 0) {
            int *rawA = reinterpret_cast<int *>(lds_k1), *rawB = rawA + VS_PAIR_MAX;
            int *common = reinterpret_cast<int *>(lds_v1);
            if (tid < 2) vs_bad[tid] = 0;
            if (tid < vs_na) rawA[tid] = vs_head_a * LIST_SCALE;
            if (tid < vs_nb) rawB[tid] = vs_head_b * LIST_SCALE;
            for (int i = tid + NT; i < vs_na; i += NT) rawA[i] = ga[i] * LIST_SCALE;
            for (int i = tid + NT; i < vs_nb; i += NT) rawB[i] = gb[i] * LIST_SCALE;
            __syncthreads();
            // waves 0 and 1 look up list A in list B, waves 2 and 3 list B in list A.  Entry i of `mine` goes to
            // common[#hits before i] when `other` holds it too (written once, by the first pair), else to
            // only[i - #hits before i].  The look-ups need strictly ascending lists, which is checked along the way:
            // in other lists they find something or other, inside the list's bounds, and nothing of it is used
            const int *mine = half ? rawB : rawA, *other = half ? rawA : rawB;
            const int nmine = half ? vs_nb : vs_na, nother = half ? vs_na : vs_nb;
            int *only = vs_only + half * VS_ONLY_MAX;
            const unsigned long long lt = (1ull << lane) - 1ull;
            bool bad = false;
            int carry = 0;
            for (int base = 0; base < max(vs_na, vs_nb); base += NTHREADS) {      // uniform trip count
                const int i = base + (tid & (NTHREADS - 1));
                const bool valid = i < nmine;
                const int x = valid ? mine[i] : 0;
                bad |= valid && i > 0 && mine[max(i - 1, 0)] >= x;
                int lo = 0, hi = nother;                           // first entry of `other` >= x
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (other[mid] < x) lo = mid + 1; else hi = mid;
                }
                const bool eq = valid && lo < nother && other[lo] == x;
                const unsigned long long bal = __ballot(eq);
                if (lane == 0) vs_wsum[wave_wg] = __builtin_popcountll(bal);
                __syncthreads();
                const int first = vs_wsum[2 * half], second = vs_wsum[2 * half + 1];
                const int pre = carry + (wave ? first : 0) + __builtin_popcountll(bal & lt);
                if (valid) {
                    if (eq) { if (!half) common[pre] = x; }
                    else if (i - pre < VS_ONLY_MAX) only[i - pre] = x;
                }
                carry += first + second;
                if (base + NTHREADS >= max(vs_na, vs_nb) && __any(bad) && lane == 0) vs_bad[0] = 1;
                if (base + NTHREADS >= max(vs_na, vs_nb) && tid == 0) vs_bad[1] = carry;
                __syncthreads();
            }
            // (the last barrier also orders these LDS lists before their readers)
            vs_nc = __builtin_amdgcn_readfirstlane(vs_bad[1]);
            vs_merged = !__builtin_amdgcn_readfirstlane(vs_bad[0]) && vs_nc > 0 && vs_na - vs_nc <= VS_ONLY_MAX && vs_nb - vs_nc <= VS_ONLY_MAX;
            if (!vs_merged) vs_nc = 0;
        }
    }
    // paired vertical-slash: vs_nc common steps, then the split steps: per half its leftover block
    // entries (from LDS when the lists were split, else its whole list from global memory) and its
    // gathered column tiles.  The barriers are the workgroup's: both halves make max(A, B) split
    // steps and a half without a tile only keeps the barriers.
    [[maybe_unused]] int vs_nb_mine = 0, vs_cc_mine = 0, vs_nt_mine = 0;
    if constexpr (VSP) {
        const int nb_a = vs_na - vs_nc, nb_b = vs_nb - vs_nc;
        const int nt_a = nb_a + ((vs_cca + BN - 1) >> 6), nt_b = nb_b + ((vs_ccb + BN - 1) >> 6);
        vs_nb_mine = half ? nb_b : nb_a;
        vs_cc_mine = half ? vs_ccb : vs_cca;
        vs_nt_mine = have_rows ? (half ? nt_b : nt_a) : 0;
    }
    auto more_tiles = [&](int it) -> bool { return it < it_end; };   // is there a tile number `it` ?
    // paired vertical-slash: entry it+1 of the common list sits in a scalar when step `it` starts; the
    // LDS read of entry it+2 is issued at the top of step `it` (no tile copy is in flight there: the
    // list shares an LDS object with the V tiles and must not wait for one) and turns into the next
    // scalar at the end of the step, its latency hidden behind the tile's work
    [[maybe_unused]] int vs_entry = 0, vs_pref = 0;
    // this row block's own list in global memory (walked directly when the lists were not split)
    [[maybe_unused]] const cint_ptr sp_list = as_const(list_base) + (((long long)b * p.index_heads + hs) * list_rows + min(m, p.rows - 1)) * list_w;
    auto vs_list = [&](int i) -> int { return reinterpret_cast<const int *>(lds_v1)[min(i, 2 * VS_PAIR_MAX - 1)]; };
    auto tile_of = [&](int it) -> Tile {      // called with it = it_begin, it_begin + 1, ... in order
        if constexpr (VSP) {
            Tile t;
            t.gathered = 0;
            t.nvalid = BN;
            if (it < vs_nc) {
                t.split = 0;
                t.on_a = t.on_b = 1;
                t.start = vs_entry;                        // common entry `it`, fetched a step ahead
            } else {
                const int j = it - vs_nc;
                t.split = 1;
                t.on_a = t.on_b = j < vs_nt_mine;          // (this half's own flag)
                t.start = 0;
                if (j < vs_nb_mine) {
                    if (vs_merged) t.start = __builtin_amdgcn_readfirstlane(vs_only[half * VS_ONLY_MAX + j]);
                    else t.start = sp_list[j] * LIST_SCALE;
                } else if (j < vs_nt_mine) {
                    t.gathered = 1;
                    t.start = (j - vs_nb_mine) * BN;
                    t.nvalid = min(BN, vs_cc_mine - t.start);
                }
            }
            return t;
        } else {
            Tile t;
            t.gathered = 0;
            t.nvalid = BN;
            t.on_a = t.on_b = 1;
            t.start = pair_tile_start<MODE>(p, mA, mB, nblk, it);
            return t;
        }
    };

    // ---- global -> LDS copies without a register round trip (global_load_lds_dwordx4): every lane
    // fetches 16 bytes from its own global address and the wave's 64 x 16 B land contiguously in
    // LDS at a wave-uniform base (lane i -> base + 16*i), i.e. one instruction fills 4 tile rows;
    // wave w owns rows 32*w .. 32*w+31 (8 instructions per matrix; 16 rows, 4 instructions when paired).  The 16-byte chunks of a row
    // are permuted for conflict-free reads (K: chunk ^ row%16, V: chunk ^ 4*(row%4)); the
    // permutation is applied on the global side: lane (row, c') loads global chunk c' ^ swz(row).
    // Rows that do not exist (past seqlen, or padding of a gathered tile) are read from a clamped,
    // valid address: their scores are masked to -inf, so their probabilities are exactly 0.
    const int cp_r = lane / NCH;                 // row inside the group of RPI rows one instruction fills
    const int cp_c = lane % NCH;                 // LDS chunk
    // gathered tiles: lane l holds the token id of tile row l (one load per lane, issued an
    // iteration ahead); the copy fetches the ids of its own rows with wave shuffles
    // (per-lane offsets of the buffer-form copies: the K permutation repeats every 16 rows, i.e. every
    // KL copy instructions, the V permutation every 4 rows: every VL instructions)
    constexpr int KL = RPI >= 4 ? 4 : 16 / RPI, VL = RPI >= 4 ? 1 : 4 / RPI;
    int k_lane[KL], v_lane[VL];
#pragma unroll
    for (int jj = 0; jj < KL; ++jj) k_lane[jj] = cp_r * (int)k_row + ((cp_c ^ swz_k(RPI * jj + cp_r)) << 4);
#pragma unroll
    for (int jj = 0; jj < VL; ++jj) v_lane[jj] = cp_r * (int)v_row + ((cp_c ^ swz_v(RPI * jj + cp_r)) << 4);
    auto gather_ids = [&](const Tile &t) -> int {
        if (MODE == MODE_VS && t.gathered) return p.ci[ridx * p.nnz_v + t.start + min(lane, max(t.nvalid, 1) - 1)];
        return 0;
    };
    // rows_c: tile rows copied by one wave (16: the four waves of a pair share the tile, 32: the
    // two waves of a row block copy it); wsel: which part of the tile this wave copies
    auto copy_rows = [&](const Tile &t, const char *base, long long rowstride, auto is_v_c, int idv,
                         char *ldsbuf, auto rows_c, const int wsel, auto whole_c) {
        constexpr bool is_v = decltype(is_v_c)::value;
        constexpr int CROWS = decltype(rows_c)::value;
        const bool gathered = MODE == MODE_VS && t.gathered;
        if (decltype(whole_c)::value || (!gathered && t.start >= 0 && t.start + BN <= seqlen)) {
            // buffer form: descriptor of the 64 tile rows (scalar), one of five per-lane offsets (the V
            // swizzle does not depend on j, the K swizzle only on j % 4) and a scalar row offset
            const char *tb = base + (long long)t.start * rowstride;      // wave-uniform
            const __amdgpu_buffer_rsrc_t srd = __builtin_amdgcn_make_buffer_rsrc((void *)tb, 0, BN * (int)rowstride, 0x00020000);
            // first row offset and step of this wave's part; in the paired vertical-slash kernel (two
            // copy shapes, K and V strides) they are made opaque so that the per-copy offsets are formed
            // with one scalar add each instead of living in two dozen loop-invariant scalar registers
            int soff0 = CROWS * wsel * (int)rowstride, sstep = RPI * (int)rowstride;
            int lds0 = (int)(unsigned)(unsigned long long)(__attribute__((address_space(3))) char *)ldsbuf + CROWS * wsel * ROW_BYTES;
            if constexpr (VSP) asm volatile("" : "+s"(soff0), "+s"(sstep), "+s"(lds0));
#pragma unroll
            for (int j = 0; j < CROWS / RPI; ++j) {
                const int voff = is_v ? v_lane[j & (VL - 1)] : k_lane[j & (KL - 1)];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(srd, (__attribute__((address_space(3))) void *)(unsigned long long)(unsigned)(lds0 + RPI * j * ROW_BYTES),
                                                         16, voff, soff0 + j * sstep, 0, 0);
            }
            return;
        }
        // three straight-line variants (a per-row select would turn into sixteen tiny branches).
        // The two rare ones recompute their per-lane rows and chunks on the spot (the empty asm
        // keeps the compiler from hoisting a dozen loop-invariant registers out of the tile loop).
        int cp_r = lane / NCH, cp_c = lane % NCH;
        asm volatile("" : "+v"(cp_r), "+v"(cp_c));
        if (gathered) {
#pragma unroll
            for (int j = 0; j < CROWS / RPI; ++j) {
                const int r = CROWS * wsel + RPI * j + cp_r;        // tile row
                const int tk = max(0, min(__shfl(idv, r), seqlen - 1));
                const int c = is_v ? (cp_c ^ swz_v(r)) : (cp_c ^ swz_k(r));
                const char *gp = base + tk * rowstride + c * 16;
                copy16_to_lds(gp, ldsbuf + (CROWS * wsel + RPI * j) * ROW_BYTES);
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < CROWS / RPI; ++j) {
            const int r = CROWS * wsel + RPI * j + cp_r;
            const int tk = max(0, min(t.start + r, seqlen - 1));
            const int c = is_v ? (cp_c ^ swz_v(r)) : (cp_c ^ swz_k(r));
            const char *gp = base + tk * rowstride + c * 16;
            copy16_to_lds(gp, ldsbuf + (CROWS * wsel + RPI * j) * ROW_BYTES);
        }
    };
    auto copy_tile = [&](const Tile &t, const char *base, long long rowstride, auto is_v_c, int idv, char *ldsbuf) {
        if constexpr (VSP) {
            if (t.split) {
                if (t.on_a) copy_rows(t, base, rowstride, is_v_c, idv, ldsbuf + half * TILE_BYTES, std::integral_constant<int, 32>{}, wave, std::false_type{});
                return;
            }
        }
        copy_rows(t, base, rowstride, is_v_c, idv, ldsbuf, std::integral_constant<int, CROWS>{}, wave_wg, std::false_type{});
    };

    // ---- accumulators -------------------------------------------------------
    f32x16_t oacc[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    float m_i = -INFINITY;   // running max (log2 domain, scaled)
    int sm_steps = 0;        // tiles this wave has put through the softmax
    int sm_prev_start = -(1 << 30);   // first key of the previous one (wave-uniform)
    bool sm_prev_masked = false;      // ... and whether it was a boundary tile (some rows may have seen none of its keys)
    float l_i = 0.f;         // this lane's share of the running sum

    // LDS read addresses that do not depend on the tile
    // K: row 32*blk + l32, logical chunk 2*ks + g -> physical chunk ^ (row % 16)
    int k_rd_off[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_rd_off[ks] = l32 * ROW_BYTES + (((2 * ks + g) ^ swz_k(l32)) << 4);
    // V transpose read: row = 16*s + 8*jj + 4*g + rsub (row % 4 == rsub), logical chunk
    // 4*db + vc -> physical 4*(db ^ rsub) + vc
    const int v_rd_rsub = (lane & 15) >> 2;
    const int v_rd_vc = (((lane >> 4) & 1) << 1) + ((lane & 3) >> 1);
    int v_rd_off[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
        v_rd_off[db] = (4 * g + v_rd_rsub) * ROW_BYTES + ((((db << 2) + v_rd_vc) ^ swz_v(v_rd_rsub)) << 4) + ((lane & 1) << 3);

    // ---- S^T = K . Q^T for this wave's 32 query rows; K tile in kbuf.
    auto qk_block = [&](const char *kbuf, f32x16_t &s0, f32x16_t &s1) {
        Frag a0[KS], a1[KS];
        __builtin_amdgcn_s_setprio(2);
#pragma unroll
        for (int r = 0; r < 16; ++r) { s0[r] = 0.f; s1[r] = 0.f; }
        // K fragments are fetched QK_AHEAD k-steps before the MFMAs that consume them; the
        // scheduling fences keep the compiler from sinking the reads back to their use
#pragma unroll
        for (int ks = 0; ks < QK_AHEAD; ++ks) {
            a0[ks].u = *reinterpret_cast<const u32x4_t *>(kbuf + k_rd_off[ks]);
            a1[ks].u = *reinterpret_cast<const u32x4_t *>(kbuf + k_rd_off[ks] + 32 * ROW_BYTES);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if (ks + QK_AHEAD < KS) {
                a0[ks + QK_AHEAD].u = *reinterpret_cast<const u32x4_t *>(kbuf + k_rd_off[ks + QK_AHEAD]);
                a1[ks + QK_AHEAD].u = *reinterpret_cast<const u32x4_t *>(kbuf + k_rd_off[ks + QK_AHEAD] + 32 * ROW_BYTES);
            }
            s0 = Mma<T>::mfma(frag_as<T>(a0[ks]), frag_as<T>(qf[ks]), s0);
            s1 = Mma<T>::mfma(frag_as<T>(a1[ks]), frag_as<T>(qf[ks]), s1);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
    };

    // ---- mask, V^T fragment reads, online softmax, O^T += V^T . P^T
    // (PLAIN: a tile none of whose keys is masked, right after another such tile)
    auto sm_pv_block = [&](const Tile &cur, const char *vbuf, f32x16_t &s0, f32x16_t &s1, auto plain_c) {
        constexpr bool PLAIN = decltype(plain_c)::value;
        // (head_dim 256: the 64 registers of a whole tile's V^T fragments do not fit next to O^T and Q;
        // that form reads a fragment two MFMAs ahead of its own)
        constexpr bool VF_AHEAD = HD <= 128;
        constexpr bool SUM_LAST = HD == 128 || (HD == 64 && PLAIN);      // (see the row sums below)
        constexpr int VALU_PER_MFMA = SUM_LAST ? 5 : 6;
        Frag vf[VF_AHEAD ? 4 : 1][NDB];
        // element (blk, r) of this lane is tile-local key tk = tkc + 4*g with the compile-time
        // part tkc = 32*blk + 8*(r/4) + r%4.  keep <=> tk <= hi && (tk > wlo || tk < slim).
        bool need_mask = false;
        const int wrow_lo = row0 + wave * 32, wrow_hi = wrow_lo + 31;
        int hi = 0, wlo = -1, slim = 0;  // per-lane bounds on tkc (4*g already subtracted)
        if (PLAIN) {
        } else if (MODE == MODE_VS && cur.gathered) {
            need_mask = cur.nvalid < BN;
            hi = cur.nvalid - 1 - 4 * g;
        } else {
            hi = min(qrow, seqlen - 1) - cur.start - 4 * g;
            if constexpr (MODE == MODE_ASHAPE) {
                const int c_lo = cur.start, c_hi = cur.start + BN - 1;
                const bool causal_ok = c_hi <= wrow_lo && c_hi < seqlen;
                const bool in_window = (wrow_hi - c_lo) < p.n_local;
                const bool in_sink = c_hi < p.n_init;
                const bool all_dense = wrow_lo >= p.dense_from, none_dense = wrow_hi < p.dense_from;
                need_mask = all_dense ? !causal_ok : (none_dense ? !(causal_ok && (in_window || in_sink)) : true);
                wlo = qrow >= p.dense_from ? -(1 << 30) : qrow - cur.start - p.n_local - 4 * g;
                slim = p.n_init - cur.start - 4 * g;
            } else {
                // (a list entry below zero is no key at all: the reference would read out of bounds)
                need_mask = (cur.start + BN - 1 > wrow_lo) || (cur.start + BN > seqlen) || cur.start < 0;
                wlo = -cur.start - 4 * g - 1;
            }
        }
        if (MODE == MODE_DENSE && need_mask) {               // one bound: a compare and a select
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int tkc = 8 * (r >> 2) + (r & 3);
                s0[r] = tkc <= hi ? s0[r] : -INFINITY;
                s1[r] = tkc + 32 <= hi ? s1[r] : -INFINITY;
            }
        } else if (need_mask) {
            // up to three bounds per key: as a 64-bit mask of the tile's keys, two instructions a score (its bit
            // spread over a word, a select) where three compares, two mask operations and a select took six.  An
            // A-shape walk has up to five boundary tiles, half of it where the window is short: 16 heads, 49152
            // tokens, window 128: head_dim 64 122.5 -> 116.6 us, 128 218.6 -> 208.4; lists 0.3 % at 16001 tokens, 800 slashes
            auto below = [](int n) -> unsigned { return n >= 32 ? ~0u : (1u << max(n, 0)) - 1u; };      // bits t < n
            unsigned keep0 = ~below(wlo + 1), keep1 = ~below(wlo - 31);
            if constexpr (MODE == MODE_ASHAPE) { keep0 |= below(slim); keep1 |= below(slim - 32); }
            keep0 &= below(hi + 1);
            keep1 &= below(hi - 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int tkc = 8 * (r >> 2) + (r & 3);
                const unsigned m0 = (unsigned)((int)(keep0 << (31 - tkc)) >> 31), m1 = (unsigned)((int)(keep1 << (31 - tkc)) >> 31);
                s0[r] = __uint_as_float((__float_as_uint(s0[r]) & m0) | (0xff800000u & ~m0));
                s1[r] = __uint_as_float((__float_as_uint(s1[r]) & m1) | (0xff800000u & ~m1));
            }
        }

        {
        // All V^T fragments of the tile are read here, in one scheduling region with the row-max
        // chain: the PV block below is bound by its vector instructions, so every LDS read moved out
        // of it shortens it (+3 % for the 24 reads that used to sit between its MFMAs), and the reads
        // fill the dependency gaps of the max chain (+0.7 % over reading them before the K copy).
        if constexpr (VF_AHEAD) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
                vf[s][db].s4[jj] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) short4_t *)(vbuf + v_rd_off[db] + (16 * s + 8 * jj) * ROW_BYTES));
        }
        }
        // ---- online softmax (exp2 domain) -------------------------------------
        // The reference maximum m_i of a row only has to keep exp2 inside the range of fp32 (bf16 has the
        // same exponent range), so most tiles take it as it is: no row maximum, no rescale factor.  It
        // is recomputed where a row has none yet (first tile, fully masked tiles), every MAX_PERIOD steps,
        // and for every tile of a walk that is run again because a row sum left the safe range (which
        // takes a row whose scores rise by more than a hundred powers of two within MAX_PERIOD tiles).
        float alpha = 1.0f, m_use = m_i;
        // ... and wherever the walk jumps (the first tile of a run of blocks, the first window tile after
        // the sink tiles, every gathered tile): scores move smoothly along a run of neighbouring keys
        // but may differ by any amount across a jump.  A tile after a masked one counts as a jump too:
        // a row that saw none of the masked tile's keys (the window starts a tile later for the last
        // rows of a row block) still carries the maximum from before the jump.
        const bool jump = PLAIN ? VSP && cur.start != sm_prev_start + BN :
                          (MODE == MODE_VS && cur.gathered) || cur.start != sm_prev_start + BN || sm_prev_masked;
        sm_prev_start = cur.start;
        sm_prev_masked = need_mask;
        if (every_max || ((sm_steps++ & (MAX_PERIOD - 1)) == 0) || jump || __any(m_i == -INFINITY)) {
        float mx;
        {
            // four independent chains of three-operand maxima (8 scores each)
            float m4[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                m4[c] = fmaxf(fmaxf(s0[4 * c], s1[4 * c]), s0[4 * c + 1]);
                m4[c] = fmaxf(fmaxf(m4[c], s1[4 * c + 1]), s0[4 * c + 2]);
                m4[c] = fmaxf(fmaxf(m4[c], s1[4 * c + 2]), s0[4 * c + 3]);
                m4[c] = fmaxf(m4[c], s1[4 * c + 3]);
            }
            mx = fmaxf(fmaxf(fmaxf(m4[0], m4[1]), m4[2]), m4[3]);
        }
        { const unsigned u = __float_as_uint(mx); auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false); mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])); }
        const float cand = mx * sc_l2;
        // lazy: raised only when a tile exceeds it by more than LAZY_MAX powers of two (probabilities of
        // f16 operands must stay inside the f16 range: 2^8 leaves room for the row sums)
        constexpr float LAZY_MAX = std::is_same<T, __bf16>::value ? LAZY_MAX_BF16 : 8.0f;
        const bool grow = cand > m_i + LAZY_MAX;
        const float m_new = grow ? cand : m_i;
        m_use = (m_new == -INFINITY) ? 0.f : m_new;
        // `alpha` is the SQUARE ROOT of the rescale factor and is applied twice.  With a maximum that
        // is looked at only now and then, the sums accumulated under the old one may be as large as
        // 2^127 (probabilities far above 1 that have not overflowed), so a factor below 2^-126 does
        // not mean that they are negligible -- and exp2 of such an exponent is flushed to zero.  Half
        // the exponent twice is exact down to 2^-252, beyond which nothing finite is left of them.
        alpha = grow ? __builtin_amdgcn_exp2f(fmaxf(0.5f * (m_i - m_use), -126.0f)) : 1.0f;
        m_i = m_new;
        }
        float psum = 0.f;
        Frag pfr[4];
        // probabilities of key group q (16 keys): registers 8*(q%2) .. +7 of s0 (q < 2) / s1
        auto probs = [&](int q) {
            const f32x16_t &sx = q < 2 ? s0 : s1;
            float pv[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) pv[r] = __builtin_amdgcn_exp2f(fmaf(sx[8 * (q & 1) + r], sc_l2, -m_use));
            cvt8<T>(&pv[0], pfr[q]);
            if constexpr (!SUM_LAST) psum = pair_sum<T>(pfr[q], psum);
        };
        probs(0);
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int i = 0; i < NDB; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[i][r] = (oacc[i][r] * alpha) * alpha;
        }

        __builtin_amdgcn_s_setprio(2);
        // ---- O^T += V^T . P^T; the exponentials of key group q+1 run under the MFMAs of group q ----
        {
            probs(1);
            probs(2);
            probs(3);
            if constexpr (!SUM_LAST) l_i = (l_i * alpha) * alpha + psum;
            if constexpr (VF_AHEAD) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int db = 0; db < NDB; ++db)
                    oacc[db] = Mma<T>::mfma(frag_as<T>(vf[s][db]), frag_as<T>(pfr[s]), oacc[db]);
            // the softmax instructions of key groups 1..3 are spread behind the MFMAs of groups 0..2
#pragma unroll
            for (int i = 0; i < 4 * NDB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (i < 3 * NDB) __builtin_amdgcn_sched_group_barrier(VALU_MASK, VALU_PER_MFMA * 4 / NDB, 0);
            }
            } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int jj = 0; jj < 2; ++jj)
                        vf[0][db].s4[jj] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (__attribute__((address_space(3))) short4_t *)(vbuf + v_rd_off[db] + (16 * s + 8 * jj) * ROW_BYTES));
#pragma unroll
                for (int db = 0; db < NDB; ++db)
                    oacc[db] = Mma<T>::mfma(frag_as<T>(vf[0][db]), frag_as<T>(pfr[s]), oacc[db]);
            }
            // one MFMA, the reads of the fragment two MFMAs ahead, softmax instructions of the next key groups.  Left to
            // the compiler the order turned with every change elsewhere in the kernel (1 wave per SIMD: nothing hides a
            // wait): dense, 16 heads of 20000 tokens, bf16 3640 us, 3715 after one to the epilogue, 3518 in this order;
            // fp16 3834, 3808, 3739; A-shape, window 1000, bf16 588, 561, 538
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int i = 0; i < 4 * NDB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (i < 4 * NDB - 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                if (i < 3 * NDB) __builtin_amdgcn_sched_group_barrier(VALU_MASK, VALU_PER_MFMA * 4 / NDB, 0);
            }
            }
        }
        // The row sums of the whole tile in one go behind the last product: a v_dot2 between two MFMAs takes about 11
        // cycles of the matrix pipe's (a product with the tile's share of fma, exp and cvt behind it 35 cycles, with half
        // a v_dot2 as well 41; four in a row 12 in all).  A batch behind each key group's products took, dense, 16384
        // tokens, 32 / 8 heads 1882 us against 1832 (on zeros 1365 : 1315); plain adds of the unpacked halves 2000.
        // (Not at head_dim 256, 7 % slower, whose one wave has nothing else to run meanwhile, and not in the general form
        // at 64: A-shape, window 512, 1 to 2 % slower.  Those add the tile's sum to the row's before the products: behind
        // them it kept two more values alive through the chain, and tri-shape calls of one 64-wide head that are a chain
        // of such steps took 22.4 us for 21.3, 1000 tokens, and 54.2 for 51.1, 2816.)
        if constexpr (SUM_LAST) {
#pragma unroll
            for (int q = 0; q < 4; ++q) psum = pair_sum<T>(pfr[q], psum);
            l_i = (l_i * alpha) * alpha + psum;
        }
        __builtin_amdgcn_s_setprio(0);
    };

    // Single K and V buffers, two barriers per tile:
    //   [own K(it) copies landed] barrier B1 (also: every wave is done with V(it-1))
    //   issue V(it) copy; fetch gathered ids of tile it+1; S^T = K.Q^T
    //   [own V(it) copies landed] barrier B2 (also: every wave is done with K(it))
    //   issue K(it+1) copy; softmax; O^T += V^T.P^T
    Tile cur, nxt;
    int gt_cur = 0, gt_nxt = 0;
    [[maybe_unused]] bool vs_shifted = false;
    bool have_cur = more_tiles(it_begin);
    if (have_cur) {
        if constexpr (VSP) vs_entry = __builtin_amdgcn_readfirstlane(vs_list(it_begin));
        cur = tile_of(it_begin);
        if constexpr (VSP) vs_entry = __builtin_amdgcn_readfirstlane(vs_list(it_begin + 1));
        gt_cur = gather_ids(cur);
        copy_tile(cur, k_base, k_row, std::false_type{}, gt_cur, lds_k);
    }

    // One step of the walk, in four forms (COMMON and SPLIT for the paired list walks only):
    // general (kind 0) -- any tile, any successor, every mode;
    // PLAIN (kind 3) -- a tile of which both row blocks see every key, after another such tile or as a list's first, and the
    // next one alike or at least unmasked up to the pair's first row: in list walks both are common entries (the next one may
    // lie anywhere behind this one), else the next one is this one's neighbour.  Both lie below the pair's first row, hence before
    // the end of the sequence: they are copied without a look at it, and no mask and, but for a list's, no jump is asked for;
    // COMMON (kind 1) -- this tile and the next one are both on the list of common entries: shared,
    // contiguous, never gathered;
    // SPLIT (kind 2) -- this step and the next one are both split steps in which each row block
    // visits a block entry of its own, fetched a step ahead: a leftover from the split lists in LDS
    // or, when the lists were not split, an entry of its list in global memory.
    // In the special forms everything that deals with the other cases drops out of the
    // instruction stream (the general form costs about 1.7 times a COMMON step).
    [[maybe_unused]] int sp_entry = 0;
    auto step = [&](const int it, auto kind_c) {
        constexpr int KIND = decltype(kind_c)::value;
        constexpr bool COMMON = KIND == 1 || (VSP && KIND == 3), SPLIT = KIND == 2, PLAIN = KIND == 3;
        __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): this wave's part of K(it) is in LDS
        __syncthreads();
        bool have_nxt;
        if constexpr (COMMON) {
            vs_pref = vs_list(it + 2);
            have_nxt = true;
            nxt.gathered = 0; nxt.nvalid = BN; nxt.on_a = nxt.on_b = 1; nxt.split = 0;
            nxt.start = vs_entry;
            gt_nxt = 0;
            cur.gathered = 0; cur.nvalid = BN; cur.on_a = cur.on_b = 1; cur.split = 0;
            copy_rows(cur, v_base, v_row, std::true_type{}, 0, lds_v, std::integral_constant<int, CROWS>{}, wave_wg, std::integral_constant<bool, PLAIN>{});
        } else if constexpr (SPLIT) {
            const int j = it - vs_nc;                      // this step's position in the leftover lists
            if (vs_merged) vs_pref = vs_only[half * VS_ONLY_MAX + min(j + 2, VS_ONLY_MAX - 1)];
            else vs_pref = sp_list[min(j + 2, list_w - 1)] * LIST_SCALE;
            have_nxt = true;
            nxt.gathered = 0; nxt.nvalid = BN; nxt.on_a = nxt.on_b = 1; nxt.split = 1;
            nxt.start = sp_entry;
            gt_nxt = 0;
            cur.gathered = 0; cur.nvalid = BN; cur.on_a = cur.on_b = 1; cur.split = 1;
            copy_rows(cur, v_base, v_row, std::true_type{}, 0, lds_v + half * TILE_BYTES, std::integral_constant<int, 32>{}, wave, std::false_type{});
        } else if constexpr (PLAIN) {
            have_nxt = true;
            cur.gathered = 0; cur.nvalid = BN; cur.on_a = cur.on_b = 1; cur.split = 0;
            nxt = cur;
            nxt.start = cur.start + BN;
            gt_nxt = 0;
            copy_rows(cur, v_base, v_row, std::true_type{}, 0, lds_v, std::integral_constant<int, CROWS>{}, wave_wg, std::true_type{});
        } else if constexpr (VSP) {
            // the merged list shares an LDS object with the V tiles: its entry is read while no copy
            // is in flight, so that the read never waits for one
            vs_pref = vs_list(it + 2);
            have_nxt = more_tiles(it + 1);
            nxt = have_nxt ? tile_of(it + 1) : cur;
            gt_nxt = gather_ids(nxt);
            copy_tile(cur, v_base, v_row, std::true_type{}, gt_cur, lds_v);
            if (cur.split && !vs_shifted) {
                // first split step: row block B reads the second tiles from here on (the LDS read
                // offsets move in place, once)
                vs_shifted = true;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) k_rd_off[ks] += half * TILE_BYTES;
#pragma unroll
                for (int db = 0; db < NDB; ++db) v_rd_off[db] += half * TILE_BYTES;
            }
        } else {
            copy_tile(cur, v_base, v_row, std::true_type{}, gt_cur, lds_v);
            have_nxt = more_tiles(it + 1);
            nxt = have_nxt ? tile_of(it + 1) : cur;
            gt_nxt = gather_ids(nxt);
        }

        // is this tile on the list of this wave's row block ?
        bool active = true;
        if constexpr (COMMON || SPLIT || PLAIN) active = have_rows;
        else if constexpr (VSP) active = have_rows && (half ? cur.on_b : cur.on_a);   // (split steps: on_a == on_b == own flag)
        else active = have_rows && tile_on_list<MODE>(p, m, cur.start);
        f32x16_t s0, s1;
        if (active) qk_block(lds_k, s0, s1);
        __builtin_amdgcn_s_waitcnt(0x0f70);          // vmcnt(0): this wave's part of V(it) is in LDS
        __syncthreads();
        if constexpr (COMMON) copy_rows(nxt, k_base, k_row, std::false_type{}, 0, lds_k, std::integral_constant<int, CROWS>{}, wave_wg, std::integral_constant<bool, PLAIN>{});
        else if constexpr (SPLIT) copy_rows(nxt, k_base, k_row, std::false_type{}, 0, lds_k + half * TILE_BYTES, std::integral_constant<int, 32>{}, wave, std::false_type{});
        else if constexpr (PLAIN) copy_rows(nxt, k_base, k_row, std::false_type{}, 0, lds_k, std::integral_constant<int, CROWS>{}, wave_wg, std::true_type{});
        else if (have_nxt) copy_tile(nxt, k_base, k_row, std::false_type{}, gt_nxt, lds_k);
        if (active) sm_pv_block(cur, lds_v, s0, s1, std::integral_constant<bool, PLAIN>{});
        if constexpr (SPLIT) sp_entry = __builtin_amdgcn_readfirstlane(vs_pref);
        else if constexpr (VSP) vs_entry = __builtin_amdgcn_readfirstlane(vs_pref);
        cur = nxt;
        gt_cur = gt_nxt;
        have_cur = have_nxt;
    };
    int it = it_begin;
    if constexpr (VSP) {
        // (a first step exists whenever there is a common entry; steps 0 .. vs_nc-2 have a common successor)
        const int common_end = min(vs_nc, it_end);
        // the common entries ascend: all but the last few are tiles of which both row blocks see every key
        if (vs_nc > 1) {
            const int back = vs_nc - 1 - lane;
            const unsigned long long late = __ballot(back >= 0 && vs_list(max(back, 0)) > mA * BM - BN);
            const int nlate = __builtin_popcountll(late);
            const int plain_end = nlate < 64 && __builtin_amdgcn_readfirstlane(vs_list(0)) >= 0 ? min(vs_nc - nlate, it_end) : 0;
            for (; it + 1 < plain_end; ++it) step(it, std::integral_constant<int, 3>{});
        }
        for (; it + 1 < common_end; ++it) step(it, std::integral_constant<int, 1>{});
        // block entries of their own that both row blocks still have (leftovers of the split, or the
        // whole lists when they were not split): these steps run in the SPLIT form
        const int split_end = min(min(vs_na, vs_nb), it_end);
        if (split_end - max(it_begin, vs_nc) >= 3 && have_cur) {
            if (it < vs_nc) {                              // from the last common tile to the first split step
                step(it, std::integral_constant<int, 0>{});
                ++it;
            }
            // cur is now an entry of each row block's own list, its K copy is on the way
            if (!vs_shifted) {
                vs_shifted = true;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) k_rd_off[ks] += half * TILE_BYTES;
#pragma unroll
                for (int db = 0; db < NDB; ++db) v_rd_off[db] += half * TILE_BYTES;
            }
            const int j1 = it - vs_nc + 1;
            sp_entry = vs_merged ? __builtin_amdgcn_readfirstlane(vs_only[half * VS_ONLY_MAX + j1]) : sp_list[j1] * LIST_SCALE;
            for (; it + 1 < split_end; ++it) step(it, std::integral_constant<int, 2>{});
        }
    }
    // From one such tile on, at head_dim 64 too: where that form began at eight tiles and was left out of segments, us before
    // and now, tri-shape with a window of 3968, one head 6000 tokens 75.3 : 64.4, 12000 80.5 : 70.8, 16 heads 24000 461 :
    // 448; with a window of 512 (five tiles), 16 heads 24000 tokens 116.0 : 115.5; A-shape of that window, 32 / 8 heads,
    // 48538 tokens 363 : 354.
    if constexpr (!VSP && HD <= 128) {
        // tiles of which both row blocks see every key, after another such tile and before one that both visit or mask
        const bool causal = MODE == MODE_DENSE || mA * BM >= p.dense_from;
        const bool windowed = MODE == MODE_ASHAPE && mB * BM + BM - 1 < p.dense_from;
        if (causal || windowed) {
            int first = 1, shift = 0;                      // tile number of the first such tile; tile number - step
            if (windowed) {
                shift = pair_tile_start<MODE>(p, mA, mB, nblk, nblk) / BN - nblk;
                first = max((mB * BM + BM - p.n_local + BN - 1) >> 6, shift + nblk) + 1;
            }
            const int lo = max(first - shift, it_begin + 1), hi = min(mA - 1 - shift, it_end - 1);
            if (lo < hi) {
                for (; it < lo; ++it) step(it, std::integral_constant<int, 0>{});
                for (; it < hi; ++it) step(it, std::integral_constant<int, 3>{});
            }
        }
    }
    for (; have_cur; ++it) step(it, std::integral_constant<int, 0>{});

    // ---- epilogue: O = O^T / l, transposed through LDS so that every global store is 16 bytes
    // of one row and 16 lanes cover a whole 256-byte row ---------------------------------------
    {
        float l_tot = l_i + __shfl_xor(l_i, 32);
        const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
        constexpr int OP = ROW_BYTES;
        auto check_range = [&]() {
            // a row sum at 2^100 or beyond (or infinite, or no number at all): some probability may have
            // overflowed.  Compared on the bit pattern: the library is compiled without NaN semantics, which
            // lets the compiler turn !(l < x) into l >= x -- false for the NaN that inf * 0 leaves in a
            // row sum when the maximum is raised after an overflow
            // ... and an accumulator that is infinite or no number: O^T sums twice as many terms per tile
            // as a lane's share of the row sum (and terms scaled by |v|), so it can overflow while the row
            // sum still fits, and a later rescale then hides the size of the sum but not the inf / NaN
            if constexpr (!every_max) {
                unsigned obits = 0;
#pragma unroll
                for (int i = 0; i < NDB; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) obits = max(obits, __float_as_uint(oacc[i][r]) & 0x7fffffffu);
                const bool suspect = (__float_as_uint(l_tot) & 0x7fffffffu) >= __float_as_uint(0x1p100f) || obits >= 0x7f800000u;
                if (__any(suspect) && lane == 0) lds_redo = 1;
            }
        };
        if (CUT && slot) {                               // a segment: the sums as they are (16 bytes per lane, contiguous)
            char *acc = slot + (wave_wg * NDB * 4 * 64 + lane) * 16;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int rq = 0; rq < 4; ++rq)
                    *reinterpret_cast<float4 *>(acc + (db * 4 + rq) * 1024) =
                        make_float4(oacc[db][rq * 4], oacc[db][rq * 4 + 1], oacc[db][rq * 4 + 2], oacc[db][rq * 4 + 3]);
            *(reinterpret_cast<float2 *>(slot + SplitSlot<HD>::ACC) + tid) = make_float2(m_i, l_tot);
            check_range();
            __syncthreads();
            return !every_max && lds_redo != 0;           // (workgroup-uniform)
        }
        // 32 rows per wave, in the K tiles: everyone was done with those at the last step's second barrier, so a
        // wave need not wait for the others' last softmax (tri-shape, 16 heads of 64, 24000 tokens 137.4 -> 135.8 us,
        // dense, 2 x 6144 tokens, 32 / 8 heads 591 -> 587)
        char *ot = lds_k + wave_wg * 32 * OP;
        // the 16-byte chunks of a row are permuted like those of a K tile: at a row's own pitch all 32 rows' writes of
        // one instruction went to one pair of banks, and a workgroup's epilogue took 5.1 us of its 34 (A-shape, window
        // 512, head_dim 128) where it takes 3.4 now: 16 heads of 64, 24000 tokens, window 512 138.5 -> 134.9 us; dense,
        // 2 x 6144 tokens, 32 / 8 heads 594 -> 588; A-shape, 100000 tokens, window 3968 6486 -> 6430 (hardly beyond noise)
        const bool live = qrow < seqlen;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
                union { T e[4]; u32x2_t u; } out4;
#pragma unroll
                for (int e = 0; e < 4; ++e) out4.e[e] = (T)(oacc[db][rq * 4 + e] * inv);
                if (!live) out4.u = u32x2_t{0u, 0u};
                *reinterpret_cast<u32x2_t *>(ot + l32 * OP + (((4 * db + rq) ^ swz_k(l32)) << 4) + 8 * g) = out4.u;
            }
        __builtin_amdgcn_wave_barrier();
        // lane -> (row = RPI*i + lane/NCH, chunk = lane%NCH)
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i) {
            const int r = RPI * i + lane / NCH;
            const int grow = row0 + wave * 32 + r;
            const u32x4_t val = *reinterpret_cast<const u32x4_t *>(ot + r * OP + (((lane % NCH) ^ swz_k(r)) << 4));
            if (grow < p.n && have_rows) *reinterpret_cast<u32x4_t *>(o_base + (long long)grow * p.os[2] * 2 + (lane % NCH) * 16) = val;
        }
        check_range();                                    // (while the stores are on their way)
    }
    if constexpr (every_max) return false;
    __syncthreads();                                      // (the flag is known)
    return !every_max && lds_redo != 0;                   // (workgroup-uniform)
}

// (head_dim 256: O^T, Q and the V^T fragments of a wave need more than 256 registers, so that form
// runs one wave per SIMD with the accumulators in the second half of the register file)
template <typename T> constexpr int dtype_code() { return std::is_same<T, __bf16>::value ? MINF_BF16 : MINF_F16; }
// workgroup `wg` of a launch
template <typename T, int MODE, int HD, bool CUT>
__device__ __forceinline__ void attn_workgroup(const AttnParams &p, const unsigned wg, char (&lds_k)[AttnLds<MODE, HD>::NK],
                                               char (&lds_v)[AttnLds<MODE, HD>::NV], int (&vs_only)[AttnLds<MODE, HD>::NONLY]) {
    __shared__ int vs_wsum[4];
    __shared__ int vs_bad[2];                // paired list walks: a list is not ascending, number of common entries
    __shared__ int lds_redo;
    if (threadIdx.x == 0) lds_redo = 0;      // (ordered before its readers by the barriers of the walk)
    if constexpr (std::is_same<T, __bf16>::value) {
        if (attn_walk<T, MODE, HD, false, CUT>(p, wg, lds_k, lds_v, vs_only, vs_wsum, vs_bad, lds_redo)) {
            __syncthreads();                 // everyone has read the flag and is done with LDS
            attn_walk<T, MODE, HD, true, CUT>(p, wg, lds_k, lds_v, vs_only, vs_wsum, vs_bad, lds_redo);
        }
    } else {
        // f16 probabilities have no headroom above the lazy threshold: the maximum of every tile
        attn_walk<T, MODE, HD, true, CUT>(p, wg, lds_k, lds_v, vs_only, vs_wsum, vs_bad, lds_redo);
    }
}

// CHOSEN: the number under which attn_walk, for which XCDs keep their places and all groups are one set, finds the deal of
// workgroup `wg` -> false: it has none (padding of the last round).  The choice is every workgroup's own, from four heads'
// counts, and so the same in all of them.  A form of the kernel of its own: as a branch of the walk's decoding, or before it, it
// cost launches that choose nothing 1 to 3 % (one head 10555 tokens 217.5 us, 220.3 and 224.7; 4 heads 11055 tokens 183.1, 187.3
// and 186.3), the compiler then making one loop of the three general steps it makes otherwise, with more spilled scalars.
__device__ __forceinline__ bool chosen_place(const AttnParams &p, unsigned &wg) {
    unsigned turn = 0;
    if (p.far_turn) {
        const cint_ptr last = as_const(p.bc) + p.rows - 1;       // (four loads on their way together)
        const int quarter = p.hq >> 2, most = p.rows >> 3;
        const int c0 = last[0], c1 = last[(long long)quarter * p.rows], c2 = last[2ll * quarter * p.rows], c3 = last[3ll * quarter * p.rows];
        if ((c0 > most) + (c1 > most) + (c2 > most) + (c3 > most) > 2) turn = (unsigned)p.far_turn;
    }
    const unsigned round = fast_quot(wg >> 3, p.by_deal), in_deal = (wg >> 3) - round * p.by_deal.d;
    const unsigned place = 8u * round + ((wg + (round >> turn)) & 7u);
    const unsigned row = fast_quot(place, p.by_set), set = fast_quot(row, p.by_chunks);
    const unsigned groups = (unsigned)p.batch * p.by_heads.d, g = set * p.by_set.d + place - row * p.by_set.d;
    if (g >= groups) return false;
    const unsigned deal = (row - set * p.by_chunks.d) * groups + g;
    wg = (((deal >> 3) * p.by_deal.d + in_deal) << 3) + (deal & 7u);
    return true;
}

template <typename T, int MODE, int HD, bool CUT, bool CHOSEN = false>
__global__ __launch_bounds__(2 * NTHREADS, HD > 128 ? 1 : 2) void attn_fwd_kernel(const AttnParams p) {
    typedef AttnLds<MODE, HD> L;
    if (p.select && *as_const(p.select) != dtype_code<T>()) return;
    __shared__ __attribute__((aligned(16))) char lds_k[L::NK];
    __shared__ __attribute__((aligned(16))) char lds_v[L::NV];
    __shared__ int vs_only[L::NONLY];        // paired list walks: [row block][entries the other list lacks]
    unsigned wg = blockIdx.x;
    if constexpr (CHOSEN)
        if (!chosen_place(p, wg)) return;
    attn_workgroup<T, MODE, HD, CUT>(p, wg, lds_k, lds_v, vs_only);
}

// The pattern types of a layer in one launch: workgroups [0, first_bs) walk vertical-slash lists, [first_bs, first_as)
// block-sparse lists, the rest A-shape windows (each part a multiple of 8 workgroups, see plan_launch).  As three launches
// each waited for the last walks of the one before on a chip that was emptying.
// Table of unlike patterns, 32 / 8 heads, whole layer, us: 9000 tokens 774 -> 692, 20000 fp16 1898 -> 1802, of 64 1059 ->
// 995, 50000 4531 -> 4482, 100000 9316 -> 9243; 28 / 4 heads 20000 tokens 1390 -> 1352; 8 / 2 heads 12000 tokens 331 -> 328.
// (bf16 at head_dim 128: 254 registers, the most of its three forms, no vector spills.)
struct MixedParams {
    AttnParams vs, bs, as;
    unsigned first_bs, first_as;
};
template <typename T, int HD>
__global__ __launch_bounds__(2 * NTHREADS, 2) void attn_mixed_kernel(const MixedParams p) {
    typedef AttnLds<MODE_VS, HD> L;
    typedef AttnLds<MODE_ASHAPE, HD> A;
    static_assert(A::NK == L::NK && A::NV <= L::NV && A::NONLY <= L::NONLY, "an A-shape walk fits the LDS of a list walk");
    __shared__ __attribute__((aligned(16))) char lds_k[L::NK];
    __shared__ __attribute__((aligned(16))) char lds_v[L::NV];
    __shared__ int vs_only[L::NONLY];
    if (blockIdx.x < p.first_bs) attn_workgroup<T, MODE_VS, HD, false>(p.vs, blockIdx.x, lds_k, lds_v, vs_only);
    else if (blockIdx.x < p.first_as) attn_workgroup<T, MODE_BS, HD, false>(p.bs, blockIdx.x - p.first_bs, lds_k, lds_v, vs_only);
    else attn_workgroup<T, MODE_ASHAPE, HD, false>(p.as, blockIdx.x - p.first_as, lds_k, reinterpret_cast<char (&)[A::NV]>(lds_v),
                                                   reinterpret_cast<int (&)[A::NONLY]>(vs_only));
}

// Folds the segments of a split pair: one workgroup per (batch, head position, pair, 32 query rows), a
// wave per 32-column block of O^T (same lane layout as the walk's accumulators), segments in ascending
// order.  The weights are exp2(m_s - M) with M the largest m_s + log2(l_s), so that no product leaves the
// fp32 range whatever a segment's (lazily raised) maximum was.  A segment is left out only where its row sum
// is the zero of an unused or fully masked one, by bit pattern: a NaN among the keys makes the row sum NaN,
// and the row is to be NaN, as a whole walk leaves it.  Latency-bound and small: it reads what the
// segments wrote (66 KB each at head_dim 128, from L2) and writes the rows once.  The statistics of all segments (up
// to 16) are loaded together and kept, then the sums of UP of them: two round trips to L2 up to UP segments, where
// statistics by eight, then statistics again and sums by four took eight for nine segments.  Vertical-slash, one head
// of 4096 tokens, 500 columns and 700 slashes, fp16, index given 27.2 -> 25.5 us; dense, one head 8000 tokens
// 35.6 -> 34.3.  Up to four segments, where the folds of many pairs fill the chip, they take the registers of four
// (with those of eight, 8 / 2 heads 8000 tokens, dense 149 -> 150).
constexpr int MERGE_FEW = 4, MERGE_HELD = 16;
template <int HD, bool FEW>
__global__ __launch_bounds__(256) void attn_merge_kernel(const AttnParams p) {
    constexpr int NDB = HD / 32, ROW_BYTES = HD * 2, NCH = ROW_BYTES / 16;
    __shared__ __attribute__((aligned(16))) char lds_o[32 * ROW_BYTES];
    const bool to_bf16 = (p.select ? *as_const(p.select) : p.dtype) == MINF_BF16;
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const int l32 = lane & 31, g = lane >> 5;
    const int heads = p.head_list ? p.index_heads : p.hq;
    const int rows_wg = (p.rows + 1) >> 1, npairs = rows_wg - p.split_first;
    unsigned rest = blockIdx.x;
    const int part = (int)(rest & 3u); rest >>= 2;                     // 32-row part of the pair
    const int pair = (int)(rest % (unsigned)npairs); rest /= (unsigned)npairs;
    const int hs = (int)(rest % (unsigned)heads), b = (int)(rest / (unsigned)heads);
    const int h = p.head_list ? p.head_list[hs] : hs;
    const int seqlen = p.seqlens ? min(p.seqlens[b], p.n) : p.n;
    const int row0 = (p.split_first + pair) * 2 * BM + part * 32;
    if (row0 >= p.n) return;
    char *o_base = p.o + ((long long)b * p.os[0] + (long long)h * p.os[1]) * 2;
    const char *slots = p.part + ((long long)(b * heads + hs) * npairs + pair) * p.nseg * SplitSlot<HD>::BYTES;
    // (a pair that starts past the sequence was not walked at all)
    const int nseg = (p.split_first + pair) * 2 * BM < seqlen ? p.nseg : 0;
    auto stat = [&](int s) { return *(reinterpret_cast<const float2 *>(slots + (long long)s * SplitSlot<HD>::BYTES + SplitSlot<HD>::ACC) + part * 64 + lane); };
    constexpr int HELD = FEW ? MERGE_FEW : MERGE_HELD;
    float2 held[HELD];
    float top = -INFINITY;
    auto look = [&](const float2 &ml) {
        const bool number = (__float_as_uint(ml.y) & 0x7fffffffu) <= 0x7f800000u;
        if (__float_as_uint(ml.y) != 0 && number) top = fmaxf(top, ml.x + __builtin_amdgcn_logf(ml.y));
    };
    if (nseg <= HELD) {
#pragma unroll
        for (int u = 0; u < HELD; ++u) held[u] = u < nseg ? stat(u) : make_float2(-INFINITY, 0.f);
#pragma unroll
        for (int u = 0; u < HELD; ++u) look(held[u]);
    } else {
        for (int s0 = 0; s0 < nseg; s0 += HELD) {
#pragma unroll
            for (int u = 0; u < HELD; ++u) held[u] = stat(min(s0 + u, nseg - 1));
#pragma unroll
            for (int u = 0; u < HELD; ++u) look(held[u]);
        }
    }
    const bool live = row0 + l32 < seqlen;
    float l_tot = 0.f;
    float4 acc[NDB > 4 ? 2 : 1][4];
#pragma unroll
    for (int i = 0; i < (NDB > 4 ? 2 : 1); ++i)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) acc[i][rq] = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr int UP = (FEW ? 4 : 8) / (NDB > 4 ? 2 : 1), NI = NDB > 4 ? 2 : 1;
    auto fold = [&](const float2 (&ml)[UP], int s0) {
        bool any[UP];
        bool some = false;
#pragma unroll
        for (int u = 0; u < UP; ++u) some |= any[u] = s0 + u < nseg && __any(__float_as_uint(ml[u].y) != 0);
        if (!some) return;
        // (an unused slot holds nothing and is not read)
        float4 x[UP][NI][4];
#pragma unroll
        for (int u = 0; u < UP; ++u)
            if (any[u])
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int db = wave + 4 * i;
                    if (db < NDB) {
                        const char *src = slots + (long long)(s0 + u) * SplitSlot<HD>::BYTES + ((part * NDB + db) * 4 * 64 + lane) * 16;
#pragma unroll
                        for (int rq = 0; rq < 4; ++rq) x[u][i][rq] = *reinterpret_cast<const float4 *>(src + rq * 1024);
                    }
                }
#pragma unroll
        for (int u = 0; u < UP; ++u) {
            if (!any[u]) continue;
            const float w = __float_as_uint(ml[u].y) != 0 ? __builtin_amdgcn_exp2f(ml[u].x - top) : 0.f;
            l_tot = fmaf(w, ml[u].y, l_tot);
#pragma unroll
            for (int i = 0; i < NI; ++i)
                if (wave + 4 * i < NDB)
#pragma unroll
                    for (int rq = 0; rq < 4; ++rq) {
                        float4 &o = acc[i][rq];
                        const float4 v = x[u][i][rq];
                        o.x = fmaf(w, v.x, o.x); o.y = fmaf(w, v.y, o.y); o.z = fmaf(w, v.z, o.z); o.w = fmaf(w, v.w, o.w);
                    }
        }
    };
    if (nseg <= HELD) {
#pragma unroll
        for (int s0 = 0; s0 < HELD; s0 += UP) {
            float2 ml[UP];
#pragma unroll
            for (int u = 0; u < UP; ++u) ml[u] = held[s0 + u];
            if (s0 < nseg) fold(ml, s0);
        }
    } else {
        for (int s0 = 0; s0 < nseg; s0 += UP) {
            float2 ml[UP];
#pragma unroll
            for (int u = 0; u < UP; ++u) ml[u] = stat(min(s0 + u, nseg - 1));
            fold(ml, s0);
        }
    }
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
#pragma unroll
    for (int i = 0; i < (NDB > 4 ? 2 : 1); ++i) {
        const int db = wave + 4 * i;
        if (db < NDB)
#pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
                union { __bf16 b[4]; _Float16 h[4]; u32x2_t u; } out4;
                const float x[4] = {acc[i][rq].x, acc[i][rq].y, acc[i][rq].z, acc[i][rq].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float y = live ? x[e] * inv : 0.f;
                    if (to_bf16) out4.b[e] = (__bf16)y; else out4.h[e] = (_Float16)y;
                }
                *reinterpret_cast<u32x2_t *>(lds_o + l32 * ROW_BYTES + (32 * db + 8 * rq + 4 * g) * 2) = out4.u;
            }
    }
    __syncthreads();
    for (int c = (int)threadIdx.x; c < 32 * NCH; c += 256) {
        const int r = c / NCH, ch = c % NCH;
        if (row0 + r < p.n)
            *reinterpret_cast<u32x4_t *>(o_base + (long long)(row0 + r) * p.os[2] * 2 + ch * 16) =
                *reinterpret_cast<const u32x4_t *>(lds_o + r * ROW_BYTES + ch * 16);
    }
}

int check_tensors(const minf_qkvo *t, bool allow_256 = false) {
    if (!t) return MINF_ERR_INVALID_ARG;
    if (t->batch < 0 || t->heads_q <= 0 || t->heads_kv <= 0 || t->n < 0) return MINF_ERR_INVALID_ARG;
    // empty problems (no batch or no tokens) have no storage: nothing to check, nothing is launched
    const bool empty = t->batch == 0 || t->n == 0;
    if (!empty && (!t->q || !t->k || !t->v || !t->o)) return MINF_ERR_INVALID_ARG;
    if (t->heads_q % t->heads_kv != 0) return MINF_ERR_INVALID_ARG;
    if (t->head_list && t->index_heads <= 0) return MINF_ERR_INVALID_ARG;
    if (t->head_dim != 128 && t->head_dim != 64 && !(allow_256 && t->head_dim == 256)) return MINF_ERR_UNSUPPORTED;
    if (t->dtype == MINF_16BIT_SELECT) { if (!empty && !t->dtype_select) return MINF_ERR_INVALID_ARG; }
    else if (t->dtype != MINF_BF16 && t->dtype != MINF_F16) return MINF_ERR_UNSUPPORTED;
    const void *ptrs[4] = {t->q, t->k, t->v, t->o};
    const int64_t *strides[4] = {t->q_stride, t->k_stride, t->v_stride, t->o_stride};
    for (int i = 0; i < 4; ++i) {
        if (((uintptr_t)ptrs[i]) & 15) return MINF_ERR_ALIGNMENT;
        for (int j = 0; j < 3; ++j)
            if (strides[i][j] < 0 || (strides[i][j] & 7)) return MINF_ERR_ALIGNMENT;
        // 64 rows x token stride is formed in 32 bits inside the tile copies
        if (strides[i][2] > (1 << 23)) return MINF_ERR_UNSUPPORTED;
        // rows must not overlap (expanded or interleaved views): the tile copies describe 64 rows of
        // a tile by one buffer descriptor of 64 x token stride bytes
        if (t->n > 1 && strides[i][2] < t->head_dim) return MINF_ERR_UNSUPPORTED;
    }
    return MINF_OK;
}

void fill_params(AttnParams &p, const minf_qkvo *t) {
    p.q = (const char *)t->q; p.k = (const char *)t->k; p.v = (const char *)t->v; p.o = (char *)t->o;
    for (int j = 0; j < 3; ++j) {
        p.qs[j] = t->q_stride[j]; p.ks[j] = t->k_stride[j];
        p.vs[j] = t->v_stride[j]; p.os[j] = t->o_stride[j];
    }
    p.batch = t->batch; p.hq = t->heads_q; p.hk = t->heads_kv; p.n = t->n;
    p.seqlens = t->seqlens;
    p.scale_log2 = t->sm_scale * 1.4426950408889634f;
    p.scale_log2_dense = p.scale_log2;
    p.rows = (t->n + BM - 1) / BM;
    p.bc = p.bo = p.cc = p.ci = nullptr; p.nnz_s = p.nnz_v = 0;
    p.bidx = nullptr; p.max_blocks = 0; p.bidx_rows = 0;
    p.n_init = p.n_local = 0; p.dense_from = 0x7fffffff;
    p.head_list = t->head_list;
    p.index_heads = t->head_list ? t->index_heads : t->heads_q;
    p.chunk = 1; p.turn = p.far_turn = 0;      // set by the launcher
    p.by_deal = p.by_group = p.by_groups = p.by_heads = p.by_set = p.by_chunks = fast_div(1);      // set by the launcher
    p.descending = 0;
    p.split_first = (p.rows + 1) / 2; p.nseg = 1; p.seg_len = 1; p.part = nullptr;
    p.dtype = t->dtype;
    p.select = t->dtype == MINF_16BIT_SELECT ? t->dtype_select : nullptr;
}

// Which walks to split, and how.  `slots` workgroups fit the chip at once, a slot's share of the launch is
// `share` steps.  The longest walk sets the time of a launch whose share is much smaller; cut, it costs a
// fixed part per segment (about five steps), and its sums travel through memory to the fold (0.02 us per
// segment of a full chip).  Segments of 1.4 shares were the best or within 5 % of it wherever splitting
// paid at all (lengths 8 .. 128 swept): dense, 8 / 2 heads 8192 tokens 180 -> 162 us, 4 heads 16384 tokens
// 350 -> 301, one head 24000 tokens 439 -> 175, 8 heads of 64, 6000 tokens 87 -> 61; vertical-slash,
// 4 heads 5000 tokens 95 -> 56, 4 heads 8000 tokens 177 -> 95, 16 heads 2570 tokens 68 -> 62; block-sparse
// 8 heads 6000 tokens 145 -> 100; A-shape 8 heads 6000 tokens 117 -> 97.  Where a share is nearly the
// longest walk the whole walks win, longest first (dense: 16 heads of 64, 12000 tokens 310 against 345 us,
// 16 heads 6000 tokens 161 : 174), and so they do where a walk is too short for what a cut costs (dense,
// 32 / 8 heads 2048 tokens 53 : 58; 32 heads 1000 tokens 26 : 32; block-sparse, 28 heads 2000 tokens 57 :
// 64): the steps saved have to be worth it.
//  * Dense walks and the dense last rows of tri-shape have any number of steps.
//  * Lists are not known on the host, only their widths: a walk is taken to be as long as its list is wide, up to
//    the diagonal.  Up to 100 slashes are taken to be neighbours (the estimation always selects the last 100
//    diagonals first): two or three blocks.  A longer walk than was taken is cut into the same number of segments.
//    Taken as dense, short lists paid for segments that do not exist and for the fold: block-sparse, top-10,
//    one head 8192 tokens 24 whole, 30 split, 4 heads 25 : 34 us; top-20, 4 heads 6000 tokens 39 : 47; 50
//    slashes and 30 columns, one head 8192 tokens 18 : 27.
//  * A-shape walks end at their window.
//  * Lists and A-shape are split up to 64 row-block pairs per head only: beyond, a head has the same bits
//    whatever heads it is launched with.  Up to there the number of segments follows the launch's load, and a head's
//    bits (the order of its fp32 sums) with it.  Up to 64 pairs in all, segments have SEG_MIN steps
//    whatever else the launch holds.
constexpr int SEG_MIN = 8;
constexpr int ADJACENT_SLASHES = 100;
SplitPlan plan_split(int mode, const AttnParams &p, int head_dim) {
    const int pairs = (p.rows + 1) / 2;
    const SplitPlan none{pairs, 1, 1};
    const long long heads = (long long)p.batch * (p.head_list ? p.index_heads : p.hq);
    const int slots = head_dim == 256 ? 256 : (head_dim == 128 ? 512 : 768);
    // walks of pairs 0 .. k-1: pair i has 2 i + 2 steps, at most `most`
    int window = 0x7fffffff;
    if (mode == MODE_ASHAPE) window = (int)(((long long)p.n_local + BM - 1) / BN + 2 + ((long long)p.n_init + BN - 1) / BN);
    if (mode == MODE_BS && p.max_blocks > 0) window = p.max_blocks;
    if (mode == MODE_VS && p.nnz_s > 0) {
        const long long blocks = p.nnz_s <= ADJACENT_SLASHES ? (p.nnz_s + BN - 1) / BN + 1 : p.nnz_s;
        const long long both = blocks + ((long long)p.nnz_v + BN - 1) / BN;
        window = both < 0x7fffffff ? (int)both : 0x7fffffff;
    }
    auto steps = [&](int k, int most) -> double {
        const double grown = most / 2 < k ? most / 2 : k;
        return grown * (grown + 1) + (k - grown) * most;
    };
    const int first_dense = mode == MODE_DENSE ? 0 : (mode == MODE_ASHAPE && p.dense_from < p.n ? p.dense_from / (2 * BM) : pairs);
    const bool dense = first_dense < pairs;
    if (!dense && pairs > 64) return none;
    const int first = dense ? first_dense : 0;
    const int longest = dense ? p.rows : (p.rows < window ? p.rows : window);
    const int others = first > 0 ? (2 * first < window ? 2 * first : window) : 0;      // longest of the walks that stay whole
    const double total = dense ? steps(pairs, 0x7fffffff) - steps(first, 0x7fffffff) + (first > 0 ? steps(first, window) : 0.) : steps(pairs, window);
    const double share = total * (double)heads / slots;
    if (!dense && heads * pairs <= 64) {
        const int most = longest + (mode == MODE_VS ? SEG_MIN : 0);                    // (gathered columns)
        const int nseg = (most + SEG_MIN - 1) / SEG_MIN;
        return longest < 2 * SEG_MIN ? none : SplitPlan{0, nseg, SEG_MIN};
    }
    double want = 1.4 * share + 2;
    // dense rows at the end of a launch of shorter walks would finish last: segments of one share (16 heads of
    // 64, fp16, 24000 tokens, 128 dense rows: whole 434 us; 145, 133, 129, 152 us with 16, 48, 64, 96 steps)
    // and at least two (32 / 8 heads, 8000 tokens, window 3968: 550 -> 460 us)
    if (others > 0) want = share;
    if (others > 0 && want > (longest + 1) / 2) want = (longest + 1) / 2 > window ? (longest + 1) / 2 : window;
    if (want >= longest) return none;
    const int len = want > SEG_MIN ? (int)want : SEG_MIN;
    int nseg = (longest + (mode == MODE_VS ? SEG_MIN : 0) + len - 1) / len;
    if (nseg > 64) nseg = 64;
    const int cut = (longest + nseg - 1) / nseg;
    // (a launch of more than 400 workgroups fills most of the chip already: vertical-slash, 16 heads of scattered
    // lists, 4096 tokens, 512 workgroups, 32 of 64 steps saved: 110 -> 116 us)
    const long long wgs = heads * (pairs - first);
    if (longest - (cut > others ? cut : others) < (wgs <= 400 ? 4 + wgs / 24 : wgs / 13)) return none;
    return SplitPlan{first, nseg, len};
}

size_t split_bytes(const SplitPlan &s, const AttnParams &p, int head_dim) {
    const size_t pairs = (size_t)((p.rows + 1) / 2 - s.first) * p.batch * (p.head_list ? p.index_heads : p.hq);
    const size_t slot = head_dim == 256 ? SplitSlot<256>::BYTES : (head_dim == 128 ? SplitSlot<128>::BYTES : SplitSlot<64>::BYTES);
    return pairs * s.nseg * slot;
}

// Fills in how a launch is split and dealt out, -> its workgroups (beyond 2^31 - 1: it cannot be made)
template <int MODE, int HD> long long plan_launch(AttnParams &p, const minf_qkvo *t) {
    if (t->workspace && ((uintptr_t)t->workspace & 15) == 0) {
        const SplitPlan s = plan_split(MODE, p, HD);
        if (s.nseg > 1 && split_bytes(s, p, HD) <= t->workspace_bytes) {
            p.split_first = s.first; p.nseg = s.nseg; p.seg_len = s.len;
            p.part = (char *)t->workspace;
        }
    }
    // heads of the grid: all of them, or the selected ones rounded up to whole chunks of hq / hk
    const int group = p.hq / p.hk;
    const long long grid_heads = p.head_list ? (long long)((p.index_heads + group - 1) / group) * group : p.hq;
    const int split_pairs = (p.rows + 1) / 2 - p.split_first;
    const long long units = p.split_first + (long long)split_pairs * p.nseg;
    // The launch is a sequence of deals, `chunk` units (row-block pairs, or segments) of one kv group each: the first
    // units of every group of a set, then the next ones, ..., then the next set.  Consecutive deals go to the 8 XCDs in
    // turn, so every XCD gets an equal part of every stretch of the sequence, and where it matters (`turn`) of every group:
    // where each worked through an eighth of the launch (or of a few groups), the one with the longest walks or the densest
    // heads was left working alone.  32 / 8 heads with a table of unlike patterns, 50000 tokens 5.54 -> 4.60 ms (28 / 4 heads 4.70 ->
    // 3.79), 20000 tokens 2.22 -> 1.86 (1.78 -> 1.40); vertical-slash, 32 / 8 heads, 131072 tokens 14.86 -> 13.96 ms, 500
    // columns and 700 slashes 4.41 -> 4.04 (28 / 4 heads 120000 tokens 3.87 -> 3.08); 9000 tokens, 8 / 2 heads,
    // vertical-slash 359 -> 214 us, block-sparse 318 -> 202, A-shape 224 -> 142.  A launch that fits the chip at
    // once gains little and may lose (vertical-slash, 4 heads 13000 tokens 218 -> 186 us, 15000 234 -> 225, 16384 223 -> 232):
    // there, and at two or three workgroups a slot, it is chance which walks end up last.  In deals of an eighth those three
    // take 252, 257 and 229, in deals of 8 one group after the other 196, 232 and 201.  8 / 2 heads, 20763 tokens 506 -> 526, in
    // deals of 8 workgroups 495; but these take 8 heads, 16443 tokens, from 408 to 438 (426 in eighths).  No order serves all.
    // A deal's workgroups share K/V through an L2, but it has to be small beside what an XCD gets in all:
    //  * 32 workgroups for whole layers of vertical-slash lists: 32 / 8 heads, 65000 tokens, 500 columns and 700 slashes, deals
    //    of 16, 32, 64, 128: 2016, 1996, 1991, 1996 us; 16 heads 30000 tokens, of 1, 2, 4, 8, 16: 1710, 1574, 1543, 1523,
    //    1520; 12 / 3 heads 9000 tokens, of 4, 8, 16, 32: 240, 239, 241, 271;
    //  * 16 for heads of a list (32 / 8 heads, 50000 tokens, of 4, 8, 16, 32, 64: 4788, 4625, 4582, 4645, 4739 us) and
    //    block-sparse or A-shape walks in ascending order;
    //  * 8 in launches of up to two rounds of workgroups (block-sparse, 7 heads 9000 tokens, of 8, 16: 177 and 201 us;
    //    A-shape, 4 heads 18000 tokens, 164 and 206);
    //  * 4 where the longest walks go first, so that the last ones stay short: A-shape, 16 heads 10000 tokens, of 1, 4,
    //    16: 269, 273, 290 us; 28 / 4 heads 9000 tokens, of 7, 28, 56: 407, 417, 433;
    //  * one unit in dense and split walks.  Dense, 8 / 2 heads 16384 tokens, of 1, 2, 4, 8 units 492, 499, 512, 553 us;
    //  * one head of up to 131072 tokens: an eighth (vertical-slash, 65536 tokens 204 us, in deals of 16 225; 100000
    //    tokens 366 : 394).
    // turn: an XCD takes another place from time to time, so that with 2, 4 or 8 groups it meets all of them.  Heads of a
    // list are unlike (another place in every round), and so are the slashes of a layer's heads: 32 / 8 heads, 65000 tokens,
    // 500 columns, 700 slashes 2.13 -> 1.93 ms.  Equal heads keep an XCD to its groups (A-shape, 70000 tokens 4.44 : 4.58 ms).
    // But while it keeps its place, it works on neighbours of one group, and lists of scattered slashes live on neighbours
    // that reach a tile at the same time: 600 scattered slashes, 32 / 8 heads, 131072 tokens, another place in every round and
    // every 2, 4, 8, 16, never: 59.7, 59.2, 59.2, 58.3, 56.5, 56.0 ms.  Lists of neighbouring diagonals gain nothing by it and lose
    // the balance: 500 columns and 700 slashes, 131072 tokens 3.81, 3.80, 3.80, 3.82, 3.86, 4.00 ms, 100000 tokens 2.63, 2.65,
    // 2.66, 2.74, 2.78, 2.93 (1000 and 6096, 131072 tokens 13.16, 13.16, 13.19, 13.19, 13.18, 13.35).  So a launch of 48 rounds and
    // more goes through the eight places once, in steps of a power of two, if three of four heads keep more than an eighth of
    // the blocks in the last row (scattered 26 % of all blocks, 1000 and 6096 11 %, 500 and 700 3 %): the workgroups see that
    // from the counts.  Where a place is no single group's it stays as it was (16 heads, scattered, 25.2 : 25.7 ms).
    // Split walks: every round, but eight groups of one head, every fourth: 8192 tokens, 500 columns and 700 slashes 101 ->
    // 89.5 us, 6000 85.9 -> 83.8 (32 / 8 heads, 6000, 187 : 194).
    // set: in a batch of more than sixteen groups (of several heads), eight or the next number that divides theirs, where
    // walks are not split and differ.  An XCD that goes through all the groups with every deal has K/V of as many under way: 8 sequences, 32 / 8
    // heads, 16000 tokens, 500 columns and 700 slashes 5102 -> 4836 us, 1000 and 6096 11.80 -> 11.42 ms.  The heads of one sequence
    // go together (32 heads, 100000 tokens, scattered 36.2 : 38.2 ms), so do ungrouped ones (4 times 16, 10000 tokens, 1000 and
    // 6096 1564 : 1590 us) and split walks (16 heads, 8192 tokens 260 : 281).
    const long long groups = (long long)p.batch * (grid_heads / group);
    const int most = MODE == MODE_BS ? p.max_blocks :
                     MODE == MODE_ASHAPE ? (int)(((long long)p.n_local + p.n_init) / BN) + 2 : p.rows;    // steps of a full walk (lists: unknown)
    const long long wgs = groups * group * units;
    // Longest walks first wherever they grow with the row block over much of the sequence.  A-shape and
    // block-sparse, 32 / 8 heads: 3000 tokens 107 -> 91 and 118 -> 92 us, 6000 tokens 336 -> 315 (6824) and
    // 333 -> 308, 12000 tokens 702 -> 677 and 921 -> 897, 24000 tokens 1508 -> 1487 and (32768) 2947 -> 2920;
    // neither order wins past 60000 tokens, and with fewer than two rounds of workgroups and walks that are
    // full-length early the first rows finish last (A-shape, 8 / 2 heads, 12000 tokens 227 -> 234 us).
    p.descending = MODE == MODE_DENSE || (MODE == MODE_VS ? p.rows <= 1024 :
                   p.rows <= most || (p.rows <= 8ll * most && wgs >= 1024));
    const int share = MODE != MODE_VS && p.descending ? 4 : (wgs <= 1024 ? 8 : (MODE == MODE_VS && !p.head_list ? 32 : 16));
    long long chunk = MODE == MODE_DENSE || split_pairs > 0 || group >= share ? 1 : share / group;
    if (MODE != MODE_DENSE && split_pairs == 0 && groups * group == 1 && units <= 1024) chunk = (units + 7) / 8;
    if (chunk > units) chunk = units;
    p.chunk = (int)chunk;
    const long long deal = chunk * group, chunks = (units + chunk - 1) / chunk, deals = chunks * groups;
    const bool whole_lists = MODE == MODE_VS && !p.head_list && split_pairs == 0;
    long long set = groups;
    if (whole_lists && p.batch > 1 && group > 1 && groups > 16)
        for (set = 8; groups % set; ++set) {}
    p.turn = p.head_list || MODE == MODE_VS ? 0 : 31;
    p.far_turn = 0;
    if (whole_lists && 8 % set == 0 && chunks * set >= 8 * 48)
        while (2ll << p.far_turn <= chunks * set / 64) ++p.far_turn;
    if (p.far_turn || set < groups) p.turn = 31;               // (lists: a CHOSEN launch)
    if (MODE == MODE_VS && !p.head_list && split_pairs > 0 && groups == 8 && group == 1) p.turn = 2;
    p.by_group = fast_div((unsigned)group);
    p.by_deal = fast_div((unsigned)deal);
    p.by_groups = fast_div((unsigned)groups);
    p.by_set = fast_div((unsigned)set);
    p.by_chunks = fast_div((unsigned)chunks);
    p.by_heads = fast_div((unsigned)(grid_heads / group));
    return (deals + 7) / 8 * 8 * deal;
}

template <int MODE, int HD> int launch_hd(AttnParams p, const minf_qkvo *t, void *stream) {
    if (p.batch == 0 || p.rows == 0) return MINF_OK;
    const int dtype = t->dtype;
    const long long grid = plan_launch<MODE, HD>(p, t);
    if (grid > 0x7fffffffLL) return MINF_ERR_UNSUPPORTED;
    const int split_pairs = (p.rows + 1) / 2 - p.split_first;
    const dim3 block(2 * NTHREADS);
    hipStream_t st = (hipStream_t)stream;
    const bool chosen = MODE == MODE_VS && p.turn == 31;
#define MINF_LAUNCH_ATTN(T)                                                                                      \
    do {                                                                                                         \
        if (p.nseg > 1) hipLaunchKernelGGL((attn_fwd_kernel<T, MODE, HD, true>), dim3((unsigned)grid), block, 0, st, p); \
        else if (chosen) hipLaunchKernelGGL((attn_fwd_kernel<T, MODE, HD, false, MODE == MODE_VS>), dim3((unsigned)grid), block, 0, st, p); \
        else hipLaunchKernelGGL((attn_fwd_kernel<T, MODE, HD, false>), dim3((unsigned)grid), block, 0, st, p);   \
    } while (0)
    if (dtype != MINF_F16) MINF_LAUNCH_ATTN(__bf16);
    if (dtype != MINF_BF16) MINF_LAUNCH_ATTN(_Float16);
#undef MINF_LAUNCH_ATTN
    const int status = minf_launch_status();
    if (status != MINF_OK || p.nseg == 1) return status;
    const unsigned merge_wgs = (unsigned)(4ll * split_pairs * p.batch * (p.head_list ? p.index_heads : p.hq));
    if (p.nseg <= MERGE_FEW) hipLaunchKernelGGL((attn_merge_kernel<HD, true>), dim3(merge_wgs), dim3(256), 0, st, p);
    else hipLaunchKernelGGL((attn_merge_kernel<HD, false>), dim3(merge_wgs), dim3(256), 0, st, p);
    return minf_launch_status();
}

template <int MODE> int launch(const AttnParams &p, const minf_qkvo *t, void *stream) {
    if constexpr (MODE == MODE_ASHAPE || MODE == MODE_DENSE)
        if (t->head_dim == 256) return launch_hd<MODE, 256>(p, t, stream);
    if (t->head_dim == 256) return MINF_ERR_UNSUPPORTED;
    return t->head_dim == 64 ? launch_hd<MODE, 64>(p, t, stream) : launch_hd<MODE, 128>(p, t, stream);
}

}  // namespace

// the arguments of the entry points, checked (`p` is filled in on MINF_OK)
static int vs_params(AttnParams &p, const minf_qkvo *t, const int32_t *block_count, const int32_t *block_offset,
                     const int32_t *column_count, const int32_t *column_index, int rows, int nnz_s, int nnz_v) {
    const int st = check_tensors(t);
    if (st) return st;
    if (!block_count || !block_offset || !column_count || !column_index) return MINF_ERR_INVALID_ARG;
    if (nnz_s < 1 || nnz_v < 1) return MINF_ERR_INVALID_ARG;
    fill_params(p, t);
    if (rows != p.rows) return MINF_ERR_INVALID_ARG;
    p.bc = block_count; p.bo = block_offset; p.cc = column_count; p.ci = column_index;
    p.nnz_s = nnz_s; p.nnz_v = nnz_v;
    return MINF_OK;
}

static int bs_params(AttnParams &p, const minf_qkvo *t, const int32_t *block_index, int rows, int max_blocks) {
    const int st = check_tensors(t);
    if (st) return st;
    if (!block_index || max_blocks < 1) return MINF_ERR_INVALID_ARG;
    fill_params(p, t);
    if (rows < p.rows) return MINF_ERR_INVALID_ARG;
    // block_index may have more rows than ceil(n/64) (the reference pads n first)
    p.bidx = block_index; p.max_blocks = max_blocks; p.bidx_rows = rows;
    return MINF_OK;
}

static int ashape_params(AttnParams &p, const minf_qkvo *t, int n_init, int n_local) {
    const int st = check_tensors(t, true);
    if (st) return st;
    if (n_init < 0 || n_local < 1) return MINF_ERR_INVALID_ARG;
    fill_params(p, t);
    p.n_init = n_init; p.n_local = n_local;
    return MINF_OK;
}

extern "C" int minf_vs_attn_fwd(const minf_qkvo *t, const int32_t *block_count,
                                const int32_t *block_offset, const int32_t *column_count,
                                const int32_t *column_index, int rows, int nnz_s, int nnz_v,
                                void *stream) {
    AttnParams p;
    const int st = vs_params(p, t, block_count, block_offset, column_count, column_index, rows, nnz_s, nnz_v);
    return st ? st : launch<MODE_VS>(p, t, stream);
}

extern "C" int minf_bs_attn_fwd(const minf_qkvo *t, const int32_t *block_index, int rows,
                                int max_blocks, void *stream) {
    AttnParams p;
    const int st = bs_params(p, t, block_index, rows, max_blocks);
    return st ? st : launch<MODE_BS>(p, t, stream);
}

extern "C" int minf_ashape_attn_fwd(const minf_qkvo *t, int n_init, int n_local, void *stream) {
    AttnParams p;
    const int st = ashape_params(p, t, n_init, n_local);
    return st ? st : launch<MODE_ASHAPE>(p, t, stream);
}

namespace {

// The parts of a layer (null: absent) in one launch -> whether it was made: not where a walk is split, nothing is to be
// done, or only one part is there
template <typename T, int HD> bool launch_mixed(const AttnParams &vs, const minf_qkvo *vs_t, const AttnParams &bs, const minf_qkvo *bs_t,
                                                const AttnParams &as, const minf_qkvo *as_t, void *stream) {
    MixedParams m;
    memset(&m, 0, sizeof(m));
    long long vs_wgs = 0, bs_wgs = 0, as_wgs = 0;
    if (vs_t) { m.vs = vs; vs_wgs = plan_launch<MODE_VS, HD>(m.vs, vs_t); }
    if (m.vs.turn == 31) m.vs.turn = 0;           // (no CHOSEN form of this kernel)
    if (bs_t) { m.bs = bs; bs_wgs = plan_launch<MODE_BS, HD>(m.bs, bs_t); }
    if (as_t) { m.as = as; as_wgs = plan_launch<MODE_ASHAPE, HD>(m.as, as_t); }
    if ((vs_t && m.vs.nseg > 1) || (bs_t && m.bs.nseg > 1) || (as_t && m.as.nseg > 1)) return false;
    if (vs_wgs + bs_wgs + as_wgs > 0x7fffffffLL) return false;
    m.first_bs = (unsigned)vs_wgs;
    m.first_as = (unsigned)(vs_wgs + bs_wgs);
    hipLaunchKernelGGL((attn_mixed_kernel<T, HD>), dim3((unsigned)(vs_wgs + bs_wgs + as_wgs)), dim3(2 * NTHREADS), 0, (hipStream_t)stream, m);
    return true;
}

}  // namespace

extern "C" int minf_mixed_attn_fwd(const minf_qkvo *vs, const int32_t *block_count, const int32_t *block_offset,
                                   const int32_t *column_count, const int32_t *column_index, int rows, int nnz_s, int nnz_v,
                                   const minf_qkvo *bs, const int32_t *block_index, int block_rows, int max_blocks,
                                   const minf_qkvo *ashape, int n_init, int n_local, void *stream) {
    AttnParams vs_p, bs_p, as_p;
    int st = MINF_OK;
    if (vs) st = vs_params(vs_p, vs, block_count, block_offset, column_count, column_index, rows, nnz_s, nnz_v);
    if (st == MINF_OK && bs) st = bs_params(bs_p, bs, block_index, block_rows, max_blocks);
    if (st == MINF_OK && ashape) st = ashape_params(as_p, ashape, n_init, n_local);
    if (st != MINF_OK) return st;
    const minf_qkvo *const parts[3] = {vs, bs, ashape};
    const minf_qkvo *first = nullptr;
    int count = 0;
    bool alike = true;
    for (const minf_qkvo *t : parts) {
        if (!t) continue;
        ++count;
        if (!first) first = t;
        alike = alike && t->head_dim == first->head_dim && t->dtype == first->dtype && t->batch > 0 && t->n > 0;
    }
    if (count > 1 && alike && first->head_dim <= 128 && first->dtype != MINF_16BIT_SELECT) {
        bool made;
        if (first->head_dim == 128)
            made = first->dtype == MINF_BF16 ? launch_mixed<__bf16, 128>(vs_p, vs, bs_p, bs, as_p, ashape, stream)
                                             : launch_mixed<_Float16, 128>(vs_p, vs, bs_p, bs, as_p, ashape, stream);
        else
            made = first->dtype == MINF_BF16 ? launch_mixed<__bf16, 64>(vs_p, vs, bs_p, bs, as_p, ashape, stream)
                                             : launch_mixed<_Float16, 64>(vs_p, vs, bs_p, bs, as_p, ashape, stream);
        if (made) return minf_launch_status();
    }
    if (vs) st = launch<MODE_VS>(vs_p, vs, stream);
    if (st == MINF_OK && bs) st = launch<MODE_BS>(bs_p, bs, stream);
    if (st == MINF_OK && ashape) st = launch<MODE_ASHAPE>(as_p, ashape, stream);
    return st;
}

extern "C" int minf_trishape_attn_fwd(const minf_qkvo *t, int n_init, int n_local, int n_last,
                                      float sm_scale_last, void *stream) {
    int st = check_tensors(t, true);
    if (st) return st;
    uint32_t scale_bits;
    memcpy(&scale_bits, &sm_scale_last, sizeof(scale_bits));          // (negative, infinite or NaN: refused)
    if (n_init < 0 || n_local < 1 || n_last < 0 || (scale_bits >> 31) || (scale_bits & 0x7f800000u) == 0x7f800000u)
        return MINF_ERR_INVALID_ARG;
    AttnParams p;
    fill_params(p, t);
    if (sm_scale_last > 0.f) p.scale_log2_dense = sm_scale_last * 1.4426950408889634f;
    p.n_init = n_init; p.n_local = n_local;
    p.dense_from = n_last < t->n ? t->n - n_last : 0;
    return launch<MODE_ASHAPE>(p, t, stream);
}

extern "C" int minf_dense_attn_fwd(const minf_qkvo *t, void *stream) {
    int st = check_tensors(t, true);
    if (st) return st;
    AttnParams p;
    fill_params(p, t);
    return launch<MODE_DENSE>(p, t, stream);
}

extern "C" size_t minf_attn_workspace_bytes(const minf_qkvo *t, int op, int n_init, int n_local, int n_last) {
    if (!t || t->batch <= 0 || t->n <= 0 || t->heads_q <= 0 || op < MINF_OP_VERTICAL_SLASH || op > MINF_OP_DENSE) return 0;
    AttnParams p;
    fill_params(p, t);
    if (op == MINF_OP_ASHAPE) {
        p.n_init = n_init; p.n_local = n_local;
        p.dense_from = n_last > 0 ? (n_last < t->n ? t->n - n_last : 0) : p.dense_from;
    }
    if (op == MINF_OP_BLOCK_SPARSE) p.max_blocks = n_local;
    if (op == MINF_OP_VERTICAL_SLASH) { p.nnz_v = n_init > 0 ? n_init : 0; p.nnz_s = n_local; }
    const SplitPlan s = plan_split(op, p, t->head_dim);
    return s.nseg > 1 ? split_bytes(s, p, t->head_dim) : 0;
}
