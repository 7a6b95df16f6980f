// Offline pattern search for gfx950: how much of the exact causal softmax mass does a candidate
// sparse pattern keep?  (reference minference/modules/minference_forward.py:129-227, where the
// whole N x N probability matrix is materialised and multiplied by N x N masks).
//
// Here nothing of size N x N exists.  A candidate is described by three flag arrays per head, one
// bit per candidate (up to 8 candidates are scored in one sweep):
//   col_flags[c]        bit t set: candidate t keeps key column c              (verticals, sinks)
//   diag_flags[o]       bit t set: candidate t keeps the diagonal query - key = o  (slashes, windows)
//   block_flags[R][C]   bit t set: candidate t keeps the 32 x 32 block (R, C)  (block-sparse)
// and element (r, c), c <= r, belongs to candidate t iff any of its three bits t is set.
//
//   pattern_recall_kernel  one workgroup per (head, 128 query rows), heavy row tiles first: 2 waves per
//                     64 rows, which take every second causal key block (32 keys each).  S^T = K.Q^T on
//                     v_mfma_f32_32x32x16, K copied to LDS and read from there in
//                     operand layout: lane <-> query row, registers <-> keys; online softmax with a
//                     running maximum per row.  The row sum and the masked sums are matrix products
//                     too (see the kernel).  Waves are merged through LDS; a 64-row tile's sum of
//                     masked/total ratios over its rows >= row_begin goes to a partial buffer.
//   pattern_recall_finalize  sums the partials of a head in a fixed order and divides by the
//                     number of rows (deterministic; no atomics).
//   flags_set_indices / flags_set_range  build the flag arrays from top-k index lists / ranges.
#include "minf_common.h"
#include <math.h>

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4_t;

constexpr int HD = 128;
constexpr int NC = 8;            // candidates per sweep (bits of a flag byte)
constexpr int TILE = 64;         // query rows per wave pair (two tiles per workgroup)
constexpr int KB = 32;           // keys per block
constexpr int DW = (2 * TILE + 2 * KB) / 4;   // words of diagonal flags that 128 rows and 64 keys touch

union Frag {
    u32x4_t u;
    bf16x8_t b;
    f16x8_t h;
};

template <typename T> __device__ __forceinline__ f32x16_t mma(const Frag &a, const Frag &b, f32x16_t c);
template <> __device__ __forceinline__ f32x16_t mma<__bf16>(const Frag &a, const Frag &b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.b, b.b, c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x16_t mma<_Float16>(const Frag &a, const Frag &b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.h, b.h, c, 0, 0, 0);
}

struct RecallParams {
    const char *q, *k;
    long long qs[3], ks[3];      // element strides batch, head, token
    int batch, hq, hk, n;
    float scale_log2;            // of |sm_scale|: the maximum is taken before the scale,
    unsigned q_flip;             // and the sign bits of Q are turned for a negative one
    const unsigned char *col, *diag, *blk;   // blk may be null
    long long flag_pitch;        // bytes between heads of col / diag (>= n rounded up to 64)
    long long blk_pitch;         // bytes between block rows; a head has ceil(n/32) block rows
    int row_begin, tiles;
    int stripes;                 // the row tiles of a kv group are dealt to this many XCD ranges
    unsigned total_wg;
    float *partial;              // [batch*hq, tiles, NC]
};

// rows of one 32-row block of one head (or keys of a key block): row = first + lane%32, clamped;
// d = 16*ks + 8*(lane/32) + 0..7
__device__ __forceinline__ void load_frag(const char *base, long long tok_stride, int first, int n, int lane,
                                          Frag (&f)[8]) {
    const int row = min(first + (lane & 31), n - 1);
    const char *rp = base + (long long)row * tok_stride * 2 + (lane >> 5) * 16;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) f[ks].u = *reinterpret_cast<const u32x4_t *>(rp + ks * 32);
}

// D[t][row] = A[t] . B[row] + C[t][row] for 16 groups of 4 lanes: a lane's B belongs to its own row, its A is row
// t = lane % 4 of its group's A, its D are rows 0..3 of its own column
__device__ __forceinline__ f32x4_t mma4(float a, float b, f32x4_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
#else
    return c;
#endif
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

struct RowState {
    float m, z, zm[NC];
};

__device__ __forceinline__ void merge_into(RowState &a, float m, float z, const float (&zm)[NC]) {
    const float mn = fmaxf(a.m, m);
    const float mu = mn == -INFINITY ? 0.f : mn;
    const float fa = fast_exp2(a.m - mu), fb = fast_exp2(m - mu);
    a.z = a.z * fa + z * fb;
#pragma unroll
    for (int t = 0; t < NC; ++t) a.zm[t] = a.zm[t] * fa + zm[t] * fb;
    a.m = mn;
}

// What all 63 diagonals of a 32 x 32 block have in common, per candidate: the block at distance d (in
// blocks) from the diagonal holds the offsets 32 d - 31 .. 32 d + 31.  Per aligned group of 32 offsets the
// table holds the OR and the AND of its flag bytes, and the same without the group's first offset.
constexpr int DIAG_GROUPS = 8192;            // (262144 tokens; farther blocks are treated as mixed)
constexpr int DIAG_GROUPS_SMALL = 4096;      // (131072 tokens: three workgroups fit a CU's LDS)

// The masked sums as matrix products.  Per 32-key block and row,  Z_t = sum_c mask_t(c) e(c)  over the columns that
// candidate t keeps, e the block's exponentials in fp32 straight from the S^T accumulators: v_mfma_f32_4x4x1 takes one
// e per lane as its own row's B, its A is one key's flags of four candidates, so the products are exact and the sums
// stay with the lane that owns the row.  A block that a candidate keeps as a whole (a block of its list, one all of
// whose diagonals it keeps: most of a window, of a run of slashes) adds the block's row sum instead.  Only
// candidates with SOME of a block's diagonals are added element by element (without the columns, which are in the
// product already).  A block's sums start from zero and are added once to the running ones.
// Relative error of the scores against fp64 sums, 4096 .. 16384 tokens, bf16 and fp16: up to 6.8e-8 (three bf16 terms per
// exponential on 32x32x16 products, which this replaces: 6.8e-8), under a sink of 14 nats 3.3e-8 (1.8e-7); shares of
// candidates without a sink of 14 .. 80 nats 1.9e-6 at most (6.5e-6; 3.1e-7 against 2.2e-7 at 14): there the rounding of
// the scale in fp32 bounds it.
// Bound by its vector instructions, 131 per 32 x 32 block (fma and exp 32, of which the exp take four times as long;
// maximum, row sum) and 40 per candidate with mixed diagonals, and by its matrix products, which overlap little with them.
// 32 / 8 heads, 16384 tokens, the six candidates of the reference: 2.73 -> 1.79 ms against the bf16 terms (56 conversions
// per block; masks built in registers by every wave, where one of a workgroup's threads now writes them to LDS once; two
// waves per SIMD, now three, since neither accumulators with nine used rows of 32 nor masks occupy registers).  0.18 ms
// of it: no value that a step fetches for the next is touched before the next barrier (a wait for a flag byte was a wait
// for the K rows before it), one LDS read for the four distances of a step, fragment addresses by XOR from one register.
// Beyond 131072 tokens the table of diagonals leaves LDS for two waves per SIMD.
template <typename T, int DG> __global__ __launch_bounds__(256, DG > DIAG_GROUPS_SMALL ? 2 : 3) void pattern_recall_kernel(const RecallParams p) {
    __shared__ unsigned dtab[DG];                       // bytes: OR, AND, OR without the first, AND without the first
    // two steps of two 32-key blocks each (one per key parity), 256-byte rows whose 16-byte chunks are
    // XOR-permuted (chunk ^ row % 16) so that the fragment reads of 32 rows hit distinct banks
    __shared__ __attribute__((aligned(16))) char kt[2][2 * KB * HD * 2];
    // ... and their column flags: as fp32 ones and zeros by candidate and key (chunks of four keys permuted: chunk ^
    // 2 (candidate % 4)), and as they are; and the flags of the diagonals a step touches, the farthest first
    __shared__ __attribute__((aligned(16))) float cmask[2][NC][2 * KB];
    __shared__ __attribute__((aligned(16))) unsigned cbytes[2][2 * KB / 4], dbytes[2][DW];
    float (*const lds)[TILE][NC + 2] = reinterpret_cast<float (*)[TILE][NC + 2]>(&kt[0][0]);   // after the sweep
    static_assert(sizeof(float) * 4 * TILE * (NC + 2) <= sizeof(kt), "the waves' shares take the place of K");
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    // XCD-aware order: every XCD works through one contiguous eighth of (batch, kv head, stripe, row tile,
    // query head in the group), so that the tiles and heads that read one kv head share an L2
    const unsigned per_xcd = p.total_wg >> 3;
    unsigned rest = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    const int group = p.hq / p.hk, tps = (p.tiles + 1) / 2, per_stripe = (tps + p.stripes - 1) / p.stripes;
    const int hin = (int)(rest % (unsigned)group); rest /= (unsigned)group;
    const int in_stripe = (int)(rest % (unsigned)per_stripe); rest /= (unsigned)per_stripe;
    const int ti = in_stripe * p.stripes + (int)(rest % (unsigned)p.stripes); rest /= (unsigned)p.stripes;
    if (ti >= tps || rest >= (unsigned)(p.batch * p.hk)) return;   // padding
    const int tp = tps - 1 - ti;                                   // heavy (late) row tiles first
    const int hkv = (int)(rest % (unsigned)p.hk), b = (int)(rest / (unsigned)p.hk), h = hkv * group + hin;
    const int head_lin = b * p.hq + h;
    const int half = wave & 1, kpar = wave >> 1;
    const int rt = 2 * tp + half;                                  // this wave's 64-row tile
    const char *qb = p.q + ((long long)b * p.qs[0] + (long long)h * p.qs[1]) * 2;
    const char *kbase = p.k + ((long long)b * p.ks[0] + (long long)hkv * p.ks[1]) * 2;
    const unsigned char *col = p.col + (long long)head_lin * p.flag_pitch;
    const unsigned char *diag = p.diag + (long long)head_lin * p.flag_pitch;
    const int brows = (p.n + KB - 1) / KB;
    const unsigned char *blk = p.blk ? p.blk + (long long)head_lin * brows * p.blk_pitch : nullptr;
    float *const out = p.partial + ((long long)head_lin * p.tiles + rt) * NC;
    if ((tp + 1) * 2 * TILE <= p.row_begin) {                      // no row of the tiles counts
        if (kpar == 0 && rt < p.tiles && lane < NC) out[lane] = 0.f;
        return;
    }

    const int groups = min(min(4 * tp + 4, brows), DG);
    for (int i = tid; i < groups; i += 256) {
        const unsigned *w = reinterpret_cast<const unsigned *>(diag + 32ll * i);
        unsigned o = 0u, an = 0xffffffffu, w0 = w[0];
#pragma unroll
        for (int j = 1; j < 8; ++j) { const unsigned x = w[j]; o |= x; an &= x; }
        auto fold_or = [](unsigned x) { x |= x >> 16; return (x | (x >> 8)) & 0xffu; };
        auto fold_and = [](unsigned x) { x &= x >> 16; return (x & (x >> 8)) & 0xffu; };
        dtab[i] = fold_or(o | w0) | (fold_and(an & w0) << 8) | (fold_or(o | (w0 & ~0xffu)) << 16) | (fold_and(an & (w0 | 0xffu)) << 24);
    }
    __syncthreads();

    Frag qf[2][8];
    load_frag(qb, p.qs[2], rt * TILE, p.n, lane, qf[0]);
    load_frag(qb, p.qs[2], rt * TILE + 32, p.n, lane, qf[1]);
    if (p.q_flip)
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                qf[0][ks].u[i] ^= p.q_flip;
                qf[1][ks].u[i] ^= p.q_flip;
            }

    constexpr float LAZY = 6.f;                        // exponentials reach 2^-1 .. 2^LAZY
    float m[2] = {-INFINITY, -INFINITY};               // running maximum of the lane's row (same in both lane halves)
    float zs[2] = {0.f, 0.f}, zc[2][NC];               // this lane's share (its keys) of the row sum and the masked sums
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int t = 0; t < NC; ++t) zc[nb][t] = 0.f;

    const bool counts = rt < p.tiles && (rt + 1) * TILE > p.row_begin;
    const int last_kb = counts ? min(2 * rt + 1, brows - 1) : -1;  // last key block any row of the tile sees
    const int last_any = min(4 * tp + 3, brows - 1);               // ... and any row of the workgroup
    // the 64 keys of a step, copied by the four waves together (16 rows each, 4 per instruction; rows past
    // the sequence read a valid row instead: no row of a head sees those keys)
    const int cp_r = lane >> 4, cp_c = lane & 15;
    const int row_bytes = (int)p.ks[2] * 2;
    const int cp_row = cp_r * row_bytes, cp_chunk = (cp_c ^ cp_r) << 4;
    auto copy_k = [&](int kb0, int buf) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the builtins do not exist in the host pass)
        if ((kb0 + 2) * KB <= p.n && p.ks[2] >= 0 && p.ks[2] <= (1 << 22)) {       // (the copies' offsets are 32-bit and unsigned)
            // the extent of 64 rows: the last one ends HD elements past its start, however close the rows lie (rows
            // that overlap, one row for every key: token stride 0)
            const int extent = (2 * KB - 1) * row_bytes + HD * 2;
            const __amdgpu_buffer_rsrc_t srd = __builtin_amdgcn_make_buffer_rsrc((void *)(kbase + (long long)kb0 * KB * row_bytes), 0, extent, 0x00020000);
            const int lds0 = (int)(unsigned)(unsigned long long)(__attribute__((address_space(3))) char *)kt[buf] + 16 * wave * HD * 2;
            int chunk = cp_chunk;
            asm volatile("" : "+v"(chunk));            // (one instruction per copy rather than a register)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(srd, (__attribute__((address_space(3))) void *)(unsigned long long)(unsigned)(lds0 + 4 * j * HD * 2),
                                                         16, (chunk ^ (64 * j)) + cp_row, (16 * wave + 4 * j) * row_bytes, 0, 0);
            return;
        }
#endif
        int ln = lane;
        asm volatile("" : "+v"(ln));                   // (or the addresses of this rare form occupy registers throughout the sweep)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 16 * wave + 4 * j + (ln >> 4);
            const char *src = kbase + (long long)min(kb0 * KB + r, p.n - 1) * p.ks[2] * 2 + (((ln & 15) ^ (r & 15)) << 4);
            copy16_to_lds(src, kt[buf] + (16 * wave + 4 * j) * HD * 2);
        }
    };
    // what the next step needs beside K, fetched a step ahead: the flags of four keys around kb0 * 32 + lane, four diagonal flags
    // per thread (word w of a step holds offsets top - 4 w - 3 .. top - 4 w, top = 128 tp + 127 - 32 kb0; offsets below 0
    // lie above the diagonal), the block bytes of this wave's two row blocks
    unsigned cb_next = 0u, dw_next = 0u, bb_next[2] = {0u, 0u};
    auto fetch_flags = [&](int kb0) {
        cb_next = *reinterpret_cast<const unsigned *>(col + min(kb0 * KB + (lane & ~3), brows * KB - 4));   // (its byte is taken when it is used: no wait here)
        if (tid < DW) {
            const int at = 2 * TILE * tp + 2 * TILE - 4 - KB * kb0 - 4 * tid;
            dw_next = at >= 0 && at + 4 <= (int)p.flag_pitch ? *reinterpret_cast<const unsigned *>(diag + at) : 0u;
        }
        if (blk)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) bb_next[nb] = blk[(long long)min(2 * rt + nb, brows - 1) * p.blk_pitch + min(kb0 + kpar, brows - 1)];
    };
    copy_k(0, 0);
    fetch_flags(0);
    for (int kb0 = 0; kb0 <= last_any; kb0 += 2) {
        const int buf = (kb0 >> 1) & 1, kb = kb0 + kpar, n0 = kb * KB;
        const unsigned cb = (cb_next >> (8 * (lane & 3))) & 0xffu, bb[2] = {bb_next[0], bb_next[1]};
        // (nobody reads these buffers: their last readers were done before the last barrier)
#pragma unroll
        for (int t = 0; t < NC; t += 4)
            cmask[buf][t + wave][(((lane >> 2) ^ (2 * wave)) << 2) | (lane & 3)] = (float)((cb >> (t + wave)) & 1u);
        if (wave == 3) reinterpret_cast<unsigned char *>(cbytes[buf])[lane] = (unsigned char)cb;
        if (tid < DW) dbytes[buf][tid] = __builtin_bswap32(dw_next);
        const unsigned long long kept_lo = __ballot((cb & 0x0fu) != 0u), kept_hi = __ballot((cb & 0xf0u) != 0u);
        const bool cols[2] = {(unsigned)(kept_lo >> (32 * kpar)) != 0u, (unsigned)(kept_hi >> (32 * kpar)) != 0u};   // candidates 0..3, 4..7
        __builtin_amdgcn_s_waitcnt(0x0f70);            // vmcnt(0): this wave's share of the step is in LDS
        __syncthreads();                               // ... and everybody's; everyone is done with the step before
        if (kb0 + 2 <= last_any) {
            copy_k(kb0 + 2, buf ^ 1);
            fetch_flags(kb0 + 2);
        }
        if (kb > last_kb) continue;                    // (wave-uniform; no barrier below)
        unsigned full[2], mixed[2];                    // candidates that keep all / some of a block, by its row block
        // (one read for the two distances and the ones before them: lane 2 nb + 1 - x holds distance d(nb) - x)
        const int d0 = 2 * rt - kb;
        const unsigned near_ = dtab[min(max(d0 - 1 + (lane & 1) + ((lane >> 1) & 1), 0), DG - 1)];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const int d = d0 + nb;
            const unsigned here = __builtin_amdgcn_readlane(near_, 2 * nb + 1);
            unsigned before = __builtin_amdgcn_readlane(near_, 2 * nb) >> 16;
            if (d <= 0) before = 0xff00u;              // (nothing before the main diagonal)
            unsigned any = (here | before) & 0xffu, all = (here & before) >> 8;
            if (d >= DG) { any = 0xffu; all = 0u; }
            full[nb] = __builtin_amdgcn_readfirstlane(bb[nb]) | (all & 0xffu);
            mixed[nb] = any & ~full[nb];
        }
        f32x16_t acc[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) { acc[0][r] = 0.f; acc[1][r] = 0.f; }
        const int kat = ((buf * 2 + kpar) * KB + l32) * HD * 2 + ((g ^ (l32 & 15)) << 4);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            Frag kf;
            kf.u = *reinterpret_cast<const u32x4_t *>(&kt[0][0] + (kat ^ (32 * ks)));
            acc[0] = mma<T>(kf, qf[0][ks], acc[0]);
            acc[1] = mma<T>(kf, qf[1][ks], acc[1]);
        }

#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const int rb = 2 * rt + nb;                            // 32-row block of this half
            if (kb > rb) continue;                                 // wholly above the diagonal
            const int row = rb * 32 + l32;
            if (kb == rb) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (n0 + 8 * (r >> 2) + 4 * g + (r & 3) > row) acc[nb][r] = -INFINITY;
            }
            float mx = fmaxf(fmaxf(acc[nb][0], acc[nb][1]), acc[nb][2]);
#pragma unroll
            for (int r = 3; r + 1 < 16; r += 2) mx = fmaxf(fmaxf(mx, acc[nb][r]), acc[nb][r + 1]);
            mx = fmaxf(mx, acc[nb][15]);
            { const unsigned u = __float_as_uint(mx); auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false); mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])); }
            const float cand = mx * p.scale_log2;
            const bool grow = cand > m[nb] + LAZY;                 // (raised only when it has to be)
            if (__any(grow)) {
                // (a whole number: the rescale is exact, so that what was summed under one maximum
                // and what is summed under the next are in proportion to the last bit)
                const float up = ceilf(cand), alpha = grow ? fast_exp2(m[nb] - up) : 1.0f;
                m[nb] = grow ? up : m[nb];
                zs[nb] *= alpha;
#pragma unroll
                for (int t = 0; t < NC; ++t) zc[nb][t] *= alpha;
            }
            float e[16];
            const float off = m[nb] == -INFINITY ? 0.f : -m[nb];           // (no key yet whose score is above -inf)
#pragma unroll
            for (int r = 0; r < 16; ++r) e[r] = fast_exp2(fmaf(acc[nb][r], p.scale_log2, off));
            // the block's sums from zero: row sum, columns of each candidate
            f32x4_t zb[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (cols[c])
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t a = *reinterpret_cast<const f32x4_t *>(&cmask[buf][4 * c + (lane & 3)][((8 * kpar + 2 * j + g) ^ (2 * (lane & 3))) << 2]);
#pragma unroll
                        for (int i = 0; i < 4; ++i) zb[c] = mma4(a[i], e[4 * j + i], zb[c]);
                    }
            const float sum = (((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7])))
                + (((e[8] + e[9]) + (e[10] + e[11])) + ((e[12] + e[13]) + (e[14] + e[15])));
            zs[nb] += sum;
            if (mixed[nb]) {
                // diagonal flags of keys n0 + 8j + 4g + 0..3, without the kept columns.  They begin at any byte: two words
                // and a byte shift, since an LDS read off its alignment took about a hundred cycles (32 / 8 heads, 4096
                // tokens: 325 -> 300 us, 16384 1890 -> 1795; one head, 6000 tokens 324 -> 308)
                unsigned pm[4];
                const int at = (2 * TILE * tp + 2 * TILE - 1 - KB * kb0) - (row - n0 - 4 * g);      // (in bytes; 0 .. 4 DW - 32 + 7)
                const unsigned *const dp = dbytes[buf] + (at >> 2);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    pm[j] = __builtin_amdgcn_alignbyte(dp[2 * j + 1], dp[2 * j], at & 3) & ~cbytes[buf][8 * kpar + 2 * j + g];
#pragma unroll
                for (int t = 0; t < NC; ++t)
                    if ((mixed[nb] >> t) & 1u) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            unsigned x = (pm[j] >> t) & 0x01010101u;
                            asm("" : "+v"(x));         // (four conversions of its bytes, not a bit field and a conversion for each)
                            float z = zb[t >> 2][t & 3];
#pragma unroll
                            for (int i = 0; i < 4; ++i) z = fmaf((float)((x >> (8 * i)) & 0xffu), e[4 * j + i], z);
                            zb[t >> 2][t & 3] = z;
                        }
                    }
            }
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (cols[c] || (((full[nb] | mixed[nb]) >> (4 * c)) & 0xfu))
#pragma unroll
                    for (int t = 4 * c; t < 4 * c + 4; ++t) zc[nb][t] += (full[nb] >> t) & 1u ? sum : zb[c][t & 3];
        }
    }

    // merge the two lanes of a row, then the two waves
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
        float *dst = lds[wave][nb * 32 + l32];
        const float total = zs[nb] + __shfl_xor(zs[nb], 32);
        if (g == 0) {
            dst[0] = m[nb];
            dst[1] = total;
        }
        float own[NC];
#pragma unroll
        for (int t = 0; t < NC; ++t) own[t] = zc[nb][t] + __shfl_xor(zc[nb][t], 32);
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[2 + 4 * g + r] = g ? own[4 + r] : own[r];
    }
    __syncthreads();
    if (kpar == 0 && rt < p.tiles) {
        RowState a;
        a.m = lds[wave][lane][0];
        a.z = lds[wave][lane][1];
#pragma unroll
        for (int t = 0; t < NC; ++t) a.zm[t] = lds[wave][lane][2 + t];
        float zm[NC];
#pragma unroll
        for (int t = 0; t < NC; ++t) zm[t] = lds[wave + 2][lane][2 + t];
        merge_into(a, lds[wave + 2][lane][0], lds[wave + 2][lane][1], zm);
        const int row = rt * TILE + lane;
        const bool counted = row < p.n && row >= p.row_begin && a.z > 0.f;
        const float inv = counted ? 1.0f / a.z : 0.f;
#pragma unroll
        for (int t = 0; t < NC; ++t) {
            float x = a.zm[t] * inv;
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d);     // fixed butterfly order
            if (lane == 0) out[t] = x;
        }
    }
}

__global__ __launch_bounds__(64) void pattern_recall_finalize(const float *partial, int tiles, int n, int row_begin,
                                                              float *recall) {
    const int head_lin = (int)blockIdx.x, lane = (int)threadIdx.x;
    const float *src = partial + (long long)head_lin * tiles * NC;
    for (int t = 0; t < NC; ++t) {
        double x = 0.;
        for (int i = lane; i < tiles; i += 64) x += (double)src[(long long)i * NC + t];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d);
        // no rows to average over -> NaN, like the mean of an empty slice in the reference
        // (written as a bit pattern: the library is built without NaN semantics, under which the constant
        // itself is undefined)
        if (lane == 0) recall[head_lin * NC + t] = n > row_begin ? (float)(x / (double)(n - max(row_begin, 0))) : __uint_as_float(0x7fc00000u);
    }
}

__global__ void flags_set_indices_kernel(const int32_t *idx, long long idx_stride, int rows, int k, unsigned bit,
                                         unsigned char *flags, long long pitch, int limit) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= k) return;
    for (int row = (int)blockIdx.y; row < rows; row += (int)gridDim.y) {
        const int x = idx[(long long)row * idx_stride + i];
        if (x < 0 || x >= limit) continue;
        const long long off = (long long)row * pitch + x;
        atomicOr(reinterpret_cast<unsigned *>(flags + (off & ~3ll)), (1u << bit) << (8 * (int)(off & 3)));
    }
}

__global__ void flags_set_range_kernel(int begin, int end, int rows, unsigned bit, unsigned char *flags,
                                       long long pitch) {
    const int x = begin + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (x >= end) return;
    for (int row = (int)blockIdx.y; row < rows; row += (int)gridDim.y) {
        const long long off = (long long)row * pitch + x;
        atomicOr(reinterpret_cast<unsigned *>(flags + (off & ~3ll)), (1u << bit) << (8 * (int)(off & 3)));
    }
}

}  // namespace

extern "C" size_t minf_pattern_recall_workspace_bytes(int batch, int heads_q, int n) {
    if (batch <= 0 || heads_q <= 0 || n <= 0) return 0;
    return (size_t)batch * heads_q * ((n + TILE - 1) / TILE) * NC * sizeof(float);
}

extern "C" int minf_pattern_recall(const void *q, const void *k, const int64_t *q_stride, const int64_t *k_stride,
                                   int batch, int heads_q, int heads_kv, int n, int head_dim, int dtype,
                                   float sm_scale, const uint8_t *col_flags, const uint8_t *diag_flags,
                                   int64_t flag_pitch, const uint8_t *block_flags, int64_t block_pitch,
                                   int row_begin, float *recall, void *workspace, size_t workspace_bytes,
                                   void *stream) {
    if (!q || !k || !q_stride || !k_stride || !col_flags || !diag_flags || !recall) return MINF_ERR_INVALID_ARG;
    if (batch < 0 || heads_q <= 0 || heads_kv <= 0 || n <= 0 || row_begin < 0) return MINF_ERR_INVALID_ARG;
    if (heads_q % heads_kv != 0) return MINF_ERR_INVALID_ARG;
    if (head_dim != HD) return MINF_ERR_UNSUPPORTED;
    if (dtype != MINF_BF16 && dtype != MINF_F16) return MINF_ERR_UNSUPPORTED;
    if (((uintptr_t)q | (uintptr_t)k) & 15) return MINF_ERR_ALIGNMENT;
    for (int i = 0; i < 3; ++i)
        if ((q_stride[i] | k_stride[i]) & 7) return MINF_ERR_ALIGNMENT;
    const int tiles = (n + TILE - 1) / TILE;
    if (flag_pitch < (int64_t)tiles * TILE || (flag_pitch & 3) || flag_pitch > 0x7fffffffLL) return MINF_ERR_INVALID_ARG;
    if (((uintptr_t)col_flags | (uintptr_t)diag_flags) & 3) return MINF_ERR_ALIGNMENT;
    if (block_flags && block_pitch < (n + KB - 1) / KB) return MINF_ERR_INVALID_ARG;
    if (batch == 0) return MINF_OK;
    const size_t need = minf_pattern_recall_workspace_bytes(batch, heads_q, n);
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 3)) return MINF_ERR_WORKSPACE;

    RecallParams p;
    p.q = (const char *)q;
    p.k = (const char *)k;
    for (int i = 0; i < 3; ++i) {
        p.qs[i] = q_stride[i];
        p.ks[i] = k_stride[i];
    }
    p.batch = batch;
    p.hq = heads_q;
    p.hk = heads_kv;
    p.n = n;
    p.scale_log2 = fabsf(sm_scale) * 1.4426950408889634f;
    p.q_flip = sm_scale < 0.f ? 0x80008000u : 0u;
    p.col = col_flags;
    p.diag = diag_flags;
    p.blk = block_flags;
    p.flag_pitch = flag_pitch;
    p.blk_pitch = block_pitch;
    p.row_begin = row_begin;
    p.tiles = tiles;
    p.partial = (float *)workspace;
    hipStream_t st = (hipStream_t)stream;
    const long long groups = (long long)batch * heads_kv;
    p.stripes = 1;
    while (p.stripes < 8 && groups * p.stripes % 8) p.stripes *= 2;
    const long long per_stripe = ((tiles + 1) / 2 + p.stripes - 1) / p.stripes;
    const long long wgs = (groups * p.stripes * per_stripe * (heads_q / heads_kv) + 7) / 8 * 8;
    if (wgs > 0x7fffffffLL) return MINF_ERR_UNSUPPORTED;
    p.total_wg = (unsigned)wgs;
    const dim3 grid((unsigned)wgs);
    const bool small = (n + KB - 1) / KB <= DIAG_GROUPS_SMALL;
    if (dtype == MINF_BF16 && small)
        hipLaunchKernelGGL((pattern_recall_kernel<__bf16, DIAG_GROUPS_SMALL>), grid, dim3(256), 0, st, p);
    else if (dtype == MINF_BF16)
        hipLaunchKernelGGL((pattern_recall_kernel<__bf16, DIAG_GROUPS>), grid, dim3(256), 0, st, p);
    else if (small)
        hipLaunchKernelGGL((pattern_recall_kernel<_Float16, DIAG_GROUPS_SMALL>), grid, dim3(256), 0, st, p);
    else
        hipLaunchKernelGGL((pattern_recall_kernel<_Float16, DIAG_GROUPS>), grid, dim3(256), 0, st, p);
    int status = minf_launch_status();
    if (status != MINF_OK) return status;
    hipLaunchKernelGGL(pattern_recall_finalize, dim3(batch * heads_q), dim3(64), 0, st, p.partial, tiles, n,
                       row_begin, recall);
    return minf_launch_status();
}

extern "C" int minf_flags_set_indices(const int32_t *idx, int rows, int k, int64_t idx_stride, int bit,
                                      uint8_t *flags, int64_t flag_pitch, int limit, void *stream) {
    if (!idx || !flags || rows < 0 || k < 0 || bit < 0 || bit >= NC || limit < 0) return MINF_ERR_INVALID_ARG;
    if (limit > flag_pitch || (flag_pitch & 3) || ((uintptr_t)flags & 3)) return MINF_ERR_INVALID_ARG;
    if (rows == 0 || k == 0) return MINF_OK;
    hipLaunchKernelGGL(flags_set_indices_kernel, dim3((k + 255) / 256, rows < 65535 ? rows : 65535), dim3(256), 0,
                       (hipStream_t)stream, idx, (long long)idx_stride, rows, k, (unsigned)bit, flags,
                       (long long)flag_pitch, limit);
    return minf_launch_status();
}

extern "C" int minf_flags_set_range(int begin, int end, int rows, int bit, uint8_t *flags, int64_t flag_pitch,
                                    void *stream) {
    if (!flags || rows < 0 || bit < 0 || bit >= NC || begin < 0) return MINF_ERR_INVALID_ARG;
    if (end > flag_pitch || (flag_pitch & 3) || ((uintptr_t)flags & 3)) return MINF_ERR_INVALID_ARG;
    if (rows == 0 || end <= begin) return MINF_OK;
    hipLaunchKernelGGL(flags_set_range_kernel, dim3((end - begin + 255) / 256, rows < 65535 ? rows : 65535),
                       dim3(256), 0, (hipStream_t)stream, begin, end, rows, (unsigned)bit, flags,
                       (long long)flag_pitch);
    return minf_launch_status();
}
