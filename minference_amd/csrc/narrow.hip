// fp32 tensors on 16-bit matrix operands, without a host read in between.
//
// The attention kernels compute on 16-bit operands with fp32 accumulation (the reference picks fp16 operands for
// every input that is not bf16, pit_sparse_flash_attention_v2.py:175).  fp32 q/k/v become fp16 when the
// largest |value| of the three lies in [2^-10, 32768], else bf16 (fp16 would overflow, or flush most of
// the tensor).  The choice is made here, on the device: a first kernel converts, to fp16 or, in large tensors, to the
// format that one or two rows of each ask for, and leaves the largest |value| of each of its workgroups, every workgroup of
// the second one folds those, one of them leaves the dtype code that the attention launches and the widening kernel
// read (minf_qkvo.dtype_select), and where the code is not the format written they convert once more, over what the first
// kernel wrote.  Bound by bytes: q, k and v are read and written once.
// With a pass for the largest |value| alone before the conversion (8192 tokens, 4 heads of 128, 3 x 16.8 MB)
// the two took 22.2 us, now 15.1; 32768 tokens, 16 heads 363 -> 223, 65536 tokens, 32 / 8 heads 741 -> 447, 5.4 TB/s.
// Tensors that need bf16 took, with that pass, converted to fp16 whatever the values, and sampled first: 8192 tokens, 4
// heads 22.2, 26.8, 15.7 us, 14 heads 65.5, 78.3, 44, 32 / 8 heads 75.7, 122, 53.4, 32768 tokens, 16 heads 366, 451, 223,
// 65536 tokens, 32 / 8 heads 744, 1007, 448.  The sample lengthens a call by one to two microseconds all the same (it is on its
// way behind the first step's loads, at addresses from the host; operator, 5000 tokens, 8 / 2 heads, 123.9 -> 125.8, two times
// 1427 tokens, 28 / 4 heads, 100.4 -> 101.8), so smaller tensors, which lose 4 to 13 to the second conversion, go without.  Where it does not show what the tensors ask for, one value
// above 32768, they are converted twice: 102, 443 and 886 us.
// With the choice read back by the host (three reductions, a synchronisation, three conversions) the GPU
// idled about 60 us per call.
#include "minf_common.h"

namespace {

constexpr int NARROW_THREADS = 256;
constexpr int UNDER_WAY = 2;     // steps of 8 elements a thread has under way
constexpr int NARROW_PARTIALS = MINF_NARROW_WORKSPACE_INTS - 1;      // workgroups of a launch, a third per tensor
constexpr int NARROW_WGS = NARROW_PARTIALS / 3;
constexpr long long SAMPLED_FROM = 1 << 21;      // vectors of the largest tensor
static_assert(NARROW_WGS * 3 == NARROW_PARTIALS, "the same number of workgroups for each tensor");

struct NarrowTensor {
    const float *in;
    char *out;                   // [batch, heads, n, dim_out] 16-bit, contiguous
    long long stride[3];         // elements: batch, head, token
    long long rows;              // batch * heads * n
    int heads;
    const float *sample;         // the rows that are looked at first: the first one, elements from one to the next
    long long sample_step;
    FastDiv by_n, by_heads;
};
struct NarrowParams {
    NarrowTensor t[3];
    int dim, sampled, lanes_log2;      // whether rows are looked at first, lanes that read one
    FastDiv by_dim_out;          // vectors of 8 elements per output row
    int *ws;                     // [0]: the dtype code, then the partial maxima (bit patterns)
};

// (I: 32-bit numbers of vectors wherever they fit, placed by multiplications; else 64-bit ones, placed by divisions)
__device__ __forceinline__ unsigned quot(unsigned x, const FastDiv &f) { return fast_quot(x, f); }
__device__ __forceinline__ unsigned long long quot(unsigned long long x, const FastDiv &f) { return x / f.d; }

// where vector i of a row-wise walk of a tensor lies, `width` elements per vector
template <typename I> __device__ __forceinline__ const float *vector_ptr(const NarrowTensor &t, const FastDiv &per_row, int width, I i, int &d) {
    const I row = quot(i, per_row), bh = quot(row, t.by_n), b = quot(bh, t.by_heads);
    d = width * (int)(i - row * per_row.d);
    return t.in + (long long)b * t.stride[0] + (long long)(bh - b * t.by_heads.d) * t.stride[1] + (long long)(row - bh * t.by_n.d) * t.stride[2] + d;
}

// largest bit pattern of |x| (NaN above infinity above every number) over the workgroup, in thread 0 .. 255
__device__ __forceinline__ unsigned wg_max(unsigned m, unsigned (&part)[NARROW_THREADS / 64]) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) m = max(m, (unsigned)__shfl_xor((int)m, s));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NARROW_THREADS / 64; ++w) m = max(m, part[w]);
    return m;
}

// bit patterns of the largest and smallest |x| that a tensor's largest may be for fp16
constexpr unsigned MOST_F16 = 0x47000000u, LEAST_F16 = 0x3a800000u;      // 32768, 2^-10

// Loads of one step: UNDER_WAY vectors of 8 elements from number i on.
template <typename I> struct Step {
    float4 x[UNDER_WAY][2];
    I at[UNDER_WAY];
};
template <typename I> __device__ __forceinline__ void load_step(const NarrowParams &p, const NarrowTensor &t, I i, I total, Step<I> &s) {
    const I step = (I)NARROW_WGS * NARROW_THREADS;
#pragma unroll
    for (int u = 0; u < UNDER_WAY; ++u) {
        s.at[u] = min(i + u * step, total - 1);        // (the last vector again, past the end)
        int d;
        const float *src = vector_ptr<I>(t, p.by_dim_out, 8, s.at[u], d);
#pragma unroll
        for (int h = 0; h < 2; ++h) s.x[u][h] = d + 4 * h < p.dim ? *reinterpret_cast<const float4 *>(src + 4 * h) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}
// converted to T and written; -> the largest bit pattern of |x| read, or m
template <typename T, typename I> __device__ __forceinline__ unsigned store_step(const NarrowTensor &t, const Step<I> &s, unsigned m) {
#pragma unroll
    for (int u = 0; u < UNDER_WAY; ++u) {
        const float v[8] = {s.x[u][0].x, s.x[u][0].y, s.x[u][0].z, s.x[u][0].w, s.x[u][1].x, s.x[u][1].y, s.x[u][1].z, s.x[u][1].w};
        union { T e[8]; uint4 u4; } o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            o.e[e] = (T)v[e];
            m = max(m, __float_as_uint(v[e]) & 0x7fffffffu);
        }
        *reinterpret_cast<uint4 *>(t.out + (long long)s.at[u] * 16) = o.u4;
    }
    return m;
}

// One pass over a workgroup's share of a tensor from number i on, the step at i loaded; the largest bit pattern of |x| read.
template <typename T, typename I> __device__ __forceinline__ unsigned convert_share(const NarrowParams &p, const NarrowTensor &t, I i, I total, Step<I> &s) {
    unsigned m = 0;
    while (i < total) {
        m = store_step<T, I>(t, s, m);
        i += (I)UNDER_WAY * NARROW_WGS * NARROW_THREADS;
        if (i < total) load_step<I>(p, t, i, total, s);
    }
    return m;
}

// The sampled rows of each tensor (their first 256 values, a vector per lane), and whether they ask for fp16: the same answer
// in every wavefront.
struct Sample { uint4 x[3]; };
__device__ __forceinline__ Sample load_sample(const NarrowParams &p) {
    Sample s;
    const int lane = minf_lane(), d = 4 * min(lane & ((1 << p.lanes_log2) - 1), p.dim / 4 - 1);
#pragma unroll
    for (int i = 0; i < 3; ++i) s.x[i] = *reinterpret_cast<const uint4 *>(p.t[i].sample + (lane >> p.lanes_log2) * p.t[i].sample_step + d);
    return s;
}
__device__ __forceinline__ bool takes_f16(const Sample &s) {
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        m = max(max(max(m, s.x[i].x & 0x7fffffffu), s.x[i].y & 0x7fffffffu), max(s.x[i].z & 0x7fffffffu, s.x[i].w & 0x7fffffffu));
    return __any(m >= LEAST_F16) && !__any(m > MOST_F16);
}

// leaves the largest bit pattern it read, with the sign bit where it wrote bf16
template <typename I> __global__ __launch_bounds__(NARROW_THREADS) void narrow_kernel(const NarrowParams p) {
    __shared__ unsigned part[NARROW_THREADS / 64];
    const NarrowTensor &t = p.t[blockIdx.y];
    const I total = (I)t.rows * p.by_dim_out.d, i = (I)blockIdx.x * NARROW_THREADS + threadIdx.x;
    Step<I> s;
    load_step<I>(p, t, min(i, total - 1), total, s);                     // (under way before the sample is looked at)
    const bool f16 = !p.sampled || takes_f16(load_sample(p));
    const unsigned m = wg_max(f16 ? convert_share<_Float16, I>(p, t, i, total, s) : convert_share<__bf16, I>(p, t, i, total, s), part);
    if (threadIdx.x == 0) p.ws[1 + blockIdx.y * NARROW_WGS + blockIdx.x] = (int)(f16 ? m : m | 0x80000000u);
}

template <typename I> __global__ __launch_bounds__(NARROW_THREADS) void narrow_choose_kernel(const NarrowParams p) {
    __shared__ unsigned part[NARROW_THREADS / 64];
    unsigned m = 0;
    for (int i = (int)threadIdx.x; i < NARROW_PARTIALS; i += NARROW_THREADS) m = max(m, (unsigned)p.ws[1 + i] & 0x7fffffffu);
    const bool is_f16 = p.ws[1] >= 0;
    m = wg_max(m, part);
    const bool f16 = m >= LEAST_F16 && m <= MOST_F16;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) p.ws[0] = f16 ? MINF_F16 : MINF_BF16;
    if (f16 == is_f16) return;
    const NarrowTensor &t = p.t[blockIdx.y];
    const I total = (I)t.rows * p.by_dim_out.d, i = (I)blockIdx.x * NARROW_THREADS + threadIdx.x;
    Step<I> s;
    if (i < total) load_step<I>(p, t, i, total, s);
    if (f16) convert_share<_Float16, I>(p, t, i, total, s);
    else convert_share<__bf16, I>(p, t, i, total, s);
}

__global__ __launch_bounds__(NARROW_THREADS) void widen_kernel(const char *__restrict__ in, float *__restrict__ out, long long rows,
                                                              int dim, int dim_in, const int *__restrict__ code) {
    const bool f16 = *code == MINF_F16;
    const unsigned per_row = (unsigned)dim / 4u;
    const long long total = rows * per_row;
    for (long long i = (long long)blockIdx.x * NARROW_THREADS + threadIdx.x; i < total; i += (long long)gridDim.x * NARROW_THREADS) {
        const long long row = i / per_row;
        const int d = 4 * (int)(i - row * per_row);
        union { _Float16 h[4]; __bf16 b[4]; uint2 u; } x;
        x.u = *reinterpret_cast<const uint2 *>(in + (row * dim_in + d) * 2);
        float4 o;
        if (f16) o = make_float4((float)x.h[0], (float)x.h[1], (float)x.h[2], (float)x.h[3]);
        else o = make_float4((float)x.b[0], (float)x.b[1], (float)x.b[2], (float)x.b[3]);
        *reinterpret_cast<float4 *>(out + i * 4) = o;
    }
}

unsigned narrow_grid(long long vectors) {
    const long long wgs = (vectors + 4 * NARROW_THREADS - 1) / (4 * NARROW_THREADS);
    return (unsigned)(wgs < 1 ? 1 : (wgs > 2048 ? 2048 : wgs));
}

}  // namespace

extern "C" int minf_narrow_qkv(const minf_qkvo *t, int dim_in, void *q16, void *k16, void *v16, int32_t *workspace, void *stream) {
    if (!t || !t->q || !t->k || !t->v || !q16 || !k16 || !v16 || !workspace) return MINF_ERR_INVALID_ARG;
    if (t->batch <= 0 || t->heads_q <= 0 || t->heads_kv <= 0 || t->n <= 0 || dim_in <= 0 || t->head_dim < dim_in) return MINF_ERR_INVALID_ARG;
    if ((dim_in & 3) || (t->head_dim & 7)) return MINF_ERR_ALIGNMENT;
    if ((long long)t->batch * t->heads_q > 0x7fffffffLL) return MINF_ERR_UNSUPPORTED;
    NarrowParams p;
    const void *in[3] = {t->q, t->k, t->v};
    void *out[3] = {q16, k16, v16};
    const int64_t *strides[3] = {t->q_stride, t->k_stride, t->v_stride};
    p.dim = dim_in;
    p.lanes_log2 = 0;
    while (p.lanes_log2 < 6 && 4 << p.lanes_log2 < dim_in) ++p.lanes_log2;
    for (int i = 0; i < 3; ++i) {
        if ((((uintptr_t)in[i]) | ((uintptr_t)out[i])) & 15) return MINF_ERR_ALIGNMENT;
        for (int j = 0; j < 3; ++j) {
            if (strides[i][j] < 0 || (strides[i][j] & 3)) return MINF_ERR_ALIGNMENT;
            p.t[i].stride[j] = strides[i][j];
        }
        p.t[i].in = (const float *)in[i];
        p.t[i].out = (char *)out[i];
        p.t[i].heads = i == 0 ? t->heads_q : t->heads_kv;
        p.t[i].rows = (long long)t->batch * p.t[i].heads * t->n;
        // as many rows as a wavefront holds: the middle head's tokens, evenly spread from the middle one to the last
        const long long head = (long long)t->batch * p.t[i].heads / 2, sampled = 64ll >> p.lanes_log2;
        p.t[i].sample = p.t[i].in + head / p.t[i].heads * strides[i][0] + head % p.t[i].heads * strides[i][1] + t->n / 2 * strides[i][2];
        p.t[i].sample_step = sampled > 1 ? (t->n - 1 - t->n / 2) / (sampled - 1) * strides[i][2] : 0;
        p.t[i].by_n = fast_div((unsigned)t->n);
        p.t[i].by_heads = fast_div((unsigned)p.t[i].heads);
    }
    p.by_dim_out = fast_div((unsigned)t->head_dim / 8u);
    p.ws = workspace;
    hipStream_t st = (hipStream_t)stream;
    // (multiplications place numbers below 2^31, and so must the steps past the end be)
    const long long most = p.t[0].rows > p.t[1].rows ? p.t[0].rows : p.t[1].rows;
    p.sampled = most * p.by_dim_out.d >= SAMPLED_FROM;
    const bool small = most * p.by_dim_out.d < 0x7fffffffLL - 2ll * UNDER_WAY * NARROW_WGS * NARROW_THREADS;
    const dim3 grid(NARROW_WGS, 3), block(NARROW_THREADS);
    if (small) hipLaunchKernelGGL(narrow_kernel<unsigned>, grid, block, 0, st, p);
    else hipLaunchKernelGGL(narrow_kernel<unsigned long long>, grid, block, 0, st, p);
    const int status = minf_launch_status();
    if (status != MINF_OK) return status;
    if (small) hipLaunchKernelGGL(narrow_choose_kernel<unsigned>, grid, block, 0, st, p);
    else hipLaunchKernelGGL(narrow_choose_kernel<unsigned long long>, grid, block, 0, st, p);
    return minf_launch_status();
}

extern "C" int minf_widen_out(const void *o16, float *out, int64_t rows, int dim, int dim_in, const int32_t *dtype_code, void *stream) {
    if (rows < 0 || dim <= 0 || dim_in < dim) return MINF_ERR_INVALID_ARG;
    if (rows == 0) return MINF_OK;
    if (!o16 || !out || !dtype_code) return MINF_ERR_INVALID_ARG;
    if ((dim & 3) || (dim_in & 3) || ((uintptr_t)o16 & 15) || ((uintptr_t)out & 15)) return MINF_ERR_ALIGNMENT;
    hipLaunchKernelGGL(widen_kernel, dim3(narrow_grid(rows * (dim / 4))), dim3(NARROW_THREADS), 0, (hipStream_t)stream,
                       (const char *)o16, out, (long long)rows, dim, dim_in, dtype_code);
    return minf_launch_status();
}
