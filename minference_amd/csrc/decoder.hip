// The element-wise passes of a decoder layer around the attention path, one kernel each: residual add +
// RMSNorm, rotary embedding of Q and K in place, SiLU(gate) * up.  (reference minference/patch.py:500-558
// chunked norms, :688-693 chunked MLP; the reference runs them as chains of torch ops.)
//
// All three are bound by the bytes they move.  As torch op chains they went over memory 6, 9 and 5 times
// with fp32 copies in between; values are rounded to the tensor dtype exactly where those chains round
// (the norm before its weight, SiLU before the product, the residual sum before the norm).
// 32768 tokens of 4096 / 14336 wide bf16 rows: add + norm 166 us (6.5 TB/s), rotary embedding of 32 + 8 heads
// 100 us (6.7 TB/s), SiLU * up 450 us (6.3 TB/s), where a large copy reaches 4.6 and a fill 6.8; a two-layer
// prefill of that length went from 44.7 to 36.3 ms.
#include "minf_common.h"
#include <math.h>
#include <type_traits>

namespace {

template <typename T, int W = 16 / (int)sizeof(T)> struct Vec {        // W elements moved by one instruction
    static constexpr int N = W;
    T e[N];
};
template <typename V, typename T> __device__ __forceinline__ V load_vec(const T *p) {
    if constexpr (V::N == 1) return V{{*p}};
    else {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        union { u32x4 u; V v; } x;
        x.u = *reinterpret_cast<const u32x4 *>(p);
        return x.v;
    }
}
template <typename V, typename T> __device__ __forceinline__ void store_vec(T *p, const V &v) {
    if constexpr (V::N == 1) *p = v.e[0];
    else {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        union { u32x4 u; V v; } x;
        x.v = v;
        *reinterpret_cast<u32x4 *>(p) = x.u;
    }
}

// One workgroup per row.  x (+ delta, rounded and written back to x) -> out = round(x * rsqrt(mean(x^2) + eps)) * w.
// fp32 tensors: the sum and its root in fp64, where rounding them shows in the result (relative error against
// fp64 4.3e-8 for rows of 1000 .. 16384; summed in fp32 5.1e-8 .. 5.3e-8, torch's chain 4.8e-8 .. 5.6e-8; 4096 rows
// of 4096 22 us either way).
// V: 16-byte vectors, or single elements for rows that are not whole vectors.  NV of them per thread stay in
// registers between the two passes (0: rows too long for that are read again).
constexpr int RMS_THREADS = 256;
template <typename T, typename V, int NV>
__global__ __launch_bounds__(RMS_THREADS) void rms_norm_kernel(T *__restrict__ x, const T *__restrict__ delta,
                                                               const T *__restrict__ w, T *__restrict__ out, int dim, float eps) {
    typedef typename std::conditional<sizeof(T) == 4, double, float>::type S;
    __shared__ S part[RMS_THREADS / 64];
    const int tid = (int)threadIdx.x;
    constexpr int VN = V::N;
    const long long row = (long long)blockIdx.x * dim;
    const int nvec = dim / VN;
    V keep[NV ? NV : 1];
    S ss = 0;
    auto one = [&](int v) -> V {
        V a = load_vec<V>(x + row + (long long)v * VN);
        if (delta) {
            const V d = load_vec<V>(delta + row + (long long)v * VN);
#pragma unroll
            for (int i = 0; i < VN; ++i) a.e[i] = (T)((float)a.e[i] + (float)d.e[i]);
            store_vec(x + row + (long long)v * VN, a);
        }
#pragma unroll
        for (int i = 0; i < VN; ++i) ss = fma((S)a.e[i], (S)a.e[i], ss);
        return a;
    };
    if constexpr (NV > 0) {
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (j * RMS_THREADS + tid < nvec) keep[j] = one(j * RMS_THREADS + tid);
    } else {
        for (int v = tid; v < nvec; v += RMS_THREADS) one(v);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) ss += __shfl_xor(ss, d);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    S tot = 0;
#pragma unroll
    for (int i = 0; i < RMS_THREADS / 64; ++i) tot += part[i];
    float r;
    if constexpr (sizeof(T) == 4) r = (float)(1.0 / sqrt(tot / dim + (double)eps));
    else r = rsqrtf(tot / (float)dim + eps);
    auto scaled = [&](T a, T wt) -> T { return (T)((float)(T)((float)a * r) * (float)wt); };
    auto finish = [&](int v, const V &a) {
        const V wv = load_vec<V>(w + (long long)v * VN);
        V o;
#pragma unroll
        for (int i = 0; i < VN; ++i) o.e[i] = scaled(a.e[i], wv.e[i]);
        store_vec(out + row + (long long)v * VN, o);
    };
    if constexpr (NV > 0) {
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (j * RMS_THREADS + tid < nvec) finish(j * RMS_THREADS + tid, keep[j]);
    } else {
        for (int v = tid; v < nvec; v += RMS_THREADS) finish(v, load_vec<V>(x + row + (long long)v * VN));   // (each thread what it wrote)
    }
}

// Rotary embedding in place: head rows of Q [tokens, hq, d] and K [tokens, hk, d], pairs (i, i + d/2) turned
// by the token's angle i (cos / sin [tokens, d/2] fp32, read once per token and shared by its heads from cache).
template <typename T>
__global__ __launch_bounds__(256) void rope_kernel(T *__restrict__ q, T *__restrict__ k, const float *__restrict__ cs,
                                                   const float *__restrict__ sn, int hq, int hk, int d, int per_head, unsigned total) {
    const unsigned id = blockIdx.x * 256u + threadIdx.x;       // (32-bit: three 64-bit divisions per 16 bytes would show)
    if (id >= total) return;
    constexpr int VN = Vec<T>::N;
    const int part = (int)(id % (unsigned)per_head);
    const unsigned th = id / (unsigned)per_head;
    const int head = (int)(th % (unsigned)(hq + hk));
    const long long tok = th / (unsigned)(hq + hk);
    const int half = d / 2, i0 = part * VN;
    T *base = head < hq ? q + (tok * hq + head) * d : k + (tok * hk + head - hq) * d;
    const float *c = cs + tok * half + i0, *s = sn + tok * half + i0;
    if (half % VN == 0) {                                 // (uniform: whole vectors, rows 16-byte aligned)
        const Vec<T> a = load_vec<Vec<T>>(base + i0), b = load_vec<Vec<T>>(base + half + i0);
        Vec<T> oa, ob;
#pragma unroll
        for (int i = 0; i < VN; ++i) {
            oa.e[i] = (T)((float)a.e[i] * c[i] - (float)b.e[i] * s[i]);
            ob.e[i] = (T)((float)b.e[i] * c[i] + (float)a.e[i] * s[i]);
        }
        store_vec(base + i0, oa);
        store_vec(base + half + i0, ob);
    } else {
        for (int i = 0; i < VN && i0 + i < half; ++i) {
            const float a = (float)base[i0 + i], b = (float)base[half + i0 + i];
            base[i0 + i] = (T)(a * c[i] - b * s[i]);
            base[half + i0 + i] = (T)(b * c[i] + a * s[i]);
        }
    }
}

template <typename T> __device__ __forceinline__ T silu_times(T g, T u) {
    const float x = (float)g;
    // (expf for the 16-bit types too, the bits of the torch chain for every gate: __expf rounds x log2(e) first, a
    // relative error of |x| 2^-24, and is no faster here, where bytes are the bound: 476 us either way)
    return (T)((float)(T)(x / (1.0f + expf(-x))) * (float)u);
}

// gate <- round(silu(gate)) * up, 16 bytes per thread and step
template <typename T>
__global__ __launch_bounds__(256) void silu_mul_kernel(T *__restrict__ gate, const T *__restrict__ up, long long n) {
    constexpr int VN = Vec<T>::N;
    const long long nvec = n / VN;
    const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
    if (v < nvec) {
        Vec<T> g = load_vec<Vec<T>>(gate + v * VN);
        const Vec<T> u = load_vec<Vec<T>>(up + v * VN);
#pragma unroll
        for (int i = 0; i < VN; ++i) g.e[i] = silu_times(g.e[i], u.e[i]);
        store_vec(gate + v * VN, g);
    } else {
        const long long i = nvec * VN + (v - nvec);
        if (i < n) gate[i] = silu_times(gate[i], up[i]);
    }
}

template <typename F> int with_dtype(int dtype, F f) {
    if (dtype == MINF_BF16) return f((__bf16 *)nullptr);
    if (dtype == MINF_F16) return f((_Float16 *)nullptr);
    if (dtype == MINF_F32) return f((float *)nullptr);
    return MINF_ERR_UNSUPPORTED;
}

}  // namespace

extern "C" int minf_rms_norm(void *x, const void *delta, const void *weight, void *out, int64_t rows, int dim, float eps,
                             int dtype, void *stream) {
    if (!x || !weight || !out || rows < 0 || dim <= 0) return MINF_ERR_INVALID_ARG;
    if (rows == 0) return MINF_OK;
    if (rows > 0x7fffffffLL) return MINF_ERR_UNSUPPORTED;
    const uintptr_t all = (uintptr_t)x | (uintptr_t)delta | (uintptr_t)weight | (uintptr_t)out;
    return with_dtype(dtype, [&](auto *tag) -> int {
        typedef typename std::remove_pointer<decltype(tag)>::type T;
        const dim3 g((unsigned)rows), b(RMS_THREADS);
        hipStream_t st = (hipStream_t)stream;
        T *px = (T *)x, *po = (T *)out;
        const T *pd = (const T *)delta, *pw = (const T *)weight;
        const bool whole = !(all & 15) && dim % Vec<T>::N == 0;
        const int nv = (dim / Vec<T>::N + RMS_THREADS - 1) / RMS_THREADS;
        if (!whole) hipLaunchKernelGGL((rms_norm_kernel<T, Vec<T, 1>, 0>), g, b, 0, st, px, pd, pw, po, dim, eps);
        else if (nv <= 1) hipLaunchKernelGGL((rms_norm_kernel<T, Vec<T>, 1>), g, b, 0, st, px, pd, pw, po, dim, eps);
        else if (nv <= 2) hipLaunchKernelGGL((rms_norm_kernel<T, Vec<T>, 2>), g, b, 0, st, px, pd, pw, po, dim, eps);
        else if (nv <= 4) hipLaunchKernelGGL((rms_norm_kernel<T, Vec<T>, 4>), g, b, 0, st, px, pd, pw, po, dim, eps);
        else hipLaunchKernelGGL((rms_norm_kernel<T, Vec<T>, 0>), g, b, 0, st, px, pd, pw, po, dim, eps);
        return minf_launch_status();
    });
}

extern "C" int minf_rope(void *q, void *k, const float *cos_table, const float *sin_table, int64_t tokens, int heads_q,
                         int heads_kv, int head_dim, int dtype, void *stream) {
    if (!q || !k || !cos_table || !sin_table || tokens < 0 || heads_q <= 0 || heads_kv <= 0 || head_dim <= 0 || head_dim % 2)
        return MINF_ERR_INVALID_ARG;
    if (((uintptr_t)q | (uintptr_t)k) & 15) return MINF_ERR_ALIGNMENT;
    if (tokens == 0) return MINF_OK;
    return with_dtype(dtype, [&](auto *tag) -> int {
        typedef typename std::remove_pointer<decltype(tag)>::type T;
        const int per_head = (head_dim / 2 + Vec<T>::N - 1) / Vec<T>::N;
        const long long total = tokens * (heads_q + heads_kv) * per_head, grid = (total + 255) / 256;
        if (total > 0xffffff00LL) return MINF_ERR_UNSUPPORTED;
        hipLaunchKernelGGL((rope_kernel<T>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, (T *)q, (T *)k,
                           cos_table, sin_table, heads_q, heads_kv, head_dim, per_head, (unsigned)total);
        return minf_launch_status();
    });
}

extern "C" int minf_silu_mul(void *gate, const void *up, int64_t n, int dtype, void *stream) {
    if (!gate || !up || n < 0) return MINF_ERR_INVALID_ARG;
    if (((uintptr_t)gate | (uintptr_t)up) & 15) return MINF_ERR_ALIGNMENT;
    if (n == 0) return MINF_OK;
    return with_dtype(dtype, [&](auto *tag) -> int {
        typedef typename std::remove_pointer<decltype(tag)>::type T;
        const long long grid = (n / Vec<T>::N + n % Vec<T>::N + 255) / 256;
        if (grid > 0x7fffffffLL) return MINF_ERR_UNSUPPORTED;
        hipLaunchKernelGGL((silu_mul_kernel<T>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, (T *)gate, (const T *)up, (long long)n);
        return minf_launch_status();
    });
}
