/* lg_fgemm.h -- token GEMMs of F16 weights and fp32 activations on fp16 MFMA
 * (lg_fgemm.hip), shared by the BERT encoder and the batched prefill. */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

/* epilogues; STORE / ADD: no bias; ADD: out +=; BIAS_GELU_SPLIT: BIAS_GELU
 * with its values split for the next F16 GEMM (lg_hgemm only) */
enum { EP_BIAS = 0, EP_BIAS_RES = 1, EP_BIAS_GELU = 2, EP_BIAS_GELU_SPLIT = 3, EP_STORE = 4, EP_ADD = 5 };

/* Split activations of T tokens of K values (a multiple of 32): each fp32
 * value times its token's power of two 1 / inv[t] as fp16 hi (rounded toward
 * zero) and lo = fp16 of the rest, laid out [t][K / 32][hi 32 | lo 32].  The
 * power puts the token's largest finite |x|, or a bound of it, in [2^14,
 * 2^15).  inv NULL: every token's is inv_all. */
struct HSplit {
    _Float16* h;
    float* inv;
    float inv_all;
};

struct BGemm {
    const uint8_t* w;          /* F16 (lg_hgemm), F32: [R][K]; BF_I8: int8 [R][K] */
    const float* wd;           /* BF_I8: [K/32][R] */
    int R, K;
    const float* x;            /* fp32 activations [T][ldx] (F32) */
    int ldx;
    const int8_t* q;           /* Q8_0 activations [T][K] (BF_I8) */
    const float* qd;           /* [K/32][ldd] */
    int ldd;
    int T;
    const float* bias;         /* [R] */
    const float* res;          /* [T][ldr] residual (EP_BIAS_RES) */
    int ldr;
    float* out;                /* [T][ldo] */
    int ldo;
    HSplit so;                 /* EP_BIAS_GELU_SPLIT: the output, R values a token (a multiple of 32), inv_all a power of two */
};

/* bytes of h for T tokens of K values (as many as the fp32 rows) */
static inline size_t lg_hsplit_bytes(int T, int K) { return (size_t)T * K * 4; }

int lg_hsplit(const float* x, int ldx, int K, int T, const HSplit& o, hipStream_t s);

/* out[t][r] (ep) W[r] . x[t] for F16 W [R][K] (K a multiple of 32) and split
 * x; a.x is not read */
int lg_hgemm(const BGemm& a, const HSplit& x, int ep, hipStream_t s);

#ifdef __HIPCC__
/* k of a token's scale 2^k from its largest finite |x| (0: any) */
__host__ __device__ __forceinline__ int lg_split_exp(float amax)
{
    const int k = 141 - (int)(__builtin_bit_cast(uint32_t, amax) >> 23);   /* amax 2^k in [2^14, 2^15) */
    return k > 126 ? 126 : k;                                               /* both 2^k and 2^-k normal */
}

__host__ __device__ __forceinline__ float lg_pow2(int k) { return __builtin_bit_cast(float, (uint32_t)(127 + k) << 23); }

/* 1 / x of a power of two whose reciprocal is normal too */
__host__ __device__ __forceinline__ float lg_recip_pow2(float x)
{
    return __builtin_bit_cast(float, 0x7f000000u - __builtin_bit_cast(uint32_t, x));
}

/* ---- device side of the split, for the kernels that produce activations ---- */

/* |x| for the maximum: infinities and NaN take no part */
__device__ __forceinline__ float lg_finite_abs(float x)
{
    const float a = fabsf(x);
    return a < INFINITY ? a : 0.0f;
}

typedef _Float16 lg_h2 __attribute__((ext_vector_type(2)));

/* two values into hi and lo (packed halves).  hi rounds toward zero, so lo
 * has x's sign, and a part that would be zero under a nonzero x becomes the
 * smallest fp16 of that sign (2^-39 of the token's largest): an infinite
 * weight then gives hi W + lo W = the infinity that x W is, never inf - inf
 * or inf 0.  An infinite x keeps hi infinite; NaN stays NaN. */
__device__ __forceinline__ uint32_t lg_nonzero_half(uint32_t h, float v)
{
    return (h & 0x7fffu) || v == 0.0f ? h : h | 1u | ((__float_as_uint(v) >> 16) & 0x8000u);
}

__device__ __forceinline__ void lg_split2(float x0, float x1, float s, uint32_t& hi, uint32_t& lo)
{
    const float v0 = x0 * s, v1 = x1 * s;
    const auto h = __builtin_amdgcn_cvt_pkrtz(v0, v1);
    const float r0 = v0 - (float)h[0], r1 = v1 - (float)h[1];   /* NaN for an infinite x */
    const lg_h2 l = {(_Float16)(r0 == r0 ? r0 : 0.0f), (_Float16)(r1 == r1 ? r1 : 0.0f)};
    const uint32_t hb = __builtin_bit_cast(uint32_t, h), lb = __builtin_bit_cast(uint32_t, l);
    hi = lg_nonzero_half(hb & 0xffffu, v0) | (lg_nonzero_half(hb >> 16, v1) << 16);
    lo = lg_nonzero_half(lb & 0xffffu, v0) | (lg_nonzero_half(lb >> 16, v1) << 16);
}

/* one value: hi in the low half, lo in the high half */
__device__ __forceinline__ uint32_t lg_split1(float x, float s)
{
    uint32_t hi, lo;
    lg_split2(x, 0.0f, s, hi, lo);
    return (hi & 0xffffu) | (lo << 16);
}

/* gelu (fast/lil_math.cpp:978-984) */
__device__ __forceinline__ float lg_gelu(float g)
{
    return 0.5f * g * (1.0f + tanhf(0.7978845608f * (g + 0.044715f * g * g * g)));
}

/* four values i .. i + 3 (i a multiple of 4) of token t into the split rows */
__device__ __forceinline__ void lg_split_store4(const float v[4], float s, const HSplit& o, int K, int t, int i)
{
    uint2 hi, lo;
    lg_split2(v[0], v[1], s, hi.x, lo.x);
    lg_split2(v[2], v[3], s, hi.y, lo.y);
    _Float16* p = o.h + (size_t)t * 2 * K + (size_t)(i >> 5) * 64 + (i & 31);
    *(uint2*)p = hi;
    *(uint2*)(p + 32) = lo;
}
#endif
