/* lg_fgemm.hip -- token GEMMs of F16 weights and fp32 activations on fp16
 * MFMA: out[t][r] = W[r] . x[t] (dot_f16_f32, fast/lil_math.cpp:403-409, for
 * many tokens at once).
 *
 * The fp32 MFMA multiplies at 157 TFLOP/s, the fp16 one at 2.5 PFLOP/s, and
 * the weights are fp16 already: each activation goes in as two fp16 parts
 * (HSplit in lg_fgemm.h: 22 bits of it), so x W = hi W + lo W with every
 * product exact and fp32 accumulation.  Against 64 bits the sums come out
 * closer than the fp32 MFMA's, whose longer chain of roundings weighs more
 * than the two bits (see the test). */
#include <math.h>

#include <algorithm>

#include "lg_common.h"
#include "lg_fgemm.h"

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));

/* token t = blockIdx.x: largest finite |x|, then the split row */
__global__ __launch_bounds__(256) void k_hsplit(const float* __restrict__ x, int ldx, int K, HSplit o)
{
    __shared__ float s_m[4];
    const int t = blockIdx.x, tid = threadIdx.x;
    const float* xr = x + (size_t)t * ldx;
    float m = 0.0f;
    for (int i = 4 * tid; i < K; i += 1024) {
        const float4 v = *(const float4*)(xr + i);
        m = fmaxf(m, fmaxf(fmaxf(lg_finite_abs(v.x), lg_finite_abs(v.y)), fmaxf(lg_finite_abs(v.z), lg_finite_abs(v.w))));
    }
    m = lg_wave_max_nn(m);
    if ((tid & 63) == 0) s_m[tid >> 6] = m;
    __syncthreads();
    const int k = lg_split_exp(fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3])));
    const float s = lg_pow2(k);
    if (tid == 0) o.inv[t] = lg_pow2(-k);
    for (int i = 4 * tid; i < K; i += 1024) {
        const float4 f = *(const float4*)(xr + i);
        const float v[4] = {f.x, f.y, f.z, f.w};
        lg_split_store4(v, s, o, K, t, i);
    }
}

int lg_hsplit(const float* x, int ldx, int K, int T, const HSplit& o, hipStream_t s)
{
    hipLaunchKernelGGL(k_hsplit, dim3(T), dim3(256), 0, s, x, ldx, K, o);
    return lg_check_launch("activation split");
}

/* one output: the sum `acc` of token t (t >= T: not stored) and weight row
 * `row`; the lanes of a 32-lane half hold consecutive rows */
template <int EP>
__device__ __forceinline__ void hg_emit(const BGemm& a, float acc, float inv, float bias, int t, int row)
{
    const float o = acc * inv;
    if constexpr (EP == EP_BIAS_GELU_SPLIT) {
        /* a lane and its neighbour hold two rows of a token: the even one
         * stores both high parts, the odd one both low ones */
        const uint32_t w = lg_split1(lg_gelu(o + bias), lg_recip_pow2(a.so.inv_all));
        const uint32_t n = (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0xb1, 0xf, 0xf, true);   /* lane ^ 1 */
        const int odd = row & 1;
        uint32_t* p = (uint32_t*)(a.so.h + (size_t)(row >> 5) * 64 + (row & 30) + 32 * odd);
        if (t < a.T) p[(size_t)t * a.R] = odd ? (n >> 16) | (w & 0xffff0000u) : (w & 0xffffu) | (n << 16);
        return;
    }
    if (t >= a.T) return;
    float* p = a.out + (size_t)t * a.ldo + row;
    if constexpr (EP == EP_STORE) *p = o;
    else if constexpr (EP == EP_ADD) *p = *p + o;
    else if constexpr (EP == EP_BIAS) *p = o + bias;
    else if constexpr (EP == EP_BIAS_RES) *p = o + (bias + a.res[(size_t)t * a.ldr + row]);
    else *p = lg_gelu(o + bias);
}

/* A workgroup computes 32 MR WR weight rows x 32 MT WT tokens: WR x WT waves
 * of MR x MT tiles of 32 x 32 (v_mfma_f32_32x32x16_f16, A = tokens, B =
 * weight rows: lane l holds token / row l % 32, values 8 (l / 32) .. +7 of a
 * 16-value step), and WK groups of such waves take consecutive parts of K
 * with stages of their own, summed in group order through LDS at the end,
 * where each group finishes its share of the tile.  With one group doing that
 * alone, and loads past a short part waited for, the 32 x 32 tile took 2 to 3
 * us longer (128 x 512 with GELU, 120 tokens: 7.7 -> 4.5; the fp32 MFMA, which
 * small models ran on before, 4.2).
 *
 * Per step of 32 values both operands go through LDS, double-buffered, a
 * step's loads in flight while the two steps before compute (one step ahead
 * 240 instead of 229 us at 24576 x 4096, 500 tokens).  A row's 32 weights are four 16-byte pieces, a token's hi and lo
 * eight; piece p of row or token j lies in the 1 KiB fragment (32 rows x 16
 * values) it belongs to at lane slot 32 (p % 2) + (j ^ swz(p)): the 8
 * threads that store a row's pieces hit 8 different 16-byte bank groups, and
 * so do the lanes that read a fragment.
 *
 * What bounds it: 128 x 128 with 64 x 64 per wave reads 96 bytes of LDS a
 * clock of the 128 possible at full MFMA rate and writes 48, so LDS holds it
 * below ~70 % of that rate; 256 x 128 reads less but one workgroup of it a
 * CU hides less of the loads' latency (267 against 229 us). */
template <int MR, int MT, int WR, int WT, int WK, int EP>
__global__ __launch_bounds__(64 * WR * WT * WK) __attribute__((amdgpu_waves_per_eu(2))) void k_hgemm(BGemm a, HSplit x)
{
    constexpr int TR = 32 * MR * WR, TT = 32 * MT * WT, NG = 64 * WR * WT;
    constexpr int WB = TR * 64, XB = TT * 128, SB = WB + XB;   /* bytes of a stage */
    constexpr int NW = TR * 4 / NG, NX = TT * 8 / NG;          /* pieces per thread */
    static_assert(NW * NG == TR * 4 && NX * NG == TT * 8, "whole pieces");
    __shared__ __attribute__((aligned(16))) uint8_t s_st[WK][2][SB];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kg = WK == 1 ? wave / (WR * WT) : __builtin_amdgcn_readfirstlane(wave / (WR * WT)), wr = wave % (WR * WT) / WT, wt = wave % WT, gt = threadIdx.x % NG;
    const int h = lane >> 5, j = lane & 31;
    const int nt = (a.T + TT - 1) / TT;
    /* the token tiles of a row block on one XCD, 8 indices apart: its
     * weights come from HBM once */
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int rb = (slot / nt) * 8 + xcd;
    if (rb * TR >= a.R) return;   /* padding of the row blocks (whole workgroup) */
    const int r0 = rb * TR, t0 = (slot % nt) * TT;
    const int ns = a.K >> 5, nsg = (ns + WK - 1) / WK;
    const int k0 = kg * nsg, kn = min(nsg, ns - k0);   /* this group's steps (kn may be <= 0) */

    uint8_t(*st)[SB] = s_st[kg];
    const uint8_t* wp[NW];
    const uint8_t* xp[NX];
    int ws[NW], xs[NX];
#pragma unroll
    for (int u = 0; u < NW; u++) {
        const int q = gt + NG * u, r = q >> 2, p = q & 3;
        wp[u] = a.w + (size_t)min(r0 + r, a.R - 1) * a.K * 2 + 16 * p;
        ws[u] = ((r >> 5) * 2 + (p >> 1)) * 1024 + (32 * (p & 1) + ((r & 31) ^ (2 * p))) * 16;
    }
#pragma unroll
    for (int u = 0; u < NX; u++) {
        const int q = gt + NG * u, t = q >> 3, p = q & 7;
        xp[u] = (const uint8_t*)x.h + (size_t)min(t0 + t, a.T - 1) * a.K * 4 + 16 * p;
        xs[u] = WB + ((t >> 5) * 4 + (p >> 1)) * 1024 + (32 * (p & 1) + ((t & 31) ^ p)) * 16;
    }
    struct Stg {
        v4i w[NW], x[NX];
    };
    auto load = [&](Stg& s, int i) __attribute__((always_inline)) {
        const int k = max(min(k0 + i, ns - 1), 0);
#pragma unroll
        for (int u = 0; u < NW; u++) s.w[u] = *(const v4i*)(wp[u] + (size_t)k * 64);
#pragma unroll
        for (int u = 0; u < NX; u++) s.x[u] = *(const v4i*)(xp[u] + (size_t)k * 128);
    };
    auto store = [&](const Stg& s, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NW; u++) *(v4i*)(st[buf] + ws[u]) = s.w[u];
#pragma unroll
        for (int u = 0; u < NX; u++) *(v4i*)(st[buf] + xs[u]) = s.x[u];
    };
    v16f acc[MR][MT];
#pragma unroll
    for (int i = 0; i < MR; i++)
#pragma unroll
        for (int u = 0; u < MT; u++) acc[i][u] = (v16f){};
    auto compute = [&](int buf) __attribute__((always_inline)) {
        const uint8_t* sw = st[buf] + wr * MR * 2048;
        const uint8_t* sx = st[buf] + WB + wt * MT * 4096;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            v8h wf[MR];
#pragma unroll
            for (int i = 0; i < MR; i++)
                wf[i] = *(const v8h*)(sw + i * 2048 + s * 1024 + (32 * h + (j ^ (4 * s + 2 * h))) * 16);
#pragma unroll
            for (int u = 0; u < MT; u++) {
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const v8h xf = *(const v8h*)(sx + u * 4096 + (2 * p + s) * 1024 + (32 * h + (j ^ (4 * p + 2 * s + h))) * 16);
#pragma unroll
                    for (int i = 0; i < MR; i++)
                        acc[i][u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf, wf[i], acc[i][u], 0, 0, 0);
                }
            }
        }
    };

    /* the encoder's products add the same four parts of K in the same order
     * in every tile, so that a text's embedding has the same bits alone and
     * in a batch */
    constexpr bool PO = EP <= EP_BIAS_GELU_SPLIT && WK == 1;
    static_assert(EP > EP_BIAS_GELU_SPLIT || WK == 1 || WK == 4, "four parts");
    v16f tot[PO ? MR : 1][PO ? MT : 1];
    const int np = (ns + 3) / 4;
    int next = np;
#pragma unroll
    for (int m = 0; m < (PO ? MR : 1); m++)
#pragma unroll
        for (int u = 0; u < (PO ? MT : 1); u++) tot[m][u] = (v16f){};
    auto part = [&](int i) __attribute__((always_inline)) {
        if (i != next) return;
        next += np;
#pragma unroll
        for (int m = 0; m < (PO ? MR : 1); m++)
#pragma unroll
            for (int u = 0; u < (PO ? MT : 1); u++) {
                tot[m][u] += acc[m][u];
                acc[m][u] = (v16f){};
            }
    };

    Stg s0, s1;
    load(s0, 0);
    load(s1, 1);
    store(s0, 0);
    __syncthreads();
    int i = 0;
    for (; i < (WK == 4 ? nsg - 3 : nsg); i += 2) {
        load(s0, i + 2);
        if (PO) part(i);
        if (i < kn) compute(0);
        store(s1, 1);
        __syncthreads();
        load(s1, i + 3);
        if (PO) part(i + 1);
        if (i + 1 < kn) compute(1);
        store(s0, 0);
        __syncthreads();
    }
    if constexpr (WK == 4) {
        /* the last one to three steps: where a group has only a handful, no load
         * past the last is waited for */
        if (i + 2 < nsg) load(s0, i + 2);
        if (i < kn) compute(0);
        if (i + 1 < nsg) {
            store(s1, 1);
            __syncthreads();
            if (i + 1 < kn) compute(1);
            if (i + 2 < nsg) {
                store(s0, 0);
                __syncthreads();
                if (i + 2 < kn) compute(0);
            }
        }
        __syncthreads();
    }
    if constexpr (PO) {
#pragma unroll
        for (int i = 0; i < MR; i++)
#pragma unroll
            for (int u = 0; u < MT; u++) acc[i][u] = tot[i][u] + acc[i][u];
    }
    /* Each group ends up with 1 / WK of the tile's registers: it gives the others
     * theirs through LDS (all stages are consumed), adds its own groups' in
     * order, and finishes those -- the epilogue's work on all waves, not on
     * one group's */
    constexpr int NR = MR * MT * 16, NP = NR / WK;
    static_assert(NR % WK == 0, "a part each");
    float* const red = (float*)s_st;   /* [group][register][thread] */
    if constexpr (WK > 1) {
        static_assert(WK * NR * NG * 4 <= (int)sizeof(s_st), "the groups' sums fit the stages");
#pragma unroll
        for (int f = 0; f < NR; f++)
            if (f / NP != kg) red[(kg * NR + f) * NG + gt] = acc[f / 16 / MT][f / 16 % MT][f % 16];
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < WK; c++) {
        if (WK > 1 && c != kg) continue;   /* (wave-uniform; the registers are named at compile time) */
#pragma unroll
        for (int u = 0; u < MT; u++) {
            const int tb = t0 + (wt * MT + u) * 32 + 4 * h;   /* register r: token tb + 8 (r / 4) + r % 4 */
            float inv[16];
#pragma unroll
            for (int r = 0; r < 16; r++) inv[r] = x.inv ? x.inv[min(tb + 8 * (r >> 2) + (r & 3), a.T - 1)] : x.inv_all;
#pragma unroll
            for (int i = 0; i < MR; i++) {
                const int row = r0 + (wr * MR + i) * 32 + j;
                if (row >= a.R) continue;
                const float bias = EP <= EP_BIAS_GELU_SPLIT ? a.bias[row] : 0.0f;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int f = (i * MT + u) * 16 + r;
                    if (f / NP != c) continue;
                    float o = c == 0 ? acc[i][u][r] : red[f * NG + gt];
#pragma unroll
                    for (int g = 1; g < WK; g++) o += c == g ? acc[i][u][r] : red[(g * NR + f) * NG + gt];
                    hg_emit<EP>(a, o, inv[r], bias, tb + 8 * (r >> 2) + (r & 3), row);
                }
            }
        }
    }
}

template <int MR, int MT, int WR, int WT, int WK>
static void hgemm_launch(const BGemm& a, const HSplit& x, int ep, hipStream_t s)
{
    const int nrb = ((a.R + 32 * MR * WR - 1) / (32 * MR * WR) + 7) & ~7, nt = (a.T + 32 * MT * WT - 1) / (32 * MT * WT);
    const dim3 grid((unsigned)(nrb * nt)), blk(64 * WR * WT * WK);
#define HG(E) hipLaunchKernelGGL((k_hgemm<MR, MT, WR, WT, WK, E>), grid, blk, 0, s, a, x)
    if constexpr (MR == MT && WK != 2) {   /* the encoder's tiles (lg_hgemm) */
        switch (ep) {
        case EP_BIAS: HG(EP_BIAS); return;
        case EP_BIAS_RES: HG(EP_BIAS_RES); return;
        case EP_BIAS_GELU: HG(EP_BIAS_GELU); return;
        case EP_BIAS_GELU_SPLIT: HG(EP_BIAS_GELU_SPLIT); return;
        }
    }
    if (ep == EP_ADD) HG(EP_ADD);
    else HG(EP_STORE);
#undef HG
}

/* The tile by how many workgroups it gives the 256 CUs (us at that tile /
 * the next candidates, weights cycled through more than the caches hold):
 * 128 x 128 while it fills them -- 24576 x 4096, 500 tokens 229 (881 TFLOP/s
 * of the two products; 256 x 128 267, 128 x 64 264), 1152 x 384, 4096 tokens
 * 21 -- then 128 x 64 (24576 x 4096, 150 tokens 117 / 129), with K in two
 * parts where a CU would hold one workgroup only (4096 x 4096, 500 tokens 50
 * / 54 unsplit), then 64 x 64 (384 x 1536, 4096 tokens 32 / 35; split:
 * 4096 x 4096, 150 tokens 32 / 34), and 32 x 32 with K in four parts for the
 * smallest (384 x 1536, 512 tokens 7.7 / 13) and for up to 32 tokens, where
 * the weights' stream is the bound (24576 x 4096, 13 tokens 48, 4.2 TB/s;
 * 64 x 64 60).
 *
 * The encoder's matrices are narrow, and every tile must add K's four parts
 * in one order (PO above): 32 x 32 up to 384 such tiles (384 x 1536, 25
 * tokens 7.5 / 64 x 64 16.1, 1000 tokens 14.0 / 16.6; 1152 x 384, 260 tokens
 * 5.3 / 7.1), 64 x 64 above (1536 x 384, 1000 tokens 11.1 / 9.6; 4096 tokens: 1152 x 384 24.3, 384 x 384 15.6,
 * 1536 x 384 25.9, 384 x 1536 35.4; 128 x 128 25.0, 30.7, 30.0, 50.2), and
 * 128 x 128 once it gives every CU two: two layers of 1024 / 4096, 4096 and
 * 8192 tokens 1006 and 1635 us (64 x 64 throughout 1143 and 2157), of 768 /
 * 3072 755 and 1380 (804 and 1471). */
int lg_hgemm(const BGemm& a, const HSplit& x, int ep, hipStream_t s)
{
    auto wgs = [&](int tr, int tt) { return (long)((a.R + tr - 1) / tr) * ((a.T + tt - 1) / tt); };
    if (ep <= EP_BIAS_GELU_SPLIT) {
        if (wgs(32, 32) <= 384) hgemm_launch<1, 1, 1, 1, 4>(a, x, ep, s);
        else if (wgs(128, 128) >= 512) hgemm_launch<2, 2, 2, 2, 1>(a, x, ep, s);
        else hgemm_launch<1, 1, 2, 2, 1>(a, x, ep, s);
    } else if (a.T <= 32) hgemm_launch<1, 1, 1, 1, 4>(a, x, ep, s);
    else if (wgs(128, 128) >= 256) hgemm_launch<2, 2, 2, 2, 1>(a, x, ep, s);
    else if (wgs(128, 64) >= 384) hgemm_launch<2, 1, 2, 2, 1>(a, x, ep, s);
    else if (wgs(128, 64) >= 224) hgemm_launch<2, 1, 2, 2, 2>(a, x, ep, s);
    else if (wgs(64, 64) >= 320) hgemm_launch<1, 1, 2, 2, 1>(a, x, ep, s);
    else if (wgs(64, 64) >= 128) hgemm_launch<1, 1, 2, 2, 2>(a, x, ep, s);
    else hgemm_launch<1, 1, 1, 1, 4>(a, x, ep, s);
    return lg_check_launch("fp16 gemm");
}
