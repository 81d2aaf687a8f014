/* lg_pfattn.hip -- causal attention of a prefill pass
 * (fast/ligguf_fast_qk.cpp:64-105 for T query tokens at once): 32 query
 * tokens x one KV head per workgroup on 32 x 32 x 16 fp16 MFMA. */
#include <math.h>

#include <algorithm>

#include "lg_common.h"
#include "lg_prefill.h"

typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

/* One wave per query head of the KV head's group and per key half: 32 query
 * tokens are the columns of both products,
 *   S^T[key][q]  = sum_d K[key][d] Q[q][d]     A = K, B = Q^T (16 dims a step)
 *   O^T[d][q]   += sum_key V^T[d][key] P[key][q]   A = V^T, B = P
 * The cache rows are fp16; each fp32 operand goes in as two fp16 parts x =
 * hi + lo (hi = fp16(x), lo = fp16(x - hi)), so every product is exact in
 * fp32 and ~22 bits of q and p survive; p <= 1 is held times 2^15, so p down
 * to 2^-29 keeps a normal hi.  A query's own key and value are its fp32 k/v
 * (the cache has them in fp16), as in the token-sequential step: the own
 * score is an fp32 dot, put in place of the fp16 one, and p (v32 - v16) is
 * added to the finished sum.  Online softmax per query column: c = 15 -
 * log2(e) / sqrt(HD) max is the exponent offset, p = exp2(s log2(e) /
 * sqrt(HD) + c); the sums are rescaled only where some column's maximum rose.
 *
 * Lane l of a 32 x 32 x 16 product feeds row / column l % 32, k = 8 (l / 32)
 * .. +7, and its register r of the result is row 8 (r / 4) + 4 (l / 32) +
 * r % 4 of column l % 32.  P therefore is an operand of the second product
 * as it comes out of the first: registers 8s .. 8s+7 of lane half h are keys
 * 16s + 4h + {0..3} and 16s + 8 + 4h + {0..3}, and V^T is stored with those
 * eight keys of a dim side by side (octet 2s + h), one ds_read_b128.  The
 * octets of dim d are permuted by d's low three bits xor d / 8 (reads of
 * eight consecutive dims, and the writes of dims 8 apart, fall on different
 * banks); K rows are padded 16 bytes for the same.
 *
 * Keys in tiles of KT, each half's waves take every second tile with two LDS
 * stages of their own; the next tile is in registers while one computes.
 * One barrier a tile.  Over many keys bound by the two waves of a SIMD
 * alternating between MFMA issue (64 products per 32 x 64 scores) and the
 * softmax's VALU work (~450 operations); a short prompt by its chain of first
 * loads, one tile and the exchanges at both ends.  Against the 16 x 16 x 16
 * form with 16 queries a wave that this replaces, which read twice the LDS
 * bytes per product, wrote V^T two bytes at a time and never split the keys
 * (32 heads of 128, 8 KV heads): 512 tokens after 6900..7412, 352 us -> 147
 * (410 TFLOP/s of the products asked for, 820 issued with the split parts);
 * 512 after none 30 -> 21 and 5.6 to merge.  All 64 scores of a column in one
 * softmax step rather than 32 and 32: 157 -> 147 us there.
 *
 * Long contexts split the keys over workgroups as well (nsplit chunks of ck
 * keys, merged by k_pf_attn_merge): pf_attn_split. */
template <int HD, int NREP>
struct PfAttn {
    static constexpr int SPLIT = NREP <= 4 ? 2 : 1;      /* key halves */
    static constexpr int KT = NREP >= 4 ? 64 : 32;       /* keys per tile */
    static constexpr int NTH = 64 * NREP;                /* threads of a half */
    static constexpr int NT = NTH * SPLIT;
    static constexpr int KST = HD + 8;                   /* halves per K row */
    static constexpr int NTO = (HD + 31) / 32;           /* 32-dim output tiles */
    static constexpr int NJ = HD / 16;                   /* 16-dim steps of S */
    static constexpr int SK = KT * KST, SV = NTO * 32 * KT;
    static constexpr int NK = (KT * HD / 8 + NTH - 1) / NTH;          /* 16-byte pieces of K per thread */
    static constexpr int NV = (KT / 4 * (HD / 8) + NTH - 1) / NTH;    /* 4 keys x 8 dims of V per thread */
    static constexpr int RED = SPLIT > 1 ? NREP * 64 * (2 + 16 * NTO) * 4 : 0;
    static constexpr int LDS0 = SPLIT * 2 * (SK + SV) * 2, LDS = LDS0 > RED ? LDS0 : RED;
    /* a wave's private part of it before and after the key loop, for 32 rows
     * of DW floats (+ 4): as wide as fits */
    static constexpr int PRIV = RED ? (LDS / (NREP * SPLIT) < RED / NREP ? LDS / (NREP * SPLIT) : RED / NREP) : LDS / NREP;
    static constexpr int PST = RED ? RED / NREP : PRIV & ~15;   /* distance of the parts after the loop */
    static constexpr int DW = HD == 128 && PRIV >= 32 * 132 * 4 ? 128 : HD % 64 == 0 && PRIV >= 32 * 68 * 4 ? 64
                            : HD % 32 == 0 && PRIV >= 32 * 36 * 4 ? 32 : 16;
    static constexpr int LPR = DW / 4, RPI = 64 / LPR, NI = 32 / RPI, NP = HD / DW;
    static_assert(PRIV >= 32 * (DW + 4) * 4, "a wave's rows");
};

/* a token's partial of one chunk: n_heads x hd sums, then (c, l) per head; in
 * floats, a multiple of 4 */
static __host__ __device__ __forceinline__ size_t pf_part_row(int n_heads, int hd)
{
    return ((size_t)n_heads * (hd + 2) + 3) & ~(size_t)3;
}

static __device__ __forceinline__ int pf_vt_at(int d, int oct, int kt)
{
    return d * kt + 8 * (oct ^ ((d ^ (d >> 3)) & (kt / 8 - 1)));
}

/* fp32 x0, x1 as elements i, i + 1 of the fp16 parts */
static __device__ __forceinline__ void split2(float x0, float x1, v8h& hi, v8h& lo, int i)
{
    const v2h x = __builtin_convertvector(((v2f){x0, x1}), v2h);
    const v2h y = __builtin_convertvector(((v2f){x0 - (float)x[0], x1 - (float)x[1]}), v2h);
    hi[i] = x[0];
    hi[i + 1] = x[1];
    lo[i] = y[0];
    lo[i + 1] = y[1];
}

template <int HD, int NREP>
__global__ __launch_bounds__(64 * NREP * (NREP <= 4 ? 2 : 1)) void k_pf_attn(
    const float* __restrict__ qkv, int qstride, int n_embed, int kv_dim, int n_kv, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, int pos0, int T, int ck, float* __restrict__ att, float* __restrict__ part)
{
    using C = PfAttn<HD, NREP>;
    constexpr int KT = C::KT, NTO = C::NTO, NJ = C::NJ, SPLIT = C::SPLIT, NS = KT / 32;
    __shared__ __attribute__((aligned(16))) uint8_t s_raw[C::LDS];
    /* KV head fastest: with 8 of them each XCD's L2 holds one head's rows;
     * the last query blocks (most keys) first */
    const int nqb = (T + 31) / 32;
    const int g = blockIdx.x % n_kv, sp = blockIdx.x / n_kv / nqb;
    const int t0 = 32 * (nqb - 1 - blockIdx.x / n_kv % nqb);
    const int last = pos0 + min(t0 + 31, T - 1);   /* last key position of this block */
    const int k0 = sp * ck;                        /* this chunk: keys k0 .. k1 - 1 */
    if (k0 > last) return;                         /* (whole workgroup) */
    const int k1 = min(k0 + ck, last + 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = wave % NREP, half = wave / NREP;
    const int tid = threadIdx.x % C::NTH;          /* within the half */
    const int col = lane & 31, h = lane >> 5;
    const int tq = t0 + col, qpos = pos0 + tq;
    const float scale2 = 1.44269504088896341f / sqrtf((float)HD);
    _Float16* const sK = (_Float16*)s_raw + (size_t)half * 2 * (C::SK + C::SV);
    _Float16* const sV = sK + 2 * C::SK;

    struct Tile {
        v4u k[C::NK], v[C::NV][4];
    };
    const int nit = (k1 - k0 + KT * SPLIT - 1) / (KT * SPLIT);
    auto tile_key = [&](int it) { return k0 + (max(0, min(it, nit - 1)) * SPLIT + half) * KT; };
    auto load_k = [&](Tile& P, int it) __attribute__((always_inline)) {
        const int kb = tile_key(it);
#pragma unroll
        for (int u = 0; u < C::NK; u++) {
            const int i = min(tid + u * C::NTH, KT * HD / 8 - 1), key = min(kb + i / (HD / 8), last);
            P.k[u] = *(const v4u*)(kc + (size_t)key * kv_dim + (size_t)g * HD + i % (HD / 8) * 8);
        }
    };
    auto load_v = [&](Tile& P, int it) __attribute__((always_inline)) {
        const int kb = tile_key(it);
#pragma unroll
        for (int u = 0; u < C::NV; u++) {
            const int i = min(tid + u * C::NTH, KT / 4 * (HD / 8) - 1);
#pragma unroll
            for (int n = 0; n < 4; n++) {
                const int key = min(kb + i / (HD / 8) * 4 + n, last);
                P.v[u][n] = *(const v4u*)(vc + (size_t)key * kv_dim + (size_t)g * HD + i % (HD / 8) * 8);
            }
        }
    };
    auto store_k = [&](const Tile& P, int buf) __attribute__((always_inline)) {
        _Float16* const K = sK + buf * C::SK;
#pragma unroll
        for (int u = 0; u < C::NK; u++) {
            const int i = tid + u * C::NTH;
            if ((KT * HD / 8) % C::NTH == 0 || i < KT * HD / 8)
                *(v4u*)(K + i / (HD / 8) * C::KST + i % (HD / 8) * 8) = P.k[u];
        }
    };
    auto store_v = [&](const Tile& P, int buf) __attribute__((always_inline)) {
        _Float16* const V = sV + buf * C::SV;
#pragma unroll
        for (int u = 0; u < C::NV; u++) {
            const int i = tid + u * C::NTH, kq = i / (HD / 8), d0 = i % (HD / 8) * 8;
            if ((KT / 4 * (HD / 8)) % C::NTH == 0 || i < KT / 4 * (HD / 8)) {
                const int oct = 2 * (kq >> 2) + (kq & 1), at = 4 * ((kq >> 1) & 1);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    /* dim d0 + e of the four keys: v_perm_b32 of two keys' words */
                    const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
                    uint2 w;
                    w.x = __builtin_amdgcn_perm(P.v[u][1][e >> 1], P.v[u][0][e >> 1], sel);
                    w.y = __builtin_amdgcn_perm(P.v[u][3][e >> 1], P.v[u][2][e >> 1], sel);
                    *(uint2*)(V + pf_vt_at(d0 + e, oct, KT) + at) = w;
                }
            }
        }
    };

    Tile P;
    /* Rows of 32 tokens go through LDS between the lane-per-token layout of
     * the products and whole lines of memory: read or written by the lane that
     * owns the token, every load or store touched 32 lines and the address
     * unit took about a cycle for each (20 tokens after 100: 17.4 -> 15.2 us;
     * 512 after none 26.5 -> 21.8). */
    constexpr int DW = C::DW, PR = DW + 4;
    auto rows = [&](v4f* R, int off, int tb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < C::NP * C::NI; i++)
            R[i] = *(const v4f*)(qkv + (size_t)min(tb + i % C::NI * C::RPI + lane / C::LPR, T - 1) * qstride + off +
                                 i / C::NI * DW + lane % C::LPR * 4);
    };
    auto wave_sync = [] __attribute__((always_inline)) {   /* the wave's LDS writes before its other lanes' reads */
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    /* the query row of the lane's column, dims 16j + 8h .. +7, as hi + lo;
     * the score with its own fp32 key */
    v8h qh[NJ], ql[NJ];
    float eown = 0.0f;
    {
        v4f Rq[C::NP * C::NI], Rk[C::NP * C::NI];
        rows(Rq, (g * NREP + r) * HD, t0);
        rows(Rk, n_embed + g * HD, t0);
        float* const w = (float*)(s_raw + (size_t)wave * (C::LDS / (NREP * SPLIT) & ~15));
        float* const wr = w + lane / C::LPR * PR + lane % C::LPR * 4;
        const float* const rd = w + col * PR + 8 * h;
        float qf[DW / 2];
#pragma unroll
        for (int p = 0; p < 2 * C::NP; p++) {
            /* queries, then keys, of dims p / 2 DW .. */
#pragma unroll
            for (int i = 0; i < C::NI; i++) *(v4f*)(wr + i * C::RPI * PR) = p & 1 ? Rk[p / 2 * C::NI + i] : Rq[p / 2 * C::NI + i];
            wave_sync();
#pragma unroll
            for (int e = 0; e < DW / 8; e++) {
                const v4f x = *(const v4f*)(rd + 16 * (e / 2) + 4 * (e % 2));
                if (p & 1) {
#pragma unroll
                    for (int i = 0; i < 4; i++) eown = __builtin_fmaf(qf[4 * e + i], x[i], eown);
                } else {
                    const int j = p / 2 * (DW / 16) + e / 2;
#pragma unroll
                    for (int i = 0; i < 4; i++) qf[4 * e + i] = x[i];
                    split2(x[0], x[1], qh[j], ql[j], 4 * (e % 2));
                    split2(x[2], x[3], qh[j], ql[j], 4 * (e % 2) + 2);
                }
            }
            wave_sync();
        }
        eown += lg_partner<5>(eown);
    }
    __syncthreads();   /* the first tile goes where the rows were */

    v16f o[NTO];
#pragma unroll
    for (int t = 0; t < NTO; t++) o[t] = (v16f){};
    /* finite start: a chunk may hold no key that an early column may see */
    float m = -1e30f, c = __builtin_fmaf(-m, scale2, 15.0f), l = 0.0f;   /* l: this lane half's keys only */

    for (int it = -1; it < nit; it++) {
        load_k(P, it + 1);
        const _Float16* const K = sK + (it & 1) * C::SK;
        const _Float16* const V = sV + (it & 1) * C::SV;
        const int kb = tile_key(it);
        const bool on = it >= 0 && kb < k1;   /* (wave-uniform) */
        v16f s[NS];
        if (on) {
#pragma unroll
            for (int n = 0; n < NS; n++) s[n] = (v16f){};
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int n = 0; n < NS; n++) {
                    const v8h a = *(const v8h*)(K + (32 * n + col) * C::KST + 16 * j + 8 * h);
                    s[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[j], s[n], 0, 0, 0);
                    s[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ql[j], s[n], 0, 0, 0);
                }
        }
        /* K and V of the next tile in turn: 16 registers less than both at once */
        store_k(P, (it + 1) & 1);
        load_v(P, it + 1);
        if (on) {
            if (kb + KT - 1 >= pos0 + t0) {   /* keys at or past some query's own (wave-uniform) */
#pragma unroll
                for (int n = 0; n < NS; n++) {
                    const int own = qpos - kb - 32 * n - 4 * h;   /* this lane's row of the own key: 8 (r / 4) + r % 4 */
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int k = 8 * (i >> 2) + (i & 3);
                        s[n][i] = k == own ? eown : k > own ? -INFINITY : s[n][i];
                    }
                }
            }
            float mn = m;
#pragma unroll
            for (int n = 0; n < NS; n++)
#pragma unroll
                for (int i = 0; i < 16; i++) mn = fmaxf(mn, s[n][i]);
            mn = fmaxf(mn, lg_partner<5>(mn));
            if (__builtin_amdgcn_ballot_w64(mn > m)) {
                const float cn = __builtin_fmaf(-mn, scale2, 15.0f), alpha = __builtin_amdgcn_exp2f(cn - c);
                m = mn;
                c = cn;
                l *= alpha;
#pragma unroll
                for (int t = 0; t < NTO; t++) o[t] *= alpha;
            }
#pragma unroll
            for (int st = 0; st < 2 * NS; st++) {
                float p[8];
#pragma unroll
                for (int i = 0; i < 8; i++)
                    p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[st / 2][8 * (st & 1) + i], scale2, c));
                l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
                v8h ph, pl;
#pragma unroll
                for (int i = 0; i < 8; i += 2) split2(p[i], p[i + 1], ph, pl, i);
#pragma unroll
                for (int t = 0; t < NTO; t++) {
                    const v8h a = *(const v8h*)(V + pf_vt_at(32 * t + col, 2 * st + h, KT));
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ph, o[t], 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pl, o[t], 0, 0, 0);
                }
            }
        }
        store_v(P, (it + 1) & 1);
        __syncthreads();
    }
    l += lg_partner<5>(l);
    /* the own values, in rows.  Their addresses are worked out again: taken
     * for the same expressions as the queries', they lived through the key
     * loop, which at 128 dims has no registers to spare, and 112 bytes a lane
     * went to scratch -- set up on the stream inside an engine's first prompt */
    v4f Rv[C::NP * C::NI];
    int te = t0;
    __asm__ volatile("" : "+s"(te));
    rows(Rv, n_embed + kv_dim + g * HD, te);
    if constexpr (SPLIT == 2) {
        /* the second half's (c, l, o) into the first half's lanes */
        float* x = (float*)s_raw + (size_t)r * (2 + 16 * NTO) * 64 + lane;   /* (the tiles are consumed) */
        if (half == 1) {
            x[0] = c;
            x[64] = l;
#pragma unroll
            for (int t = 0; t < NTO; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) x[64 * (2 + 16 * t + i)] = o[t][i];
        }
        __syncthreads();
        if (half == 1) return;
        const float c1 = x[0], cn = fminf(c, c1);
        const float a0 = __builtin_amdgcn_exp2f(cn - c), a1 = __builtin_amdgcn_exp2f(cn - c1);
        c = cn;
        l = lg_fma2(l, a0, x[64], a1);
#pragma unroll
        for (int t = 0; t < NTO; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) o[t][i] = lg_fma2(o[t][i], a0, x[64 * (2 + 16 * t + i)], a1);
    }
    /* p of the own key: its value in fp32 adds p (v32 - v16) */
    const float pown = qpos >= k0 && qpos < k1 ? __builtin_amdgcn_exp2f(__builtin_fmaf(eown, scale2, c)) : 0.0f;
    const int head = g * NREP + r, n_heads = n_kv * NREP;
    float* const w = (float*)(s_raw + (size_t)r * C::PST);   /* (the other half's part of it is read) */
    const size_t prow = pf_part_row(n_heads, HD);
    float* const dst = (part ? part + (size_t)sp * T * prow : att) + (size_t)head * HD;
    const size_t drow = part ? prow : (size_t)n_embed;
#pragma unroll
    for (int p = 0; p < C::NP; p++) {
#pragma unroll
        for (int d = p * DW; d < (p + 1) * DW; d += 8) {
            const int t = d / 32, a = d % 32 / 8;
            *(v4f*)(w + col * PR + d - p * DW + 4 * h) = (v4f){o[t][4 * a], o[t][4 * a + 1], o[t][4 * a + 2], o[t][4 * a + 3]};
        }
        if (h == 0) *(v2f*)(w + col * PR + DW) = (v2f){pown, part ? 1.0f : 1.0f / l};
        wave_sync();
#pragma unroll
        for (int i = 0; i < C::NI; i++) {
            const int row = i * C::RPI + lane / C::LPR, d = lane % C::LPR * 4;
            v4f y = *(const v4f*)(w + row * PR + d);
            const v2f pw = *(const v2f*)(w + row * PR + DW);
            const v4f v = Rv[p * C::NI + i];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float f = __builtin_fmaf(pw[0], v[e] - (float)(_Float16)v[e], y[e]);
                y[e] = (pw[0] != 0.0f ? f : y[e]) * pw[1];
            }
            if (t0 + row < T) *(v4f*)(dst + (t0 + row) * drow + p * DW + d) = y;
        }
        wave_sync();
    }
    if (part && h == 0 && tq < T)
        *(v2f*)(part + ((size_t)sp * T + tq) * prow + n_heads * HD + 2 * head) = (v2f){c, l};
}

/* the chunks' partials of token t: out = sum w_i o_i / sum w_i l_i with w_i =
 * 2^(c - c_i), over the chunks that hold a key the token may see */
__global__ __launch_bounds__(256) void k_pf_attn_merge(const float* __restrict__ part, int T, int n_heads, int hd,
                                                       int pos0, int ck, float* __restrict__ att)
{
    const int t = blockIdx.y, d = 4 * (blockIdx.x * 256 + threadIdx.x), n = n_heads * hd;
    if (d >= n) return;
    const int ns = (pos0 + t) / ck + 1, head = d / hd;
    const size_t row = pf_part_row(n_heads, hd), st = T * row;
    const float* p = part + t * row;
    float c = p[n + 2 * head];
    for (int s = 1; s < ns; s++) c = fminf(c, p[s * st + n + 2 * head]);
    float l = 0.0f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s = 0; s < ns; s++) {
        const float2 ml = *(const float2*)(p + s * st + n + 2 * head);
        const float4 v = *(const float4*)(p + s * st + d);
        const float w = __builtin_amdgcn_exp2f(c - ml.x);
        l = __builtin_fmaf(ml.y, w, l);
        o.x = __builtin_fmaf(v.x, w, o.x);
        o.y = __builtin_fmaf(v.y, w, o.y);
        o.z = __builtin_fmaf(v.z, w, o.z);
        o.w = __builtin_fmaf(v.w, w, o.w);
    }
    const float inv = 1.0f / l;
    *(float4*)(att + (size_t)t * n + d) = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
}

/* Chunks of keys: as many as keep the launch within one workgroup a CU (the
 * 8-wave workgroup's registers allow no second one; a second round of them
 * would start when the first ends), each of at least PF_ATT_KEYS keys, below
 * which a chunk's start and the merge cost what they save: two 4096-wide
 * layers, 3 tokens after 6000, 367 us with 1024 keys a chunk, 342 with 512,
 * 329 with 256, 332 with 128.  Two chunks begin to pay near 512 keys: a
 * prompt of 512 after none 813 us in one or two, of 64 after 450 367 / 361,
 * 300 after 600 680 / 666 (in three). */
constexpr int PF_ATT_WGS = 256, PF_ATT_KEYS = 256;
static int pf_attn_split(int T, int keys, int n_kv)
{
    return std::max(1, std::min(PF_ATT_WGS / ((T + 31) / 32 * n_kv), keys / PF_ATT_KEYS));
}

size_t lg_prefill_attn_part(int n_ctx, int n_heads, int n_kv, int head_dim)
{
    if (n_ctx < 2 * PF_ATT_KEYS || 2 * n_kv > PF_ATT_WGS) return 0;   /* never split */
    /* chunks x tokens <= 32 chunks x query blocks */
    return (size_t)32 * (PF_ATT_WGS / n_kv) * pf_part_row(n_heads, head_dim);
}

int lg_prefill_attn_supported(int head_dim, int nrep)
{
    return (head_dim == 48 || head_dim == 64 || head_dim == 128) && nrep >= 1 && nrep <= 8;
}

int lg_prefill_attn(const PfModel& M, const float* qkv, int qs, const uint16_t* kc, const uint16_t* vc, int T, int pos0,
                    float* att, float* part, size_t part_floats, hipStream_t s)
{
    const int nrep = M.n_heads / M.n_kv;
    if (!lg_prefill_attn_supported(M.head_dim, nrep)) {
        lg_set_error("prefill attention: head_dim %d with %d query heads per KV head", M.head_dim, nrep);
        return LG_ERR_TYPE;
    }
    const int keys = pos0 + T;
    /* chunks that the partials have room for */
    const size_t room = part_floats / (T * pf_part_row(M.n_heads, M.head_dim));
    int ns = (int)std::min<size_t>(pf_attn_split(T, keys, M.n_kv), std::max<size_t>(room, 1));
    const int ck = ((keys + ns - 1) / ns + 127) & ~127;   /* whole tiles of both halves */
    ns = (keys + ck - 1) / ck;
    if (ns == 1) part = nullptr;
    const dim3 grid((unsigned)((T + 31) / 32 * M.n_kv * ns));
#define PFA(HD, NR)                                                                                          \
    hipLaunchKernelGGL((k_pf_attn<HD, NR>), grid, dim3(PfAttn<HD, NR>::NT), 0, s, qkv, qs, M.n_embed, M.kv_dim, M.n_kv, kc, vc, \
                       pos0, T, ck, att, part)
#define PFA_HD(HD)                    \
    switch (nrep) {                   \
    case 1: PFA(HD, 1); break;        \
    case 2: PFA(HD, 2); break;        \
    case 3: PFA(HD, 3); break;        \
    case 4: PFA(HD, 4); break;        \
    case 5: PFA(HD, 5); break;        \
    case 6: PFA(HD, 6); break;        \
    case 7: PFA(HD, 7); break;        \
    default: PFA(HD, 8); break;       \
    }
    switch (M.head_dim) {
    case 48: PFA_HD(48); break;
    case 64: PFA_HD(64); break;
    default: PFA_HD(128); break;
    }
#undef PFA_HD
#undef PFA
    if (part)
        hipLaunchKernelGGL(k_pf_attn_merge, dim3((M.n_heads * M.head_dim / 4 + 255) / 256, T), dim3(256), 0, s, part, T,
                           M.n_heads, M.head_dim, pos0, ck, att);
    return lg_check_launch("prefill attention");
}
