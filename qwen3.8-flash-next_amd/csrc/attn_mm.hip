/*
 * attn_mm.hip -- the attention part of attention_forward (reference
 * c/src/model.c:951-1143: scaled scores, causal and block mask, softmax,
 * weighted sum of v, sigmoid gate) for calls of many tokens, on bf16 MFMA at
 * fp32 precision, in three or four launches:
 *
 *   k_am_prep  the cached k and v rows as three bf16 parts each (hi + mid +
 *              lo, 24 bits) in the operand order of the matrix
 *              instructions, one image of 32 keys after the other, and a
 *              flag per image that holds a value the parts cannot carry;
 *   k_am_mask  (block mask on) one bit per (token, key);
 *   k_am_attn  workgroup = 128 (token, query head) rows of one kv head x a
 *              range of keys: scores, running maximum and sum, O;
 *   k_am_comb  the key ranges merged, times sigmoid(gate), as the operand
 *              planes of o_proj.
 *
 * Precision: a product of two fp32 numbers in three bf16 parts each needs
 * six of the nine partial products (the other three are below 2^-24 of it);
 * sums are fp32.  So scores, probabilities and outputs keep fp32 accuracy.
 * Six bf16 products run at 417 TFLOP/s against 157 for the fp32 matrix
 * instructions and 79 for the vector ALU.
 */
#include "qk_device.h"
#include "mfma_parts.h"

typedef float qm_f32x16 __attribute__((ext_vector_type(16)));
#define AM_MFMA(A, B, C) __builtin_amdgcn_mfma_f32_32x32x16_bf16((A), (B), (C), 0, 0, 0)

#define AM_KT 32      /* keys per image */
#define AM_ROWS 128   /* (token, head) rows per workgroup */
#define AM_BIG 1e15f  /* parts and products of values up to this stay finite */

struct AmArgs {
    const float *qn;       /* [n, h, hd] */
    const float *k, *v;    /* [T, kvh, hd] */
    const uint32_t *keep;  /* [n, kw] or NULL */
    uint4 *img;            /* [kvh, tiles, 2, hd * 12] */
    int *flag;             /* [kvh, tiles] */
    uint32_t *mask;        /* [n, tiles] (keep set) */
    float *po;             /* [n, h, nch, hd] */
    float2 *pml;           /* [n, h, nch]: maximum (log2 units), sum */
    const float *qg;       /* [n, h, 2, hd] */
    qk_planes pl;          /* of h * hd columns */
    int n, h, kvh, hd, T, tiles, offset, comp, nb, kw, nch, ctiles, nqb;
};

/* two fp32 -> three bf16 pairs */
__device__ __forceinline__ void am_split2(float a, float b, uint32_t w[3]) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
        w[i] = qk_cvt_pk_bf16(a, b);
        a = a - qk_bf16_lo(w[i]);
        b = b - qk_bf16_hi(w[i]);
    }
}
__device__ __forceinline__ void am_split8(const float x[8], uint4 w[3]) {
    uint32_t p[4][3];
#pragma unroll
    for (int j = 0; j < 4; j++) am_split2(x[2 * j], x[2 * j + 1], p[j]);
#pragma unroll
    for (int i = 0; i < 3; i++) w[i] = make_uint4(p[0][i], p[1][i], p[2][i], p[3][i]);
}
__device__ __forceinline__ bool am_bad8(const float x[8]) {
    bool b = false;
#pragma unroll
    for (int j = 0; j < 8; j++) b |= !(fabsf(x[j]) <= AM_BIG);
    return b;
}

/*
 * grid (tiles, kvh).  The images are exactly what a wave's operand reads
 * take, 16 bytes per lane and fragment, so the copy into LDS and the reads
 * there are linear.  k image: fragment (part, K-step s of 16 dims), lane l =
 * key l%32, dims 16 s + 8 (l/32) + 0..7.  v image (transposed): fragment
 * (part, 32 dims dt, K-step s of 16 keys), lane l = dim 32 dt + l%32, the
 * keys 16 s + 8 a + 4 (l/32) + b at 4 a + b: the order in which the scores'
 * accumulators hold the keys of a row.  Keys past T are zero.  Bound: HBM /
 * L2 writes (6 bytes out per 4 in).
 */
__global__ __launch_bounds__(256) void k_am_prep(AmArgs a) {
    const int tile = blockIdx.x, kh = blockIdx.y, tid = threadIdx.x;
    const int c8 = a.hd >> 3, ks = a.hd >> 4;
    const size_t kvw = (size_t)a.kvh * a.hd;
    uint4 *ki = a.img + ((size_t)kh * a.tiles + tile) * 2 * (a.hd * 12), *vi = ki + a.hd * 12;
    bool bad = false;
    for (int i = tid; i < AM_KT * c8; i += 256) {
        const int key = i / c8, ch = i - key * c8, kk = tile * AM_KT + key;
        float x[8];
        const float4 *src = (const float4 *)(a.k + (size_t)min(kk, a.T - 1) * kvw + (size_t)kh * a.hd) + 2 * ch;
        const float4 x0 = qk_ld(src), x1 = qk_ld(src + 1);
        x[0] = x0.x; x[1] = x0.y; x[2] = x0.z; x[3] = x0.w;
        x[4] = x1.x; x[5] = x1.y; x[6] = x1.z; x[7] = x1.w;
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = kk < a.T ? x[j] : 0.0f;
        bad |= am_bad8(x);
        uint4 w[3];
        am_split8(x, w);
#pragma unroll
        for (int p = 0; p < 3; p++) ki[(p * ks + (ch >> 1)) * 64 + (ch & 1) * 32 + key] = w[p];
    }
    for (int i = tid; i < a.hd * 4; i += 256) {
        const int g = i / a.hd, d = i - g * a.hd, s = g >> 1, h = g & 1;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int kk = tile * AM_KT + 16 * s + 8 * (j >> 2) + 4 * h + (j & 3);
            const float v = qk_ld(a.v + (size_t)min(kk, a.T - 1) * kvw + (size_t)kh * a.hd + d);
            x[j] = kk < a.T ? v : 0.0f;
        }
        bad |= am_bad8(x);
        uint4 w[3];
        am_split8(x, w);
#pragma unroll
        for (int p = 0; p < 3; p++) vi[((p * (a.hd >> 5) + (d >> 5)) * 2 + s) * 64 + h * 32 + (d & 31)] = w[p];
    }
    const int any = __syncthreads_or(bad);
    if (tid == 0) a.flag[kh * a.tiles + tile] = any;
}

/* one thread per (token, 32 keys): bit j = key may be seen (at or before the
 * token, and in a kept block or in the token's own tail block) */
__global__ __launch_bounds__(256) void k_am_mask(AmArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int t = i / a.tiles, tile = i - t * a.tiles;
    if (t >= a.n) return;
    const int qpos = a.offset + t, own = (qpos + 1) / a.comp * a.comp;
    const uint32_t *kp = a.keep + (size_t)t * a.kw;
    uint32_t w = 0;
    int blk = -1;
    bool kept = false;
    for (int j = 0; j < 32; j++) {
        const int kk = tile * 32 + j;
        if (kk > qpos || kk >= a.T) break;
        const int b = kk / a.comp;
        if (b != blk) {
            blk = b;
            kept = b < a.nb && ((qk_ld(kp + (b >> 5)) >> (b & 31)) & 1u);
        }
        if (kept || kk >= own) w |= 1u << j;
    }
    a.mask[i] = w;
}

/* bits of the keys 32 tile + 0..31 that token position qpos sees */
__device__ __forceinline__ uint32_t am_causal(int qpos, int tile) {
    const int d = qpos - 32 * tile;
    return d >= 31 ? 0xFFFFFFFFu : (d < 0 ? 0u : (2u << d) - 1u);
}

/* score * this -> log2 units */
__device__ __forceinline__ float am_scale(int hd) { return 1.4426950408889634f / sqrtf((float)hd); }

/*
 * A workgroup whose keys or queries hold a value the bf16 parts cannot carry
 * (not finite, or past AM_BIG): one row at a time per wave in fp32 on the
 * vector ALU, so masked keys and keys of weight 0 are never multiplied and
 * an infinity or NaN reaches the rows that see it and no others.
 */
template <int HD>
__device__ void am_slow(const AmArgs &a, int kh, int row0, int kt0, int kt1, int c) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int G = a.h / a.kvh;
    const size_t kvw = (size_t)a.kvh * HD;
    const float c1 = am_scale(HD);
    for (int r = row0 + 32 * wave; r < min(row0 + 32 * wave + 32, a.n * G); r++) {
        const int t = r / G, hh = kh + a.kvh * (r - t * G), qpos = a.offset + t;
        const float *q = a.qn + ((size_t)t * a.h + hh) * HD;
        const int k1 = min(min(kt1 * AM_KT, a.T), qpos + 1);
        auto score = [&](int kk) {
            bool live = kk < k1;
            if (live && a.keep) live = (qk_ld(a.mask + (size_t)t * a.tiles + (kk >> 5)) >> (kk & 31)) & 1u;
            float s = 0.0f;
            if (live) {
                const float4 *kr = (const float4 *)(a.k + (size_t)kk * kvw + (size_t)kh * HD);
                for (int i = 0; i < HD / 4; i++) {
                    const float4 x = qk_ld(kr + i), y = qk_ld((const float4 *)q + i);
                    s = fmaf(y.x, x.x, s);
                    s = fmaf(y.y, x.y, s);
                    s = fmaf(y.z, x.z, s);
                    s = fmaf(y.w, x.w, s);
                }
            }
            return live ? s * c1 : -INFINITY;
        };
        float m = -INFINITY;
        for (int k0 = kt0 * AM_KT; k0 < k1; k0 += 64) {
            const float s = score(k0 + lane);
            m = fmaxf(m, s);
        }
        for (int o = 1; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, QK_WAVE));
        float l = 0.0f, acc[HD / 64];
#pragma unroll
        for (int e = 0; e < HD / 64; e++) acc[e] = 0.0f;
        for (int k0 = kt0 * AM_KT; k0 < k1; k0 += 64) {
            const float s = score(k0 + lane);
            /* a NaN score must reach the sum although the maximum passes it by */
            const float p = m == -INFINITY && s == s ? 0.0f : exp2f(s - m);
            l += p;
            for (int j = 0; j < min(64, k1 - k0); j++) {
                const float pj = __shfl(p, j, QK_WAVE);
                if (pj == 0.0f) continue;
                const float *vr = a.v + (size_t)(k0 + j) * kvw + (size_t)kh * HD;
#pragma unroll
                for (int e = 0; e < HD / 64; e++) acc[e] = fmaf(pj, qk_ld(vr + lane + 64 * e), acc[e]);
            }
        }
        l = qk_group_sum<64>(l);
        const size_t u = ((size_t)t * a.h + hh) * a.nch + c;
#pragma unroll
        for (int e = 0; e < HD / 64; e++) qk_st(a.po + u * HD + lane + 64 * e, acc[e]);
        if (lane == 0) a.pml[u] = make_float2(m, l);
    }
}

/*
 * grid (nqb * kvh * nch).  Wave = 32 rows (columns of the instructions: all
 * scores and outputs of a row sit in lanes l and l + 32), transposed
 * products: S^T = K Q^T leaves lane l the scores of its row for keys
 * 8 a + 4 (l/32) + b, which is the B operand of O^T = V^T P^T as it is, so
 * the probabilities never leave the registers.  Q stays in registers as
 * three parts.  The images go through a ring of three LDS buffers, copied
 * straight from memory two half-steps (k, then v of a tile) ahead, one
 * barrier per half-step; 72 KB at head dim 128, so two workgroups share a
 * CU and one's softmax runs under the other's matrix products.
 *
 * Bound: matrix cores, 12 * 32 * 32 * hd * 2 flop issued per wave and tile.
 * 4096 tokens in two calls of 2048 (16 heads of 128 on 2 kv heads): 437 us,
 * 940 TFLOP/s issued; the per-token kernels (k_at_attn, k_at_comb) 4590 us.
 */
template <int HD>
__global__ __launch_bounds__(256, HD <= 128 ? 2 : 1) void k_am_attn(AmArgs a) {
    constexpr int KS = HD / 16, DT = HD / 32, IMG = HD * 12; /* uint4 per image */
    constexpr int NL = IMG / 256;                            /* copies per wave and image */
    __shared__ __attribute__((aligned(16))) uint4 ring[3][IMG];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = a.nqb * a.kvh;
    const int c = blockIdx.x / per, rem = blockIdx.x - c * per;
    const int kh = rem / a.nqb, row0 = (rem - kh * a.nqb) * AM_ROWS;
    const int G = a.h / a.kvh, nrow = a.n * G;
    const int tmax = (min(row0 + AM_ROWS, nrow) - 1) / G;
    const int kt0 = c * a.ctiles;
    const int kt1 = min(min(kt0 + a.ctiles, a.tiles), (a.offset + tmax) / AM_KT + 1);
    if (kt0 >= kt1) return; /* every key of the range is after every row */

    const int r = min(row0 + 32 * wave + (lane & 31), nrow - 1);
    const int t = r / G, hh = kh + a.kvh * (r - t * G), qpos = a.offset + t;
    uint4 q[3][KS];
    bool bad = false;
    {
        const float4 *src = (const float4 *)(a.qn + ((size_t)t * a.h + hh) * HD + 8 * (lane >> 5));
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const float4 x0 = qk_ld(src + 4 * s), x1 = qk_ld(src + 4 * s + 1);
            const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            uint4 w[3];
            bad |= am_bad8(x);
            am_split8(x, w);
#pragma unroll
            for (int p = 0; p < 3; p++) q[p][s] = w[p];
        }
        for (int i = kt0 + tid; i < kt1; i += 256) bad = bad || a.flag[kh * a.tiles + i] != 0;
    }
    if (__syncthreads_or(bad)) {
        am_slow<HD>(a, kh, row0, kt0, kt1, c);
        return;
    }

    const uint4 *src = a.img + ((size_t)kh * a.tiles + kt0) * 2 * IMG + 64 * NL * wave + lane;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(qm_lptr)&ring[0][0] + 1024 * NL * wave);
    auto copy = [&](int hs) {
        const uint4 *p = src + (size_t)hs * IMG;
        const uint32_t d = lds0 + (uint32_t)(hs % 3) * (IMG * 16);
#pragma unroll
        for (int i = 0; i < NL; i += 3) { /* NL = 3, 6, 9 or 12 */
            qm_copy<0>(p + 64 * i, d + 1024 * i);
            qm_copy<1024>(p + 64 * i, d + 1024 * i);
            qm_copy<2048>(p + 64 * i, d + 1024 * i);
        }
    };
    const int nhs = 2 * (kt1 - kt0);
    copy(0);
    copy(1);
    float m = -INFINITY, l = 0.0f;
    const float c1 = am_scale(HD);
    const uint32_t *mp = a.keep ? a.mask + (size_t)t * a.tiles : (const uint32_t *)a.flag;
    qm_f32x16 o[DT];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[d][i] = 0.0f;

    for (int kt = kt0; kt < kt1; kt++) {
        const int hs = 2 * (kt - kt0);
        const uint32_t ml = qk_ld(mp + kt); /* used after the scores, so its wait finds the copies done */
        /* image hs is in LDS once this wave's older copies are done and every
         * wave has said so; the ring slot of hs + 2 was last read in hs - 1 */
        qm_sync<NL>();
        if (hs + 2 < nhs) copy(hs + 2);
        qm_f32x16 st;
#pragma unroll
        for (int i = 0; i < 16; i++) st[i] = 0.0f;
        {
            const uint4 *kb = ring[hs % 3] + lane;
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const qm_bf16x8 k0 = __builtin_bit_cast(qm_bf16x8, kb[s * 64]),
                                k1 = __builtin_bit_cast(qm_bf16x8, kb[(KS + s) * 64]),
                                k2 = __builtin_bit_cast(qm_bf16x8, kb[(2 * KS + s) * 64]);
                const qm_bf16x8 q0 = __builtin_bit_cast(qm_bf16x8, q[0][s]), q1 = __builtin_bit_cast(qm_bf16x8, q[1][s]),
                                q2 = __builtin_bit_cast(qm_bf16x8, q[2][s]);
                st = AM_MFMA(k2, q0, st);
                st = AM_MFMA(k1, q1, st);
                st = AM_MFMA(k0, q2, st);
                st = AM_MFMA(k1, q0, st);
                st = AM_MFMA(k0, q1, st);
                st = AM_MFMA(k0, q0, st);
            }
        }
        /* running maximum over the row's keys so far, both halves alike */
        uint32_t mw = a.keep ? ml : am_causal(qpos, kt);
        mw >>= 4 * (lane >> 5);
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            st[i] = (mw >> (8 * (i >> 2) + (i & 3))) & 1u ? st[i] * c1 : -INFINITY;
            mx = fmaxf(mx, st[i]);
        }
        mx = fmaxf(mx, __uint_as_float(qk_xor32_u(__float_as_uint(mx))));
        const float mn = fmaxf(m, mx);
        if (__any(mn > m)) {
            const float f = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            l *= f;
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[d][i] *= f;
            m = mn;
        }
        const float ms = m == -INFINITY ? 0.0f : m; /* no key yet: every score is -inf */
#pragma unroll
        for (int i = 0; i < 16; i++) {
            st[i] = __builtin_amdgcn_exp2f(st[i] - ms);
            l += st[i];
        }
        /* image hs + 1, as above */
        if (hs + 2 < nhs) qm_sync<NL>();
        else qm_sync<0>();
        if (hs + 3 < nhs) copy(hs + 3);
        const uint4 *vb = ring[(hs + 1) % 3] + lane;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const float x[8] = {st[8 * s], st[8 * s + 1], st[8 * s + 2], st[8 * s + 3],
                                st[8 * s + 4], st[8 * s + 5], st[8 * s + 6], st[8 * s + 7]};
            uint4 w[3];
            am_split8(x, w);
            const qm_bf16x8 p0 = __builtin_bit_cast(qm_bf16x8, w[0]), p1 = __builtin_bit_cast(qm_bf16x8, w[1]),
                            p2 = __builtin_bit_cast(qm_bf16x8, w[2]);
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const qm_bf16x8 v0 = __builtin_bit_cast(qm_bf16x8, vb[(2 * d + s) * 64]),
                                v1 = __builtin_bit_cast(qm_bf16x8, vb[(2 * (DT + d) + s) * 64]),
                                v2 = __builtin_bit_cast(qm_bf16x8, vb[(2 * (2 * DT + d) + s) * 64]);
                o[d] = AM_MFMA(v2, p0, o[d]);
                o[d] = AM_MFMA(v1, p1, o[d]);
                o[d] = AM_MFMA(v0, p2, o[d]);
                o[d] = AM_MFMA(v1, p0, o[d]);
                o[d] = AM_MFMA(v0, p1, o[d]);
                o[d] = AM_MFMA(v0, p0, o[d]);
            }
        }
    }
    l += __uint_as_float(qk_xor32_u(__float_as_uint(l)));
    if (row0 + 32 * wave + (lane & 31) >= nrow) return;
    const size_t u = ((size_t)t * a.h + hh) * a.nch + c;
    float *po = a.po + u * HD + 4 * (lane >> 5);
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            qk_st((float4 *)(po + 32 * d + 8 * i), make_float4(o[d][4 * i], o[d][4 * i + 1], o[d][4 * i + 2], o[d][4 * i + 3]));
    if (lane < 32) a.pml[u] = make_float2(m, l);
}

/* a wave per 8 tokens x 64 columns of the attention output: the key ranges up
 * to the token's own merged, the gate, and the planes.  Bound: HBM / L2, the
 * partial outputs read once. */
__global__ __launch_bounds__(256) void k_am_comb(AmArgs a) {
    const int G = a.h * a.hd / 64, lane = threadIdx.x & 63;
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6), rb = w / G, gr = w - rb * G;
    if (8 * rb >= a.n) return;
    const int t = min(8 * rb + (lane & 7), a.n - 1), col = 64 * gr + 8 * (lane >> 3), hh = col / a.hd, d = col - hh * a.hd;
    const int live = min((a.offset + t) / (AM_KT * a.ctiles) + 1, a.nch);
    const size_t u = ((size_t)t * a.h + hh) * a.nch;
    float M = -INFINITY, L = 0.0f, x[8];
    for (int c = 0; c < live; c++) M = fmaxf(M, qk_ld((const float *)(a.pml + u + c)));
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = 0.0f;
    for (int c = 0; c < live; c++) {
        const float2 ml = a.pml[u + c];
        const float4 *p = (const float4 *)(a.po + (u + c) * a.hd + d);
        const float4 p0 = qk_ld(p), p1 = qk_ld(p + 1);
        /* a range with every key masked has maximum -inf and zero sums */
        const float f = ml.x == -INFINITY && ml.y == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(ml.x - M);
        L = fmaf(ml.y, f, L);
        x[0] = fmaf(p0.x, f, x[0]); x[1] = fmaf(p0.y, f, x[1]); x[2] = fmaf(p0.z, f, x[2]); x[3] = fmaf(p0.w, f, x[3]);
        x[4] = fmaf(p1.x, f, x[4]); x[5] = fmaf(p1.y, f, x[5]); x[6] = fmaf(p1.z, f, x[6]); x[7] = fmaf(p1.w, f, x[7]);
    }
    const float inv = 1.0f / L;
    const float4 *g = (const float4 *)(a.qg + ((size_t)t * a.h + hh) * 2 * a.hd + a.hd + d);
    const float4 g0 = qk_ld(g), g1 = qk_ld(g + 1);
    const float gv[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = (x[j] * inv) * qk_sigmoid(gv[j]);
    qm_pack_store(a.pl, 8 * rb + (lane & 7), a.n, gr, G, x);
}

/* ------------------------------------------------------------ host side */

/* bytes of the images, flags and mask words for cap cached rows and n tokens */
extern "C" size_t qk_am_img_bytes(const qk_at_shape *s) {
    return (size_t)s->kvh * ((s->cap + AM_KT - 1) / AM_KT) * ((size_t)2 * s->hd * 192 + 4);
}
extern "C" size_t qk_am_mask_bytes(const qk_at_shape *s, int n) {
    return (size_t)n * ((s->cap + AM_KT - 1) / AM_KT) * 4;
}

/* keys per workgroup, in images: 1024 keys (the partial outputs of shorter
 * ranges cost more than the better balance gives), fewer while the grid would
 * leave CUs idle, at least 128 */
static int am_ctiles(int units, int tiles) {
    int ct = 32;
    while (ct > 4 && (long long)units * ((tiles + ct - 1) / ct) < 768) ct >>= 1;
    return ct;
}

extern "C" int qk_launch_attn_mm(const qk_at_shape *s, int n, int offset, int T, const float *qn, const float *qg,
                                 const float *k_cache, const float *v_cache, const uint32_t *keep, int nb, int kw,
                                 const qk_at_scratch *sc, void *stream) {
    hipStream_t st = (hipStream_t)stream;
    AmArgs a;
    a.qn = qn; a.k = k_cache; a.v = v_cache; a.keep = keep;
    a.n = n; a.h = s->h; a.kvh = s->kvh; a.hd = s->hd; a.T = T;
    a.tiles = (T + AM_KT - 1) / AM_KT;
    a.offset = offset; a.comp = s->comp; a.nb = nb; a.kw = kw;
    a.nqb = (n * (s->h / s->kvh) + AM_ROWS - 1) / AM_ROWS;
    a.ctiles = am_ctiles(a.nqb * s->kvh, a.tiles);
    a.nch = (a.tiles + a.ctiles - 1) / a.ctiles;
    /* the partials take n * nch units of hd + 2 floats per head */
    while ((long long)n * a.nch > sc->part_units) {
        if (a.nch == 1) return (int)hipErrorInvalidValue;
        a.ctiles *= 2;
        a.nch = (a.tiles + a.ctiles - 1) / a.ctiles;
    }
    a.img = (uint4 *)sc->img;
    a.flag = (int *)(a.img + (size_t)s->kvh * a.tiles * 2 * (s->hd * 12));
    a.mask = sc->kmask;
    a.po = sc->part;
    a.pml = (float2 *)(sc->part + (size_t)n * s->h * a.nch * s->hd);
    a.qg = qg;
    a.pl = sc->pl;
    hipLaunchKernelGGL(k_am_prep, dim3(a.tiles, s->kvh), dim3(256), 0, st, a);
    int rc = QK_CHECK_LAUNCH();
    if (rc) return rc;
    if (keep) {
        hipLaunchKernelGGL(k_am_mask, dim3((unsigned)(((long long)n * a.tiles + 255) / 256)), dim3(256), 0, st, a);
        rc = QK_CHECK_LAUNCH();
        if (rc) return rc;
    }
    const dim3 grid((unsigned)(a.nqb * s->kvh * a.nch));
    switch (s->hd) {
    case 64: hipLaunchKernelGGL(k_am_attn<64>, grid, dim3(256), 0, st, a); break;
    case 128: hipLaunchKernelGGL(k_am_attn<128>, grid, dim3(256), 0, st, a); break;
    case 192: hipLaunchKernelGGL(k_am_attn<192>, grid, dim3(256), 0, st, a); break;
    case 256: hipLaunchKernelGGL(k_am_attn<256>, grid, dim3(256), 0, st, a); break;
    default: return (int)hipErrorInvalidValue;
    }
    rc = QK_CHECK_LAUNCH();
    if (rc) return rc;
    hipLaunchKernelGGL(k_am_comb, dim3(qm_pack_wgs(n, s->h * s->hd / 64)), dim3(256), 0, st, a);
    return QK_CHECK_LAUNCH();
}
