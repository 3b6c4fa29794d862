/*
 * dn_chunk.hip -- the DeltaNet recurrence of many tokens (reference
 * c/src/model.c:1177-1248: conv, silu, l2 norms, decay, delta rule) in
 * chunks of 32 tokens, two launches per 2048 tokens instead of a serial step
 * per token.  The method is the chunked delta rule of Yang, Wang, Zhang, Shen
 * and Kim, "Parallelizing Linear Transformers with the Delta Rule over
 * Sequence Length" (2024), with the decay of Yang, Kautz and Hatamizadeh,
 * "Gated Delta Networks" (2024).
 *
 * With the decay products g_1..g_t = exp(G_t) inside a chunk and S the state
 * before it, the rule S <- g S; S += beta (v - S k) k^T gives
 *     u_t = beta_t (v_t - exp(G_t) S k_t - sum_{j<t} exp(G_t - G_j) (k_t.k_j) u_j)
 *     o_t = exp(G_t) S q_t + sum_{j<=t} exp(G_t - G_j) (q_t.k_j) u_j
 *     S'  = exp(G_C) S + sum_j exp(G_C - G_j) u_j k_j^T.
 * k_dc_prep does what does not depend on S, one workgroup per (chunk, value
 * head): the conv and norms, A_tj = beta_t exp(G_t - G_j) (k_t.k_j), and by
 * forward substitution on I + A the columns U0 (from beta v) and W (from
 * beta exp(G) k), so u = U0 - W S^T.  k_dc_seq carries S through the chunks,
 * one workgroup per 16 state rows of a head: three products per chunk.
 * Everything is fp32 (v_mfma_f32_16x16x4_f32); G is summed and subtracted in
 * fp64, so a strong decay earlier in the chunk costs the later ratios
 * nothing.
 *
 * A chunk whose inputs are not finite or past DC_BIG is stepped token by
 * token by k_dc_seq (dn_rec.h): a matrix product would spread a NaN or an
 * infinity to the chunk's earlier tokens.
 *
 * Layout of 16x16x4: A lane l holds row l%16, B lane l column l%16, K element
 * l/16; D lane l column l%16, rows 4*(l/16) + i.  K elements are dealt to the
 * lane quarters in runs, so a lane's operands of a product are contiguous.
 */
#include "dn_rec.h"

#define DC_C 32       /* tokens per chunk */
#define DC_SEG 2048   /* tokens per pair of launches (bounds the scratch) */
#define DC_BIG 1e15f
#define DC_VB 128     /* columns per round of the substitution */
#define DC_LP 4       /* LDS row padding, floats */

typedef float dc_f32x4 __attribute__((ext_vector_type(4)));
#define DC_MFMA(A, B, C) __builtin_amdgcn_mfma_f32_16x16x4f32((A), (B), (C), 0, 0, 0)

/* per (value head, chunk) of a segment.  All in the order in which k_dc_seq's
 * lanes take them, 16 bytes per lane l and load (r = l % 16, kq = l / 16), so
 * a wave's load is one run of 1 KB: read as rows, its lanes touched 64 lines
 * each time and the address path of the CU, not the products, set the pace
 * (206 us a 2048-token segment against 165). */
struct DcArgs {
    DnRecArgs r;
    float *w;   /* [2 token halves][dk/16][64][4]: -W, token 16 half + r, column kq dk/4 + 4 i + e */
    float *q;   /* the same of exp(G_t) q_t */
    float *kt;  /* [dk/16][2][64][4]: exp(G_C - G_j) k_j, column 16 i + r, token 8 kq + 4 half + e */
    float *u0;  /* [dv/16][2 token halves][64][4]: token 16 half + r, row 16 i + 4 kq + e */
    float *p;   /* [2 token halves][2][64][4]: exp(G_t - G_j) (q_t.k_j), 0 for j > t;
                 * t = 16 half + r, j = 8 kq + 4 i + e */
    float *gam; /* [1]: exp(G_C) */
    int *flag;  /* [1] */
    int t0, chunks; /* the segment */
};

/* silu(conv) of channel ch at tokens tb .. tb + nt - 1 of the chunk at t0 (0
 * from n on; nt a
 * multiple of CB) into dst[0], dst[ld], .., the sums of dn_conv_silu; bad
 * is set by a value past DC_BIG or not finite.  A round's loads are all in
 * flight; row j of [conv_state; mixed] past the end repeats the last one. */
template <int CB>
__device__ __forceinline__ void dc_conv(const DnRecArgs &a, int ch, int t0, int tb, int nt, float *dst, int ld, bool &bad) {
    const int k1 = a.kc - 1, last = a.n - 1 + k1;
    /* a chunk inside mixed (uniform over the workgroup) steps by whole rows */
    const bool inner = t0 >= k1 && t0 + DC_C - 1 + k1 <= last;
    const float *mp = a.mixed + (size_t)max(tb - k1, 0) * a.conv_dim + ch;
    auto row = [&](int j) {
        if (inner) return qk_ld(mp + (size_t)(uint32_t)(j - tb) * (uint32_t)a.conv_dim);
        j = min(j, last);
        return qk_ld(j < k1 ? a.conv_state + (size_t)j * a.conv_dim + ch : a.mixed + (size_t)(j - k1) * a.conv_dim + ch);
    };
    float w[4], x[CB + 3];
    const bool four = a.kc == 4;
    if (four) {
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = qk_bf16(qk_ld(a.conv_w + (size_t)ch * 4 + i));
#pragma unroll
        for (int i = 0; i < 3; i++) x[CB + i] = row(tb + i);
    }
#pragma unroll 1
    for (int u0 = 0; u0 < nt; u0 += CB) {
        float o[CB];
        if (four) {
#pragma unroll
            for (int i = 0; i < 3; i++) x[i] = x[CB + i];
#pragma unroll
            for (int u = 0; u < CB; u++) x[3 + u] = row(tb + u0 + u + 3);
#pragma unroll
            for (int u = 0; u < CB; u++)
                o[u] = fmaf(x[u + 3], w[3], fmaf(x[u + 2], w[2], fmaf(x[u + 1], w[1], fmaf(x[u], w[0], 0.0f))));
        } else {
#pragma unroll
            for (int u = 0; u < CB; u++) o[u] = 0.0f;
#pragma unroll 1
            for (int i = 0; i < a.kc; i++) {
                const float wi = qk_bf16(qk_ld(a.conv_w + (size_t)ch * a.kc + i));
#pragma unroll
                for (int u = 0; u < CB; u++) o[u] = fmaf(row(tb + u0 + u + i), wi, o[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < CB; u++) {
            const float v = tb + u0 + u < a.n ? qk_silu(o[u]) : 0.0f;
            bad |= !(fabsf(v) <= DC_BIG);
            dst[(u0 + u) * ld] = v;
        }
    }
}

/*
 * grid (chunks, hv), 256 threads.  Bound: the vector ALU (the substitution,
 * 496 fmas for each of dk + dv columns) and the reads of mixed, three times
 * over its rows for the value heads that share a key head.  103 us for 2048
 * tokens, 32 heads of 128 x 128.  Chunks of 64 would halve k_dc_seq's
 * barriers but double the substitution per token and leave room for one
 * workgroup per CU.
 */
template <int DK>
__global__ __launch_bounds__(256, 2) void k_dc_prep(DcArgs c) {
    constexpr int LD = DK + DC_LP, LV = DC_VB + DC_LP;
    __shared__ __attribute__((aligned(16))) float s_q[DC_C][LD], s_k[DC_C][LD];
    __shared__ __attribute__((aligned(16))) float s_at[DC_C][DC_C + DC_LP]; /* [j][t] = -A_tj */
    __shared__ __attribute__((aligned(16))) float s_v[DC_C][DC_VB + DC_LP];
    __shared__ __attribute__((aligned(16))) float s_p[DC_C][DC_C + DC_LP];
    __shared__ double s_g[DC_C];
    __shared__ float s_b[DC_C], s_eg[DC_C], s_ec[DC_C], s_n[2][DC_C];
    const DnRecArgs &a = c.r;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ck = blockIdx.x, h = blockIdx.y, t0 = c.t0 + DC_C * ck;
    const int kh = h / (a.hv / a.hk), key_dim = a.hk * DK;
    const size_t hc = (size_t)h * c.chunks + ck;
    bool bad = false;

    /* q and k channels */
    constexpr int NT = DK / 4 < DC_C ? DK / 4 : DC_C; /* tokens per thread and channel */
    for (int i = tid; i < 2 * DK * (DC_C / NT); i += 256) {
        const int chl = i % (2 * DK), tb = i / (2 * DK) * NT;
        const int ch = chl < DK ? kh * DK + chl : key_dim + kh * DK + (chl - DK);
        dc_conv<NT < 16 ? NT : 16>(a, ch, t0, t0 + tb, NT, chl < DK ? &s_q[tb][chl] : &s_k[tb][chl - DK], LD, bad);
    }
    auto conv_v = [&](int c0) {
        const int nv = min(DC_VB, a.dv - c0); /* 32, 64 or 128 */
        for (int i = tid; i < nv * 2; i += 256) {
            const int cl = i & (nv - 1), tb = i >= nv ? DC_C / 2 : 0;
            dc_conv<16>(a, 2 * key_dim + h * a.dv + c0 + cl, t0, t0 + tb, DC_C / 2, &s_v[tb][cl], LV, bad);
        }
    };
    conv_v(0);
    /* decays and beta: log g as the per-token path has it, floored where g is
     * long 0 in fp32; a token past the end changes nothing (g = 1, beta = 0) */
    if (tid < 64) {
        const int t = t0 + tid;
        double G = 0.0;
        float beta = 0.0f;
        if (tid < DC_C && t < a.n) {
            const float av = qk_ld(a.a + (size_t)t * a.hv + h), bv = qk_ld(a.b + (size_t)t * a.hv + h);
            const float al = expf(qk_ld(a.a_log + h));
            const float lg = -al * log1pf(expf(av + qk_ld(a.dt_bias + h)));
            bad |= !(fabsf(av) <= DC_BIG) || !(fabsf(bv) <= DC_BIG) || lg != lg;
            G = (double)fmaxf(lg, -200.0f);
            beta = 1.0f / (1.0f + expf(-bv));
        }
#pragma unroll
        for (int o = 1; o < DC_C; o <<= 1) {
            const double v = __shfl_up(G, o, QK_WAVE);
            if (lane >= o) G += v;
        }
        if (tid < DC_C) {
            s_g[tid] = G;
            s_eg[tid] = expf((float)G);
            s_b[tid] = beta;
            s_ec[tid] = expf((float)(__shfl(G, DC_C - 1, QK_WAVE) - G));
        }
    }
    __syncthreads();
    {
        /* four threads per (q or k, token) */
        const int which = tid >> 7, t = (tid >> 2) & 31, part = tid & 3;
        const float *row = which ? s_k[t] : s_q[t];
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < DK / 16; i++) {
            const float4 v = *(const float4 *)(row + 4 * (part + 4 * i));
            ss = fmaf(v.x, v.x, ss);
            ss = fmaf(v.y, v.y, ss);
            ss = fmaf(v.z, v.z, ss);
            ss = fmaf(v.w, v.w, ss);
        }
        ss = qk_group_sum<4>(ss);
        if (part == 0) s_n[which][t] = 1.0f / sqrtf(ss + 1e-6f);
    }
    __syncthreads();
    const float scale_q = 1.0f / sqrtf((float)DK);
    for (int i = tid; i < DC_C * DK; i += 256) {
        const int t = i / DK, d = i - t * DK;
        const float qv = (s_q[t][d] * s_n[0][t]) * scale_q;
        s_q[t][d] = qv;
        s_k[t][d] *= s_n[1][t];
    }
    __syncthreads();
    for (int i = tid; i < DC_C * DK / 4; i += 256) {
        const int l = i & 63, f = (i >> 6) % (DK / 16), t = 16 * ((i >> 6) / (DK / 16)) + (l & 15);
        const float4 v = *(const float4 *)&s_q[t][(l >> 4) * (DK / 4) + 4 * f];
        const float e = s_eg[t];
        qk_st((float4 *)(c.q + hc * DC_C * DK) + i, make_float4(e * v.x, e * v.y, e * v.z, e * v.w));
    }

    /* tiles 0..2: k.k of token blocks (0,0), (1,0), (1,1); 3..5: q.k; the
     * block (0,1) is zero */
    for (int id = wave; id < 7; id += 4) {
        if (id == 6) {
            *(float4 *)&s_p[lane >> 2][16 + 4 * (lane & 3)] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            continue;
        }
        const int tp = id >= 3 ? id - 3 : id, ti = tp > 0, tj = tp == 2;
        const int r = lane & 15, kq = lane >> 4;
        const float *ap = (id >= 3 ? s_q[16 * ti + r] : s_k[16 * ti + r]) + kq * (DK / 4), *bp = s_k[16 * tj + r] + kq * (DK / 4);
        dc_f32x4 acc[2];
#pragma unroll
        for (int i = 0; i < 4; i++) acc[0][i] = acc[1][i] = 0.0f;
#pragma unroll
        for (int s = 0; s < DK / 16; s++) {
            const dc_f32x4 av = *(const dc_f32x4 *)(ap + 4 * s), bv = *(const dc_f32x4 *)(bp + 4 * s);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e & 1] = DC_MFMA(av[e], bv[e], acc[e & 1]);
        }
        const int j = 16 * tj + r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = 16 * ti + 4 * kq + i;
            const float d = (acc[0][i] + acc[1][i]) * expf((float)(s_g[t] - s_g[min(j, t)]));
            if (id < 3) s_at[j][t] = j < t ? -s_b[t] * d : 0.0f;
            else s_p[t][j] = j <= t ? d : 0.0f;
        }
    }
    __syncthreads();

    {
        const int l = tid & 63, t = 16 * (tid >> 7) + (l & 15), j = 8 * (l >> 4) + 4 * ((tid >> 6) & 1);
        qk_st((float4 *)(c.p + hc * DC_C * DC_C) + tid, *(const float4 *)&s_p[t][j]);
    }
    /* (I + A) X = B, a column per thread: columns of -W (threads 0..127) and
     * of U0 (128..255), 128 of each a round */
    for (int c0 = 0; c0 < max(DK, a.dv); c0 += DC_VB) {
        if (c0 > 0) {
            __syncthreads(); /* the round before is out */
            if (c0 < a.dv) conv_v(c0);
            __syncthreads();
        }
        const bool isk = tid < DC_VB;
        const int col = c0 + (isk ? tid : tid - DC_VB), width = isk ? DK : a.dv;
        if (col < width) {
            float x[DC_C];
#pragma unroll
            for (int t = 0; t < DC_C; t++) x[t] = isk ? -(s_b[t] * s_eg[t]) * s_k[t][min(col, DK - 1)] : s_b[t] * s_v[t][tid & (DC_VB - 1)];
#pragma unroll
            for (int j = 0; j < DC_C - 1; j++) {
#pragma unroll
                for (int t4 = (j + 1) / 4; t4 < DC_C / 4; t4++) {
                    const float4 m = *(const float4 *)&s_at[j][4 * t4];
                    if (4 * t4 > j) x[4 * t4] = fmaf(m.x, x[j], x[4 * t4]);
                    if (4 * t4 + 1 > j) x[4 * t4 + 1] = fmaf(m.y, x[j], x[4 * t4 + 1]);
                    if (4 * t4 + 2 > j) x[4 * t4 + 2] = fmaf(m.z, x[j], x[4 * t4 + 2]);
                    if (4 * t4 + 3 > j) x[4 * t4 + 3] = fmaf(m.w, x[j], x[4 * t4 + 3]);
                }
            }
            /* over the queries and the v columns, both used up */
            float *dst = isk ? &s_q[0][min(col, DK - 1)] : &s_v[0][tid & (DC_VB - 1)];
            const int ld = isk ? LD : LV;
#pragma unroll
            for (int t = 0; t < DC_C; t++) dst[t * ld] = x[t];
        }
        if (c0 < a.dv) {
            __syncthreads();
            const int nv = min(DC_VB, a.dv - c0);
            for (int i = tid; i < nv * (DC_C / 4); i += 256) {
                const int l = i & 63, t = 16 * ((i >> 6) & 1) + (l & 15);
                qk_st((float4 *)(c.u0 + hc * DC_C * a.dv + (size_t)DC_C * c0) + i,
                      *(const float4 *)&s_v[t][16 * (i >> 7) + 4 * (l >> 4)]);
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < DC_C * DK / 4; i += 256) {
        const int l = i & 63, f = (i >> 6) % (DK / 16), t = 16 * ((i >> 6) / (DK / 16)) + (l & 15);
        qk_st((float4 *)(c.w + hc * DC_C * DK) + i, *(const float4 *)&s_q[t][(l >> 4) * (DK / 4) + 4 * f]);
    }
    /* exp(G_C - G_j) k_j, transposed */
    for (int i = tid; i < DK * (DC_C / 4); i += 256) {
        const int l = i & 63, d = 16 * (i >> 7) + (l & 15), j = 8 * (l >> 4) + 4 * ((i >> 6) & 1);
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = s_ec[j + u] * s_k[j + u][d];
        qk_st((float4 *)(c.kt + hc * DK * DC_C) + i, make_float4(v[0], v[1], v[2], v[3]));
    }
    const int any = __syncthreads_or(bad);
    if (tid == 0) {
        c.gam[hc] = s_eg[DC_C - 1];
        c.flag[hc] = any;
    }
}

__device__ __forceinline__ float dc_at(const float4 (&v)[2], int e) {
    const float4 x = v[e >> 2];
    return (e & 3) == 0 ? x.x : (e & 3) == 1 ? x.y : (e & 3) == 2 ? x.z : x.w;
}

/*
 * Workgroup = 16 state rows of a value head, through the segment's chunks.
 * Waves 0, 1 form u of the chunk's token halves, waves 2, 3 the state's part
 * of o; after a barrier waves 2, 3 add the u part and write o, and all four
 * update the state's 16-column tiles.  The state lives in registers (the
 * accumulator layout) and in LDS (the operand); a chunk's other operands go
 * from L2 straight to the registers of the one wave that uses them, loaded a
 * chunk ahead.  o is written without its gate, which k_dn_pack applies: here
 * its exponentials would sit in the chain.  Bound: the serial chain, dk/4 +
 * 24 fp32 matrix instructions and two barriers per chunk: 142 us for the 64
 * chunks of 2048 tokens (32 heads of 128 x 128), matrix cores busy a third.
 */
template <int DK>
__global__ __launch_bounds__(256, 1) void k_dc_seq(DcArgs c) {
    constexpr int NTL = DK / 16, OT = NTL >= 8 ? (NTL >= 16 ? 3 : 1) : 0, UT = NTL / 2 - OT; /* tiles per wave */
    constexpr int KF = DK / 16; /* float4s of a lane's dk run */
    constexpr int EPL = DK / 16;
    __shared__ __attribute__((aligned(16))) float s_s[DN_RB][DK + DC_LP];
    __shared__ __attribute__((aligned(16))) float s_u[DN_RB][DC_C + DC_LP];
    __shared__ DnRecSmem<DK> sh;
    const DnRecArgs &a = c.r;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, kq = lane >> 4, kind = wave >> 1, tt = wave & 1;
    /* the row blocks of one head on one XCD: they share its operands in L2 */
    const int nrb = a.dv / DN_RB;
    const int h = (blockIdx.x & 7) + 8 * (blockIdx.x / (8 * nrb)), rb = (blockIdx.x >> 3) % nrb * DN_RB;
    if (h >= a.hv) return;
    const int vd = a.hv * a.dv;
    const int cnt = kind ? OT : UT, d0 = 16 * (kind ? 2 * UT + tt * OT : tt * UT);
    const int tl = 16 * tt + r; /* this lane's token of the chunk */

    float *srow = a.rec_state + ((size_t)h * a.dv + rb) * DK;
    for (int i = tid; i < DN_RB * DK / 4; i += 256) {
        const int row = i / (DK / 4), d4 = i - row * (DK / 4);
        *(float4 *)&s_s[row][4 * d4] = qk_ld((const float4 *)(srow + (size_t)row * DK) + d4);
    }
    __syncthreads();
    dc_f32x4 S[UT];
    auto load_state = [&]() {
#pragma unroll
        for (int j = 0; j < UT; j++)
            if (j < cnt)
#pragma unroll
                for (int i = 0; i < 4; i++) S[j][i] = s_s[4 * kq + i][d0 + 16 * j + r];
    };
    load_state();

    struct Op {
        float4 b[KF], x, p[2], kt[UT][2];
        float g;
        int flag;
    };
    auto load = [&](Op &o, int ck) {
        const size_t hc = (size_t)h * c.chunks + ck;
        const float4 *bp = (const float4 *)((kind ? c.q : c.w) + hc * DC_C * DK) + tt * KF * 64 + lane;
#pragma unroll
        for (int i = 0; i < KF; i++) o.b[i] = qk_ld(bp + 64 * i);
        o.x = qk_ld((const float4 *)(c.u0 + hc * DC_C * a.dv + (size_t)DC_C * rb) + tt * 64 + lane); /* waves 0, 1 */
        const float4 *pp = (const float4 *)(c.p + hc * DC_C * DC_C) + tt * 128 + lane;
        o.p[0] = qk_ld(pp);
        o.p[1] = qk_ld(pp + 64);
#pragma unroll
        for (int j = 0; j < UT; j++) {
            const float4 *kp = (const float4 *)(c.kt + hc * DK * DC_C) + min(d0 / 16 + j, DK / 16 - 1) * 128 + lane;
            o.kt[j][0] = qk_ld(kp);
            o.kt[j][1] = qk_ld(kp + 64);
        }
        o.g = qk_ld(c.gam + hc);
        o.flag = qk_ld(c.flag + hc);
    };
    /* a chunk's outputs are stored at the next one's start, before its loads:
     * the loads are waited for at a chunk's end, and with them every store
     * issued before (one counter), which there has had a chunk's time */
    float4 out = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float out_ss = 0.0f;
    int out_t = a.n;
    auto store_out = [&]() {
        if (out_t < a.n) {
            qk_st((float4 *)(a.core + (size_t)out_t * vd + (size_t)h * a.dv + rb + 4 * kq), out);
            if (kq == 0) qk_st(a.ssp + ((size_t)out_t * a.hv + h) * nrb + rb / DN_RB, out_ss);
        }
        out_t = a.n;
    };
    auto step = [&](const Op &cur, Op &nxt, int ck) {
        store_out();
        load(nxt, min(ck + 1, c.chunks - 1));
        const int tg = c.t0 + DC_C * ck;
        if (__builtin_amdgcn_readfirstlane(cur.flag)) {
            const int row = tid >> 4, i0 = (tid & 15) * EPL;
            float s[EPL];
#pragma unroll
            for (int e = 0; e < EPL; e++) s[e] = s_s[row][i0 + e];
            dn_rec_tokens<EPL, true>(a, h, rb, tg, min(tg + DC_C, a.n), s, sh);
#pragma unroll
            for (int e = 0; e < EPL; e++) s_s[row][i0 + e] = s[e];
            __syncthreads();
            load_state();
            return;
        }
        /* u^T = U0^T + S (-W)^T, or the state's part of o^T = S Q'^T */
        dc_f32x4 acc[2], av[KF];
#pragma unroll
        for (int s = 0; s < KF; s++) av[s] = *(const dc_f32x4 *)&s_s[r][kq * (DK / 4) + 4 * s];
        __builtin_amdgcn_sched_barrier(0); /* every read out before the first product */
#pragma unroll
        for (int i = 0; i < 4; i++) acc[1][i] = 0.0f;
        acc[0] = kind ? acc[1] : dc_f32x4{cur.x.x, cur.x.y, cur.x.z, cur.x.w};
#pragma unroll
        for (int s = 0; s < KF; s++) {
            acc[0] = DC_MFMA(av[s][0], cur.b[s].x, acc[0]);
            acc[1] = DC_MFMA(av[s][1], cur.b[s].y, acc[1]);
            acc[0] = DC_MFMA(av[s][2], cur.b[s].z, acc[0]);
            acc[1] = DC_MFMA(av[s][3], cur.b[s].w, acc[1]);
        }
        if (!kind)
#pragma unroll
            for (int i = 0; i < 4; i++) s_u[4 * kq + i][tl] = acc[0][i] + acc[1][i];
        qk_lds_barrier();
        const dc_f32x4 u0 = *(const dc_f32x4 *)&s_u[r][8 * kq], u1 = *(const dc_f32x4 *)&s_u[r][8 * kq + 4];
        const float uu[8] = {u0[0], u0[1], u0[2], u0[3], u1[0], u1[1], u1[2], u1[3]};
#pragma unroll
        for (int j = 0; j < UT; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) S[j][i] *= cur.g;
        /* the tiles' chains side by side; kind is uniform over a wave */
        if (kind) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                acc[e & 1] = DC_MFMA(uu[e], dc_at(cur.p, e), acc[e & 1]);
#pragma unroll
                for (int j = 0; j < OT; j++) S[j] = DC_MFMA(uu[e], dc_at(cur.kt[j], e), S[j]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
#pragma unroll
                for (int j = 0; j < UT; j++) S[j] = DC_MFMA(uu[e], dc_at(cur.kt[j], e), S[j]);
        }
        /* the state's new operand copy: its last readers passed the barrier */
#pragma unroll
        for (int j = 0; j < UT; j++)
            if (j < cnt)
#pragma unroll
                for (int i = 0; i < 4; i++) s_s[4 * kq + i][d0 + 16 * j + r] = S[j][i];
        if (kind) {
            float ss = 0.0f, v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v[i] = acc[0][i] + acc[1][i];
                ss = fmaf(v[i], v[i], ss);
            }
            ss += __uint_as_float(qk_xor16_u(__float_as_uint(ss)));
            ss += __uint_as_float(qk_xor32_u(__float_as_uint(ss)));
            out = make_float4(v[0], v[1], v[2], v[3]);
            out_ss = ss;
            out_t = tg + tl;
        }
        qk_lds_barrier();
    };
    Op p0, p1; /* turn about, so nothing is moved between them */
    load(p0, 0);
    for (int ck = 0; ck < c.chunks; ck += 2) {
        step(p0, p1, ck);
        if (ck + 1 < c.chunks) step(p1, p0, ck + 1);
    }
    store_out();
#pragma unroll
    for (int j = 0; j < UT; j++)
        if (j < cnt)
#pragma unroll
            for (int i = 0; i < 4; i++) qk_st(srow + (size_t)(4 * kq + i) * DK + d0 + 16 * j + r, S[j][i]);
}

/* ------------------------------------------------------------ host side */

static size_t dc_floats(const qk_dn_shape *s, size_t chunks) {
    return (size_t)s->hv * chunks * ((size_t)DC_C * (3 * s->dk + s->dv) + DC_C * DC_C + 2);
}

extern "C" size_t qk_dn_chunk_bytes(const qk_dn_shape *s, int max_n) {
    const int n = max_n < DC_SEG ? max_n : DC_SEG;
    return dc_floats(s, (size_t)((n + DC_C - 1) / DC_C)) * 4;
}

template <int DK>
static int dc_launch(DcArgs &c, hipStream_t st) {
    const int hv = c.r.hv, n = c.r.n;
    float *base = c.w;
    for (c.t0 = 0; c.t0 < n; c.t0 += DC_SEG) {
        c.chunks = ((n - c.t0 < DC_SEG ? n - c.t0 : DC_SEG) + DC_C - 1) / DC_C;
        const size_t hc = (size_t)hv * c.chunks;
        c.w = base;
        c.q = c.w + hc * DC_C * DK;
        c.kt = c.q + hc * DC_C * DK;
        c.u0 = c.kt + hc * DC_C * DK;
        c.p = c.u0 + hc * DC_C * c.r.dv;
        c.gam = c.p + hc * DC_C * DC_C;
        c.flag = (int *)(c.gam + hc);
        hipLaunchKernelGGL(k_dc_prep<DK>, dim3(c.chunks, hv), dim3(256), 0, st, c);
        int rc = QK_CHECK_LAUNCH();
        if (rc) return rc;
        hipLaunchKernelGGL(k_dc_seq<DK>, dim3((hv + 7) / 8 * 8 * (c.r.dv / DN_RB)), dim3(256), 0, st, c);
        rc = QK_CHECK_LAUNCH();
        if (rc) return rc;
    }
    return 0;
}

extern "C" int qk_launch_dn_chunks(const void *rec_args, float *scratch, void *stream) {
    DcArgs c = {};
    c.r = *(const DnRecArgs *)rec_args;
    c.w = scratch;
    hipStream_t st = (hipStream_t)stream;
    switch (c.r.dk) {
    case 32: return dc_launch<32>(c, st);
    case 64: return dc_launch<64>(c, st);
    case 128: return dc_launch<128>(c, st);
    case 256: return dc_launch<256>(c, st);
    default: return (int)hipErrorInvalidValue;
    }
}
