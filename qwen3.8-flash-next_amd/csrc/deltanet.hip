/*
 * deltanet.hip -- the gated DeltaNet mixer (linear attention) on gfx950,
 * replacing deltanet_forward of the reference C port (c/src/model.c:
 * 1146-1278) for n tokens in three launches:
 *
 *   k_dn_in   one wave per four rows of [in_proj_qkv | in_proj_z | in_proj_a
 *             | in_proj_b]: the q4 rows with the per-group identity of
 *             gemm_q4 (kernel.c:279-282, gemv_parts.h), the bf16 rows as
 *             dot products of bf16 pairs; x (f32) enters as bf16 hi + lo
 *             pairs.  Writes mixed [n, conv_dim], z [n, value_dim], a, b
 *             [n, hv].
 *   k_dn_rec  one workgroup per (value head, block of 16 state rows), the
 *             state rows in registers across the tokens: per token the
 *             causal depthwise conv over [conv_state; mixed] (kernel.c:
 *             311-324) + silu for the head's q and k channels and its v
 *             rows, l2norm(q)*dk^-1/2 and l2norm(k) (kernel.c:73-78), the
 *             decay exp(-exp(A_log) softplus(a + dt_bias)) and beta =
 *             sigmoid(b), then per row S <- g S; kv = S.k; S += k (beta
 *             (v - kv)); o = S.q (model.c:1225-1248).  Writes o [n, value_dim]
 *             and the new recurrent state.
 *             The gated norm rmsnorm(o_h) * norm_w * sigmoid(z_h) (model.c:
 *             1263-1274) is split: k_dn_rec writes o * norm_w * sigmoid(z)
 *             per row and the sum of o^2 over its rows.
 *   k_dn_out  one wave per two rows of out_proj (q4); each lane scales its
 *             own columns by the head's 1/sqrt(sum(o^2)/dv + eps); also
 *             moves the conv state on by n tokens (its old rows are read by
 *             k_dn_rec, so it changes only here).
 *
 * From QK_DN_MM_N tokens on the projections run on MFMA instead (proj_mm.hip):
 * x packed once into operand planes, one grouped product for qkv | z and one
 * for a | b, and k_dn_pack in place of k_dn_out's scaling and conv state.
 * The GEMVs above walk the tokens one after another and convert x again in
 * every wave: at 2048 tokens (hidden 2048, heads 16/32 of 128) 10050 us for
 * k_dn_in and 5830 for k_dn_out, against 240 + 11 and 100 + 24.
 * From qk_dn_chunk_n tokens on k_dn_rec gives way to dn_chunk.hip (3225 us
 * there against 103 + 142).
 *
 * Sums run in parallel orders (lane trees), so results match the reference
 * to rounding, not bit for bit.
 */
#include "qk_device.h"
#include "gemv_parts.h"
#include "dn_rec.h"
#include "mfma_parts.h"

#define DN_RPW 4   /* rows per wave in the two GEMV kernels */

struct DnInArgs {
    const uint32_t *qkv_q, *z_q;
    const uint16_t *qkv_s, *qkv_b, *z_s, *z_b;
    const uint16_t *a_w, *b_w;
    const float *x;  /* [n, d] */
    float *mixed;    /* [n, conv_dim] */
    float *z;        /* [n, value_dim] */
    float *a, *b;    /* [n, hv] */
    int d, n, conv_dim, value_dim, hv;
};

template <int P>
__global__ __launch_bounds__(256) void k_dn_in(DnInArgs a) {
    const int lane = threadIdx.x & 63;
    const int r0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * DN_RPW;
    const int R1 = a.conv_dim, R2 = R1 + a.value_dim, R3 = R2 + a.hv, R = R3 + a.hv;
    const int CH = a.d >> 5, G = a.d >> 6;
    const size_t wrow = (size_t)a.d >> 3;
    __shared__ XWg<P> sh;
    XWgRaw<P> xr;
    load_xwg<P>(a.x, a.d, xr);
    /* q4 rows: codes, scales and biases of the wave's rows stay in registers */
    uint4 wq[DN_RPW][P];
    float ws[DN_RPW][P], wb[DN_RPW][P];
    if (r0 < R2) {
#pragma unroll
        for (int j = 0; j < DN_RPW; j++) {
            const int r = min(r0 + j, R2 - 1);
            const bool z = r >= R1;
            const int rr = z ? r - R1 : r;
            const uint32_t *q = (z ? a.z_q : a.qkv_q) + (size_t)rr * wrow;
            const uint16_t *s = (z ? a.z_s : a.qkv_s) + (size_t)rr * G;
            const uint16_t *bb = (z ? a.z_b : a.qkv_b) + (size_t)rr * G;
#pragma unroll
            for (int ps = 0; ps < P; ps++) {
                const int c0 = ps * 64 + lane;
                const bool ok = c0 < CH;
                const int c = ok ? c0 : 0;
                wq[j][ps] = qk_ld((const uint4 *)(q + 4 * (size_t)c));
                ws[j][ps] = ok ? qk_bf16(qk_ld(s + (c >> 1))) : 0.0f;
                wb[j][ps] = ok ? qk_bf16(qk_ld(bb + (c >> 1))) : 0.0f;
                if (!ok) wq[j][ps] = make_uint4(0u, 0u, 0u, 0u);
            }
        }
    }
    for (int t = 0; t < a.n; t++) {
        store_xwg<P>(xr, a.d, sh);
        qk_lds_barrier();
        if (t + 1 < a.n) load_xwg<P>(a.x + (size_t)(t + 1) * a.d, a.d, xr);
        XPairs<64, P, false> xp;
        read_xwg<P>(sh, lane, xp);
        if (r0 < R2) {
#pragma unroll
            for (int j = 0; j < DN_RPW; j++) {
                /* the codes stay codes: widened before the token loop, four rows
                 * of P = 2 took 288 registers, one wave a SIMD, and at P = 4
                 * they spilled.  One token of the mixer, us: hidden 4096, heads
                 * 32/32 40.5 -> 29.2, hidden 8192, heads 8/32 96 -> 89 */
                if (P >= 2)
#pragma unroll
                    for (int ps = 0; ps < P; ps++)
                        asm volatile("" : "+v"(wq[j][ps].x), "+v"(wq[j][ps].y), "+v"(wq[j][ps].z), "+v"(wq[j][ps].w));
                const float v = qk_group_sum<64>(row_part<64, P, false>(wq[j], ws[j], wb[j], xp));
                const int r = r0 + j;
                if (lane == 0 && r < R2) {
                    if (r < R1) qk_st(a.mixed + (size_t)t * a.conv_dim + r, v);
                    else qk_st(a.z + (size_t)t * a.value_dim + (r - R1), v);
                }
            }
        } else if (r0 < R) {
            /* bf16 rows (in_proj_a, in_proj_b): w pairs against the x pairs */
#pragma unroll
            for (int j = 0; j < DN_RPW; j++) {
                const int r = r0 + j;
                const int rc = min(r, R - 1);
                const bool isb = rc >= R3;
                const uint16_t *w = (isb ? a.b_w : a.a_w) + (size_t)(isb ? rc - R3 : rc - R2) * a.d;
                float part = 0.0f;
#pragma unroll
                for (int ps = 0; ps < P; ps++) {
                    const int c0 = ps * 64 + lane;
                    const bool ok = c0 < CH;
                    const uint4 *src = (const uint4 *)(w + 32 * (size_t)(ok ? c0 : 0));
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        uint32_t wp[4];
                        qk_bf16x8_to_pairs(qk_ld(src + g), wp);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const uint32_t w2 = ok ? wp[i] : 0u;
                            part = qk_dot2(xp.hi[ps][4 * g + i], w2, part);
                            part = qk_dot2(xp.lo[ps][4 * g + i], w2, part);
                        }
                    }
                }
                const float v = qk_group_sum<64>(part);
                if (lane == 0 && r < R) {
                    if (r < R3) qk_st(a.a + (size_t)t * a.hv + (r - R2), v);
                    else qk_st(a.b + (size_t)t * a.hv + (r - R3), v);
                }
            }
        }
        if (t + 1 < a.n) qk_lds_barrier(); /* sh is rewritten for the next token */
    }
}

/* ------------------------------------------------------------ recurrence */

template <int EPL>
__global__ __launch_bounds__(256) void k_dn_rec(DnRecArgs a) {
    constexpr int DK = 16 * EPL;
    __shared__ DnRecSmem<DK> sh;
    const int tid = threadIdx.x;
    const int h = blockIdx.y, rb = blockIdx.x * DN_RB;
    const int row = rb + (tid >> 4), i0 = (tid & 15) * EPL;
    float *srow = a.rec_state + ((size_t)h * a.dv + row) * DK + i0;
    float s[EPL];
    if (EPL % 4 == 0) {
#pragma unroll
        for (int e = 0; e < EPL; e += 4) {
            const float4 v = qk_ld((const float4 *)(srow + e));
            s[e] = v.x; s[e + 1] = v.y; s[e + 2] = v.z; s[e + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int e = 0; e < EPL; e++) s[e] = qk_ld(srow + e);
    }
    dn_rec_tokens<EPL, false>(a, h, rb, 0, a.n, s, sh);
    if (EPL % 4 == 0) {
#pragma unroll
        for (int e = 0; e < EPL; e += 4)
            qk_st((float4 *)(srow + e), make_float4(s[e], s[e + 1], s[e + 2], s[e + 3]));
    } else {
#pragma unroll
        for (int e = 0; e < EPL; e++) qk_st(srow + e, s[e]);
    }
}

/* ------------------------------------------------------------ out_proj */

struct DnOutArgs {
    const uint32_t *out_q;
    const uint16_t *out_s, *out_b;
    const float *core;         /* [n, value_dim]: o * norm_w * sigmoid(z) */
    const float *ssp;          /* [n, hv, dv/16] */
    const float *mixed;        /* [n, conv_dim] */
    float *conv_state;         /* [kc-1, conv_dim], moved on by n tokens */
    float *out;                /* [n, d] */
    float *hyper;              /* INJ: [n, hc, d], hyper[t, j] += inject[t, j] * out[t] */
    const float *inject;       /* INJ: [n, hc] */
    int n, d, value_dim, dv, kc, conv_dim, ch_per_wg, hc;
};

#define DN_ORW 2 /* out_proj rows per wave */

#define DN_KCMAX 16 /* conv taps at most */
#define DN_NBU 16   /* sums-of-squares partials per head loaded at once */

/*
 * One wave per DN_ORW rows of out_proj.  The gated norm's head factor
 * r = 1/sqrt(sum(o^2)/dv + eps) comes from the per-block sums of squares
 * of k_dn_rec (dv/16 of them per head, loaded together and added in
 * order); each thread scales its units (8 columns of one head) and
 * splits them into bf16 hi + lo pairs for the workgroup (XWg).  The code
 * words are loaded first; the conv state moves on at the end (its stores
 * would otherwise hold the loads back).
 */
template <int P, bool INJ>
__global__ __launch_bounds__(256) void k_dn_out(DnOutArgs a) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int K = a.value_dim, CH = K >> 5, G = K >> 6;
    const size_t wrow = (size_t)K >> 3;

    /* the conv state: channels [c0, c0 + ch_per_wg) move on by n tokens;
     * every new value is read now, written at the end */
    const int cc = blockIdx.x * a.ch_per_wg + tid;
    const bool cthr = tid < a.ch_per_wg && cc < a.conv_dim;
    float cv[DN_KCMAX - 1];
    if (cthr) {
#pragma unroll
        for (int j = 0; j < DN_KCMAX - 1; j++)
            if (j < a.kc - 1) {
                const int m = a.n + j;
                cv[j] = m < a.kc - 1 ? a.conv_state[(size_t)m * a.conv_dim + cc]
                                     : qk_ld(a.mixed + (size_t)(m - (a.kc - 1)) * a.conv_dim + cc);
            }
    }

    const int r0 = (blockIdx.x * 4 + (tid >> 6)) * DN_ORW;
    const int nb = a.dv / DN_RB;
    __shared__ XWg<P> sh;
    uint4 wq[DN_ORW][P];
    float ws[DN_ORW][P], wb[DN_ORW][P];
#pragma unroll
    for (int j = 0; j < DN_ORW; j++) {
        const int r = min(r0 + j, a.d - 1);
#pragma unroll
        for (int ps = 0; ps < P; ps++) {
            const int c0 = ps * 64 + lane;
            const bool ok = c0 < CH;
            const int c = ok ? c0 : 0;
            wq[j][ps] = qk_ld((const uint4 *)(a.out_q + (size_t)r * wrow + 4 * (size_t)c));
            ws[j][ps] = ok ? qk_bf16(qk_ld(a.out_s + (size_t)r * G + (c >> 1))) : 0.0f;
            wb[j][ps] = ok ? qk_bf16(qk_ld(a.out_b + (size_t)r * G + (c >> 1))) : 0.0f;
            if (!ok) wq[j][ps] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    for (int t = 0; t < a.n; t++) {
        /* INJ: lane (row, copy) has the copy's inject weight and the hyper
         * value of the row, loaded before the row sums (a load per copy and
         * row, every lane the same address: 7.9 us among other layers, 7.2 so) */
        const int ir = lane / QK_INJECT_MAX_HC, iq = lane % QK_INJECT_MAX_HC;
        const bool il = INJ && ir < DN_ORW && iq < a.hc && r0 + ir < a.d;
        float iv = 0.0f, hv = 0.0f;
        float *hp = INJ ? a.hyper + ((size_t)t * a.hc + (il ? iq : 0)) * a.d + (il ? r0 + ir : 0) : nullptr;
        if (il) {
            iv = qk_ld(a.inject + (size_t)t * a.hc + iq);
            hv = qk_ld(hp);
        }
        XWgRaw<P> xr;
        load_xwg<P>(a.core + (size_t)t * K, K, xr);
#pragma unroll
        for (int k = 0; k < P; k++) {
            const int u = tid + 256 * k, c8 = u < (K >> 3) ? 8 * u : 0;
            const float *sp = a.ssp + ((size_t)t * (K / a.dv) + c8 / a.dv) * nb;
            float ss = 0.0f;
            for (int j0 = 0; j0 < nb; j0 += DN_NBU) {
                float pv[DN_NBU];
#pragma unroll
                for (int j = 0; j < DN_NBU; j++) pv[j] = qk_ld(sp + min(j0 + j, nb - 1));
#pragma unroll
                for (int j = 0; j < DN_NBU; j++) ss = ss + (j0 + j < nb ? pv[j] : 0.0f);
            }
            const float r = 1.0f / sqrtf(ss / (float)a.dv + 1e-6f);
#pragma unroll
            for (int w = 0; w < 2; w++) {
                const float4 v = xr.f[k][w];
                xr.f[k][w] = make_float4(v.x * r, v.y * r, v.z * r, v.w * r);
            }
        }
        store_xwg<P>(xr, K, sh);
        qk_lds_barrier();
        XPairs<64, P, false> xp;
        read_xwg<P>(sh, lane, xp);
#pragma unroll
        for (int j = 0; j < DN_ORW; j++) {
            const float v = qk_group_sum<64>(row_part<64, P, false>(wq[j], ws[j], wb[j], xp));
            const int rr = r0 + j;
            if (lane == 0 && rr < a.d) {
                if (a.out) qk_st(a.out + (size_t)t * a.d + rr, v);
            }
            if (il && ir == j) qk_st(hp, fmaf(iv, v, hv));
        }
        if (t + 1 < a.n) qk_lds_barrier(); /* sh is rewritten for the next token */
    }
    if (cthr) {
#pragma unroll
        for (int j = 0; j < DN_KCMAX - 1; j++)
            if (j < a.kc - 1) a.conv_state[(size_t)j * a.conv_dim + cc] = cv[j];
    }
}

/*
 * Many tokens: core scaled by its head's 1/sqrt(sum(o^2)/dv + eps) as
 * operand planes of out_proj; the workgroups past the planes move the conv state
 * on by n tokens.
 */
struct DnPackArgs {
    const float *core, *ssp, *mixed;
    const float *z, *norm_w; /* z set: core is o itself (the chunked recurrence), gated here */
    float *conv_state;
    qk_planes pl;
    int n, value_dim, dv, kc, conv_dim;
};

__global__ __launch_bounds__(256) void k_dn_pack(DnPackArgs a) {
    const int G = a.value_dim / 64;
    const unsigned pack_wgs = qm_pack_wgs(a.n, G);
    if (blockIdx.x >= pack_wgs) {
        const int cc = (int)(blockIdx.x - pack_wgs) * 256 + threadIdx.x;
        if (cc >= a.conv_dim) return;
        float cv[DN_KCMAX - 1];
#pragma unroll
        for (int j = 0; j < DN_KCMAX - 1; j++)
            if (j < a.kc - 1) {
                const int m = a.n + j;
                cv[j] = m < a.kc - 1 ? a.conv_state[(size_t)m * a.conv_dim + cc]
                                     : qk_ld(a.mixed + (size_t)(m - (a.kc - 1)) * a.conv_dim + cc);
            }
#pragma unroll
        for (int j = 0; j < DN_KCMAX - 1; j++)
            if (j < a.kc - 1) a.conv_state[(size_t)j * a.conv_dim + cc] = cv[j];
        return;
    }
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int rb = u / G, g = u - rb * G, t = 8 * rb + (lane & 7);
    if (8 * rb >= a.n) return;
    const int tc = min(t, a.n - 1), col = 64 * g + 8 * (lane >> 3), nb = a.dv / DN_RB;
    const size_t i = ((size_t)tc * a.value_dim + col) / 8;
    const float4 a0 = qk_ld((const float4 *)a.core + 2 * i), a1 = qk_ld((const float4 *)a.core + 2 * i + 1);
    const float *sp = a.ssp + ((size_t)tc * (a.value_dim / a.dv) + col / a.dv) * nb;
    float ss = 0.0f;
    for (int j0 = 0; j0 < nb; j0 += 8) {
        float pv[8];
#pragma unroll
        for (int j = 0; j < 8; j++) pv[j] = qk_ld(sp + min(j0 + j, nb - 1));
#pragma unroll
        for (int j = 0; j < 8; j++) ss = ss + (j0 + j < nb ? pv[j] : 0.0f);
    }
    const float r = 1.0f / sqrtf(ss / (float)a.dv + 1e-6f);
    float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
    if (a.z) {
        const float4 z0 = qk_ld((const float4 *)a.z + 2 * i), z1 = qk_ld((const float4 *)a.z + 2 * i + 1);
        const float4 *np = (const float4 *)(a.norm_w + col % a.dv);
        const float4 n0 = qk_ld(np), n1 = qk_ld(np + 1);
        const float zv[8] = {z0.x, z0.y, z0.z, z0.w, z1.x, z1.y, z1.z, z1.w};
        const float nv[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = (v[j] * nv[j]) * (1.0f / (1.0f + expf(-zv[j])));
    }
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] *= r;
    qm_pack_store(a.pl, t, a.n, g, G, v);
}

/* ------------------------------------------------------------ host side */

extern "C" int qk_dn_shape_ok(const qk_dn_shape *s) {
    const int key_dim = s->hk * s->dk, value_dim = s->hv * s->dv;
    const int conv_dim = 2 * key_dim + value_dim;
    if (s->d <= 0 || s->d % 64 || s->d > 8192) return 0;
    if (s->hk <= 0 || s->hv <= 0 || s->hv % s->hk) return 0;
    if (!(s->dk == 32 || s->dk == 64 || s->dk == 128 || s->dk == 256)) return 0;
    /* dv: a power-of-two count (<= 64) of 32-column chunks */
    if (!(s->dv == 32 || s->dv == 64 || s->dv == 128 || s->dv == 256 || s->dv == 512 ||
          s->dv == 1024 || s->dv == 2048))
        return 0;
    /* out_proj takes value_dim inputs in q4 groups of 64 */
    if (value_dim > 8192 || value_dim % 64) return 0;
    if (s->kc < 1 || s->kc > 16) return 0;
    if (conv_dim <= 0) return 0;
    return 1;
}

/* conv-state channels that each workgroup of k_dn_out moves on */
static int dn_ch_per_wg(int d, int conv_dim, int &owgs) {
    owgs = (d + 4 * DN_ORW - 1) / (4 * DN_ORW);
    return (conv_dim + owgs - 1) / owgs;
}

extern "C" int qk_launch_dn(const qk_dn_shape *s, const qk_dn_dev *W, const float *x, int n, float *out,
                            float *conv_state, float *rec_state, float *mixed, float *z, float *av,
                            float *bv, float *core, float *ssp, const qk_planes *pl, float *chunk,
                            const qk_inject *inj_in, void *stream) {
    if (n <= 0) return 0;
    if (!qk_dn_shape_ok(s)) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    const int key_dim = s->hk * s->dk, value_dim = s->hv * s->dv;
    const int conv_dim = 2 * key_dim + value_dim;
    const bool inj = inj_in && inj_in->hyper;
    if (inj && (inj_in->hc < 1 || inj_in->hc > QK_INJECT_MAX_HC || !inj_in->inject)) return (int)hipErrorInvalidValue;
    /* more conv channels to a row of out_proj than k_dn_out can move: refused
     * at every token count, before anything is launched */
    int owgs;
    const int ch_per_wg = dn_ch_per_wg(s->d, conv_dim, owgs);
    if (ch_per_wg > 256) return (int)hipErrorInvalidValue;
    int rc;
    const bool mm = n >= QK_DN_MM_N;
    if (mm) {
        if (!pl || !pl->a || !pl->pg) return (int)hipErrorInvalidValue;
        rc = qk_launch_proj_pack(x, n, s->d, pl, stream);
        if (rc) return rc;
        qk_proj p = {};
        p.seg[0] = {W->qkv_q, W->qkv_s, W->qkv_b, mixed, conv_dim, conv_dim};
        p.seg[1] = {W->z_q, W->z_s, W->z_b, z, value_dim, value_dim};
        p.nseg = 2;
        p.pl = *pl;
        p.K = s->d; p.n = n;
        p.bw[0] = W->a_w; p.bw[1] = W->b_w;
        p.bout[0] = av; p.bout[1] = bv;
        p.brows = s->hv;
        rc = qk_launch_proj(&p, stream);
        if (rc) return rc;
    } else {
    DnInArgs ia;
    ia.qkv_q = W->qkv_q; ia.qkv_s = W->qkv_s; ia.qkv_b = W->qkv_b;
    ia.z_q = W->z_q; ia.z_s = W->z_s; ia.z_b = W->z_b;
    ia.a_w = W->a_w; ia.b_w = W->b_w;
    ia.x = x; ia.mixed = mixed; ia.z = z; ia.a = av; ia.b = bv;
    ia.d = s->d; ia.n = n; ia.conv_dim = conv_dim; ia.value_dim = value_dim; ia.hv = s->hv;
    const int rows = conv_dim + value_dim + 2 * s->hv;
    const int waves = (rows + DN_RPW - 1) / DN_RPW;
    const dim3 igrid((waves + 3) / 4);
    const int p_in = (s->d / 32 + 63) / 64;
    switch (p_in) {
    case 1: hipLaunchKernelGGL(k_dn_in<1>, igrid, dim3(256), 0, st, ia); break;
    case 2: hipLaunchKernelGGL(k_dn_in<2>, igrid, dim3(256), 0, st, ia); break;
    case 3: hipLaunchKernelGGL(k_dn_in<3>, igrid, dim3(256), 0, st, ia); break;
    default: hipLaunchKernelGGL(k_dn_in<4>, igrid, dim3(256), 0, st, ia); break;
    }
    rc = QK_CHECK_LAUNCH();
    if (rc) return rc;
    }

    DnRecArgs ra;
    ra.mixed = mixed; ra.a = av; ra.b = bv;
    ra.conv_state = conv_state; ra.conv_w = W->conv_w;
    ra.a_log = W->a_log; ra.dt_bias = W->dt_bias;
    ra.z = z; ra.norm_w = W->norm_w;
    ra.rec_state = rec_state; ra.core = core; ra.ssp = ssp;
    ra.n = n; ra.hk = s->hk; ra.hv = s->hv; ra.dk = s->dk; ra.dv = s->dv; ra.kc = s->kc;
    ra.conv_dim = conv_dim;
    const dim3 rgrid(s->dv / DN_RB, s->hv);
    const bool chunks = n >= qk_dn_chunk_n(s);
    if (chunks) {
        if (!chunk) return (int)hipErrorInvalidValue;
        rc = qk_launch_dn_chunks(&ra, chunk, stream);
        if (rc) return rc;
    } else switch (s->dk) {
    case 32: hipLaunchKernelGGL(k_dn_rec<2>, rgrid, dim3(256), 0, st, ra); break;
    case 64: hipLaunchKernelGGL(k_dn_rec<4>, rgrid, dim3(256), 0, st, ra); break;
    case 128: hipLaunchKernelGGL(k_dn_rec<8>, rgrid, dim3(256), 0, st, ra); break;
    default: hipLaunchKernelGGL(k_dn_rec<16>, rgrid, dim3(256), 0, st, ra); break;
    }
    rc = QK_CHECK_LAUNCH();
    if (rc) return rc;

    if (mm) {
        const DnPackArgs ka = {core, ssp, mixed, chunks ? z : nullptr, W->norm_w, conv_state, *pl, n, value_dim, s->dv, s->kc, conv_dim};
        hipLaunchKernelGGL(k_dn_pack, dim3(qm_pack_wgs(n, value_dim / 64) + (unsigned)(conv_dim + 255) / 256),
                           dim3(256), 0, st, ka);
        rc = QK_CHECK_LAUNCH();
        if (rc) return rc;
        qk_proj p = {};
        p.seg[0] = {W->out_q, W->out_s, W->out_b, out, s->d, s->d};
        p.nseg = 1;
        p.pl = *pl;
        p.K = value_dim; p.n = n;
        if (inj) { p.hyper = inj_in->hyper; p.inject = inj_in->inject; p.hc = inj_in->hc; }
        return qk_launch_proj(&p, stream);
    }

    DnOutArgs oa;
    oa.out_q = W->out_q; oa.out_s = W->out_s; oa.out_b = W->out_b;
    oa.core = core; oa.ssp = ssp; oa.mixed = mixed;
    oa.conv_state = conv_state; oa.out = out;
    oa.hyper = inj ? inj_in->hyper : nullptr;
    oa.inject = inj ? inj_in->inject : nullptr;
    oa.hc = inj ? inj_in->hc : 1;
    oa.n = n; oa.d = s->d; oa.value_dim = value_dim; oa.dv = s->dv; oa.kc = s->kc;
    oa.conv_dim = conv_dim;
    oa.ch_per_wg = ch_per_wg;
    const int p_out = (value_dim / 32 + 63) / 64;
    switch (p_out) {
#define DN_OUT_L(P)                                                                          \
    do {                                                                                     \
        if (inj) hipLaunchKernelGGL((k_dn_out<P, true>), dim3(owgs), dim3(256), 0, st, oa);  \
        else hipLaunchKernelGGL((k_dn_out<P, false>), dim3(owgs), dim3(256), 0, st, oa);     \
    } while (0)
    case 1: DN_OUT_L(1); break;
    case 2: DN_OUT_L(2); break;
    case 3: DN_OUT_L(3); break;
    default: DN_OUT_L(4); break;
#undef DN_OUT_L
    }
    return QK_CHECK_LAUNCH();
}

/* a fill kernel for the state (graph capture records no memset node) */
__global__ __launch_bounds__(256) void k_dn_zero(float *p, size_t count) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < count) p[i] = 0.0f;
}

extern "C" int qk_launch_dn_zero(float *p, size_t count, void *stream) {
    if (count == 0) return 0;
    hipLaunchKernelGGL(k_dn_zero, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       p, count);
    return QK_CHECK_LAUNCH();
}
