/*
 * dn_rec.h -- the DeltaNet recurrence token by token for one workgroup: 16
 * state rows of one value head, shared by the one-launch recurrence
 * (deltanet.hip) and the chunked one (dn_chunk.hip, for chunks whose values
 * its matrix products cannot carry).
 */
#ifndef DN_REC_H
#define DN_REC_H

#include "qk_device.h"

#define DN_RB 16   /* state rows per recurrence workgroup */

struct DnRecArgs {
    const float *mixed, *a, *b;  /* [n, conv_dim], [n, hv], [n, hv] */
    const float *conv_state;     /* [kc-1, conv_dim], the state before these tokens */
    const uint16_t *conv_w;      /* [conv_dim, kc] */
    const float *a_log, *dt_bias;
    const float *z;              /* [n, value_dim] */
    const float *norm_w;         /* [dv] */
    float *rec_state;            /* [hv, dv, dk] */
    float *core;                 /* [n, value_dim]: o * norm_w * sigmoid(z) */
    float *ssp;                  /* [n, hv, dv/16]: sums of o^2 over each block's rows */
    int n, hk, hv, dk, dv, kc, conv_dim;
};

/* silu(conv) of channels ch[0..NC) at token t: sum over taps i of
 * w[c, i] * seq[t+i, c] with seq = [conv_state rows; mixed rows], the fma
 * chain over i ascending.  The taps come four at a time with every load of
 * a round (all NC channels) in flight: a loop with a runtime trip count
 * would wait on each load.  Past kc the last tap is read again, unused. */
template <int NC>
__device__ __forceinline__ void dn_conv_silu(const DnRecArgs &a, int t, const int (&ch)[NC], float (&out)[NC]) {
    float acc[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) acc[c] = 0.0f;
    for (int i0 = 0; i0 < a.kc; i0 += 4) {
        float sv[NC][4];
        uint16_t wv[NC][4];
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = min(i0 + u, a.kc - 1), j = t + i;
                const float *src = j < a.kc - 1 ? a.conv_state + (size_t)j * a.conv_dim + ch[c]
                                                : a.mixed + (size_t)(j - (a.kc - 1)) * a.conv_dim + ch[c];
                sv[c][u] = qk_ld(src);
                wv[c][u] = qk_ld(a.conv_w + (size_t)ch[c] * a.kc + i);
            }
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (i0 + u < a.kc) acc[c] = fmaf(sv[c][u], qk_bf16(wv[c][u]), acc[c]);
    }
#pragma unroll
    for (int c = 0; c < NC; c++) out[c] = qk_silu(acc[c]);
}

template <int DK>
struct DnRecSmem {
    alignas(16) float ch[2 * DK + DN_RB]; /* q, k, v of the block's rows, read 16 bytes at a time */
    float sc[4];              /* q and k norms, decay, beta */
    float o[DN_RB];           /* the block's outputs of this token */
};

/* tokens [t0, t1) on the state rows rb.. of head h: thread = row rb + tid/16,
 * columns (tid % 16) * EPL + 0..EPL-1 of it in s.  RAW: core gets o itself */
template <int EPL, bool RAW>
__device__ __forceinline__ void dn_rec_tokens(const DnRecArgs &a, int h, int rb, int t0, int t1, float (&s)[EPL],
                                              DnRecSmem<16 * EPL> &sh) {
    constexpr int DK = 16 * EPL;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kh = h / (a.hv / a.hk);
    const int key_dim = a.hk * DK, value_dim = a.hv * a.dv;
    const int row = rb + (tid >> 4), i0 = (tid & 15) * EPL;
    const float al = expf(qk_ld(a.a_log + h)), dtb = qk_ld(a.dt_bias + h);
    const float scale_q = 1.0f / sqrtf((float)DK);
    for (int t = t0; t < t1; t++) {
        /* what the token's later steps read, loaded with the channels' taps
         * (every thread loads them; the addresses are shared) */
        const size_t zi = (size_t)t * value_dim + (size_t)h * a.dv + row;
        const float zv = qk_ld(a.z + zi), nwv = qk_ld(a.norm_w + row);
        const float av = qk_ld(a.a + (size_t)t * a.hv + h), bv = qk_ld(a.b + (size_t)t * a.hv + h);
        {
            /* the block's q, k, v channels, NCC per thread (all their loads
             * in flight); past the last one a thread repeats it */
            constexpr int NCC = (2 * DK + DN_RB + 255) / 256;
            int ch[NCC];
#pragma unroll
            for (int u = 0; u < NCC; u++) {
                const int c = min(tid + 256 * u, 2 * DK + DN_RB - 1);
                ch[u] = c < DK ? kh * DK + c
                      : c < 2 * DK ? key_dim + kh * DK + (c - DK)
                                   : 2 * key_dim + h * a.dv + rb + (c - 2 * DK);
            }
            float v[NCC];
            dn_conv_silu<NCC>(a, t, ch, v);
#pragma unroll
            for (int u = 0; u < NCC; u++)
                if (tid + 256 * u < 2 * DK + DN_RB) sh.ch[tid + 256 * u] = v[u];
        }
        __syncthreads();
        if (wave < 2) {
            /* wave 0: |q|^2, wave 1: |k|^2 */
            float ss = 0.0f;
            for (int i = lane; i < DK; i += 64) {
                const float v = sh.ch[wave * DK + i];
                ss = fmaf(v, v, ss);
            }
            ss = qk_group_sum<64>(ss);
            if (lane == 0) sh.sc[wave] = 1.0f / sqrtf(ss + 1e-6f);
        } else if (tid == 128) {
            sh.sc[2] = expf(-al * log1pf(expf(av + dtb)));
            sh.sc[3] = 1.0f / (1.0f + expf(-bv));
        }
        __syncthreads();
        const float rq = sh.sc[0], rk = sh.sc[1], g = sh.sc[2], beta = sh.sc[3];
        float kk[EPL], qq[EPL];
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            kk[e] = sh.ch[DK + i0 + e] * rk;
            qq[e] = (sh.ch[i0 + e] * rq) * scale_q;
        }
        float kv = 0.0f;
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            s[e] = s[e] * g;
            kv = fmaf(s[e], kk[e], kv);
        }
        kv = qk_group_sum<16>(kv);
        const float delta = (sh.ch[2 * DK + (tid >> 4)] - kv) * beta;
        float o = 0.0f;
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            s[e] = fmaf(kk[e], delta, s[e]);
            o = fmaf(s[e], qq[e], o);
        }
        o = qk_group_sum<16>(o);
        if ((tid & 15) == 0) {
            /* the gated norm's row factors here, its head factor (from the
             * sums of squares) in k_dn_out */
            qk_st(a.core + zi, RAW ? o : (o * nwv) * (1.0f / (1.0f + expf(-zv))));
            sh.o[tid >> 4] = o;
        }
        __syncthreads();
        if (tid == 0) {
            float ss = 0.0f;
            for (int j = 0; j < DN_RB; j++) ss = fmaf(sh.o[j], sh.o[j], ss);
            qk_st(a.ssp + ((size_t)t * a.hv + h) * (a.dv / DN_RB) + rb / DN_RB, ss);
        }
        __syncthreads(); /* s_ch, s_sc, s_o are rewritten for the next token */
    }
}

#endif
