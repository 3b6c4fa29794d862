/*
 * proj_mm.hip -- the mixers' q4 projections for many tokens on bf16 MFMA
 * (v_mfma_f32_32x32x16_bf16): out[t, r] = x[t] . W[r] for the row segments
 * of one input (DeltaNet in_proj_qkv | in_proj_z, and out_proj; attention
 * q | k | v, and o_proj), replacing the per-token GEMVs of linear_forward
 * (reference c/src/model.c:193-202 -> gemm_q4, kernel.c:230-309).
 *
 * The arithmetic is the expert GEMM's (ffn_mfma.hip): f32 activations as
 * bf16 hi + lo planes in (x_i, x_{i+4}) pair order (qk_planes), codes as
 * the exact bf16 numbers 16 + q, every 64-column group's accumulator
 * started at -16 sum(x) so it ends at sum x q, one fp32 fma per output
 * and group for the scale, and the bias term sum_g b_g X_g as a K = G
 * product at the end.  Accumulation is fp32 throughout, as in the GEMV.
 *
 * Bound: matrix cores (n = 2048: 103 GFLOP for qkv | z, twice that issued
 * for hi + lo).  Measured 240 us there, 430 TFLOP/s (860 issued); the matrix
 * cores are busy 40 % of the time, the rest goes to the decode, the scale
 * fmas and the waits between them.  The address path comes next: a load whose
 * lanes sit in different rows touches a line per row, so the planes lie in
 * operand order (qk_planes; as rows, staged through registers, 272 us), the
 * group sums by group and the scales come eight at a time (one at a time with
 * a sum per row 315).
 *
 * 32x32x16 lane layout: A lane l holds row l%32, B lane l column l%32, both
 * eight K elements of half h = l/32; D lane l holds column l%32, rows
 * 8*(i/4) + 4*h + i%4.  K-step j of a group gives half h the chunk 4*h + j
 * (8 columns, one code word), so a lane's four code words of a group are
 * one 16-byte load.
 */
#include "qk_device.h"
#include "mfma_parts.h"

typedef float qm_f32x16 __attribute__((ext_vector_type(16)));

#define PJ_THREADS 256
#define QK_PROJ_FEW_N 320

/* the segment and local first row of column block cb (64 columns); false
 * past the last one */
__device__ __forceinline__ bool pj_segment(const qk_proj &a, int cb, const uint32_t *&q, const uint16_t *&s,
                                           const uint16_t *&b, float *&out, int &ostride, int &r0) {
    int sg = 0, base = 0;
    if (a.nseg > 1 && cb >= a.end64[0]) { sg = 1; base = a.end64[0]; }
    if (a.nseg > 2 && cb >= a.end64[1]) { sg = 2; base = a.end64[1]; }
    q = a.seg[0].q; s = a.seg[0].s; b = a.seg[0].b; out = a.seg[0].out; ostride = a.seg[0].ostride;
    if (sg == 1) { q = a.seg[1].q; s = a.seg[1].s; b = a.seg[1].b; out = a.seg[1].out; ostride = a.seg[1].ostride; }
    if (sg == 2) { q = a.seg[2].q; s = a.seg[2].s; b = a.seg[2].b; out = a.seg[2].out; ostride = a.seg[2].ostride; }
    r0 = (cb - base) * 64;
    return cb < a.end64[a.nseg - 1];
}

/* eight group sums P of a row (pg: of group 0, the next group ld on) from
 * group k0 on (0 past G) as X = P / -128 in three bf16 parts, 24 bits: with a zero point inside the code range the
 * bias term is as large as the code term and cancels most of it, so two
 * parts (2^-17 of it) would show in the result */
__device__ __forceinline__ void pj_bias_x(const float *pg, size_t ld, int k0, int G, qm_bf16x8 (&X)[3]) {
    uint32_t w[3][4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float p0 = qk_ld(pg + ld * min(k0 + 2 * j, G - 1)), p1 = qk_ld(pg + ld * min(k0 + 2 * j + 1, G - 1));
        float x0 = k0 + 2 * j < G ? p0 * (-1.0f / 128.0f) : 0.0f;
        float x1 = k0 + 2 * j + 1 < G ? p1 * (-1.0f / 128.0f) : 0.0f;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            w[i][j] = qk_cvt_pk_bf16(x0, x1);
            x0 = x0 - qk_bf16_lo(w[i][j]);
            x1 = x1 - qk_bf16_hi(w[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < 3; i++) X[i] = __builtin_bit_cast(qm_bf16x8, make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]));
}

/* the bias words b[col][k0 .. k0+8) (0 past G), one load each: a row of
 * biases is only 2-byte aligned when G is odd */
__device__ __forceinline__ qm_bf16x8 pj_bias_w(const uint16_t *bp, int k0, int G) {
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t b0 = qk_ld(bp + min(k0 + 2 * j, G - 1)), b1 = qk_ld(bp + min(k0 + 2 * j + 1, G - 1));
        w[j] = (k0 + 2 * j < G ? b0 : 0u) | ((k0 + 2 * j + 1 < G ? b1 : 0u) << 16);
    }
    return __builtin_bit_cast(qm_bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}

#define PJ_MFMA(A, B, C) __builtin_amdgcn_mfma_f32_32x32x16_bf16((A), (B), (C), 0, 0, 0)

/* one output: the store, and with INJ the gated residual's update */
template <bool INJ>
__device__ __forceinline__ void pj_store(const qk_proj &a, float *out, int ostride, int t, int r, float v) {
    if (out) qk_st(out + (size_t)t * ostride + r, v);
    if (INJ)
        for (int j = 0; j < a.hc; j++) {
            float *hp = a.hyper + ((size_t)t * a.hc + j) * ostride + r;
            qk_st(hp, fmaf(qk_ld(a.inject + (size_t)t * a.hc + j), v, qk_ld(hp)));
        }
}

/*
 * Tiles of BM = 32*RT*WR tokens x BN = 64*(4/WR) columns; wave (wr, wc) owns
 * RT row tiles and two column tiles.  Per group the rows' planes are copied
 * into LDS as they lie (two buffers, one barrier), the next group's under
 * this one's products; code words and scales come straight into registers
 * one group ahead.
 */
template <int RT, int WR, bool INJ, bool S8>
__global__ __launch_bounds__(PJ_THREADS, 2) void k_proj_mm(qk_proj a) {
    constexpr int BM = 32 * RT * WR, WC = 4 / WR;
    constexpr int NRT = RT * WR, NC = NRT * 2; /* row tiles; 1 KB copies per wave and group */
    __shared__ __attribute__((aligned(16))) uint4 s_a[2][NRT][8][64]; /* [plane, K-step][lane] */
    __shared__ __attribute__((aligned(16))) float s_p[2][BM];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 31, h = lane >> 5;
    const int wr = wave % WR, wc = wave / WR;
    /* workgroups go round-robin over the 8 XCDs: the row tiles of one column
     * tile are consecutive workgroups of one XCD and share its L2 copy of
     * the weights */
    const int per = (a.mtiles * a.ntiles + 7) >> 3;
    const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (id >= a.mtiles * a.ntiles) return;
    const int nt = id / a.mtiles, mt = id - nt * a.mtiles;
    const int m0 = mt * BM;
    const int G = a.K >> 6;
    const size_t wrow = (size_t)a.K >> 3;

    const uint32_t *q;
    const uint16_t *s, *b;
    float *out;
    int ostride, r0;
    const int cb = nt * WC + wc;
    const bool live = pj_segment(a, min(cb, a.end64[a.nseg - 1] - 1), q, s, b, out, ostride, r0) &&
                      cb < a.end64[a.nseg - 1];
    const uint32_t *wq[2];
    const uint16_t *sp[2];
#pragma unroll
    for (int ct = 0; ct < 2; ct++) {
        wq[ct] = q + (size_t)(r0 + 32 * ct + c) * wrow + 4 * h;
        sp[ct] = s + (size_t)(r0 + 32 * ct + c) * G;
    }

    /* wave w copies units NC w .. of the group's 8 NRT (a unit: 1 KB); row
     * tiles past the last repeat it */
    const size_t ldp = qk_planes_ld(a.n);
    const int lastrt = (a.n - 1) >> 5;
    const uint4 *ap = (const uint4 *)a.pl.a + (size_t)min((m0 >> 5) + NC * wave / 8, lastrt) * G * 512 + NC * wave % 8 * 64 + lane;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(qm_lptr)&s_a[0][0][0][0] + 1024 * NC * wave);
    float pr = 0.0f;
    auto copy_a = [&](int g, int buf) {
#pragma unroll
        for (int i = 0; i < NC; i += 4) {
            const uint4 *src = ap + (size_t)g * 512 + 64 * i;
            const uint32_t dst = lds0 + buf * (NRT * 8192) + 1024 * i;
            qm_copy<0>(src, dst);
            qm_copy<1024>(src, dst);
            qm_copy<2048>(src, dst);
            qm_copy<3072>(src, dst);
        }
        pr = qk_ld(a.pl.pg + ldp * g + min(m0 + min(tid, BM - 1), a.n - 1));
    };
    uint4 wv[2];
    /* scales: eight groups of a column per load where its row of scales is
     * 16-byte aligned (a load of one touches a line per column all the same),
     * shifted down a group at a time */
    uint4 s8[2], s8n[2];
    auto load_s = [&](uint4 (&d)[2], int g) {
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            if (S8) d[ct] = qk_ld((const uint4 *)(sp[ct] + min(g, G - 8)));
            else d[ct].x = qk_ld(sp[ct] + min(g, G - 1));
        }
    };
    auto load_w = [&](int g) {
#pragma unroll
        for (int ct = 0; ct < 2; ct++) wv[ct] = qk_ld((const uint4 *)(wq[ct] + 8 * g));
    };
    qm_f32x16 acc[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[rt][ct][i] = 0.0f;

    copy_a(0, 0);
    load_w(0);
    load_s(s8, 0);
    if (tid < BM) s_p[0][tid] = pr * QM_P16;
    for (int g = 0; g < G; g++) {
        const int buf = g & 1;
        qm_bf16x8 bop[2][4];
        float sc[2];
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            bop[ct][0] = qm_codes16(wv[ct].x);
            bop[ct][1] = qm_codes16(wv[ct].y);
            bop[ct][2] = qm_codes16(wv[ct].z);
            bop[ct][3] = qm_codes16(wv[ct].w);
            sc[ct] = qk_bf16_lo(s8[ct].x);
            if (S8) {
                s8[ct].x = (s8[ct].x >> 16) | (s8[ct].y << 16);
                s8[ct].y = (s8[ct].y >> 16) | (s8[ct].z << 16);
                s8[ct].z = (s8[ct].z >> 16) | (s8[ct].w << 16);
                s8[ct].w >>= 16;
            }
        }
        /* group g is in LDS; its buffer's partner was last read in group g-1,
         * before this barrier */
        qm_sync<0>();
        const int gn = min(g + 1, G - 1); /* past the end: loaded, not used */
        if (g + 1 < G) copy_a(gn, buf ^ 1); /* no copy may outlive the workgroup */
        load_w(gn);
        if (!S8) {
            load_s(s8, gn);
        } else {
            if ((g & 7) == 0) load_s(s8n, g + 8);
            if ((g & 7) == 7) {
                s8[0] = s8n[0];
                s8[1] = s8n[1];
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            qm_f32x16 p;
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                const qm_f32x4 v = *(const qm_f32x4 *)&s_p[buf][32 * (RT * wr + rt) + 8 * i4 + 4 * h];
#pragma unroll
                for (int i = 0; i < 4; i++) p[4 * i4 + i] = v[i];
            }
            qm_f32x16 t[2];
#pragma unroll
            for (int tm = 0; tm < 2; tm++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const qm_bf16x8 A = __builtin_bit_cast(qm_bf16x8, s_a[buf][RT * wr + rt][4 * tm + j][lane]);
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) t[ct] = PJ_MFMA(A, bop[ct][j], (tm == 0 && j == 0) ? p : t[ct]);
                }
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[rt][ct][i] = fmaf(sc[ct], t[ct][i], acc[rt][ct][i]);
        }
        if (tid < BM) s_p[buf ^ 1][tid] = pr * QM_P16;
    }

    /* bias term: acc += sum_g b[col][g] X[row][g] */
    for (int k0 = 0; k0 < G; k0 += 16) {
        qm_bf16x8 bb[2];
#pragma unroll
        for (int ct = 0; ct < 2; ct++) bb[ct] = pj_bias_w(b + (size_t)(r0 + 32 * ct + c) * G, k0 + 8 * h, G);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            qm_bf16x8 X[3];
            pj_bias_x(a.pl.pg + min(m0 + 32 * (RT * wr + rt) + c, a.n - 1), ldp, k0 + 8 * h, G, X);
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int i = 0; i < 3; i++) acc[rt][ct] = PJ_MFMA(X[i], bb[ct], acc[rt][ct]);
        }
    }
    if (!live) return;
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = m0 + 32 * (RT * wr + rt) + 8 * (i >> 2) + 4 * h + (i & 3);
            if (t < a.n)
#pragma unroll
                for (int ct = 0; ct < 2; ct++) pj_store<INJ>(a, out, ostride, t, r0 + 32 * ct + c, acc[rt][ct][i]);
        }
}

/*
 * Dense bf16 weight rows (DeltaNet in_proj_a | in_proj_b, the hyper
 * connection's inject) on the same planes: 32 tokens x 32 of the matrices'
 * rows, K dealt to WK waves.  In k_proj_few these are its last column blocks;
 * the large tiles run them as a launch of their own.
 */
template <int WK, int LDR>
__device__ __forceinline__ void pj_bf16_tile(const qk_proj &a, int m0, int tile, float (&s_r)[WK][32][LDR]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 31, h = lane >> 5;
    const int rows = a.bw[1] ? 2 * a.brows : a.brows;
    const int cc = min(tile * 32 + c, rows - 1);
    const uint16_t *wp = (cc < a.brows ? a.bw[0] + (size_t)cc * a.K : a.bw[1] + (size_t)(cc - a.brows) * a.K) + 32 * h;
    const int G = a.K >> 6;
    const uint4 *ap = (const uint4 *)a.pl.a + (size_t)(m0 >> 5) * G * 512 + lane;
    qm_f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.0f;
    uint4 av[2][4], wv[4];
    auto load = [&](int g) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            av[0][j] = qk_ld(ap + (size_t)g * 512 + 64 * j);
            av[1][j] = qk_ld(ap + (size_t)g * 512 + 256 + 64 * j);
            wv[j] = qk_ld((const uint4 *)(wp + 64 * g) + j);
        }
    };
    if (wave < G) load(wave);
    for (int g = wave; g < G; g += WK) {
        qm_bf16x8 A[2][4], B[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t p[4];
            qk_bf16x8_to_pairs(wv[j], p);
            B[j] = __builtin_bit_cast(qm_bf16x8, make_uint4(p[0], p[1], p[2], p[3]));
            A[0][j] = __builtin_bit_cast(qm_bf16x8, av[0][j]);
            A[1][j] = __builtin_bit_cast(qm_bf16x8, av[1][j]);
        }
        load(min(g + WK, G - 1));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc = PJ_MFMA(A[0][j], B[j], acc);
            acc = PJ_MFMA(A[1][j], B[j], acc);
        }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) s_r[wave][8 * (i >> 2) + 4 * h + (i & 3)][c] = acc[i];
    __syncthreads();
    for (int i = threadIdx.x; i < 32 * 32; i += 64 * WK) {
        const int row = i >> 5, r = tile * 32 + (i & 31);
        if (m0 + row >= a.n || r >= rows) continue;
        float v = s_r[0][row][i & 31];
#pragma unroll
        for (int w = 1; w < WK; w++) v += s_r[w][row][i & 31];
        const int k = r >= a.brows;
        qk_st(a.bout[k] + (size_t)(m0 + row) * a.brows + (r - k * a.brows), v);
    }
}

/*
 * Few tokens: 32 tokens x 32*CT columns per workgroup, the K groups dealt to
 * its WK waves (wave w: groups w, w + WK, ..) and their sums added through
 * LDS in wave order.  A tile of 32 rows leaves too few workgroups of the
 * tiles above to fill the chip, and each would walk the whole K alone; here
 * a wave walks K / WK with its operands read straight from the planes (the
 * workgroup's rows are L1/L2 hits), no LDS and no barrier in the loop.
 */
template <int CT, int WK, bool INJ>
__global__ __launch_bounds__(64 * WK) void k_proj_few(qk_proj a) {
    __shared__ float s_r[WK][32][32 * CT + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 31, h = lane >> 5;
    /* workgroup L runs on XCD L % 8.  While the planes are small next to an
     * XCD's L2 the row tiles of a column block stay together there (the weights
     * are read once), else the column blocks of a row tile */
    const int i8 = blockIdx.x >> 3, x8 = blockIdx.x & 7, ncb = a.ntiles + a.btiles;
    int nt, mt;
    if (a.byrow) { mt = i8 / ncb * 8 + x8; nt = i8 % ncb; }
    else { nt = i8 / a.mtiles * 8 + x8; mt = i8 % a.mtiles; }
    if (mt >= a.mtiles || nt >= ncb) return;
    const int m0 = mt * 32;
    if (nt >= a.ntiles) {
        pj_bf16_tile<WK>(a, m0, nt - a.ntiles, s_r);
        return;
    }
    const int G = a.K >> 6;
    const size_t wrow = (size_t)a.K >> 3;
    const uint32_t *q;
    const uint16_t *s, *b;
    float *out;
    int ostride, r0;
    pj_segment(a, nt * CT / 2, q, s, b, out, ostride, r0);
    if (CT == 1) r0 += 32 * (nt & 1);
    const uint32_t *wq[CT];
    const uint16_t *sp[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        wq[ct] = q + (size_t)(r0 + 32 * ct + c) * wrow + 4 * h;
        sp[ct] = s + (size_t)(r0 + 32 * ct + c) * G;
    }
    const size_t ldp = qk_planes_ld(a.n);
    const uint4 *ap = (const uint4 *)a.pl.a + (size_t)(m0 >> 5) * G * 512 + lane;
    struct Op {
        uint4 w[CT], a[2][4];
        uint16_t s[CT];
        float4 p[4];
    };
    auto load = [&](Op &o, int g) {
        g = min(g, G - 1); /* past the end: loaded, not used */
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            o.w[ct] = qk_ld((const uint4 *)(wq[ct] + 8 * g));
            o.s[ct] = qk_ld(sp[ct] + g);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            o.a[0][j] = qk_ld(ap + (size_t)g * 512 + 64 * j);
            o.a[1][j] = qk_ld(ap + (size_t)g * 512 + 256 + 64 * j);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) /* rows past n: within the leading dimension, not used */
            o.p[i] = qk_ld((const float4 *)(a.pl.pg + ldp * g + m0 + 8 * i + 4 * h));
    };
    qm_f32x16 acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[ct][i] = 0.0f;
    auto step = [&](Op &o, int g) {
        qm_bf16x8 A[2][4], bop[CT][4];
        float sc[CT];
        qm_f32x16 t[CT];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            A[0][j] = __builtin_bit_cast(qm_bf16x8, o.a[0][j]);
            A[1][j] = __builtin_bit_cast(qm_bf16x8, o.a[1][j]);
        }
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            bop[ct][0] = qm_codes16(o.w[ct].x);
            bop[ct][1] = qm_codes16(o.w[ct].y);
            bop[ct][2] = qm_codes16(o.w[ct].z);
            bop[ct][3] = qm_codes16(o.w[ct].w);
            sc[ct] = qk_bf16(o.s[ct]);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                t[ct][4 * i] = o.p[i].x * QM_P16;
                t[ct][4 * i + 1] = o.p[i].y * QM_P16;
                t[ct][4 * i + 2] = o.p[i].z * QM_P16;
                t[ct][4 * i + 3] = o.p[i].w * QM_P16;
            }
        }
        load(o, g + 2 * WK);
#pragma unroll
        for (int tm = 0; tm < 2; tm++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++) t[ct] = PJ_MFMA(A[tm][j], bop[ct][j], t[ct]);
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[ct][i] = fmaf(sc[ct], t[ct][i], acc[ct][i]);
    };
    Op o0, o1; /* two groups in flight */
    load(o0, wave);
    load(o1, wave + WK);
    for (int g = wave; g < G; g += 2 * WK) {
        step(o0, g);
        if (g + WK < G) step(o1, g + WK);
    }
    /* bias term, 16 groups per step, the steps dealt to the waves */
    for (int k0 = 16 * wave; k0 < G; k0 += 16 * WK) {
        qm_bf16x8 X[3];
        pj_bias_x(a.pl.pg + min(m0 + c, a.n - 1), ldp, k0 + 8 * h, G, X);
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            const qm_bf16x8 bb = pj_bias_w(b + (size_t)(r0 + 32 * ct + c) * G, k0 + 8 * h, G);
#pragma unroll
            for (int i = 0; i < 3; i++) acc[ct] = PJ_MFMA(X[i], bb, acc[ct]);
        }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int i = 0; i < 16; i++) s_r[wave][8 * (i >> 2) + 4 * h + (i & 3)][32 * ct + c] = acc[ct][i];
    __syncthreads();
    for (int i = threadIdx.x; i < 32 * 32 * CT; i += 64 * WK) {
        const int row = i / (32 * CT), col = i - row * (32 * CT);
        if (m0 + row >= a.n) break; /* rows ascend with i */
        float v = s_r[0][row][col];
#pragma unroll
        for (int w = 1; w < WK; w++) v = v + s_r[w][row][col];
        pj_store<INJ>(a, out, ostride, m0 + row, r0 + col, v);
    }
}

template <int WK>
__global__ __launch_bounds__(64 * WK) void k_proj_bf16(qk_proj a) {
    __shared__ float s_r[WK][32][33];
    pj_bf16_tile<WK>(a, blockIdx.y * 32, blockIdx.x, s_r);
}

/* f32 rows -> planes, a wave per 8 rows x 64 columns.  Bound: HBM / L2. */
__global__ __launch_bounds__(256) void k_proj_pack(const float *x, int n, int G, qk_planes pl) {
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int rb = u / G, g = u - rb * G, t = 8 * rb + (lane & 7);
    if (8 * rb >= n) return;
    const float4 *p = (const float4 *)x + ((size_t)min(t, n - 1) * G + g) * 16 + 2 * (lane >> 3);
    const float4 a0 = qk_ld(p), a1 = qk_ld(p + 1);
    const float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
    qm_pack_store(pl, t, n, g, G, v);
}

/* ------------------------------------------------------------ host side */

extern "C" int qk_launch_proj_pack(const float *x, int n, int K, const qk_planes *pl, void *stream) {
    if (n <= 0) return 0;
    if (K <= 0 || K % 64) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(k_proj_pack, dim3(qm_pack_wgs(n, K / 64)), dim3(256), 0, (hipStream_t)stream, x, n, K / 64, *pl);
    return QK_CHECK_LAUNCH();
}

extern "C" int qk_launch_proj(const qk_proj *in, void *stream) {
    qk_proj a = *in;
    if (a.n <= 0) return 0;
    if (a.K <= 0 || a.K % 64 || (a.bw[0] && a.brows < 1) || a.nseg < 1 || a.nseg > QK_PROJ_SEGS || (a.hyper && (a.nseg != 1 || a.hc < 1)))
        return (int)hipErrorInvalidValue;
    int end = 0;
    for (int i = 0; i < a.nseg; i++) {
        if (a.seg[i].rows <= 0 || a.seg[i].rows % 64) return (int)hipErrorInvalidValue;
        end += a.seg[i].rows / 64;
        a.end64[i] = end;
    }
    hipStream_t st = (hipStream_t)stream;
    const bool inj = a.hyper != nullptr;
    bool s8 = a.K % 512 == 0; /* G a multiple of 8, and the scales' bases aligned */
    for (int i = 0; i < a.nseg; i++) s8 = s8 && ((uintptr_t)a.seg[i].s & 15) == 0;
#define PJ_MM(RT, WR)                                                                                        \
    do {                                                                                                     \
        a.mtiles = (a.n + 32 * RT * WR - 1) / (32 * RT * WR);                                                \
        a.ntiles = (end + 4 / WR - 1) / (4 / WR);                                                            \
        const dim3 grid(((unsigned)(a.mtiles * a.ntiles) + 7) / 8 * 8);                                      \
        if (s8) {                                                                                            \
            if (inj) hipLaunchKernelGGL((k_proj_mm<RT, WR, true, true>), grid, dim3(PJ_THREADS), 0, st, a);  \
            else hipLaunchKernelGGL((k_proj_mm<RT, WR, false, true>), grid, dim3(PJ_THREADS), 0, st, a);     \
        } else {                                                                                             \
            if (inj) hipLaunchKernelGGL((k_proj_mm<RT, WR, true, false>), grid, dim3(PJ_THREADS), 0, st, a); \
            else hipLaunchKernelGGL((k_proj_mm<RT, WR, false, false>), grid, dim3(PJ_THREADS), 0, st, a);    \
        }                                                                                                    \
    } while (0)
#define PJ_FEW(CT, WK)                                                                                       \
    do {                                                                                                     \
        a.ntiles = end * 2 / CT;                                                                             \
        const int ncb = a.ntiles + bt;                                                                       \
        const dim3 grid(8u * (a.byrow ? (unsigned)(mt + 7) / 8 * ncb : (unsigned)(ncb + 7) / 8 * mt));       \
        if (inj) hipLaunchKernelGGL((k_proj_few<CT, WK, true>), grid, dim3(64 * WK), 0, st, a);              \
        else hipLaunchKernelGGL((k_proj_few<CT, WK, false>), grid, dim3(64 * WK), 0, st, a);                 \
    } while (0)
    const int mt = (a.n + 31) / 32, bt = a.bw[0] ? ((a.bw[1] ? 2 : 1) * a.brows + 31) / 32 : 0;
    a.btiles = bt;
    /* The K-split tiles while the others would leave the chip short of
     * workgroups (DeltaNet mixer of hidden 2048, both products, us without
     * the recurrence: 77 tokens 85 against 120, 256 tokens 133 / 145, 512
     * tokens 245 / 200), split the deeper the fewer tiles there are: four
     * waves from a workgroup per CU on (two fit), eight below, of 64 columns
     * while those are still 128 workgroups.  128-row tiles once they give every
     * CU four workgroups (2048 tokens: 427 together, 64-row tiles 520). */
    const long long wg64 = (long long)((a.n + 63) / 64) * ((end + 1) / 2);
    if (a.n <= QK_PROJ_FEW_N || wg64 < 256) {
        a.mtiles = mt;
        a.byrow = (size_t)a.n * a.K * 4 > ((size_t)4 << 20);
        if (end * mt >= 256 || a.K < 1024) PJ_FEW(2, 4);
        else if (8 * end * mt >= 1024) PJ_FEW(2, 8);
        else PJ_FEW(1, 8);
        return QK_CHECK_LAUNCH();
    }
    if ((long long)((a.n + 127) / 128) * ((end + 1) / 2) < 1024) PJ_MM(1, 2);
    else PJ_MM(2, 2);
#undef PJ_MM
#undef PJ_FEW
    int rc = QK_CHECK_LAUNCH();
    if (rc || !bt) return rc;
    hipLaunchKernelGGL(k_proj_bf16<8>, dim3(bt, mt), dim3(512), 0, st, a);
    return QK_CHECK_LAUNCH();
}
