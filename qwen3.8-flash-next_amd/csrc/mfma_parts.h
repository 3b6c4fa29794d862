/*
 * mfma_parts.h -- operand helpers for v_mfma_f32_16x16x32_bf16 and
 * v_mfma_f32_32x32x16_bf16 on q4 weights: the vector types, the code word ->
 * B operand conversions, copies straight to LDS with their waits, and the
 * packing of rows into operand planes.
 */
#ifndef MFMA_PARTS_H
#define MFMA_PARTS_H

#include "qk_device.h"

typedef __bf16 qm_bf16x8 __attribute__((ext_vector_type(8)));
typedef float qm_f32x4 __attribute__((ext_vector_type(4)));

/* one code word -> the B operand: bf16 128+q in (q_i, q_{i+4}) pair order,
 * as qk_codes_to_pairs, built with byte permutes: the low nibbles of the
 * four bytes (q0, q2, q4, q6) and the high ones (q1, q3, q5, q7) each give
 * two pairs by interleaving with the byte 0x43 */
__device__ __forceinline__ qm_bf16x8 qm_codes(uint32_t w) {
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
    const uint32_t k = 0x43434343u;
    return __builtin_bit_cast(qm_bf16x8,
                              make_uint4(__builtin_amdgcn_perm(k, lo, 0x04020400u), __builtin_amdgcn_perm(k, hi, 0x04020400u),
                                         __builtin_amdgcn_perm(k, lo, 0x04030401u), __builtin_amdgcn_perm(k, hi, 0x04030401u)));
}

/* the same as 16 + q (0x4180 | q << 3, exact: the ulp in [16, 32) is 1/8).
 * The offset is what the running sums carry until the group ends, so its size
 * sets their rounding: with 128 + q (one instruction fewer) the DeltaNet
 * out_proj's error against 64 bits at 4096 columns was 9.6e-6, more than the
 * per-token GEMV's 9.3e-6; with 16 + q 7.5e-6. */
__device__ __forceinline__ qm_bf16x8 qm_codes16(uint32_t w) {
    const uint32_t lo = ((w << 3) & 0x78787878u) | 0x80808080u, hi = ((w >> 1) & 0x78787878u) | 0x80808080u;
    const uint32_t k = 0x41414141u;
    return __builtin_bit_cast(qm_bf16x8,
                              make_uint4(__builtin_amdgcn_perm(k, lo, 0x04020400u), __builtin_amdgcn_perm(k, hi, 0x04020400u),
                                         __builtin_amdgcn_perm(k, lo, 0x04030401u), __builtin_amdgcn_perm(k, hi, 0x04030401u)));
}
#define QM_P16 0.125f /* a group's start -16 X from the planes' P = -128 X */

/* one copy of a wave straight from memory to LDS: 64 x 16 bytes from src + OFF
 * + 16 lane (src the lane's own address) to LDS byte lds + OFF + 16 lane.  As
 * an instruction of its own and not the builtin: the compiler waits for every
 * builtin copy in flight before the next LDS read, whichever buffer it reads;
 * qm_sync has the waits these need.  No register is written. */
template <int OFF>
__device__ __forceinline__ void qm_copy(const uint4 *src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off offset:%2"
                 :
                 : "v"(src), "s"(lds), "n"(OFF)
                 : "memory", "m0");
}
typedef __attribute__((address_space(3))) uint32_t *qm_lptr;

/* at most N copies (or loads) of this wave in flight, its LDS accesses done,
 * and every wave of the workgroup here */
template <int N>
__device__ __forceinline__ void qm_sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14)); /* vmcnt(N) lgkmcnt(0) */
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

/* A wave packs 8 rows x 64 columns (one group) into qk_planes: lane l has row
 * t = 8 block + l % 8 and the 8 columns of chunk l / 8, so each plane's store
 * is runs of 128 bytes (a lane per chunk of one row wrote 16 at a time: 2 to
 * 2.5 times as long) and the loads runs of 256.  The group sum pairs the
 * chunks as k_pack_rows does (1, 2, 4). */
__device__ __forceinline__ void qm_pack_store(const qk_planes &pl, int t, int n, int g, int G, const float v[8]) {
    const int lane = threadIdx.x & 63;
    uint32_t ph[4], pw[4];
    float s = qk_f32x8_pairs(v, ph, pw);
    s += qk_dpp<0x128>(s); /* row_ror:8 = l^8 within 16 lanes */
    s += __uint_as_float(qk_xor16_u(__float_as_uint(s)));
    s += __uint_as_float(qk_xor32_u(__float_as_uint(s)));
    if (t >= n) return;
    uint4 *o = (uint4 *)pl.a + qk_planes_at(t, 8 * g + (lane >> 3), G);
    o[0] = make_uint4(ph[0], ph[1], ph[2], ph[3]);
    o[256] = make_uint4(pw[0], pw[1], pw[2], pw[3]);
    if (lane < 8) pl.pg[(size_t)g * qk_planes_ld(n) + t] = -128.0f * s;
}
/* waves, and workgroups of four, that pack n rows of G groups */
QK_HD static inline unsigned qm_pack_wgs(int n, int G) { return (unsigned)(((size_t)(n + 7) / 8 * G + 3) / 4); }

#endif
