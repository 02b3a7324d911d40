/*
 * r9vx_thin.h -- the weight decode of the thin-tile dequant-GEMM
 * (gemm_thin.hip): one unit is one weight row's half of a 64-K step (32
 * weights), loaded from the device layout and decoded into the four fp16
 * granules that the MFMA slices of that step read.  The arithmetic is that of
 * the 256-row loop (m3_dec_unit of r9vx_mma3.h), so every weight is the same
 * fp16 bits there and here; only the unit's index within its super-block is a
 * run-time value instead of a constant.
 */
#ifndef R9VX_THIN_H
#define R9VX_THIN_H

#include "r9vx_mma3.h"

namespace r9vx {

/* Registers of one loaded unit (16 payload bytes; Q8_0 / Q6_K 32, IQ3_S 12)
 * and its block's header. */
template <int SCHEME>
struct ThinUnit {
    r9vx_u32x4 p;  /* Q4_K / IQ4_XS payload, Q6_K ql, Q8_0 quants 0-15, IQ3_S index bytes (.x .y) and sign word (.z) */
    r9vx_u32x4 p2; /* Q6_K qh, Q8_0 quants 16-31 */
    r9vx_u32x4 h;  /* block header / scales / IQ3_S side word */
    uint32_t d;    /* split layout: f16 d */
};

typedef uint32_t thin_u32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t thin_u32x2 __attribute__((ext_vector_type(2), aligned(4)));

/* Global load at a uniform base plus a 32-bit lane offset plus a constant: the
 * base goes through scalar registers, so that the address costs no vector
 * instruction (and the pointer keeps its address space: a flat load would
 * count as an LDS access too). */
template <class T>
__device__ __forceinline__ T thin_ld(const uint8_t *base, uint32_t off, int imm) {
    typedef const __attribute__((address_space(1))) char *gptr;
    const uint64_t b = (uint64_t)(uintptr_t)base;
    const uint64_t u = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32) |
                       (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
    return *(const __attribute__((address_space(1))) T *)((gptr)u + off + imm);
}

/* Unit u (0..7: step u / 2, half u % 2) of super-block blk of a weight row at
 * base + off (split layouts: its d values at sbase + soff). */
template <int SCHEME>
__device__ __forceinline__ void thin_load(const uint8_t *base, uint32_t off, const uint8_t *sbase, uint32_t soff,
                                          uint32_t blk, uint32_t u, ThinUnit<SCHEME> &t) {
    if constexpr (SCHEME == R9VX_SCHEME_Q4_K) {
        const uint8_t *const b = base + (uint64_t)blk * R9VX_Q4K_BYTES;
        t.p = thin_ld<thin_u32x4>(b, off + 16 * u, 16);
        t.h = thin_ld<thin_u32x4>(b, off, 0);
    } else if constexpr (SCHEME == R9VX_SCHEME_IQ4_XS) {
        const uint8_t *const b = base + (uint64_t)blk * R9VX_IQ4XS_BYTES;
        t.p = thin_ld<thin_u32x4>(b, off + 16 * u, 8);
        const thin_u32x2 h = thin_ld<thin_u32x2>(b, off, 0);
        t.h.x = h.x;
        t.h.y = h.y;
    } else if constexpr (SCHEME == R9VX_SCHEME_Q6_K) {
        const uint8_t *const b = base + (uint64_t)blk * R9VX_Q6K_BODY;
        t.p = thin_ld<thin_u32x4>(b, off + 16 * u, 0);
        t.p2 = thin_ld<thin_u32x4>(b, off + 32 * (u >> 2) + 16 * (u & 1), 128);
        t.h = thin_ld<thin_u32x4>(b, off, 192);
        t.d = thin_ld<uint16_t>(sbase + 2ull * blk, soff, 0);
    } else if constexpr (SCHEME == R9VX_SCHEME_Q8_0) {
        const uint8_t *const b = base + 256ull * blk;
        t.p = thin_ld<thin_u32x4>(b, off + 32 * u, 0);
        t.p2 = thin_ld<thin_u32x4>(b, off + 32 * u, 16);
        t.d = thin_ld<uint16_t>(sbase + 16ull * blk, soff + 2 * u, 0);
    } else {
        const uint8_t *const b = base + (uint64_t)blk * R9VX_IQ3S_DEV_BYTES;
        const thin_u32x2 q = thin_ld<thin_u32x2>(b, off + 8 * u, 0);
        t.p.x = q.x;
        t.p.y = q.y;
        t.p.z = thin_ld<uint32_t>(b, off + 4 * u, 64);
        t.h = thin_ld<thin_u32x4>(b, off, 96);
    }
}

/* {fp16(dl a + c), fp16(dl b + c)} of one half of each of a, b (fp16 pairs;
 * HI: the high halves), each fused and rounded once. */
template <bool HI>
__device__ __forceinline__ uint32_t thin_mix(float dl, uint32_t a, uint32_t b, float c) {
    uint32_t r;
    if constexpr (HI)
        asm("v_fma_mixlo_f16 %0, %1, %2, %4 op_sel:[0,1,0] op_sel_hi:[0,1,0]\n\t"
            "v_fma_mixhi_f16 %0, %1, %3, %4 op_sel:[0,1,0] op_sel_hi:[0,1,0]"
            : "=&v"(r) : "v"(dl), "v"(a), "v"(b), "v"(c));
    else
        asm("v_fma_mixlo_f16 %0, %1, %2, %4 op_sel_hi:[0,1,0]\n\t"
            "v_fma_mixhi_f16 %0, %1, %3, %4 op_sel_hi:[0,1,0]"
            : "=&v"(r) : "v"(dl), "v"(a), "v"(b), "v"(c));
    return r;
}

/* The unit's four granules, written to dst[64 s] for slice s as soon as each
 * is whole; mid() runs after the second. */
template <int SCHEME, class Mid>
__device__ __forceinline__ void thin_decode(const ThinUnit<SCHEME> &t, uint32_t u, const uint32_t *lut,
                                            r9vx_u32x4 *dst, Mid mid) {
    const uint32_t dw[4] = {t.p.x, t.p.y, t.p.z, t.p.w};
    if constexpr (SCHEME == R9VX_SCHEME_Q4_K) {
        const float d = r9vx_f16_to_f32((uint16_t)(t.h.x & 0xFFFF)), dmin = r9vx_f16_to_f32((uint16_t)(t.h.x >> 16));
        /* r9vx_q4k_pair_bytes with its two cases selected per bit */
        const uint32_t sel = (u & 2u) ? 0x07060302u : 0x05040100u;
        const uint32_t x = __builtin_amdgcn_perm(t.h.z, t.h.y, sel), y = __builtin_amdgcn_perm(t.h.w >> 4, t.h.w, sel);
        const uint32_t late = u >= 4 ? 0xFFFFFFFFu : 0u;
        const uint32_t b = (((y & 0x0F0F0F0Fu) | ((x >> 2) & 0x30303030u)) & late) | (x & 0x3F3F3F3Fu & ~late);
        const float dl0 = d * (float)(b & 0xFFu), dl1 = d * (float)((b >> 8) & 0xFFu);
        const float c0 = fmaf(-1024.f, dl0, -(dmin * (float)((b >> 16) & 0xFFu)));
        const float c1 = fmaf(-1024.f, dl1, -(dmin * (float)(b >> 24)));
        /* the fp16 pairs 1024 + q of bytes 0, 2 and of bytes 1, 3; their
         * halves are picked apart again by the fused scale */
        const uint32_t k1024 = 0x64006400u;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t l02 = r9vx_and_or(dw[q], 0x000F000Fu, k1024), l13 = r9vx_and_or(dw[q] >> 8, 0x000F000Fu, k1024);
            const uint32_t h02 = r9vx_and_or(dw[q] >> 4, 0x000F000Fu, k1024), h13 = r9vx_and_or(dw[q] >> 12, 0x000F000Fu, k1024);
            dst[64 * q] = r9vx_u32x4{thin_mix<false>(dl0, l02, l13, c0), thin_mix<true>(dl0, l02, l13, c0),
                                     thin_mix<false>(dl1, h02, h13, c1), thin_mix<true>(dl1, h02, h13, c1)};
            if (q == 1) mid();
        }
        return;
    }
    BScale sc{};
    uint32_t dw2[4] = {0u, 0u, 0u, 0u}, kv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) kv[i] = 0u;
    if constexpr (SCHEME == R9VX_SCHEME_IQ4_XS) {
        sc.dl0 = r9vx_f16_to_f32((uint16_t)(t.h.x & 0xFFFF)) * r9vx_iq4xs_scale(r9vx_u32x2{t.h.x, t.h.y}, u);
#pragma unroll
        for (int i = 0; i < 16; ++i) kv[i] = lut[(dw[i >> 2] >> (8 * (i & 3))) & 0xFFu];
    } else if constexpr (SCHEME == R9VX_SCHEME_Q6_K) {
        const uint32_t n = u >> 2, j = (u >> 1) & 1u, sh = 8 * (u & 3u);
        const float d = r9vx_f16_to_f32((uint16_t)t.d);
        sc.dl0 = d * (float)(int8_t)((n ? t.h.z : t.h.x) >> sh);
        sc.dl1 = d * (float)(int8_t)((n ? t.h.w : t.h.y) >> sh);
        sc.c0 = -1056.f * sc.dl0;
        sc.c1 = -1056.f * sc.dl1;
        /* the bit pairs j and 2 + j, moved to pairs 0 and 2 */
        dw2[0] = t.p2.x >> (2 * j), dw2[1] = t.p2.y >> (2 * j), dw2[2] = t.p2.z >> (2 * j), dw2[3] = t.p2.w >> (2 * j);
    } else if constexpr (SCHEME == R9VX_SCHEME_Q8_0) {
        sc.dl0 = r9vx_f16_to_f32((uint16_t)t.d);
        sc.c0 = -1152.f * sc.dl0;
        dw2[0] = t.p2.x, dw2[1] = t.p2.y, dw2[2] = t.p2.z, dw2[3] = t.p2.w;
    } else if constexpr (SCHEME == R9VX_SCHEME_IQ3_S) {
        sc.dl0 = r9vx_f16_to_f32((uint16_t)(t.h.w & 0xFFFF)) * (float)(1u + 2u * ((t.h.z >> (4 * u)) & 0xFu));
        sc.c0 = -1152.f * sc.dl0;
        const uint32_t qh = ((u < 4 ? t.h.x : t.h.y) >> (8 * (u & 3u))) & 0xFFu, sg = t.p.z;
        /* granule q, m: values 2m, 2m + 1 of indices 2q (low pair) and 2q + 1
         * (high pair), signs from bits 8q + 2m and 8q + 4 + 2m
         * (m3_init_iq3s_lut's word order) */
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t e = (((i < 4 ? t.p.x : t.p.y) >> (8 * (i & 3))) & 0xFFu) | (((qh >> i) & 1u) << 8);
#pragma unroll
            for (int m = 0; m < 2; ++m)
                kv[4 * (i >> 1) + 2 * m + (i & 1)] = lut[(e << 3) | ((uint32_t)m << 2) | ((sg >> (4 * i + 2 * m)) & 3u)];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t o[4];
#pragma unroll
        for (int m = 0; m < 2; ++m)
            m3_dec_unit<SCHEME, 0>(dw[q], dw2[q], m, sc, kv[4 * q + 2 * m], kv[4 * q + 2 * m + 1], o[m], o[2 + m]);
        dst[64 * q] = r9vx_u32x4{o[0], o[1], o[2], o[3]};
        if (q == 1) mid();
    }
}

}  // namespace r9vx

#endif
