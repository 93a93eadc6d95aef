/**
 * skinny_exact.h - The exact-integer arithmetic of the multi-row projections
 * (kernels_skinny.hip) and the layout of the tiled weights, which
 * kernels_tgemm.hip reads too.
 */
#ifndef VITNA_SKINNY_EXACT_H
#define VITNA_SKINNY_EXACT_H

#include "vitna_hip_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define SK_TOK 32

/* ---- exact-integer quants ------------------------------------------------ */
/*
 * Widths a multiple of 256 take this path. A wave owns one tile of 32 weight rows x 32 token rows over one
 * 256-column superblock (one Q4_K or Q6_K block, eight Q8_0 blocks), four units of 64 columns each: the
 * work is a few microseconds of loads a wave, so it is spread as wide as it goes and every load of the
 * wave's weights is issued at once. Within a unit every scale group (Q4_K 32 columns, Q6_K 16, Q8_0 32) keeps its own MFMA sum
 * P over its columns, and the group's scale is applied to P in fp32:
 *   Q8_0  bf16(q) exactly (signed):            acc += d P
 *   Q4_K  bf16(128 + q), q in 0..15:           acc += d sc P  -  (dmin m + 128 d sc) S
 *   Q6_K  bf16(128 + q6), q6 in 0..63:         acc += d sc P  -  160 d sc S
 * where S is the group's sum of the activations. 128 + q is the byte q under the exponent byte of 2^7 (two
 * v_perm_b32 for four weights). The S terms of eight groups go through the matrix cores too, as one
 * 32x32x8 product of the groups' sums (bf16 hi + lo, split on the host side of the pass) by their
 * coefficients, both as three bf16 pieces. S is the sum of the split activations hi + lo, so the offset
 * 128 S cancels exactly what the 128 in the weights added.
 *
 * A unit's k order: lane half kq (lane / 32) of each 16-column MFMA supplies 8 columns, and both operands
 * take them in the same order. Q4_K and Q8_0: the MFMAs of unit u cover columns 64 u + 16 kq + {0, 8} (the
 * first group) and + 32 (the second); Q4_K's byte 32 u + j holds columns 64 u + j (low nibble) and
 * 64 u + 32 + j (high). Q6_K unit u = (h, r0) = (u / 2, u % 2) covers the groups at columns
 * 128 h + 32 r + 16 s, r in {r0, r0 + 2}, s in {0, 1}, of which lane half kq takes columns + 8 kq .. + 8 kq + 7:
 * ql byte 64 h + 32 r0 + 16 s + j holds column 128 h + 32 r0 + 16 s + j (low nibble) and 128 h + 32 (r0 + 2)
 * + 16 s + j (high), qh byte 32 h + 16 s + j its high bits (bits 2 r).
 */

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t sx_u2 __attribute__((ext_vector_type(2)));

/* four bytes (each below 128) as bf16 128 + byte */
__device__ __forceinline__ sx_u2 sx_mag4(uint32_t v) {
    return sx_u2{__builtin_amdgcn_perm(0x43434343u, v, 0x04010400u), __builtin_amdgcn_perm(0x43434343u, v, 0x04030402u)};
}
__device__ __forceinline__ bf16x8 sx_join(sx_u2 a, sx_u2 b) { return __builtin_bit_cast(bf16x8, u32x4{a.x, a.y, b.x, b.y}); }
/* eight signed bytes as bf16, exactly */
__device__ __forceinline__ bf16x8 sx_i8(uint32_t a, uint32_t b) {
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r[i] = (__bf16)(float)(int8_t)(a >> (8 * i));
        r[4 + i] = (__bf16)(float)(int8_t)(b >> (8 * i));
    }
    return r;
}

/* One superblock of one 32-row tile: the lane's row's bytes for all four units. */
template <int DT> struct sx_w;
template <> struct sx_w<VITNA_DTYPE_Q4_K> { u32x4 q[4], h; };
template <> struct sx_w<VITNA_DTYPE_Q6_K> { sx_u2 ql[4][2], qh[2][2]; u32x4 sc; uint32_t d; };
template <> struct sx_w<VITNA_DTYPE_Q8_0> { u32x4 q[4][2], d; };

/* a unit's activations for the lane's token: four 8-column operands, hi and lo, and (when the unit applies
   S terms) the four group sums of the lane half */
struct sx_a {
    u32x4 h[4], l[4];
    sx_u2 sp[3];
};

/*
 * The tiled copy: per tile (32 rows; rows past the matrix repeat its last) and superblock, lane l = l32 + 32 kq
 * reads 16-byte pieces at lane-order offsets, so every load is 1 KB contiguous (512 bytes for the per-row
 * fields, which both lane halves read):
 *   Q4_K  [u][lane] q bytes 32 u + 16 kq + 0..15 (u < 4); at 4096 [l32] the 16-byte header
 *   Q6_K  [u][lane] ql bytes 64 (u / 2) + 32 (u % 2) + 16 s + 8 kq + 0..7 for s = 0, 1; at 4096 [h][lane] qh
 *         bytes 32 h + 16 s + 8 kq + 0..7 for s = 0, 1; at 6144 [l32] the 16 scales; at 6656 [l32] d
 *   Q8_0  [2 u + j][lane] q bytes 16 kq + 0..15 of block 8 b + 2 u + j; at 8192 [l32] the 8 blocks' d
 */
/* The lane's bytes of tile / superblock b from the tiled copy: 1 KB (512-byte) loads in lane order. */
template <int DT>
__device__ __forceinline__ void sx_load_w(const qmat& w, int tile, int b, int lane, sx_w<DT>& o) {
    const uint8_t* T = w.tiled + ((size_t)tile * (w.cols / 256) + b) * (DT == VITNA_DTYPE_Q4_K ? 4608 : DT == VITNA_DTYPE_Q6_K ? 6720 : 8704);
    const int l32 = lane & 31;
    if constexpr (DT == VITNA_DTYPE_Q4_K) {
#pragma unroll
        for (int u = 0; u < 4; u++) o.q[u] = *reinterpret_cast<const u32x4*>(T + u * 1024 + lane * 16);
        o.h = *reinterpret_cast<const u32x4*>(T + 4096 + l32 * 16);
    } else if constexpr (DT == VITNA_DTYPE_Q6_K) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(T + u * 1024 + lane * 16);
            o.ql[u][0] = sx_u2{v.x, v.y};
            o.ql[u][1] = sx_u2{v.z, v.w};
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(T + 4096 + h * 1024 + lane * 16);
            o.qh[h][0] = sx_u2{v.x, v.y};
            o.qh[h][1] = sx_u2{v.z, v.w};
        }
        o.sc = *reinterpret_cast<const u32x4*>(T + 6144 + l32 * 16);
        o.d = *reinterpret_cast<const uint16_t*>(T + 6656 + l32 * 2);
    } else {
#pragma unroll
        for (int v = 0; v < 8; v++) o.q[v >> 1][v & 1] = *reinterpret_cast<const u32x4*>(T + v * 1024 + lane * 16);
        o.d = *reinterpret_cast<const u32x4*>(T + 8192 + l32 * 16);
    }
}

template <int DT> struct sx_unit_sums { static constexpr bool at(int U) { return DT == VITNA_DTYPE_Q4_K ? U == 3 : DT == VITNA_DTYPE_Q6_K ? (U & 1) : false; } };

/* Unit U's operands of token tile tt, superblock b (and the S-term sums when the unit applies them), from the
   images: every load is 1 KB (512 bytes for the sums) in lane order. */
template <int DT, int U>
__device__ __forceinline__ void sx_load_a(const skinny_args& a, int tt, int K, int b, int lane, sx_a& o) {
    const u32x4* img = reinterpret_cast<const u32x4*>(DT == VITNA_DTYPE_Q6_K ? a.img[1] : a.img[0]) +
                       ((size_t)tt * (K / 256) + b) * 2048 + (size_t)U * 512 + lane;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        o.h[i] = img[i * 128];
        o.l[i] = img[i * 128 + 64];
    }
    if constexpr (sx_unit_sums<DT>::at(U)) {
        const sx_u2* sp = DT == VITNA_DTYPE_Q4_K
                              ? reinterpret_cast<const sx_u2*>(a.s32) + ((size_t)tt * (K / 256) + b) * 192 + lane
                              : reinterpret_cast<const sx_u2*>(a.s16) + ((size_t)tt * (K / 128) + 2 * b + (U >> 1)) * 192 + lane;
#pragma unroll
        for (int i = 0; i < 3; i++) o.sp[i] = sp[64 * i];
    }
}

__device__ __forceinline__ void sx_scale(f32x16& acc, float d, const f32x16& P) {
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = fmaf(d, P[r], acc[r]);
}
#define SX_MMA(A, B, C) __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, A), B, C, 0, 0, 0)

/* Q4_K scale and min of group g from the 12 scale bytes (header dwords 1..3) */
template <int G>
__device__ __forceinline__ void sx_q4k_sm(const u32x4& h, uint32_t& sc, uint32_t& mn) {
    if constexpr (G < 4) {
        sc = (h.y >> (8 * G)) & 63;
        mn = (h.z >> (8 * G)) & 63;
    } else {
        constexpr int j = G - 4;
        sc = ((h.w >> (8 * j)) & 15) | (((h.y >> (8 * j + 6)) & 3) << 4);
        mn = ((h.w >> (8 * j + 4)) & 15) | (((h.z >> (8 * j + 6)) & 3) << 4);
    }
}

/* the S terms of eight groups: the lane half's four sums times its four coefficients c, each as three bf16
   pieces, the six products down to 2^-24 of the largest (the offset part of c S cancels against the MFMA sums
   of 128 + q, so it is carried to fp32 accuracy) */
__device__ __forceinline__ void sx_sterm(const sx_a& x, const float c[4], f32x16& acc) {
    s16x4 cp[3];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const __bf16 p0 = (__bf16)c[i];
        const float r0 = c[i] - (float)p0;
        const __bf16 p1 = (__bf16)r0;
        cp[0][i] = __builtin_bit_cast(short, p0);
        cp[1][i] = __builtin_bit_cast(short, p1);
        cp[2][i] = __builtin_bit_cast(short, (__bf16)(r0 - (float)p1));
    }
    const s16x4 s0 = __builtin_bit_cast(s16x4, x.sp[0]), s1 = __builtin_bit_cast(s16x4, x.sp[1]), s2 = __builtin_bit_cast(s16x4, x.sp[2]);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(s2, cp[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(s1, cp[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(s0, cp[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(s1, cp[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(s0, cp[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(s0, cp[0], acc, 0, 0, 0);
}

/* Unit U: its groups' sums and scales into acc; cs carries the superblock's S coefficients (Q4_K) from the
   units that make them to the unit that applies them. */
template <int DT, int U>
__device__ __forceinline__ void sx_compute(const sx_w<DT>& w, const sx_a& x, int kq, f32x16& acc, float cs[8]) {
    const f32x16 Z = {};
    if constexpr (DT == VITNA_DTYPE_Q4_K) {
        constexpr uint32_t M = 0x0f0f0f0fu;
        const u32x4 q = w.q[U];
        const bf16x8 a0 = sx_join(sx_mag4(q.x & M), sx_mag4(q.y & M)), a1 = sx_join(sx_mag4(q.z & M), sx_mag4(q.w & M));
        const bf16x8 b0 = sx_join(sx_mag4((q.x >> 4) & M), sx_mag4((q.y >> 4) & M));
        const bf16x8 b1 = sx_join(sx_mag4((q.z >> 4) & M), sx_mag4((q.w >> 4) & M));
        f32x16 P0 = SX_MMA(x.h[0], a0, Z), P1 = SX_MMA(x.h[2], b0, Z);
        P0 = SX_MMA(x.h[1], a1, P0);
        P1 = SX_MMA(x.h[3], b1, P1);
        P0 = SX_MMA(x.l[0], a0, P0);
        P1 = SX_MMA(x.l[2], b0, P1);
        P0 = SX_MMA(x.l[1], a1, P0);
        P1 = SX_MMA(x.l[3], b1, P1);
        const float d = f16_bits_to_f32(w.h.x & 0xffffu), dmin = f16_bits_to_f32(w.h.x >> 16);
        uint32_t sc0, mn0, sc1, mn1;
        sx_q4k_sm<2 * U>(w.h, sc0, mn0);
        sx_q4k_sm<2 * U + 1>(w.h, sc1, mn1);
        const float d0 = d * (float)sc0, d1 = d * (float)sc1;
        sx_scale(acc, d0, P0);
        sx_scale(acc, d1, P1);
        cs[2 * U] = -fmaf(128.0f, d0, dmin * (float)mn0);
        cs[2 * U + 1] = -fmaf(128.0f, d1, dmin * (float)mn1);
        if constexpr (U == 3) {
            float c[4];
#pragma unroll
            for (int j = 0; j < 4; j++) c[j] = kq ? cs[4 + j] : cs[j];
            sx_sterm(x, c, acc);
        }
    } else if constexpr (DT == VITNA_DTYPE_Q6_K) {
        constexpr int h = U >> 1, r0 = U & 1;
        bf16x8 wq[4]; /* groups (r0, 0), (r0, 1), (r0 + 2, 0), (r0 + 2, 1) */
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int s = i & 1, hi = i >> 1, r = r0 + 2 * hi;
            uint32_t v[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t ql = hi ? (w.ql[U][s][j] >> 4) : w.ql[U][s][j];
                const uint32_t qh = w.qh[h][s][j];
                const uint32_t top = r == 0 ? qh << 4 : r == 1 ? qh << 2 : r == 2 ? qh : qh >> 2;
                v[j] = (ql & 0x0f0f0f0fu) | (top & 0x30303030u);
            }
            wq[i] = sx_join(sx_mag4(v[0]), sx_mag4(v[1]));
        }
        f32x16 P[4];
#pragma unroll
        for (int i = 0; i < 4; i++) P[i] = SX_MMA(x.h[i], wq[i], Z);
#pragma unroll
        for (int i = 0; i < 4; i++) P[i] = SX_MMA(x.l[i], wq[i], P[i]);
        const float d = f16_bits_to_f32(w.d);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int g = 8 * h + 2 * (r0 + 2 * (i >> 1)) + (i & 1); /* the group's scale index */
            sx_scale(acc, d * (float)(int8_t)(w.sc[g >> 2] >> (8 * (g & 3))), P[i]);
        }
        if constexpr (r0 == 1) {
            /* the S terms of groups 8 h .. 8 h + 7: lane half kq supplies 8 h + 4 kq .. + 3 */
            const uint32_t scw = kq ? w.sc[2 * h + 1] : w.sc[2 * h];
            const float m = -160.0f * d;
            float c[4];
#pragma unroll
            for (int j = 0; j < 4; j++) c[j] = m * (float)(int8_t)(scw >> (8 * j));
            sx_sterm(x, c, acc);
        }
    } else {
        const bf16x8 a0 = sx_i8(w.q[U][0].x, w.q[U][0].y), a1 = sx_i8(w.q[U][0].z, w.q[U][0].w);
        const bf16x8 b0 = sx_i8(w.q[U][1].x, w.q[U][1].y), b1 = sx_i8(w.q[U][1].z, w.q[U][1].w);
        f32x16 P0 = SX_MMA(x.h[0], a0, Z), P1 = SX_MMA(x.h[2], b0, Z);
        P0 = SX_MMA(x.h[1], a1, P0);
        P1 = SX_MMA(x.h[3], b1, P1);
        P0 = SX_MMA(x.l[0], a0, P0);
        P1 = SX_MMA(x.l[2], b0, P1);
        P0 = SX_MMA(x.l[1], a1, P0);
        P1 = SX_MMA(x.l[3], b1, P1);
        const uint32_t dw = w.d[U];
        sx_scale(acc, f16_bits_to_f32(dw & 0xffffu), P0);
        sx_scale(acc, f16_bits_to_f32(dw >> 16), P1);
    }
}

#endif
