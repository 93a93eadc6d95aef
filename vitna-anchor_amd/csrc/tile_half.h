/**
 * tile_half.h - Quantized weights against float32 activations on the f16
 * matrix cores, to better than float32 sums need: the arithmetic of the tiled
 * kernels of passes with many rows (kernels_tgemm.hip).
 *
 * An activation enters as f16 hi + lo of x f, f a power of two that brings
 * the row's largest value under 2^14 (22 bits of each value; what is 2^-17 of
 * the row's largest and smaller keeps an absolute 2^-39 of it, which is more
 * than bf16's hi + lo keep down to 2^-21 of the largest). A weight enters as an
 * exact integer times a power of two, so a superblock is one chain of
 * products and its scale d is applied once:
 *   Q4_K  sc q (at most 63 x 15)             acc += d 2^14 P - 64 dmin M
 *   Q6_K  sc (q - 32), as its f16 rounding   acc += d 2^9 P
 *         and what that left (-1, 0 or 1: the product has up to 13 bits)
 *   Q8_0  q                                  acc += d 2^9 P, each 32 columns
 * with M = sum of m_g S_g / 64 over the eight groups, S_g the group's sum of
 * the split activations, as two more products: S_g / 64 as an f16 hi on lane
 * half 0 and, on lane half 1, the rest 2^11 as two more f16 pieces against
 * m_g 2^-11, which holds all of float32's bits (a fast pass, whose activations
 * have 11, leaves the last piece out).
 *
 * Against the bf16 form (skinny_exact.h) a weight needs no scale a group: Q4_K
 * 50 VALU instructions a 32-row tile's unit instead of 100, of which the
 * matrix cores hide six to a product.
 *
 * Error of a layer's mixture against 64 bits (200 rows, relative 2-norm, worst
 * of Q4_K, Q6_K and Q8_0 mixes at 512 x 256 and 2048 x 768): 9e-7, where the
 * bf16 form's was 4e-5; the typical row 2e-7, where it was 4e-6.
 *
 * The quants are f16 subnormals until their scale makes them normal (the low
 * byte of each 16-bit half: q 2^-24, exactly), so four bytes are two packed
 * multiplies. That takes a dword's bytes in the order 0, 2, 1, 3, and the
 * activations' images hold each four columns in it.
 */
#ifndef VITNA_TILE_HALF_H
#define VITNA_TILE_HALF_H

#include "skinny_exact.h"

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

#define TH_MMA(A, B, C) __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, A), B, C, 0, 0, 0)

__device__ __forceinline__ h2 th_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ h2 th_both(_Float16 v) { return h2{v, v}; }
__device__ __forceinline__ h8 th_join(h2 a, h2 b, h2 c, h2 d) { return h8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y}; }

/* The power of two that brings a row's largest magnitude under 2^14 (1 for a row that is not finite, whose results are
   not either way), its inverse a normal number too. */
__device__ __forceinline__ float th_scale(float largest) {
    const int e = (int)(__float_as_uint(largest) >> 23) & 0xff;
    return e == 0xff ? 1.0f : __uint_as_float((uint32_t)(min(13 - (e - 127), 126) + 127) << 23);
}

/* 1 / f of a power of two whose inverse is normal */
__device__ __forceinline__ float th_inverse(float f) { return __uint_as_float((254u << 23) - __float_as_uint(f)); }

/* eight values times f as f16 hi and lo in the operands' order, and the sum of hi + lo (fast: of hi) */
__device__ __forceinline__ void th_split8(const float e[8], float f, bool fast, u32x4& vh, u32x4& vl, float& sum) {
    h8 h, l;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int at = (k & 4) | ((k & 1) << 1) | ((k >> 1) & 1); /* columns 0, 2, 1, 3 */
        const float v = e[k] * f;
        const _Float16 a = (_Float16)v;
        const _Float16 b = (_Float16)(v - (float)a);
        h[at] = a;
        l[at] = b;
        s += fast ? (float)a : (float)a + (float)b;
    }
    vh = __builtin_bit_cast(u32x4, h);
    vl = __builtin_bit_cast(u32x4, l);
    sum = s;
}

/* Group g's sum S of row l of a tile / superblock, for the lanes of the two M products: sums [2][64 lanes][8], lane half
   0 hi and 0, half 1 the two pieces of 2^11 (S / 64 - hi). */
__device__ __forceinline__ void th_sum(_Float16* sums, int l, int g, float S) {
    const float v = S * 0.015625f;
    const _Float16 h = (_Float16)v;
    const float r = (v - (float)h) * 2048.0f;
    const _Float16 r1 = (_Float16)r;
    sums[l * 8 + g] = h;
    sums[(l + 32) * 8 + g] = r1;
    sums[512 + l * 8 + g] = (_Float16)0.0f;
    sums[512 + (l + 32) * 8 + g] = (_Float16)(r - (float)r1);
}

/* A weight tile's operands of half a unit: its two 16-column steps (and what Q6_K's rounding left of them). */
template <int DT> struct th_b { h8 o[2]; };
template <> struct th_b<VITNA_DTYPE_Q6_K> { h8 o[2], r[2]; };

/* Half N of unit U of a weight tile's bytes. */
template <int DT, int U, int N>
__device__ __forceinline__ void th_unpack(const sx_w<DT>& w, th_b<DT>& b) {
    if constexpr (DT == VITNA_DTYPE_Q4_K) {
        constexpr uint32_t M = N ? 0x00f000f0u : 0x000f000fu;
        uint32_t sc, mn;
        sx_q4k_sm<2 * U + N>(w.h, sc, mn);
        /* q 2^-24 (q 2^-20 for the high nibbles) times sc 2^10 (sc 2^6): sc q 2^-14 */
        const h2 s = th_both((_Float16)(uint16_t)sc * (_Float16)(N ? 64.0f : 1024.0f));
        const uint32_t q[4] = {w.q[U].x, w.q[U].y, w.q[U].z, w.q[U].w};
#pragma unroll
        for (int i = 0; i < 2; i++)
            b.o[i] = th_join(th_h2(q[2 * i] & M) * s, th_h2((q[2 * i] >> 8) & M) * s, th_h2(q[2 * i + 1] & M) * s, th_h2((q[2 * i + 1] >> 8) & M) * s);
    } else if constexpr (DT == VITNA_DTYPE_Q6_K) {
        constexpr int hh = U >> 1, r = (U & 1) + 2 * N, g0 = 8 * hh + 2 * r; /* groups (r, 0), (r, 1) of half hh */
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const h2 sc = th_both((_Float16)(int16_t)(int8_t)(w.sc[g0 >> 2] >> (8 * ((g0 + s) & 3))));
            h2 wh[4], wl[4];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t ql = N ? (w.ql[U][s][j] >> 4) : w.ql[U][s][j], qh = w.qh[hh][s][j];
                const uint32_t top = r == 0 ? qh << 4 : r == 1 ? qh << 2 : r == 2 ? qh : qh >> 2;
                const uint32_t v = (ql & 0x0f0f0f0fu) | (top & 0x30303030u);
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    /* (q - 32) 2^-9, its product with sc, and what rounding that took off */
                    const h2 q = __builtin_elementwise_fma(th_h2((k ? v >> 8 : v) & 0x00ff00ffu), th_both((_Float16)32768.0f), th_both((_Float16)-0.0625f));
                    wh[2 * j + k] = q * sc;
                    wl[2 * j + k] = __builtin_elementwise_fma(q, sc, -wh[2 * j + k]);
                }
            }
            b.o[s] = th_join(wh[0], wh[1], wh[2], wh[3]);
            b.r[s] = th_join(wl[0], wl[1], wl[2], wl[3]);
        }
    } else {
        const uint32_t v[4] = {w.q[U][N].x, w.q[U][N].y, w.q[U][N].z, w.q[U][N].w};
        h2 o[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t u = v[i] ^ 0x80808080u;
#pragma unroll
            for (int k = 0; k < 2; k++)
                o[2 * i + k] = __builtin_elementwise_fma(th_h2((k ? u >> 8 : u) & 0x00ff00ffu), th_both((_Float16)32768.0f), th_both((_Float16)-0.25f));
        }
        b.o[0] = th_join(o[0], o[1], o[2], o[3]);
        b.o[1] = th_join(o[4], o[5], o[6], o[7]);
    }
}

/* The eight minimums of a Q4_K superblock, a byte each, as f16 (1024 + m, less 1024) times the lane half's 1 or 2^-11;
   and what their product is multiplied by. Other types have none. */
template <int DT>
__device__ __forceinline__ float th_dmin(const sx_w<DT>& w) {
    if constexpr (DT == VITNA_DTYPE_Q4_K) return f16_bits_to_f32(w.h.x >> 16) * -64.0f;
    else return 0.0f;
}
template <int DT>
__device__ __forceinline__ u32x4 th_header(const sx_w<DT>& w) {
    if constexpr (DT == VITNA_DTYPE_Q4_K) return w.h;
    else return u32x4{};
}
__device__ __forceinline__ h8 th_mins(const u32x4& hd, int kq) {
    const uint32_t m0 = hd.z & 0x3f3f3f3fu, m1 = ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u);
    const h2 off = th_both((_Float16)1024.0f), f = th_both(kq ? (_Float16)0.00048828125f : (_Float16)1.0f);
    const auto two = [&](uint32_t m, uint32_t bytes) { return (th_h2(__builtin_amdgcn_perm(0x64646464u, m, bytes)) - off) * f; };
    return th_join(two(m0, 0x04010400u), two(m0, 0x04030402u), two(m1, 0x04010400u), two(m1, 0x04030402u));
}

/* What a product chain is multiplied by: the superblock's scale, or for Q8_0 that of unit U's half N. */
template <int DT, int U, int N>
__device__ __forceinline__ float th_d(const sx_w<DT>& w) {
    if constexpr (DT == VITNA_DTYPE_Q4_K) return f16_bits_to_f32(w.h.x & 0xffffu) * 16384.0f;
    else if constexpr (DT == VITNA_DTYPE_Q6_K) return f16_bits_to_f32(w.d) * 512.0f;
    else return f16_bits_to_f32(N ? w.d[U] >> 16 : w.d[U] & 0xffffu) * 512.0f;
}

#endif
