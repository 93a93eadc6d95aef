/**
 * kernels_skinny.hip - Several token rows (up to 32 a tile) times a quantized
 * matrix on the bf16 matrix cores, to fp32 accuracy: the multi-row dense
 * projections of a ragged decode pass (q/k/v, o, LM head).
 *
 * Reference counterpart: rows_dot_multi model_cuda.cu:1826 and the *_multi
 * kernels :1872-2006 (the reference reads each weight row once for up to 8
 * rows, on the CUDA cores); the CPU arithmetic checked against is
 * engine/src/model.c:887-979, one row at a time.
 *
 * Two kernels:
 *   skinny_exact_kernel / skinny_wide_kernel (widths a multiple of 256): the
 *     quants enter the MFMA as exact bf16 integers, each scale group keeps its
 *     own MFMA sum and its scale is applied in fp32 (skinny_exact.h); the
 *     operands come from images in MFMA lane order
 *     (skinny_image.h) and the weights from a tiled copy, so every load of a
 *     wave is 1 KB contiguous.
 *   skinny_kernel (other widths): each weight is widened as the reference
 *     widens it (engine/src/quant.c:40-188) and split into bf16 hi + lo, the
 *     activations likewise (split_rows_kernel), and a product is
 *     hi*hi + hi*lo + lo*hi on v_mfma_f32_32x32x16_bf16: about 2^-16 relative
 *     a product. A workgroup is KS waves over one tile of 32 token rows x
 *     (32 NT) weight rows; wave w takes every KS-th 32-weight slice of K, and
 *     the waves' accumulators are added through LDS in wave order. A lane
 *     supplies weight row lane % 32 and the k-octet lane / 32 of both runs of
 *     each slice, as the activations' lanes do for token lane % 32.
 * Both stay within 1e-3 of the CPU checker; each projection alone is held to
 * 2e-5 of max |ref| against the widened matrix in float64.
 */

#include "vitna_kernels.h"
#include "skinny_image.h"
#include "skinny_exact.h"

#include <algorithm>

#define SK_NT 2 /* token tiles a block of the exact kernel takes when a pass has many */
#ifndef SK_NR
#define SK_NR 2
#endif

/* ---- activations, split ------------------------------------------------- */

__global__ void split_rows_kernel(const float* __restrict__ x, int n, int K, int xstride, uint16_t* __restrict__ xh,
                                  uint16_t* __restrict__ xl) {
    const int r = blockIdx.y;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < K; c += gridDim.x * blockDim.x) {
        const float v = x[(size_t)r * xstride + c];
        const __bf16 h = (__bf16)v;
        const __bf16 l = (__bf16)(v - (float)h);
        xh[(size_t)r * K + c] = __builtin_bit_cast(uint16_t, h);
        xl[(size_t)r * K + c] = __builtin_bit_cast(uint16_t, l);
    }
}

__device__ __forceinline__ uint16_t bf16_bits(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }

/* The operand images of a pass (skinny_image.h): block (b, tt) takes superblock b of token tile tt, thread t
   its 8-column groups t + 256 j; rows past n repeat row n - 1. */
__global__ void split_image_kernel(const float* __restrict__ x, int n, int K, int xstride, u32x4* __restrict__ imga,
                                   u32x4* __restrict__ imgb, uint16_t* __restrict__ s32, uint16_t* __restrict__ s16) {
    const int b = blockIdx.x, tt = blockIdx.y;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int item = threadIdx.x + 256 * j, l = item >> 5, c8 = 32 * b + (item & 31);
        const int tok = min(32 * tt + l, n - 1), row = 32 * tt + l;
        const float4* src = reinterpret_cast<const float4*>(x + (size_t)tok * xstride + 8 * c8);
        const float4 v0 = src[0], v1 = src[1];
        const float e[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        u32x4 vh, vl;
        float sum;
        img_split8(e, vh, vl, sum);
        img_put(imga, imgb, row, K, c8, vh, vl);
        /* the 16- and 32-column sums (the pair's, then the quad's: lanes of consecutive c8, one token) */
        const float t16 = sum + __shfl_xor(sum, 1, WAVE);
        const float t32 = t16 + __shfl_xor(t16, 2, WAVE);
        if (!(c8 & 1)) img_sum16(s16, row, K, c8 >> 1, t16);
        if (!(c8 & 3)) img_sum32(s32, row, K, c8 >> 2, t32);
    }
}

hipError_t launch_split_rows(const float* x, int n, int K, int xstride, uint16_t* xh, uint16_t* xl, uint32_t* const* img,
                             hipStream_t s) {
    if (n < 1 || K < 1) return hipErrorInvalidValue;
    if (img) {
        if (K % 256 || xstride % 4 || (uintptr_t)x % 16) return hipErrorInvalidValue;
        split_image_kernel<<<dim3(K / 256, (n + 31) / 32), 256, 0, s>>>(x, n, K, xstride, (u32x4*)img[0], (u32x4*)img[1],
                                                                        (uint16_t*)img[2], (uint16_t*)img[3]);
    } else {
        split_rows_kernel<<<dim3((K + 255) / 256, n), 256, 0, s>>>(x, n, K, xstride, xh, xl);
    }
    return hipGetLastError();
}

/* ---- weights: one lane's octets of a slice, widened ----------------------- */

/* Elements 8 kq .. 8 kq + 7 of the slice's low run (lo) and high run (hi),
   widened exactly. */
template <int DT>
__device__ __forceinline__ void widen_octets(const qraw& r, int t, int kq, float lo[8], float hi[8]) {
    if (DT == VITNA_DTYPE_Q8_0) {
        const float d = f16_bits_to_f32(r.c);
        const uint32_t a0 = kq ? r.a.z : r.a.x, a1 = kq ? r.a.w : r.a.y, b0 = kq ? r.b.z : r.b.x, b1 = kq ? r.b.w : r.b.y;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = (float)(int8_t)((a0 >> (8 * i)) & 0xff) * d;
            lo[4 + i] = (float)(int8_t)((a1 >> (8 * i)) & 0xff) * d;
            hi[i] = (float)(int8_t)((b0 >> (8 * i)) & 0xff) * d;
            hi[4 + i] = (float)(int8_t)((b1 >> (8 * i)) & 0xff) * d;
        }
    } else if (DT == VITNA_DTYPE_Q4_K) {
        const uint32_t h0 = r.b.x, s03 = r.b.y, s47 = r.b.z, s8b = r.b.w;
        const float d = f16_bits_to_f32(h0 & 0xffffu), dmin = f16_bits_to_f32(h0 >> 16);
        const int c = (t & 7) >> 1;
        uint32_t sc0, mn0, sc1, mn1;
        if (c < 2) {
            const int g0 = 2 * c, g1 = g0 + 1;
            sc0 = (s03 >> (8 * g0)) & 63; mn0 = (s47 >> (8 * g0)) & 63;
            sc1 = (s03 >> (8 * g1)) & 63; mn1 = (s47 >> (8 * g1)) & 63;
        } else {
            const int j0 = 2 * c - 4, j1 = j0 + 1;
            sc0 = ((s8b >> (8 * j0)) & 15) | (((s03 >> (8 * j0 + 6)) & 3) << 4);
            mn0 = ((s8b >> (8 * j0 + 4)) & 15) | (((s47 >> (8 * j0 + 6)) & 3) << 4);
            sc1 = ((s8b >> (8 * j1)) & 15) | (((s03 >> (8 * j1 + 6)) & 3) << 4);
            mn1 = ((s8b >> (8 * j1 + 4)) & 15) | (((s47 >> (8 * j1 + 6)) & 3) << 4);
        }
        const float d10 = d * (float)sc0, m10 = dmin * (float)mn0, d11 = d * (float)sc1, m11 = dmin * (float)mn1;
        const uint32_t w0 = kq ? r.a.z : r.a.x, w1 = kq ? r.a.w : r.a.y;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = d10 * (float)((w0 >> (8 * i)) & 15) - m10;
            lo[4 + i] = d10 * (float)((w1 >> (8 * i)) & 15) - m10;
            hi[i] = d11 * (float)((w0 >> (8 * i + 4)) & 15) - m11;
            hi[4 + i] = d11 * (float)((w1 >> (8 * i + 4)) & 15) - m11;
        }
    } else { /* Q6_K */
        const int sh = (int)(r.c >> 16);
        const float d = f16_bits_to_f32(r.d);
        const float ds0 = d * (float)(int8_t)(r.c & 0xff), ds1 = d * (float)(int8_t)((r.c >> 8) & 0xff);
        const uint32_t l0 = kq ? r.a.z : r.a.x, l1 = kq ? r.a.w : r.a.y, q0h = kq ? r.b.z : r.b.x, q1h = kq ? r.b.w : r.b.y;
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const uint32_t ql = w ? l1 : l0, hb = (w ? q1h : q0h) >> sh;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int qa = (int)(((ql >> (8 * i)) & 15) | (((hb >> (8 * i)) & 3) << 4)) - 32;
                const int qb = (int)(((ql >> (8 * i + 4)) & 15) | (((hb >> (8 * i + 4)) & 3) << 4)) - 32;
                lo[4 * w + i] = ds0 * (float)qa;
                hi[4 * w + i] = ds1 * (float)qb;
            }
        }
    }
}

__device__ __forceinline__ void split8(const float w[8], bf16x8& h, bf16x8& l) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const __bf16 b = (__bf16)w[i];
        h[i] = b;
        l[i] = (__bf16)(w[i] - (float)b);
    }
}

/* ---- the kernel --------------------------------------------------------- */

/* Block (blockIdx.x = weight-row block of matrix i, blockIdx.y = token tile). */
template <int NT>
__global__ __launch_bounds__(NT == 1 ? 1024 : 256) void skinny_kernel(skinny_args a) {
    extern __shared__ float red[]; /* [KS][NT][16][64] when KS > 1 */
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, KS = blockDim.x >> 6;
    const int l32 = lane & 31, kq = lane >> 5;
    constexpr int RB = 32 * NT; /* weight rows a block */
    int bx = blockIdx.x, mi = 0;
    for (; mi < a.nm - 1; mi++) {
        const int nb = (a.w[mi].rows + RB - 1) / RB;
        if (bx < nb) break;
        bx -= nb;
    }
    const qmat& w = a.w[mi];
    const int dt = w.dtype;
    const int row0 = bx * RB;
    const int tok0 = blockIdx.y * SK_TOK, tok = tok0 + l32;
    const bool tok_ok = tok < a.n;
    const int S = w.cols / 32;
    const uint16_t* xh = a.xh + (size_t)(tok_ok ? tok : 0) * w.cols;
    const uint16_t* xl = a.xl + (size_t)(tok_ok ? tok : 0) * w.cols;

    f32x16 acc[NT];
#pragma unroll
    for (int k = 0; k < NT; k++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[k][r] = 0.0f;

    /* one slice's operands: the activations (token tok, the lane's octet of both runs) and the NT weight rows */
    struct slice_ops {
        u32x4 ah0, al0, ah1, al1;
        qraw q[NT];
    };
    auto load = [&](int t, slice_ops& o) {
        int clo, chi;
        slice_cols(dt, t, &clo, &chi);
        o.ah0 = o.al0 = o.ah1 = o.al1 = u32x4{0, 0, 0, 0};
        if (tok_ok) {
            o.ah0 = *reinterpret_cast<const u32x4*>(xh + clo + 8 * kq);
            o.al0 = *reinterpret_cast<const u32x4*>(xl + clo + 8 * kq);
            o.ah1 = *reinterpret_cast<const u32x4*>(xh + chi + 8 * kq);
            o.al1 = *reinterpret_cast<const u32x4*>(xl + chi + 8 * kq);
        }
#pragma unroll
        for (int k = 0; k < NT; k++) {
            const int rr = min(row0 + 32 * k + l32, w.rows - 1);
            if (dt == VITNA_DTYPE_Q4_K) slice_load<VITNA_DTYPE_Q4_K>(w, 0, rr, t, o.q[k]);
            else if (dt == VITNA_DTYPE_Q6_K) slice_load<VITNA_DTYPE_Q6_K>(w, 0, rr, t, o.q[k]);
            else slice_load<VITNA_DTYPE_Q8_0>(w, 0, rr, t, o.q[k]);
        }
    };
    auto compute = [&](int t, const slice_ops& o) {
        const bf16x8 Ah0 = __builtin_bit_cast(bf16x8, o.ah0), Al0 = __builtin_bit_cast(bf16x8, o.al0);
        const bf16x8 Ah1 = __builtin_bit_cast(bf16x8, o.ah1), Al1 = __builtin_bit_cast(bf16x8, o.al1);
#pragma unroll
        for (int k = 0; k < NT; k++) {
            float wlo[8], whi[8];
            if (dt == VITNA_DTYPE_Q4_K) widen_octets<VITNA_DTYPE_Q4_K>(o.q[k], t, kq, wlo, whi);
            else if (dt == VITNA_DTYPE_Q6_K) widen_octets<VITNA_DTYPE_Q6_K>(o.q[k], t, kq, wlo, whi);
            else widen_octets<VITNA_DTYPE_Q8_0>(o.q[k], t, kq, wlo, whi);
            bf16x8 Bh0, Bl0, Bh1, Bl1;
            split8(wlo, Bh0, Bl0);
            split8(whi, Bh1, Bl1);
            acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Ah0, Bh0, acc[k], 0, 0, 0);
            acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Ah0, Bl0, acc[k], 0, 0, 0);
            acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Al0, Bh0, acc[k], 0, 0, 0);
            acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Ah1, Bh1, acc[k], 0, 0, 0);
            acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Ah1, Bl1, acc[k], 0, 0, 0);
            acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Al1, Bh1, acc[k], 0, 0, 0);
        }
    };
    /* slices wv, wv + KS, ...: the next one's loads in flight while this one computes */
    slice_ops o0, o1;
    if (wv < S) load(wv, o0);
    for (int t = wv; t < S; t += 2 * KS) {
        if (t + KS < S) load(t + KS, o1);
        compute(t, o0);
        if (t + KS >= S) break;
        if (t + 2 * KS < S) load(t + 2 * KS, o0);
        compute(t + KS, o1);
    }
    /* accumulator r of a lane: token 8 (r / 4) + 4 (lane / 32) + r % 4 of the tile, weight row lane % 32 */
    float* y = a.y[mi];
    auto put = [&](int k, int r, float v) {
        const int n = row0 + 32 * k + l32;
        const int tk = tok0 + 8 * (r >> 2) + 4 * kq + (r & 3);
        if (n < w.rows && tk < a.n) {
            float* o = y + (size_t)tk * w.rows + n;
            *o = a.add ? *o + v : v;
        }
    };
    if (KS == 1) {
#pragma unroll
        for (int k = 0; k < NT; k++)
#pragma unroll
            for (int r = 0; r < 16; r++) put(k, r, acc[k][r]);
        return;
    }
    /* the waves' sums: every wave's accumulators through LDS, then wave v adds up the registers r = v, v + KS,
       ... of every tile over the waves, in wave order */
#pragma unroll
    for (int k = 0; k < NT; k++)
#pragma unroll
        for (int r = 0; r < 16; r++) red[((wv * NT + k) * 16 + r) * 64 + lane] = acc[k][r];
    __syncthreads();
    for (int kr = wv; kr < NT * 16; kr += KS) {
        const int k = kr >> 4, r = kr & 15;
        float v = 0.0f;
        for (int u = 0; u < KS; u++) v += red[((u * NT + k) * 16 + r) * 64 + lane];
        put(k, r, v);
    }
}

/* ---- the tiled copy (its layout: skinny_exact.h) ------------------------- */

__device__ __forceinline__ uint32_t tile_src(const qmat& m, int tile, int b, int o) {
    /* the byte of the planes that byte o of tile / superblock b copies */
    const int S = m.cols / 256;
    (void)S;
    if (m.dtype == VITNA_DTYPE_Q4_K) {
        if (o < 4096) {
            const int u = o >> 10, lane = (o >> 4) & 63, j = o & 15;
            const size_t row = min(32 * tile + (lane & 31), m.rows - 1);
            return m.p[0][(row * m.nb + b) * 128 + 32 * u + 16 * (lane >> 5) + j];
        }
        const int l32 = (o - 4096) >> 4, j = o & 15;
        const size_t row = min(32 * tile + l32, m.rows - 1);
        return m.p[1][(row * m.nb + b) * 16 + j];
    } else if (m.dtype == VITNA_DTYPE_Q6_K) {
        if (o < 4096) {
            const int u = o >> 10, lane = (o >> 4) & 63, j = o & 15, sh = j >> 3, jj = j & 7;
            const size_t row = min(32 * tile + (lane & 31), m.rows - 1);
            return m.p[0][(row * m.nb + b) * 128 + 64 * (u >> 1) + 32 * (u & 1) + 16 * sh + 8 * (lane >> 5) + jj];
        }
        if (o < 6144) {
            const int q = o - 4096, h = q >> 10, lane = (q >> 4) & 63, j = q & 15, sh = j >> 3, jj = j & 7;
            const size_t row = min(32 * tile + (lane & 31), m.rows - 1);
            return m.p[1][(row * m.nb + b) * 64 + 32 * h + 16 * sh + 8 * (lane >> 5) + jj];
        }
        if (o < 6656) {
            const int l32 = (o - 6144) >> 4, j = o & 15;
            const size_t row = min(32 * tile + l32, m.rows - 1);
            return m.p[2][(row * m.nb + b) * 16 + j];
        }
        const int l32 = (o - 6656) >> 1, j = o & 1;
        const size_t row = min(32 * tile + l32, m.rows - 1);
        return m.p[3][(row * m.nb + b) * 2 + j];
    } else {
        if (o < 8192) {
            const int v = o >> 10, lane = (o >> 4) & 63, j = o & 15;
            const size_t row = min(32 * tile + (lane & 31), m.rows - 1);
            return m.p[0][(row * m.nb + 8 * b + v) * 32 + 16 * (lane >> 5) + j];
        }
        const int l32 = (o - 8192) >> 4, j = o & 15;
        const size_t row = min(32 * tile + l32, m.rows - 1);
        return m.p[1][(row * m.nb + 8 * b) * 2 + j];
    }
}

/* One block a tile / superblock, a thread a byte (the copy is made once, at upload). */
__global__ void tile_kernel(qmat m, uint8_t* __restrict__ dst) {
    const int S = m.cols / 256, tile = blockIdx.x / S, b = blockIdx.x % S;
    const int tb = (int)tile_bytes(m.dtype);
    uint8_t* out = dst + (size_t)blockIdx.x * tb;
    for (int o = threadIdx.x; o < tb; o += blockDim.x) out[o] = (uint8_t)tile_src(m, tile, b, o);
}

hipError_t launch_tile(const qmat& m, uint8_t* dst, hipStream_t s) {
    if (!tile_bytes(m.dtype) || m.cols % 256 || m.rows < 1) return hipErrorInvalidValue;
    tile_kernel<<<((m.rows + 31) / 32) * (m.cols / 256), 256, 0, s>>>(m, dst);
    return hipGetLastError();
}

/* Superblock b of the lane's weight rows of NR consecutive 32-row tiles (those of them below nr) against NT
   token tiles tt0, tt0 + 1, ... (those below mt): every weight load issued first, then each token tile's
   activations two units ahead, each unit's activations used for all NR weight tiles; the weights stay in
   registers across the token tiles, and each (weight tile, token tile)'s sums run as they would alone. */
template <int DT, int NT, int NR>
__device__ __forceinline__ void sx_superblock(const skinny_args& a, const qmat& w, int tile, int nr, int tt0, int mt, int b,
                                              int lane, f32x16 (&acc)[NR][NT]) {
    const int kq = lane >> 5;
    const int K = w.cols;
    sx_w<DT> W[NR];
#pragma unroll
    for (int r = 0; r < NR; r++)
        if (r < nr) sx_load_w<DT>(w, tile + r, b, lane, W[r]);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int tt = tt0 + t;
        if (tt >= mt) break;
        float cs[NR][8];
        sx_a x0, x1;
        sx_load_a<DT, 0>(a, tt, K, b, lane, x0);
        sx_load_a<DT, 1>(a, tt, K, b, lane, x1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < NR; r++)
            if (r < nr) sx_compute<DT, 0>(W[r], x0, kq, acc[r][t], cs[r]);
        sx_load_a<DT, 2>(a, tt, K, b, lane, x0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < NR; r++)
            if (r < nr) sx_compute<DT, 1>(W[r], x1, kq, acc[r][t], cs[r]);
        sx_load_a<DT, 3>(a, tt, K, b, lane, x1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < NR; r++)
            if (r < nr) sx_compute<DT, 2>(W[r], x0, kq, acc[r][t], cs[r]);
#pragma unroll
        for (int r = 0; r < NR; r++)
            if (r < nr) sx_compute<DT, 3>(W[r], x1, kq, acc[r][t], cs[r]);
    }
}

/*
 * Block (blockIdx.x = (32-row tile of matrix i, split), blockIdx.y = token tile): KS waves, wave v on superblock
 * 8 split + v. The waves' sums are added through LDS in wave order. A matrix wider than 8 superblocks takes
 * several splits: each block stores its tile's sum in part[], and the block that finishes a tile last (its
 * counter in cnt[]) adds the splits' sums in split order, writes the result and clears the counter, so the
 * result does not depend on which block finishes last. With a.fold (many token tiles) each split's block writes
 * its sums to its own copy of y and skinny_fold_kernel adds them, in the same order.
 */
template <int NT, int NR>
__global__ __launch_bounds__(512) void skinny_exact_kernel(skinny_args a) {
    extern __shared__ float red[]; /* [KS][16][64] */
    __shared__ int last;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, KS = blockDim.x >> 6;
    const int l32 = lane & 31, kq = lane >> 5;
    int bx = blockIdx.x, mi = 0, tile0 = 0;
    size_t fold0 = 0; /* with a.fold: the matrix's first copy in part */
    for (; mi < a.nm - 1; mi++) {
        const int nb = ((a.w[mi].rows + 31) / 32 + NR - 1) / NR * a.splits[mi];
        if (bx < nb) break;
        bx -= nb;
        tile0 += (a.w[mi].rows + 31) / 32;
        fold0 += (size_t)a.splits[mi] * a.n * a.w[mi].rows;
    }
    const qmat& w = a.w[mi];
    const int splits = a.splits[mi], sp = bx % splits, tile = bx / splits * NR;
    const int nr = min(NR, (w.rows + 31) / 32 - tile); /* this block's weight tiles */
    const int mt = (a.n + SK_TOK - 1) / SK_TOK, tt0 = blockIdx.y * NT;
    const int b = 8 * sp + wv;
    f32x16 acc[NR][NT];
#pragma unroll
    for (int r = 0; r < NR; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = f32x16{};
    if (b < w.cols / 256) {
        if (w.dtype == VITNA_DTYPE_Q4_K) sx_superblock<VITNA_DTYPE_Q4_K, NT, NR>(a, w, tile, nr, tt0, mt, b, lane, acc);
        else if (w.dtype == VITNA_DTYPE_Q6_K) sx_superblock<VITNA_DTYPE_Q6_K, NT, NR>(a, w, tile, nr, tt0, mt, b, lane, acc);
        /* (two Q8_0 weight tiles a block do not fit the registers: the launch keeps Q8_0 to one) */
        else if constexpr (NR == 1) sx_superblock<VITNA_DTYPE_Q8_0, NT, NR>(a, w, tile, nr, tt0, mt, b, lane, acc);
    }

    float* y = a.y[mi];
#pragma unroll
    for (int wr = 0; wr < NR; wr++) {
        if (wr >= nr) break;
        const int row0 = 32 * (tile + wr);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int tt = tt0 + t;
            if (tt >= mt) break;
            /* accumulator r of a lane: token 8 (r / 4) + 4 (lane / 32) + r % 4 of the tile, weight row lane % 32 */
            const int tok0 = tt * SK_TOK;
            auto put = [&](int r, float v) {
                const int n = row0 + l32;
                const int tk = tok0 + 8 * (r >> 2) + 4 * kq + (r & 3);
                if (n < w.rows && tk < a.n) {
                    float* o = y + (size_t)tk * w.rows + n;
                    *o = a.add ? *o + v : v;
                }
            };
            if (KS > 1) {
                if (t || wr) __syncthreads(); /* the previous tile's sums are read */
#pragma unroll
                for (int r = 0; r < 16; r++) red[(wv * 16 + r) * 64 + lane] = acc[wr][t][r];
                __syncthreads();
            }
            if (splits == 1) {
                if (KS == 1) {
#pragma unroll
                    for (int r = 0; r < 16; r++) put(r, acc[wr][t][r]);
                    continue;
                }
                for (int r = wv; r < 16; r += KS) {
                    float v = 0.0f;
                    for (int u = 0; u < KS; u++) v += red[(u * 16 + r) * 64 + lane];
                    put(r, v);
                }
                continue;
            }
            if (a.fold) {
                float* o = a.part + fold0 + (size_t)sp * a.n * w.rows + row0 + l32;
                for (int r = wv; r < 16; r += KS) {
                    float v = 0.0f;
                    for (int u = 0; u < KS; u++) v += red[(u * 16 + r) * 64 + lane];
                    const int tk = tok0 + 8 * (r >> 2) + 4 * kq + (r & 3);
                    if (row0 + l32 < w.rows && tk < a.n) o[(size_t)tk * w.rows] = v;
                }
                continue;
            }
            /* several splits: this block's sum of the tile into part[], then the last block of the tile adds them */
            const size_t slot = (size_t)tt * a.tiles + tile0 + tile + wr; /* the tile's counter */
            float* part = a.part + slot * a.split_max * 1024;
            /* The sums are stored as agent-scope atomics (written through this XCD's L2 to where every XCD reads);
               the counter's increment releases them and the last block's acquires them, at agent scope, so the last
               block reads every split's sums (the workgroup barrier carries thread 0's acquire to the others). */
            for (int r = wv; r < 16; r += KS) {
                float v = 0.0f;
                for (int u = 0; u < KS; u++) v += red[(u * 16 + r) * 64 + lane];
                __hip_atomic_store(part + (size_t)sp * 1024 + r * 64 + lane, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* every wave's stores complete before the barrier */
            __syncthreads();
            if (threadIdx.x == 0) last = __hip_atomic_fetch_add(a.cnt + slot, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == splits - 1;
            __syncthreads();
            if (last) {
                for (int r = wv; r < 16; r += KS) {
                    float v = 0.0f;
                    for (int u = 0; u < splits; u++)
                        v += __hip_atomic_load(part + (size_t)u * 1024 + r * 64 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    put(r, v);
                }
                if (threadIdx.x == 0) __hip_atomic_store(a.cnt + slot, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

/* y (+)= the splits' sums, in split order, four values a thread */
__global__ __launch_bounds__(256) void skinny_fold_kernel(const float* __restrict__ part, int splits, size_t n, float* __restrict__ y, int add) {
    const size_t i0 = (size_t)blockIdx.x * 1024 + threadIdx.x;
    float old[4], v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        old[j] = add && i0 + 256 * j < n ? y[i0 + 256 * j] : 0.0f;
        v[j] = 0.0f;
    }
    for (int u = 0; u < splits; u++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i0 + 256 * j < n) v[j] += part[u * n + i0 + 256 * j];
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (i0 + 256 * j < n) y[i0 + 256 * j] = add ? old[j] + v[j] : v[j];
}

/* Token tiles from which a split width's sums are added by skinny_fold_kernel. A tile's counter costs no launch, but
   each count is a release and an acquire at agent scope, which write back and invalidate an XCD's L2: with few tiles
   that hides behind the weights' reads, with many it is most of the time. A 4096-wide projection to 2048 (kernel
   trace, us), with the counters, and the kernel + the fold: 1024 rows 152, 65 + 5; 333 rows 56, 26 + 4; 128 rows 20,
   10 + 4; 96 rows 21, 12 + 4; 64 rows 12.3, 8 + 4; 32 rows 10.3, 6.5 + 2.5; 8 rows 9.8, 7 + 3: up to two tiles they
   are level in the trace, and a pass of 8 rows 562 and 567 us, of 32 rows 2.50 and 2.53 ms (the launch's gap). */
#define SK_FOLD_TILES 3

/* ---- wide matrices (the LM head): activations staged in LDS ---------------- */

#define SXW_PIECES 2048

typedef __attribute__((address_space(3))) void* sx_lds_void;
typedef __attribute__((address_space(1))) void* sx_glb_void;

/* Superblock b's image of token tile tt, copied into LDS by global-to-LDS loads (lane l of a wave lands at the
   wave's base + 16 l: a straight copy). Counted by vmcnt. */
template <int DT, int NW>
__device__ __forceinline__ void sxw_fetch(const skinny_args& a, int K, int tt, int b, u32x4* img) {
    const int wv = threadIdx.x >> 6;
    const u32x4* src = reinterpret_cast<const u32x4*>(DT == VITNA_DTYPE_Q6_K ? a.img[1] : a.img[0]) + ((size_t)tt * (K / 256) + b) * 2048;
#pragma unroll
    for (int j = 0; j < SXW_PIECES / (64 * NW); j++) {
        const int p = threadIdx.x + 64 * NW * j;
        __builtin_amdgcn_global_load_lds((sx_glb_void)(src + p), (sx_lds_void)(img + wv * 64 + 64 * NW * j), 16, 0, 0);
    }
}

template <int DT, int U>
__device__ __forceinline__ void sxw_read(const u32x4* img, const skinny_args& a, int tt, int K, int b, int lane, sx_a& o) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        o.h[i] = img[U * 512 + i * 128 + lane];
        o.l[i] = img[U * 512 + i * 128 + 64 + lane];
    }
    if constexpr (sx_unit_sums<DT>::at(U)) {
        const sx_u2* sp = DT == VITNA_DTYPE_Q4_K
                              ? reinterpret_cast<const sx_u2*>(a.s32) + ((size_t)tt * (K / 256) + b) * 192 + lane
                              : reinterpret_cast<const sx_u2*>(a.s16) + ((size_t)tt * (K / 128) + 2 * b + (U >> 1)) * 192 + lane;
#pragma unroll
        for (int i = 0; i < 3; i++) o.sp[i] = sp[64 * i];
    }
}

/* NW waves, wave v on tile NW blockIdx.x + v of the matrix, every superblock in turn: the block stages
   superblock b + 1's activations and each wave loads its weights for b + 1 while b computes. */
template <int DT, int NW>
__device__ __forceinline__ void sxw_body(const skinny_args& a, const qmat& w, int tile, int tt, u32x4* img, f32x16& acc) {
    const int lane = threadIdx.x & 63, kq = lane >> 5;
    const int K = w.cols, S = K / 256;

    sx_w<DT> W0, W1;
    float cs[8];
    sxw_fetch<DT, NW>(a, K, tt, 0, img);
    sx_load_w<DT>(w, tile, 0, lane, W0);
    auto step = [&](int b, const sx_w<DT>& W, sx_w<DT>& Wn) {
        /* image b landed (each wave waits for its own loads, the barrier for the others'); image b + 1's
           buffer was last read in step b - 1, which every wave has left */
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const u32x4* cur = img + (b & 1) * SXW_PIECES;
        if (b + 1 < S) {
            sxw_fetch<DT, NW>(a, K, tt, b + 1, img + ((b + 1) & 1) * SXW_PIECES);
            sx_load_w<DT>(w, tile, b + 1, lane, Wn);
        }
        /* one unit's operands at a time (the barriers keep the scheduler from hoisting every unit's reads) */
        sx_a x;
        sxw_read<DT, 0>(cur, a, tt, K, b, lane, x);
        sx_compute<DT, 0>(W, x, kq, acc, cs);
        __builtin_amdgcn_sched_barrier(0);
        sxw_read<DT, 1>(cur, a, tt, K, b, lane, x);
        sx_compute<DT, 1>(W, x, kq, acc, cs);
        __builtin_amdgcn_sched_barrier(0);
        sxw_read<DT, 2>(cur, a, tt, K, b, lane, x);
        sx_compute<DT, 2>(W, x, kq, acc, cs);
        __builtin_amdgcn_sched_barrier(0);
        sxw_read<DT, 3>(cur, a, tt, K, b, lane, x);
        sx_compute<DT, 3>(W, x, kq, acc, cs);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int b = 0; b < S; b += 2) {
        step(b, W0, W1);
        if (b + 1 < S) step(b + 1, W1, W0);
    }
}

/* Every matrix of the launch has dtype DT. */
template <int DT, int NW>
__global__ __launch_bounds__(64 * NW) void skinny_wide_kernel(skinny_args a) {
    __shared__ u32x4 img[2 * SXW_PIECES]; /* 64 KB */
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, l32 = lane & 31, kq = lane >> 5;
    int bx = blockIdx.x, mi = 0;
    for (; mi < a.nm - 1; mi++) {
        const int nb = ((a.w[mi].rows + 31) / 32 + NW - 1) / NW;
        if (bx < nb) break;
        bx -= nb;
    }
    const qmat& w = a.w[mi];
    const int tile = NW * bx + wv, tok0 = blockIdx.y * SK_TOK;
    f32x16 acc = {};
    sxw_body<DT, NW>(a, w, tile, blockIdx.y, img, acc);
    float* y = a.y[mi];
    const int n = 32 * tile + l32;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int tk = tok0 + 8 * (r >> 2) + 4 * kq + (r & 3);
        if (n < w.rows && tk < a.n) {
            float* o = y + (size_t)tk * w.rows + n;
            *o = a.add ? *o + acc[r] : acc[r];
        }
    }
}

static hipError_t launch_skinny_exact(const skinny_args& a0, hipStream_t s) {
    skinny_args a = a0;
    const int mt = (a.n + SK_TOK - 1) / SK_TOK;
    int blocks = 0, ks = 1, tiles = 0, split_max = 1;
    for (int i = 0; i < a.nm; i++) {
        const int S = a.w[i].cols / 256;
        a.splits[i] = (S + 7) / 8;
        ks = std::max(ks, std::min(S, 8));
        split_max = std::max(split_max, a.splits[i]);
        tiles += (a.w[i].rows + 31) / 32;
        blocks += (a.w[i].rows + 31) / 32 * a.splits[i];
    }
    a.tiles = tiles;
    a.split_max = split_max;
    bool one_dt = true;
    for (int i = 1; i < a.nm; i++) one_dt &= a.w[i].dtype == a.w[0].dtype;
    if (tiles >= 1024 && one_dt) {
        /* wide: NW tiles a block over the whole width, the activations shared through LDS (Q8_0 takes four
           waves a block: its two superblocks of weights in flight need more registers than eight allow) */
        const int dt = a.w[0].dtype, NW = dt == VITNA_DTYPE_Q8_0 ? 4 : 8;
        int wb = 0;
        for (int i = 0; i < a.nm; i++) wb += ((a.w[i].rows + 31) / 32 + NW - 1) / NW;
        const dim3 grid(wb, mt);
        if (dt == VITNA_DTYPE_Q4_K) skinny_wide_kernel<VITNA_DTYPE_Q4_K, 8><<<grid, 512, 0, s>>>(a);
        else if (dt == VITNA_DTYPE_Q6_K) skinny_wide_kernel<VITNA_DTYPE_Q6_K, 8><<<grid, 512, 0, s>>>(a);
        else skinny_wide_kernel<VITNA_DTYPE_Q8_0, 4><<<grid, 256, 0, s>>>(a);
        return hipGetLastError();
    }
    if (split_max > 1 && (!a.part || !a.cnt || (size_t)mt * tiles > a.cnt_cap || (size_t)mt * tiles * split_max * 1024 > a.part_cap))
        return hipErrorInvalidValue;
    a.fold = split_max > 1 && mt >= SK_FOLD_TILES;
    /* many token tiles (a prompt's chunk): each block takes SK_NT of them, the weights loaded once for all, or
       two weight tiles against the same token tile, each unit's activations loaded once for both */
    const size_t lds = (size_t)ks * 16 * 64 * sizeof(float);
    if (mt >= 2 * SK_NT) {
        bool q8 = false;
        for (int i = 0; i < a.nm; i++) q8 |= a.w[i].dtype == VITNA_DTYPE_Q8_0;
        if (SK_NR == 2 && !q8) {
            int b2 = 0;
            for (int i = 0; i < a.nm; i++) b2 += ((a.w[i].rows + 31) / 32 + 1) / 2 * a.splits[i];
            skinny_exact_kernel<1, 2><<<dim3(b2, mt), 64 * ks, lds, s>>>(a);
        } else {
            skinny_exact_kernel<SK_NT, 1><<<dim3(blocks, (mt + SK_NT - 1) / SK_NT), 64 * ks, lds, s>>>(a);
        }
    } else {
        skinny_exact_kernel<1, 1><<<dim3(blocks, mt), 64 * ks, lds, s>>>(a);
    }
    const float* part = a.part;
    for (int i = 0; a.fold && i < a.nm; i++) {
        const size_t y = (size_t)a.n * a.w[i].rows;
        skinny_fold_kernel<<<(unsigned)((y + 1023) / 1024), 256, 0, s>>>(part, a.splits[i], y, a.y[i], a.add);
        part += a.splits[i] * y;
    }
    return hipGetLastError();
}

hipError_t launch_skinny(const skinny_args& a, hipStream_t s) {
    if (a.nm < 1 || a.nm > 3 || a.n < 1) return hipErrorInvalidValue;
    for (int i = 0; i < a.nm; i++) {
        const int d = a.w[i].dtype;
        if (a.w[i].cols != a.w[0].cols || a.w[i].cols % 32) return hipErrorInvalidValue;
        if (d != VITNA_DTYPE_Q8_0 && d != VITNA_DTYPE_Q4_K && d != VITNA_DTYPE_Q6_K) return hipErrorInvalidValue;
    }
    bool exact = a.img[0] && a.img[1] && a.s16 && a.s32;
    for (int i = 0; i < a.nm; i++) exact &= a.w[i].cols % 256 == 0 && a.w[i].tiled;
    if (exact) return launch_skinny_exact(a, s);
    if (!a.xh || !a.xl) return hipErrorInvalidValue;
    int cus = 0, dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    const int want = 8 * cus; /* two waves a SIMD */
    const int mt = (a.n + SK_TOK - 1) / SK_TOK;
    const int S = a.w[0].cols / 32;
    int rows = 0;
    for (int i = 0; i < a.nm; i++) rows += a.w[i].rows;
    /* wide matrices (the LM head) take four 32-row tiles a wave, so each token tile's activations are read
       a quarter as often; the rest one */
    const bool wide = rows >= 32768;
    const int RB = wide ? 128 : 32, ks_max = wide ? 2 : 16;
    int blocks = 0;
    for (int i = 0; i < a.nm; i++) blocks += (a.w[i].rows + RB - 1) / RB;
    int ks = 1;
    while (ks < ks_max && ks * 2 <= S && (size_t)blocks * mt * ks < (size_t)want) ks *= 2;
    const size_t lds = ks > 1 ? (size_t)ks * (wide ? 4 : 1) * 16 * 64 * sizeof(float) : 0;
    const dim3 grid(blocks, mt);
    if (wide) skinny_kernel<4><<<grid, 64 * ks, lds, s>>>(a);
    else skinny_kernel<1><<<grid, 64 * ks, lds, s>>>(a);
    return hipGetLastError();
}

/* ---- the crowded passes' copy of the experts (kernels_tgemm.hip) ------------ */

/* One block a (expert, 32-row tile, superblock): the expert's planes as a matrix of its own. */
__global__ void gsx_tile_kernel(qmat m, int tiles, uint8_t* __restrict__ dst) {
    const int S = m.cols / 256, b = blockIdx.x % S, tile = (blockIdx.x / S) % tiles, e = blockIdx.x / (S * tiles);
    qmat me = m;
#pragma unroll
    for (int i = 0; i < 4; i++) me.p[i] = m.p[i] ? m.p[i] + (size_t)e * m.estride[i] : nullptr;
    const int tb = (int)tile_bytes(m.dtype);
    uint8_t* out = dst + (size_t)blockIdx.x * tb;
    for (int o = threadIdx.x; o < tb; o += blockDim.x) out[o] = (uint8_t)tile_src(me, tile, b, o);
}

size_t gsx_tiled_bytes(const qmat& m, int n_experts) {
    return tile_bytes(m.dtype) * (size_t)(m.rows / 32) * (m.cols / 256) * n_experts;
}

hipError_t launch_gsx_tile(const qmat& m, int n_experts, uint8_t* dst, hipStream_t s) {
    if (!tile_bytes(m.dtype) || m.cols % 256 || m.rows % 32 || n_experts < 1) return hipErrorInvalidValue;
    const int tiles = m.rows / 32;
    gsx_tile_kernel<<<n_experts * tiles * (m.cols / 256), 256, 0, s>>>(m, tiles, dst);
    return hipGetLastError();
}
