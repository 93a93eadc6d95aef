/**
 * kernels_tgemm.hip - The grouped experts of passes with many rows (a
 * prompt's chunk) on tiles of 32 pairs of one expert: float32 accuracy on the
 * f16 matrix cores (tile_half.h), in blocks of 256 weight rows x 64 pairs that
 * loop over the width, operands in an LDS ring.
 *
 * Reference counterparts: experts_in_rows_kernel model_cuda.cu:2071 and
 * experts_down_rows_kernel model_cuda.cu:2101; the CPU arithmetic checked
 * against is mixture_of_experts engine/src/model.c:745-761 and vitna_silu_mul
 * engine/src/ops.c:283, one row at a time.
 *
 * A block is eight waves, two a SIMD: wave (rg, tg) = (wave % 4, wave / 4)
 * takes the 32-row weight tiles 2 rg and 2 rg + 1 of the block's eight against
 * token tile tg of its two. The stage is a unit (64 columns, a quarter of a
 * superblock): the two token tiles' operand images (8 KB each, one contiguous
 * piece of skinny_image.h's layout), the eight weight tiles' bytes of the unit
 * (1 KB each, 2 KB for Q8_0) and, with the superblock's first unit, the block
 * headers and the activations' group sums. Everything goes to LDS by
 * global-to-LDS loads, three stages ahead in a ring of four slots (a slot a
 * unit of the superblock), waited for by count, one barrier a stage.
 *
 * What bounds it: the issue of a wave's instructions. A unit is 16 products a
 * wave (512 clocks of a SIMD's matrix core, 1024 for its two waves) beside
 * about 100 VALU instructions a wave (4 clocks each), so the order inside a
 * wave decides: with a unit's weights unpacked ahead of its products instead
 * of among them, the stage took 2200 clocks. A wave with one superblock of one
 * tile and its sums added through LDS (the kernels before) waited for its
 * first loads most of its life. One layer's experts of a 1024-row pass (top-8
 * of 128, 2048 x 768; kernel trace): gate/up in Q4_K 293 -> 167 us (163 with
 * group sums of 22 bits), down in Q6_K 243 -> 173 us; 333 rows in Q8_0 155 ->
 * 95 to 135 by how the rows fall on the experts, and 113 -> 80 us.
 *
 * A --precision fast pass takes the activations' hi alone: a wave's second
 * token tile takes the place of the first one's lo, so a block holds four
 * tiles of one expert and each weight is unpacked for two. Against the bf16
 * GEMM that widened each K-quant weight in float32 (kernels_prefill.hip): 246
 * -> 139 and 181 -> 138 us at the same sizes (135 with the first piece of the
 * group sums alone), the error against 64 bits of a two-layer pass 6e-3 -> 5e-4
 * (f16 keeps 11 bits, bf16 8).
 */

#include "vitna_kernels.h"
#include "skinny_exact.h"
#include "skinny_image.h"
#include "tile_half.h"

#include <algorithm>
#include <type_traits>

#define TG_THREADS 512
#define TG_R 8 /* 32-row weight tiles a block */
#define TG_T 2 /* token tiles a block */
#ifndef TG_VALU
#define TG_VALU 6 /* VALU instructions the scheduler puts after a product */
#endif

/* Where a block's operands lie in LDS, and what one wave loads a stage at least (the wave's share: one weight
   tile's bytes, an eighth of each token tile's). Unit n goes to slot n % 4; what a superblock has once lies after
   the slots (loaded with unit 0, Q6_K's high bits with units 0 and 2). */
template <int DT> struct tg_lds;
template <> struct tg_lds<VITNA_DTYPE_Q4_K> {
    static constexpr int TB = 4608, WU = 1024, HDR_LANES = 32;
    static constexpr int HDR = 4 * (TG_T * 8192 + TG_R * WU); /* [8][512] */
    static constexpr int SUMS = HDR + TG_R * 512;             /* [2 tiles][2 pieces][1024], FAST [4 tiles][1024] */
    static constexpr int BYTES = SUMS + 2 * TG_T * 1024;
    static constexpr int loads(int u) { return TG_T + 1 + (u == 0); }
};
template <> struct tg_lds<VITNA_DTYPE_Q6_K> {
    static constexpr int TB = 6720, WU = 1024, HDR_LANES = 36; /* scales and d */
    static constexpr int HDR = 4 * (TG_T * 8192 + TG_R * WU);  /* [8][576] */
    static constexpr int QH = HDR + TG_R * 576;                /* [2][8][1024] */
    static constexpr int SUMS = QH + 2 * TG_R * 1024;
    static constexpr int BYTES = SUMS;
    static constexpr int loads(int u) { return TG_T + 1 + (u % 2 == 0) + (u == 0); }
};
template <> struct tg_lds<VITNA_DTYPE_Q8_0> {
    static constexpr int TB = 8704, WU = 2048, HDR_LANES = 32;
    static constexpr int HDR = 4 * (TG_T * 8192 + TG_R * WU); /* [8][512] */
    static constexpr int SUMS = HDR + TG_R * 512;
    static constexpr int BYTES = SUMS;
    static constexpr int loads(int u) { return TG_T + 2 + (u == 0); }
};
#define TG_LDS_MAX (tg_lds<VITNA_DTYPE_Q8_0>::BYTES)
static_assert(TG_LDS_MAX >= tg_lds<VITNA_DTYPE_Q6_K>::BYTES && TG_LDS_MAX >= tg_lds<VITNA_DTYPE_Q4_K>::BYTES, "the largest layout");

/* A wave's sources, at the block's first superblock: its eighth of each token tile's images, its weight tile, its
   share of the group sums. */
struct tg_src {
    const uint8_t *img[TG_T], *wt, *sums;
};

/* A global-to-LDS load of 16 bytes a lane: lane l's bytes from base + off go to lds + 16 l. M0 is set here and
   nowhere else in these kernels. The compiler does not count these loads: tg_wait does. */
__device__ __forceinline__ void tg_dma(const uint8_t* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
}

/* This wave's loads but the N youngest have landed and its LDS reads are done; then every wave's. Not a fence: that
   would wait for the loads of later stages too. */
template <int N>
__device__ __forceinline__ void tg_wait() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

/* Part PART of unit U of superblock b into its slot: 0 and 1 the token tiles' images, 2 the weights and what the
   superblock has once. */
template <int DT, bool FAST, int U, int PART>
__device__ __forceinline__ void tg_part(const tg_src& s, int b, uint32_t lds, int wv, int lane) {
    typedef tg_lds<DT> L;
    const uint32_t off = 16 * lane, slot = lds + U * (TG_T * 8192 + TG_R * L::WU);
    if constexpr (PART < TG_T) {
        tg_dma(s.img[PART] + (size_t)b * (FAST ? 16384 : 32768) + U * (FAST ? 4096 : 8192), off, slot + PART * 8192 + wv * 1024);
    } else {
        const uint8_t* w = s.wt + (size_t)b * L::TB;
#pragma unroll
        for (int k = 0; k < L::WU / 1024; k++) tg_dma(w + U * L::WU + k * 1024, off, slot + TG_T * 8192 + wv * L::WU + k * 1024);
        if constexpr (DT == VITNA_DTYPE_Q6_K && U % 2 == 0)
            tg_dma(w + 4096 + (U / 2) * 1024, off, lds + L::QH + ((U / 2) * TG_R + wv) * 1024);
        if constexpr (U == 0) {
            if (lane < L::HDR_LANES) tg_dma(w + 4 * L::WU + (DT == VITNA_DTYPE_Q6_K ? 2048 : 0), off, lds + L::HDR + wv * L::HDR_LANES * 16);
            if (DT == VITNA_DTYPE_Q4_K && wv < 2 * TG_T) tg_dma(s.sums + (size_t)b * 2048, off, lds + L::SUMS + wv * 1024);
        }
    }
}
template <int DT, bool FAST, int U>
__device__ __forceinline__ void tg_issue(const tg_src& s, int b, uint32_t lds, int wv, int lane) {
    tg_part<DT, FAST, U, 0>(s, b, lds, wv, lane);
    tg_part<DT, FAST, U, 1>(s, b, lds, wv, lane);
    tg_part<DT, FAST, U, 2>(s, b, lds, wv, lane);
}

/* The lane's operands of unit U from its slot: half N of the activations of token tile tg (hi and lo of its two
   steps; FAST: hi of its two tiles), the weight tile at LDS index r. */
struct tg_a {
    u32x4 h[2], l[2];
};
template <int DT, int U, int N>
__device__ __forceinline__ void tg_read_a(const uint8_t* lds, int tg, int lane, tg_a& o) {
    const u32x4* p = reinterpret_cast<const u32x4*>(lds + U * (TG_T * 8192 + TG_R * tg_lds<DT>::WU) + tg * 8192) + lane;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        o.h[i] = p[(2 * N + i) * 128];
        o.l[i] = p[(2 * N + i) * 128 + 64];
    }
}
/* (part 0 before the unit's first half is unpacked, part 1 before its second: Q8_0's halves have bytes of their own) */
template <int DT, int U, int PART>
__device__ __forceinline__ void tg_read_w(const uint8_t* lds, int r, int lane, sx_w<DT>& o) {
    typedef tg_lds<DT> L;
    const uint8_t* p = lds + U * (TG_T * 8192 + TG_R * L::WU) + TG_T * 8192 + r * L::WU + lane * 16;
    const uint8_t* h = lds + L::HDR + r * L::HDR_LANES * 16;
    const int l32 = lane & 31;
    if constexpr (PART == 1 && DT != VITNA_DTYPE_Q8_0) {
    } else if constexpr (DT == VITNA_DTYPE_Q4_K) {
        o.q[U] = *reinterpret_cast<const u32x4*>(p);
        if constexpr (U == 0) o.h = *reinterpret_cast<const u32x4*>(h + l32 * 16);
    } else if constexpr (DT == VITNA_DTYPE_Q6_K) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(p);
        o.ql[U][0] = sx_u2{v.x, v.y};
        o.ql[U][1] = sx_u2{v.z, v.w};
        if constexpr (U % 2 == 0) {
            const u32x4 t = *reinterpret_cast<const u32x4*>(lds + L::QH + ((U / 2) * TG_R + r) * 1024 + lane * 16);
            o.qh[U / 2][0] = sx_u2{t.x, t.y};
            o.qh[U / 2][1] = sx_u2{t.z, t.w};
        }
        if constexpr (U == 0) {
            o.sc = *reinterpret_cast<const u32x4*>(h + l32 * 16);
            o.d = *reinterpret_cast<const uint16_t*>(h + 512 + l32 * 2);
        }
    } else {
        o.q[U][PART] = *reinterpret_cast<const u32x4*>(p + PART * 1024);
        if constexpr (U == 0 && PART == 0) o.d = *reinterpret_cast<const u32x4*>(h + l32 * 16);
    }
}

/* v is computed here: the compiler sinks what only a later step uses into that step, where it would stand before the
   products instead of among these. */
template <typename T>
__device__ __forceinline__ void tg_keep(T& v) { asm volatile("" : "+v"(v)); }

/* S superblocks of the wave's two weight tiles (LDS indexes r0, r0 + 1) against its token tile into acc. A wave
   that is not live (its token tile lies past the rows) loads its share and computes nothing.
   A wave issues in order, so a step (half a unit) keeps its three parts apart and interleaves them: the products
   of this step on operands made before, the unpacking of the next step's weights, and the scaling of the last
   finished products; and it reads from LDS what the next step multiplies and the one after it unpacks.
   FAST: activations in f16 alone (hi). A wave then takes two token tiles, the second's hi in the place of the first's
   lo, against weights that are unpacked once for both, and what Q6_K's rounding leaves is dropped. */
template <int DT, bool FAST>
__device__ __forceinline__ void tg_body(const tg_src& s, int S, const uint8_t* lds, uint32_t base, int wv, int lane, int r0, int tg, bool live,
                                        f32x16 (&acc)[FAST ? 2 : 1][2]) {
    typedef tg_lds<DT> L;
    constexpr bool Q4 = DT == VITNA_DTYPE_Q4_K, Q6 = DT == VITNA_DTYPE_Q6_K && !FAST, Q8 = DT == VITNA_DTYPE_Q8_0;
    constexpr int NT = FAST ? 2 : 1;
    auto top = [&](auto u, int b) {
        constexpr int U = decltype(u)::value;
        /* the next unit has landed, the loads of the one after it may still run; the unit loaded from here on goes to
           the slot of the unit before this one, which every wave has left */
        if (U < 2 || b + 1 < S) tg_wait<L::loads((U + 2) & 3)>();
        else tg_wait<0>();
    };
    auto load = [&](auto u, auto part, int b) {
        constexpr int U = decltype(u)::value, PART = decltype(part)::value;
        if constexpr (U == 0) tg_part<DT, FAST, 3, PART>(s, b, base, wv, lane);
        else if (b + 1 < S) tg_part<DT, FAST, (U + 3) & 3, PART>(s, b + 1, base, wv, lane);
    };
    std::integral_constant<int, 0> u0;
    std::integral_constant<int, 1> u1;
    std::integral_constant<int, 2> u2;
    std::integral_constant<int, 3> u3;
    tg_issue<DT, FAST, 0>(s, 0, base, wv, lane);
    tg_issue<DT, FAST, 1>(s, 0, base, wv, lane);
    tg_issue<DT, FAST, 2>(s, 0, base, wv, lane);
    tg_wait<L::loads(1) + L::loads(2)>();
    if (!live) {
        auto unit = [&](auto u, int b) {
            top(u, b);
            load(u, u0, b);
            load(u, u1, b);
            load(u, u2, b);
        };
        for (int b = 0; b < S; b++) {
            unit(u0, b);
            unit(u1, b);
            unit(u2, b);
            unit(u3, b);
        }
        return;
    }
    sx_w<DT> w[2], wn[2];
    tg_a x[2];       /* the activations of this step and the next, by the step's parity */
    th_b<DT> o[2];   /* the weights of this step */
    h8 mins[2];      /* Q4_K: a superblock's minimums */
    u32x4 sums[2];   /* and its sums: the token tile's two pieces, FAST its two tiles' */
    f32x16 P[NT][2] = {}, M[2]; /* the products, with their scale dP once they are finished, and Q4_K's of the minimums */
    float dP[2] = {0.0f, 0.0f}, dM[2] = {0.0f, 0.0f};
    auto start = [&](const sx_w<DT>(&ws)[2]) { /* a superblock's minimums and sums */
        if constexpr (Q4) {
#pragma unroll
            for (int t = 0; t < 2; t++) sums[t] = *(reinterpret_cast<const u32x4*>(lds + L::SUMS + (2 * tg + t) * 1024) + lane);
            mins[0] = th_mins(th_header(ws[0]), lane >> 5);
            mins[1] = th_mins(th_header(ws[1]), lane >> 5);
        }
    };
#pragma unroll
    for (int i = 0; i < 2; i++) {
        tg_read_w<DT, 0, 0>(lds, r0 + i, lane, w[i]);
        tg_read_w<DT, 0, 1>(lds, r0 + i, lane, w[i]);
    }
    tg_read_a<DT, 0, 0>(lds, tg, lane, x[0]);
    th_unpack<DT, 0, 0>(w[0], o[0]);
    th_unpack<DT, 0, 0>(w[1], o[1]);
    start(w);

    for (int b = 0; b < S; b++) {
        auto step = [&](auto u, auto half) {
            constexpr int U = decltype(u)::value, N = decltype(half)::value, V = (U + 1) & 3;
            constexpr bool first = U == 0 && N == 0, last = U == 3 && N == 1;
            /* the minimums' products in the first two steps: FAST a token tile's in each, its scale in the next; else the
               small piece's, then the large one's, and the scale in the third */
            constexpr int mt = Q4 && 2 * U + N < 2 ? 2 * U + N : -1;
            constexpr int ms = !Q4 ? -1 : FAST && (2 * U + N == 1 || 2 * U + N == 2) ? 2 * U + N - 1 : !FAST && 2 * U + N == 2 ? 0 : -1;
            __builtin_amdgcn_sched_barrier(0);
            sx_w<DT>(&ws)[2] = U == 3 ? wn : w; /* the next unit's */
            if constexpr (N == 0) {
                tg_read_a<DT, U, 1>(lds, tg, lane, x[1]);
            } else {
                tg_read_a<DT, V, 0>(lds, tg, lane, x[0]);
            }
            tg_read_w<DT, V, N>(lds, r0, lane, ws[0]);
            tg_read_w<DT, V, N>(lds, r0 + 1, lane, ws[1]);
            const tg_a xs = x[N];
            /* the finished products' scale */
            if constexpr (Q8 || first) {
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        sx_scale(acc[t][i], dP[i], P[t][i]);
                        tg_keep(acc[t][i]);
                        P[t][i] = f32x16{};
                    }
            }
            if constexpr (ms >= 0) {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    sx_scale(acc[ms][i], dM[i], M[i]);
                    tg_keep(acc[ms][i]);
                }
            }
            if constexpr (mt >= 0) {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    M[i] = TH_MMA(sums[FAST ? mt : 1 - mt], mins[i], !FAST && mt == 1 ? M[i] : f32x16{});
                    if (mt == 0) dM[i] = th_dmin(w[i]);
                }
            }
            /* this step's products */
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int i = 0; i < 2; i++) P[0][i] = TH_MMA(xs.h[k], o[i].o[k], P[0][i]);
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int i = 0; i < 2; i++) P[NT - 1][i] = TH_MMA(xs.l[k], o[i].o[k], P[NT - 1][i]);
            if constexpr (Q6) {
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int i = 0; i < 2; i++) P[0][i] = TH_MMA(xs.h[k], o[i].r[k], P[0][i]);
            }
            /* the next step's weights (past the last superblock, whatever the slots hold: not used) */
            th_b<DT> on[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                if constexpr (N == 0) th_unpack<DT, U, 1>(w[i], on[i]);
                else th_unpack<DT, V, 0>(ws[i], on[i]);
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
                tg_keep(on[i].o[0]);
                tg_keep(on[i].o[1]);
                if constexpr (Q6) {
                    tg_keep(on[i].r[0]);
                    tg_keep(on[i].r[1]);
                }
                if constexpr (Q8 || last) dP[i] = th_d<DT, U, N>(w[i]);
            }
            if constexpr (last) start(wn);
#pragma unroll
            for (int k = 0; k < (Q6 ? 12 : 8); k++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, TG_VALU, 0);
            }
            o[0] = on[0];
            o[1] = on[1];
            __builtin_amdgcn_sched_barrier(0);
        };
        /* the loads go out a part at a time: all eight waves' loads of a unit at once (18 clocks of the compute unit's
           memory pipeline each) would hold every wave's products up behind them */
        auto unit = [&](auto u) {
            top(u, b);
            load(u, u0, b);
            step(u, u0);
            load(u, u1, b);
            step(u, u1);
            load(u, u2, b);
        };
        unit(u0);
        unit(u1);
        unit(u2);
        unit(u3);
        w[0] = wn[0];
        w[1] = wn[1];
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < 2; i++) sx_scale(acc[t][i], dP[i], P[t][i]);
}

/* What the kernels read: the rows' operand images (img, tile_half.h's values in skinny_image.h's layout, order B for
   Q6_K; FAST: the hi pieces alone) and, for Q4_K, group sums ([tile][superblock][2][64][8] f16, th_sum). */
struct tg_images {
    const uint8_t *img, *sums;
};

/* One wave's sources: token tiles tt (two, FAST four) of S superblocks each, its weight tile. */
template <int DT, bool FAST>
__device__ __forceinline__ tg_src tg_sources(const tg_images& a, const int (&tt)[2 * TG_T], const uint8_t* tile, int S, int wv) {
    tg_src s;
#pragma unroll
    for (int j = 0; j < TG_T; j++)
        s.img[j] = FAST ? a.img + (size_t)tt[2 * j + (wv & 1)] * S * 16384 + (wv >> 1) * 1024 : a.img + (size_t)tt[j] * S * 32768 + wv * 1024;
    s.wt = tile;
    s.sums = FAST ? a.sums + (size_t)tt[wv & 3] * S * 2048 : a.sums + (size_t)tt[(wv >> 1) & 1] * S * 2048 + (wv & 1) * 1024;
    return s;
}

__device__ __forceinline__ uint32_t tg_lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)p;
}

/* Work item w of n on the block's XCD: blocks go to the eight XCDs in turn, and each takes a contiguous run of the
   items, so that neighbours (the same token tiles, or the same expert) meet in one L2. -1 past the last. */
__device__ __forceinline__ int tg_item(int n) {
    const int per = (n + 7) >> 3, slot = blockIdx.x >> 3, w = (blockIdx.x & 7) * per + slot;
    return slot < per && w < n ? w : -1;
}

/* ---- the grouped experts of crowded passes --------------------------------- */

/*
 * A pass whose experts hold many pairs each (a prompt's chunk: 1024 rows of top-8 over 128 experts, 64 pairs an
 * expert) runs its experts on tiles of 32 pairs of one expert, instead of the four-pair tiles of kernels_gmma.hip,
 * with the f16 arithmetic of tile_half.h. The pairs of each expert (launch_group's lists) are cut into tiles; tile t
 * (of one expert, te[t]) is the virtual token tile t of the operand images, which a gather writes from the
 * normalized rows. A token block is up to two tiles of one expert (a fast pass: four). Gate and up run in one block over the same
 * activations; the block writes the SwiGLU output in fp32, whose images gsx_act_image_kernel writes for down; down
 * multiplies by the pair's weight into ypart, as kernels_gmma.hip does. The weights come from a copy tiled as the
 * dense matrices' are, experts back to back (expert e's 32-row tile x is tile e I / 32 + x).
 */

bool gsx_fits(const qmat& gate, const qmat& up, const qmat& down) {
    auto dt = [](int d) { return d == VITNA_DTYPE_Q8_0 || d == VITNA_DTYPE_Q4_K || d == VITNA_DTYPE_Q6_K; };
    const int H = gate.cols, I = gate.rows;
    /* whole superblocks of the width and whole blocks of rows; experts wider than 2048 keep the four-pair kernels, as
       none has been timed here */
    return dt(gate.dtype) && up.dtype == gate.dtype && dt(down.dtype) && up.rows == I && up.cols == H && down.rows == H &&
           down.cols == I && H % 256 == 0 && I % 256 == 0 && H <= 2048 && I <= 2048;
}

int gsx_max_tiles(int n, int K, int E) { return (n * K + 31) / 32 + E; }
int gsx_max_blocks(int n, int K, int E) { return (n * K + 63) / 64 + E; }
int gsx_least_blocks(const qmat& gate, int E) { return E * std::min(gate.rows / 128, gate.cols / 256); }

__device__ __forceinline__ float gsx_largest(float m, const float4& v) {
    return fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
}

/* Tile offsets of the experts' pair lists (toff[E + 1]), the expert of each tile (te[max_tiles], -1 past the
   last) and the first tile of each token block of up to `block` tiles (tb, their number at n_tb): block 0, the first
   wave scanning the tile counts, the second the block counts, 64 experts at a time. The blocks after it take four
   rows each of the n (H wide) at x and leave the rows' powers of two in scale: beside the plan, which one block
   takes longer over. */
__global__ __launch_bounds__(256) void gsx_plan_kernel(const int* __restrict__ count, int E, int* __restrict__ toff,
                                                       int* __restrict__ te, int max_tiles, int block, int* __restrict__ tb,
                                                       int* __restrict__ n_tb, const float* __restrict__ x, int n, int H,
                                                       float* __restrict__ scale) {
    __shared__ int off[2][ROUTE_E_MAX + 1];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    if (blockIdx.x) {
        const int row = 4 * (blockIdx.x - 1) + wv;
        if (row >= n) return;
        const float4* src = reinterpret_cast<const float4*>(x + (size_t)row * H);
        float m = 0.0f;
        for (int c = lane; c < H / 4; c += 64) m = gsx_largest(m, src[c]);
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, WAVE));
        if (lane == 0) scale[row] = th_scale(m);
        return;
    }
    if (wv < 2) {
        const int per = wv ? 32 * block : 32;
        int run = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane;
            const int c = e < E ? (count[e] + per - 1) / per : 0;
            int v = c; /* inclusive scan across the wave */
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(v, d, WAVE);
                if (lane >= d) v += o;
            }
            if (e < E) off[wv][e] = run + v - c;
            run += __shfl(v, 63, WAVE);
        }
        if (lane == 0) off[wv][E] = run;
    }
    __syncthreads();
    for (int e = tid; e <= E; e += blockDim.x) toff[e] = off[0][e];
    for (int e = tid; e < E; e += blockDim.x) {
        for (int t = off[0][e]; t < off[0][e + 1]; t++) te[t] = e;
        for (int b = off[1][e]; b < off[1][e + 1]; b++) tb[b] = off[0][e] + block * (b - off[1][e]);
    }
    for (int t = off[0][E] + tid; t < max_tiles; t += blockDim.x) te[t] = -1;
    if (tid == 0) *n_tb = off[1][E];
}

/* The tiles of token block item / X: t = tb[item / X] and the next ones of its expert, up to two (FAST four), the last
   one again past them. Returns how many there are. */
template <bool FAST>
__device__ __forceinline__ int gsx_tiles(const int* __restrict__ te, int t, int T, int (&tt)[2 * TG_T]) {
    int n = 1;
#pragma unroll
    for (int j = 1; j < (FAST ? 4 : 2); j++) n += n == j && t + j < T && te[t + j] == te[t];
#pragma unroll
    for (int j = 0; j < 2 * TG_T; j++) tt[j] = t + min(j, n - 1);
    return n;
}

/* Block of (token block, row block x). act[32 t + token][32 x + row] = silu(gate . x) * (up . x): a wave's two weight
   tiles are the gate and the up rows of the same 32 columns, so both halves of an output are in one lane. */
template <int DT, bool FAST>
__global__ __launch_bounds__(TG_THREADS) void gsx_tile_in_kernel(qmat gate, qmat up, tg_images im, const int* __restrict__ te,
                                                                 const int* __restrict__ tb, const int* __restrict__ n_tb, int T,
                                                                 const float* __restrict__ inv, float* __restrict__ act) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[tg_lds<DT>::BYTES];
    constexpr int NT = FAST ? 2 : 1;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = gate.cols, I = gate.rows, X = I / 128, S0 = H / 256;
    const int item = tg_item(*n_tb * X);
    if (item < 0) return;
    const int t = tb[item / X], x = item - item / X * X, e = te[t];
    int tt[2 * TG_T];
    const int n = gsx_tiles<FAST>(te, t, T, tt);
    const int rg = wv & 3, tg = wv >> 2;
    const qmat& m = wv & 1 ? up : gate;
    const uint8_t* tile = m.tiled + ((size_t)e * (I / 32) + 4 * x + (wv >> 1)) * S0 * tg_lds<DT>::TB;
    f32x16 acc[NT][2] = {};
    tg_body<DT, FAST>(tg_sources<DT, FAST>(im, tt, tile, S0, wv), S0, lds, __builtin_amdgcn_readfirstlane(tg_lds_addr(lds)), wv, lane, 2 * rg,
                      tg, NT * tg < n, acc);
    const int l32 = lane & 31, kq = lane >> 5;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        if (NT * tg + j >= n) break;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int tok = 8 * (r >> 2) + 4 * kq + (r & 3);
            const size_t row = 32 * (t + NT * tg + j) + tok;
            const float f = inv[row], g = acc[j][0][r] * f;
            act[row * I + 32 * (4 * x + rg) + l32] = (g / (1.0f + expf(-g))) * (acc[j][1][r] * f);
        }
    }
}

/* ypart[(row K + slot) H + n] = w_slot (down_e[n] . act[pair]) for the pairs of the block's token tiles. */
template <int DT, bool FAST>
__global__ __launch_bounds__(TG_THREADS) void gsx_tile_down_kernel(qmat down, tg_images im, const int* __restrict__ te,
                                                                   const int* __restrict__ tb, const int* __restrict__ n_tb, int T,
                                                                   const int* __restrict__ toff, const int* __restrict__ count,
                                                                   const int* __restrict__ pairs, int cap,
                                                                   const route_out* __restrict__ rt, int K, const float* __restrict__ inv,
                                                                   float* __restrict__ ypart) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[tg_lds<DT>::BYTES];
    constexpr int NT = FAST ? 2 : 1;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = down.rows, X = H / 256, S0 = down.cols / 256;
    const int item = tg_item(*n_tb * X);
    if (item < 0) return;
    const int t = tb[item / X], x = item - item / X * X, e = te[t];
    int tt[2 * TG_T];
    const int n = gsx_tiles<FAST>(te, t, T, tt);
    const int rg = wv & 3, tg = wv >> 2;
    const uint8_t* tile = down.tiled + ((size_t)e * (H / 32) + TG_R * x + wv) * S0 * tg_lds<DT>::TB;
    f32x16 acc[NT][2] = {};
    tg_body<DT, FAST>(tg_sources<DT, FAST>(im, tt, tile, S0, wv), S0, lds, __builtin_amdgcn_readfirstlane(tg_lds_addr(lds)), wv, lane, 2 * rg,
                      tg, NT * tg < n, acc);
    const int l32 = lane & 31, kq = lane >> 5, c = count[e];
#pragma unroll
    for (int i = 0; i < NT; i++) {
        if (NT * tg + i >= n) break;
        const int tile_t = t + NT * tg + i, j0 = 32 * (tile_t - toff[e]);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int j = j0 + 8 * (r >> 2) + 4 * kq + (r & 3);
            if (j < c) {
                const int p = pairs[(size_t)e * cap + j], row = p / ROUTE_K_MAX, slot = p % ROUTE_K_MAX;
                const float wt = rt[row].weights[slot], f = inv[32 * tile_t + j - j0];
                float* y = ypart + ((size_t)row * K + slot) * H + 32 * (TG_R * x + 2 * rg) + l32;
                y[0] = wt * (acc[i][0][r] * f);
                y[32] = wt * (acc[i][1][r] * f);
            }
        }
    }
}

/* Columns 8 c8 .. of row `row` into the image: both pieces at img_put's place, or with fast the hi piece alone, at the
   same place of an image of half the size. */
__device__ __forceinline__ void gsx_put(u32x4* img, bool order_b, bool fast, int row, int K, int c8, const u32x4& vh, const u32x4& vl) {
    if (!fast) {
        img_put(order_b ? nullptr : img, order_b ? img : nullptr, row, K, c8, vh, vl);
        return;
    }
    const int c = 8 * (c8 & 31), r = c & (order_b ? 127 : 63);
    const int U = order_b ? 2 * (c >> 7) + ((r >> 5) & 1) : c >> 6, kq = order_b ? (r >> 3) & 1 : (r >> 4) & 1;
    const int i = order_b ? ((r >> 4) & 1) + 2 * (r >> 6) : ((r >> 5) << 1) | ((r >> 3) & 1);
    img[((size_t)(row >> 5) * (K / 256) + (c8 >> 5)) * 1024 + (U * 4 + i) * 64 + (row & 31) + 32 * kq] = vh;
}

/* The images (one column order) and, for Q4_K weights (sums not null), group sums of the virtual token tiles: block (b, t) takes
   superblock b of tile t, whose token l is pair 32 (t - toff[e]) + l of expert te[t] (past its count: the last pair
   again), row pair / ROUTE_K_MAX of x, times that row's scale, whose inverse goes to inv. */
__global__ __launch_bounds__(256) void gsx_image_kernel(const float* __restrict__ x, int K, const float* __restrict__ scale,
                                                        const int* __restrict__ pairs, const int* __restrict__ count, int cap,
                                                        const int* __restrict__ toff, const int* __restrict__ te,
                                                        u32x4* __restrict__ img, bool order_b, bool fast, _Float16* __restrict__ sums,
                                                        float* __restrict__ inv) {
    const int b = blockIdx.x, t = blockIdx.y;
    const int e = te[t];
    if (e < 0) return;
    const int j0 = 32 * (t - toff[e]), c = count[e];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int item = threadIdx.x + 256 * j, l = item >> 5, c8 = 32 * b + (item & 31);
        const size_t src_row = (size_t)(pairs[(size_t)e * cap + min(j0 + l, c - 1)] / ROUTE_K_MAX);
        const float4* src = reinterpret_cast<const float4*>(x + src_row * K + 8 * c8);
        const float4 v0 = src[0], v1 = src[1];
        const float ev[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        const float f = scale[src_row];
        if (c8 == 0) inv[32 * t + l] = th_inverse(f);
        u32x4 vh, vl;
        float sum;
        th_split8(ev, f, fast, vh, vl, sum);
        gsx_put(img, order_b, fast, 32 * t + l, K, c8, vh, vl);
        if (!sums) continue;
        const float t16 = sum + __shfl_xor(sum, 1, WAVE), t32 = t16 + __shfl_xor(t16, 2, WAVE);
        if (!(c8 & 3)) th_sum(sums + ((size_t)t * (K / 256) + b) * 1024, l, (c8 & 31) >> 2, t32);
    }
}

/* The same of the SwiGLU output's rows (row 32 t + l of x for token l of tile t), each scaled by its own power of
   two, whose inverse goes to inv: block t, eight threads a row, the row read twice. */
__global__ __launch_bounds__(256) void gsx_act_image_kernel(const float* __restrict__ x, int K, const int* __restrict__ te, u32x4* __restrict__ img,
                                                            bool order_b, bool fast, _Float16* __restrict__ sums, float* __restrict__ inv) {
    const int t = blockIdx.x;
    if (te[t] < 0) return;
    const int l = threadIdx.x >> 3, j = threadIdx.x & 7, row = 32 * t + l;
    const float4* src = reinterpret_cast<const float4*>(x + (size_t)row * K);
    float m = 0.0f;
    for (int c = j; c < K / 8; c += 8) {
        m = gsx_largest(gsx_largest(m, src[2 * c]), src[2 * c + 1]);
    }
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, WAVE));
    const float f = th_scale(m);
    if (j == 0) inv[row] = th_inverse(f);
    for (int c = j; c < K / 8; c += 8) {
        const float4 v0 = src[2 * c], v1 = src[2 * c + 1];
        const float ev[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        u32x4 vh, vl;
        float sum;
        th_split8(ev, f, fast, vh, vl, sum);
        gsx_put(img, order_b, fast, row, K, c, vh, vl);
        if (!sums) continue;
        const float t16 = sum + __shfl_xor(sum, 1, WAVE), t32 = t16 + __shfl_xor(t16, 2, WAVE);
        if (!(c & 3)) th_sum(sums + ((size_t)t * (K / 256) + (c >> 5)) * 1024, l, (c & 31) >> 2, t32);
    }
}

template <bool FAST>
static hipError_t launch_gsx_tiles(const gsx_args& a, bool in, hipStream_t s) {
    const qmat& m = in ? a.gate : a.down;
    const int X = in ? a.gate.rows / 128 : a.down.rows / 256, T = gsx_max_tiles(a.n, a.K, a.E);
    const int blocks = (gsx_max_blocks(a.n, a.K, a.E) * X + 7) / 8 * 8;
    const tg_images k = {reinterpret_cast<const uint8_t*>(in ? a.img_in : a.img_act), reinterpret_cast<const uint8_t*>(a.sums)};
    const int *tb = a.tb, *n_tb = a.tb + a.max_tiles;
    auto go = [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if (in) gsx_tile_in_kernel<DT, FAST><<<blocks, TG_THREADS, 0, s>>>(a.gate, a.up, k, a.te, tb, n_tb, T, a.inv, a.act);
        else gsx_tile_down_kernel<DT, FAST><<<blocks, TG_THREADS, 0, s>>>(a.down, k, a.te, tb, n_tb, T, a.toff, a.count, a.pairs, a.cap, a.rt, a.K, a.inv, a.ypart);
    };
    switch (m.dtype) {
    case VITNA_DTYPE_Q4_K: go(std::integral_constant<int, VITNA_DTYPE_Q4_K>()); break;
    case VITNA_DTYPE_Q6_K: go(std::integral_constant<int, VITNA_DTYPE_Q6_K>()); break;
    default:
        if constexpr (FAST) return hipErrorInvalidValue;
        else go(std::integral_constant<int, VITNA_DTYPE_Q8_0>());
        break;
    }
    return hipGetLastError();
}

hipError_t launch_gsx(const gsx_args& a, hipStream_t s) {
    if (!gsx_fits(a.gate, a.up, a.down) || !a.gate.tiled || !a.up.tiled || !a.down.tiled || a.K < 1 || a.K > ROUTE_K_MAX ||
        a.E < 1 || a.E > ROUTE_E_MAX || a.n < 1 || a.cap < a.n || a.max_tiles < gsx_max_tiles(a.n, a.K, a.E))
        return hipErrorInvalidValue;
    const int H = a.gate.cols, I = a.gate.rows, T = gsx_max_tiles(a.n, a.K, a.E);
    gsx_plan_kernel<<<1 + (a.n + 3) / 4, 256, 0, s>>>(a.count, a.E, a.toff, a.te, T, a.fast ? 4 : 2, a.tb, a.tb + a.max_tiles, a.xn, a.n, H,
                                                      a.scale);
    u32x4* ii = reinterpret_cast<u32x4*>(a.img_in);
    u32x4* ia = reinterpret_cast<u32x4*>(a.img_act);
    _Float16* sums = reinterpret_cast<_Float16*>(a.sums);
    gsx_image_kernel<<<dim3(H / 256, T), 256, 0, s>>>(a.xn, H, a.scale, a.pairs, a.count, a.cap, a.toff, a.te, ii,
                                                      a.gate.dtype == VITNA_DTYPE_Q6_K, a.fast,
                                                      a.gate.dtype == VITNA_DTYPE_Q4_K ? sums : nullptr, a.inv);
    hipError_t err = a.fast ? launch_gsx_tiles<true>(a, true, s) : launch_gsx_tiles<false>(a, true, s);
    if (err != hipSuccess) return err;
    gsx_act_image_kernel<<<T, 256, 0, s>>>(a.act, I, a.te, ia, a.down.dtype == VITNA_DTYPE_Q6_K, a.fast,
                                       a.down.dtype == VITNA_DTYPE_Q4_K ? sums : nullptr, a.inv);
    return a.fast ? launch_gsx_tiles<true>(a, false, s) : launch_gsx_tiles<false>(a, false, s);
}
