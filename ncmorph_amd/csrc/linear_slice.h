// The K-sliced small-tile product of linear_slice.hip and vq_tok.hip: one
// workgroup computes 16 RB x 16 CB outputs of A B^T, its NW wavefronts
// splitting K instead of the tile: wavefront w multiplies the whole tile over
// K tiles w, w + NW, ... (64 bf16 or 32 fp32 elements each), and the NW
// partial sums are added in wavefront order through LDS.
//
// A wavefront's operand rows go straight to its own LDS region (buffer_load
// ... lds, 8 rows x 128 bytes per instruction: whole cache lines), NST stages
// deep. No other wavefront reads that region, so the main loop has no
// barrier: each wavefront waits for its oldest stage only (vmcnt), reads the
// stage's fragments into registers and refills the stage before its MFMAs.
//
// Fragments: v_mfma_f32_16x16x32_bf16 (A = x rows, B = weight rows; lane l
// supplies 16-byte chunk 4 i + l / 16 of row l % 16 for k-step i), or for
// fp32 four v_mfma_f32_16x16x4_f32 per k-step, MFMA j taking element j of
// each lane's chunk. D: lane l, element j holds row 4 (l / 16) + j, column
// l % 16. LDS chunk c of row r sits at chunk c ^ ((r / 2) % 8), which gives
// the 16 rows of a ds_read_b128 phase distinct bank groups.
#pragma once

#include "gemm_core.h"

namespace ncm {

// RB x CB blocks of 16 x 16 outputs per workgroup, NW wavefronts, NST LDS
// stages each.
template <bool F32, int RB, int CB, int NW, int NST>
struct SliceShape {
    static constexpr int ROWS = 16 * (RB + CB);
    static constexpr int STAGE = ROWS * 128;
    static constexpr int ND = ROWS / 8;  // load instructions per stage
    static constexpr int RED = NW * RB * CB * 1024;
    static constexpr int LDS = NW * NST * STAGE > RED ? NW * NST * STAGE : RED;
    static constexpr int EPC = F32 ? 4 : 8;  // elements per 16-byte chunk
    static_assert(LDS <= 160 * 1024, "LDS budget of a gfx950 CU");
    static_assert(NST >= 1 && (NST - 1) * ND <= 63, "vmcnt range");
};

// The tile's partial sums into LDS: block b of wavefront v at ((v NB + b) 64 +
// lane) 16 bytes; the barrier that ends it makes them visible. rsx: the 16 RB
// rows of A, xstride bytes apart; rsw: 16 CB rows of B, wstride bytes apart,
// block cb at row cb BSTEP (TWO_W: the second half of the blocks from rsw2).
// Rows and K-chunks past the operands load as zero. K in elements, a multiple
// of 16 bytes.
template <bool F32, int RB, int CB, int NW, int NST, int BSTEP, bool TWO_W>
__device__ __forceinline__ void slice_partial_sums(char* lds, __amdgpu_buffer_rsrc_t rsx,
                                                   uint32_t xstride, __amdgpu_buffer_rsrc_t rsw,
                                                   __amdgpu_buffer_rsrc_t rsw2, uint32_t wstride,
                                                   int64_t K) {
    using S = SliceShape<F32, RB, CB, NW, NST>;
    constexpr int ESZ = F32 ? 4 : 2;
    constexpr int NB = RB * CB;
    constexpr int HB = CB > 1 ? CB / 2 : 1;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, grp = lane >> 4;

    // Load instruction p fills LDS rows 8 p .. 8 p + 7 (x rows, then weight
    // rows), lane l row l / 8, chunk slot l % 8; the swizzle term depends on
    // the parity of p only.
    const int drow = lane >> 3;
    const int ch0 = (lane & 7) ^ (drow >> 1), ch1 = ch0 ^ 4;
    const uint32_t x0 = drow * xstride + ch0 * 16, x1 = drow * xstride + ch1 * 16;
    const uint32_t w0 = drow * wstride + ch0 * 16, w1 = drow * wstride + ch1 * 16;
    char* region = lds + wave * (NST * S::STAGE);
    auto dma = [&](char* stage, int64_t k0) {
        // Chunks at or past K, and tiles past the last one, load as zero.
        const uint32_t kb = (uint32_t)(k0 * ESZ);
        const bool in0 = k0 + ch0 * S::EPC < K, in1 = k0 + ch1 * S::EPC < K;
        const uint32_t vx0 = in0 ? x0 + kb : kOobOffset, vx1 = in1 ? x1 + kb : kOobOffset;
        const uint32_t vw0 = in0 ? w0 + kb : kOobOffset, vw1 = in1 ? w1 + kb : kOobOffset;
#pragma unroll
        for (int p = 0; p < S::ND; ++p) {
            const bool is_x = p < 2 * RB;
            const int q = is_x ? p : p - 2 * RB;
            const int cb = TWO_W ? (q >> 1) % HB : q >> 1;
            const int row = is_x ? 8 * q : cb * BSTEP + 8 * (q & 1);
            const uint32_t off = is_x ? (p & 1 ? vx1 : vx0) + (uint32_t)row * xstride
                                      : (p & 1 ? vw1 : vw0) + (uint32_t)row * wstride;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                is_x ? rsx : (TWO_W && q >= 2 * HB ? rsw2 : rsw),
                (__attribute__((address_space(3))) void*)(stage + p * 1024), 16, off, 0, 0, 0);
        }
    };

    f32x4_t acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    constexpr int BK = 8 * S::EPC;
    const int tiles_k = (int)((K + BK - 1) / BK);
    // This wavefront's tiles: those past the last would only multiply zeros, in
    // the way of the wavefront that shares their SIMD (fp32, 200 x 3072 x 576, 18
    // tiles: 16.2 us with three for every wavefront, 13.6 so; 384 x 4096 x 384, 12
    // tiles: 21.6 -> 18.0).
    const int iters = (tiles_k - wave + NW - 1) / NW;
#pragma unroll
    for (int s = 0; s < NST; ++s) dma(region + s * S::STAGE, (int64_t)(wave + NW * s) * BK);
    const uint32_t frag = (uint32_t)(r16 * 128);
    const uint32_t c0 = (uint32_t)((grp ^ (r16 >> 1)) * 16), c1 = c0 ^ 64;
    int st = 0;
    for (int i = 0; i < iters; ++i) {
        char* base = region + st * S::STAGE;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((NST - 1) * S::ND));
        asm volatile("" ::: "memory");
        u32x4_t af[2][RB], bf[2][CB];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const uint32_t c = ks ? c1 : c0;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                af[ks][rb] = *(const u32x4_t*)(base + frag + rb * 2048 + c);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
                bf[ks][cb] = *(const u32x4_t*)(base + frag + (RB + cb) * 2048 + c);
        }
        // The stage is free once its fragments are in registers.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        dma(base, (int64_t)(wave + NW * (i + NST)) * BK);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    if constexpr (F32) {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                __uint_as_float(af[ks][rb][j]), __uint_as_float(bf[ks][cb][j]),
                                acc[rb][cb], 0, 0, 0);
                    } else {
                        acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, af[ks][rb]),
                            __builtin_bit_cast(bf16x8_t, bf[ks][cb]), acc[rb][cb], 0, 0, 0);
                    }
                }
        st = st + 1 == NST ? 0 : st + 1;
    }

    // Partial sums over the operand stages, once no load can still write
    // there; block b of wavefront v at ((v NB + b) 64 + lane) 16 bytes.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    f32x4_t* red = (f32x4_t*)lds;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) red[(wave * NB + rb * CB + cb) * 64 + lane] = acc[rb][cb];
    __syncthreads();
}

// Block b of the tile: the wavefronts' partial sums added in their order.
template <int NW, int NB>
__device__ __forceinline__ f32x4_t slice_sum(const char* lds, int b) {
    const f32x4_t* red = (const f32x4_t*)lds;
    const int lane = threadIdx.x & 63;
    f32x4_t s = red[b * 64 + lane];
#pragma unroll
    for (int v = 1; v < NW; ++v) {
        const f32x4_t p = red[(v * NB + b) * 64 + lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = s[j] + p[j];
    }
    return s;
}

// Tiles RB x CB with their LDS stages. NW is 8 for all of them: the sums of
// an output do not depend on the tile. One stage (refilled while its
// fragments are multiplied) leaves LDS for a second workgroup on the CU up to
// 5 blocks of rows and measured as fast as two or three from 1 x 2 up.
constexpr int kSliceWaves = 8;
struct SliceTile {
    int rb, cb;
};
constexpr SliceTile kSliceTiles[] = {{1, 1}, {2, 1}, {1, 2}, {2, 2}, {3, 2}, {1, 4},
                           {4, 2}, {2, 4}, {3, 4}, {4, 4}, {5, 4}};
constexpr int kSliceTileCount = sizeof(kSliceTiles) / sizeof(kSliceTiles[0]);

// fp32: the matrix core is the bound (1/16 of the bf16 rate), so a tile is
// priced in time: rounds of the CUs times the workgroup's MFMAs (0.22 us per
// block of 16 x 16 outputs and iteration of its eight wavefronts, two on each
// SIMD) plus what starting, summing and storing it takes, an eighth more past
// one round (the operands then compete for the L2), plus the launch. Fitted to
// M = 1 .. 13000, K = 384 .. 4864, within 15% where the weight stream is not the
// bound (200 rows, 576 x 576: 5.1 us; 300 rows, 4864 x 896: 32 us; 4222 rows, 384 x
// 1152: 49 us).
inline double slice_f32_tile_us(const SliceTile& s, int64_t M, int64_t N, int64_t K) {
    const int64_t tiles =
        ((M + 16 * s.rb - 1) / (16 * s.rb)) * ((N + 16 * s.cb - 1) / (16 * s.cb));
    const double iters = 0.5 * (double)(((K + 31) / 32 + 3) / 4);
    const int blocks = s.rb * s.cb;
    const double round = 0.22 * blocks * iters + 1.3 + 0.3 * blocks;
    const int64_t rounds = (tiles + 255) / 256;
    return 3.0 + (rounds > 1 ? 1.12 * (double)rounds : 1.0) * round;
}

// The other fp32 tiles' time (linear.hip, vq_tok.hip): 128 x 128 tiles by their
// rounds of the CUs (130 us for anything up to 256 tiles at K = 2048; from four
// rounds on they overlap and take a tenth less), 64 x 64 tiles by those of the
// fullest CU (within 10% over M = 64 .. 33000 at K = 384 .. 1536).
inline double f32_large_us(int64_t M, int64_t N, int64_t K) {
    const int64_t rounds = (((M + 127) / 128) * ((N + 127) / 128) + 255) / 256;
    const double us = (double)rounds * (1.95 * ((K + 31) / 32) + 6.0);
    return 3.0 + (rounds >= 4 ? 0.9 * us : us);
}

inline double f32_small_us(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
    return 6.5 + (double)((tiles + 255) / 256) * (0.5 * ((K + 31) / 32) + 0.6);
}

inline double slice_best_tile_f32(int64_t M, int64_t N, int64_t K, bool paired, int* tile) {
    double best = 1e300;
    for (int t = 0; t < kSliceTileCount; ++t) {
        if (paired && kSliceTiles[t].cb < 2) continue;
        const double us = slice_f32_tile_us(kSliceTiles[t], M, N, K);
        if (us < best) {
            best = us;
            *tile = t;
        }
    }
    return best;
}

}  // namespace ncm
