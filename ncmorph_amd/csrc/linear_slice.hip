// Linears with few rows: y = x * W^T where the 128- and 256-row tiles of
// linear.hip leave most of the chip idle or multiply mostly padding (a
// prompt of 77 tokens through a 2048-wide projection is 16 tiles for 256
// CUs). Small output tiles fill the CUs, and the wavefronts of a workgroup
// split K instead of the tile (slice_partial_sums in linear_slice.h): no
// second pass over memory, no workspace, no atomic, no barrier in the main
// loop.
//
// What bounds it: the weight stream from HBM for the smallest batches, the
// operand traffic L2 -> LDS (every column tile reads all of x, every row tile
// all of W) for the larger ones, and the matrix core for fp32.
//
// Every output is a function of its row of x and its weight row(s) alone,
// whatever the tile: the same sums for every epilogue, so the fused results
// equal the unfused kernels' bit for bit.
#include "linear.h"
#include "linear_slice.h"

namespace ncm {

namespace {

constexpr int kPlain = 0, kSwiGLU = 1, kRope = 2;

struct SliceArgs {
    const void* x;
    const void* w;
    const uint16_t* bias;  // bf16, nullable
    const float* residual;  // fp32 [M, N], nullable; may be y in the fp32 modes
    void* y;
    int64_t M, K, N;  // N: weight rows
    int out_mode, tiles_m;
    // fp32 only: the bias; SwiGLU's up rows and bias (w and bias32: gate);
    // columns n1 .. n2 - 1 go to y1 and n2 .. N - 1 to y2 (rows of their own
    // width, n1 = 0: all to y).
    const float* bias32;
    const float* w2;
    const float* bias2;
    float* y1;
    float* y2;
    int64_t n1, n2;
    // RoPE: tables [seq_len, 64], columns [0, rot_cols) rotated.
    const float* cosine;
    const float* sine;
    int64_t seq_len, rot_cols;
};

template <bool F32, int RB, int CB, int NW, int NST, int EPI>
__global__ __launch_bounds__(64 * NW) void linear_slice_kernel(SliceArgs a) {
    constexpr int ESZ = F32 ? 4 : 2;
    constexpr int NB = RB * CB;
    static_assert(EPI == kPlain || CB == 2 || CB == 4, "pairs of 16-column blocks");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, grp = lane >> 4;

    // The row tiles of one column tile are consecutive and on one XCD, so W is
    // read from HBM once.
    const int logical = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int tm = logical % a.tiles_m;
    const int tn = logical / a.tiles_m;

    const int64_t m0 = (int64_t)tm * 16 * RB;
    // First weight row. The paired epilogues (gate and up rows, or the two
    // halves of a head) need rows c and c + 32 of a 64-row group together:
    // CB = 4 takes the group, CB = 2 its rows s .. s + 15 and s + 32 .. s + 47.
    // (fp32 SwiGLU: the same CB / 2 blocks of rows from each of two matrices.)
    constexpr bool TWO_W = F32 && EPI == kSwiGLU;
    constexpr int HB = CB > 1 ? CB / 2 : 1;
    const int64_t n0 = TWO_W ? (int64_t)tn * 16 * HB
                       : EPI == kPlain || CB == 4
                           ? (int64_t)tn * 16 * CB
                           : (int64_t)(tn >> 1) * 64 + (tn & 1) * 16;
    // Rows between column blocks.
    constexpr int BSTEP = !TWO_W && EPI != kPlain && CB == 2 ? 32 : 16;
    const int64_t K = a.K;
    const __amdgpu_buffer_rsrc_t rsx =
        make_rsrc((const char*)a.x + m0 * K * ESZ, operand_bytes(a.M, m0, K, ESZ));
    const __amdgpu_buffer_rsrc_t rsw =
        make_rsrc((const char*)a.w + n0 * K * ESZ, operand_bytes(a.N, n0, K, ESZ));
    const __amdgpu_buffer_rsrc_t rsw2 =
        make_rsrc((const char*)(TWO_W ? a.w2 : a.w) + n0 * K * ESZ,
                  operand_bytes(a.N, n0, K, ESZ));

    slice_partial_sums<F32, RB, CB, NW, NST, BSTEP, TWO_W>(lds, rsx, (uint32_t)(K * ESZ), rsw,
                                                           rsw2, (uint32_t)(K * ESZ), K);
    auto sum = [&](int b) { return slice_sum<NW, NB>(lds, b); };
    auto bias_of = [&](int64_t n) {
        if (F32) return a.bias32 ? a.bias32[n] : 0.0f;
        return a.bias ? __uint_as_float((uint32_t)a.bias[n] << 16) : 0.0f;
    };
    const bool has_bias = F32 ? a.bias32 != nullptr : a.bias != nullptr;
    // fp32 output element (m, n) under the column split.
    auto out32 = [&](int64_t m, int64_t n) -> float* {
        if (a.n1 == 0) return (float*)a.y + m * a.N + n;
        if (n < a.n1) return (float*)a.y + m * a.n1 + n;
        if (n < a.n2) return a.y1 + m * (a.n2 - a.n1) + n - a.n1;
        return a.y2 + m * (a.N - a.n2) + n - a.n2;
    };

    if constexpr (EPI == kPlain) {
        for (int b = wave; b < NB; b += NW) {
            const int64_t n = n0 + 16 * (b % CB) + r16;
            f32x4_t v = sum(b);
            if (n >= a.N) continue;
            const float bv = bias_of(n);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t m = m0 + 16 * (b / CB) + 4 * grp + j;
                if (m >= a.M) continue;
                const int64_t off = m * a.N + n;
                const float f = has_bias ? v[j] + bv : v[j];
                if constexpr (F32) {
                    *out32(m, n) = a.residual ? a.residual[off] + f : f;
                } else if (a.out_mode == NCM_OUT_F32) {
                    ((float*)a.y)[off] = a.residual ? a.residual[off] + f : f;
                } else {
                    uint32_t bits = bf16_bits_rne(flush_subnormal(f));
                    if (a.residual)
                        bits = bf16_bits_rne(a.residual[off] + __uint_as_float(bits << 16));
                    if (a.out_mode == NCM_OUT_BF16_F32)
                        ((float*)a.y)[off] = __uint_as_float(bits << 16);
                    else
                        ((uint16_t*)a.y)[off] = (uint16_t)bits;
                }
            }
        }
        return;
    }
    // Pairs: column blocks cb and cb + CB / 2, 32 weight rows apart.
    for (int b = wave; b < RB * HB; b += NW) {
        const int rb = b / HB, cb = b % HB;
        const f32x4_t va = sum(rb * CB + cb), vb = sum(rb * CB + cb + HB);
        const int64_t na = n0 + 16 * cb + r16;
        if constexpr (TWO_W) {
            // silu(g) * u, unrounded (root.zig:255-261, src/decoder.zig:210-211).
            if (na >= a.N) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t m = m0 + 16 * rb + 4 * grp + j;
                if (m >= a.M) continue;
                const float g = a.bias32 ? va[j] + a.bias32[na] : va[j];
                const float u = a.bias2 ? vb[j] + a.bias2[na] : vb[j];
                const float sigmoid = 1.0f / (1.0f + expf(-g));
                const float act = g * sigmoid;
                ((float*)a.y)[m * a.N + na] = act * u;
            }
            continue;
        }
        // N % 64 == 0: the pair is in range.
        const float ba = bias_of(na), bb = bias_of(na + 32);
        if constexpr (F32 && EPI == kRope) {
            // rotate_head in f32 mode (root.zig:615-634).
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t m = m0 + 16 * rb + 4 * grp + j;
                if (m >= a.M) continue;
                float first = has_bias ? va[j] + ba : va[j];
                float second = has_bias ? vb[j] + bb : vb[j];
                if (na < a.rot_cols) {
                    const int64_t t = (m % a.seq_len) * 64 + (na & 63);
                    const float left = first * a.cosine[t];
                    const float right = -second * a.sine[t];
                    const float right2 = first * a.sine[t + 32];
                    const float left2 = second * a.cosine[t + 32];
                    first = left + right;
                    second = left2 + right2;
                }
                *out32(m, na) = first;
                *out32(m, na + 32) = second;
            }
            continue;
        }
        uint16_t* y = (uint16_t*)a.y;
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
            const int64_t m = m0 + 16 * rb + 4 * grp + j;
            if constexpr (EPI == kSwiGLU) {
                uint32_t q0, q1;
                swiglu_bits2(va[j], vb[j], va[j + 1], vb[j + 1], ba, bb, q0, q1);
                const int64_t col = (na >> 6) * 32 + (na & 31);
                if (m < a.M) y[m * (a.N / 2) + col] = (uint16_t)q0;
                if (m + 1 < a.M) y[(m + 1) * (a.N / 2) + col] = (uint16_t)q1;
            } else {
                // Two rows of the projection's bits, bf16(flush(acc + bias)).
                uint32_t fa = bf16x2_bits_rne(flush_subnormal(va[j] + ba),
                                              flush_subnormal(va[j + 1] + ba));
                uint32_t fb = bf16x2_bits_rne(flush_subnormal(vb[j] + bb),
                                              flush_subnormal(vb[j + 1] + bb));
                if (na < a.rot_cols) {
                    const int c = (int)(na & 63);
                    const float* ct0 = a.cosine + ((m < a.M ? m : 0) % a.seq_len) * 64 + c;
                    const float* ct1 = a.cosine + ((m + 1 < a.M ? m + 1 : 0) % a.seq_len) * 64 + c;
                    const float* st0 = a.sine + (ct0 - a.cosine);
                    const float* st1 = a.sine + (ct1 - a.cosine);
                    rope_bits2(fa, fb, bf16x2_rne(ct0[0], ct1[0]), bf16x2_rne(st0[0], st1[0]),
                               bf16x2_rne(ct0[32], ct1[32]), bf16x2_rne(st0[32], st1[32]));
                }
                if (m < a.M) {
                    y[m * a.N + na] = (uint16_t)fa;
                    y[m * a.N + na + 32] = (uint16_t)fb;
                }
                if (m + 1 < a.M) {
                    y[(m + 1) * a.N + na] = (uint16_t)(fa >> 16);
                    y[(m + 1) * a.N + na + 32] = (uint16_t)(fb >> 16);
                }
            }
        }
    }
}

template <bool F32, int RB, int CB, int NW, int NST, int EPI>
hipError_t launch_slice_t(SliceArgs a, hipStream_t st) {
    using S = SliceShape<F32, RB, CB, NW, NST>;
    auto kern = linear_slice_kernel<F32, RB, CB, NW, NST, EPI>;
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
    if (attr != hipSuccess) return attr;
    a.tiles_m = (int)((a.M + 16 * RB - 1) / (16 * RB));
    constexpr int COLS = F32 && EPI == kSwiGLU ? 8 * CB : 16 * CB;  // of N per workgroup
    const int64_t blocks = a.tiles_m * ((a.N + COLS - 1) / COLS);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(64 * NW), S::LDS, st, a);
    return hipGetLastError();
}

// Cost of a tile: rounds of the 256 CUs times the blocks of 16 operand rows
// that a workgroup loads (at 75 GB/s a CU, over all shapes measured: 31 us for
// 512 x 2048 x 8192 at cost 8, 18 us for 128 rows at cost 4).
int64_t tile_cost(const SliceTile& s, int64_t M, int64_t N) {
    const int64_t tiles =
        ((M + 16 * s.rb - 1) / (16 * s.rb)) * ((N + 16 * s.cb - 1) / (16 * s.cb));
    return (tiles + 255) / 256 * (s.rb + s.cb);
}

// The cheapest tile (paired: one with a partner column block).
int64_t best_tile(int64_t M, int64_t N, bool paired, int* tile) {
    int64_t best = INT64_MAX;
    for (int t = 0; t < kSliceTileCount; ++t) {
        if (paired && kSliceTiles[t].cb < 2) continue;
        const int64_t cost = tile_cost(kSliceTiles[t], M, N);
        if (cost < best) {
            best = cost;
            *tile = t;
        }
    }
    // Up to 48 rows against a head of four rounds or more: the weight stream
    // is the bound, and two workgroups a CU with two column blocks each keep
    // more of it in flight (24 rows, 151936 x 1024: 77 -> 70 us; 40 rows: 90 ->
    // 77 us; 24 rows, 128256 x 2048: 116 -> 110 us).
    const int64_t rb = (M + 15) / 16;
    if (rb <= 3 && (N + 63) / 64 > 3 * 256) *tile = rb == 1 ? 2 : (rb == 2 ? 3 : 4);
    return best;
}

template <int EPI, bool F32 = false>
hipError_t launch_slice(int tile, const SliceArgs& a, hipStream_t st) {
#define NCM_SLICE(RB, CB, NST) \
    return launch_slice_t<F32, RB, CB, kSliceWaves, NST, EPI>(a, st)
    if constexpr (EPI == kPlain) {
        if (tile == 0) NCM_SLICE(1, 1, 2);
        if (tile == 1) NCM_SLICE(2, 1, 1);
    }
    switch (tile) {
        case 2: NCM_SLICE(1, 2, 1);
        case 3: NCM_SLICE(2, 2, 1);
        case 4: NCM_SLICE(3, 2, 1);
        case 5: NCM_SLICE(1, 4, 1);
        case 6: NCM_SLICE(4, 2, 1);
        case 7: NCM_SLICE(2, 4, 1);
        case 8: NCM_SLICE(3, 4, 1);
        case 9: NCM_SLICE(4, 4, 1);
        case 10: NCM_SLICE(5, 4, 1);
        default: return hipErrorInvalidValue;
    }
#undef NCM_SLICE
}

}  // namespace

// Where this kernel takes a product, from measurements of both kernels over
// M = 1 .. 1024 and the projections of the 135M to 8B checkpoints (weights
// rotated so that they come from HBM). A round of 128 x 128 tiles costs 16 in
// tile_cost's units, so at cost 13 the small tiles still win: 2048 x 2048
// with 17 / 128 / 512 rows 17 / 21 / 21 -> 5.6 / 7.4 / 12.2 us, 2048 x 8192
// with 77 / 203 / 512 rows 58 / 58 / 63 -> 16 / 21 / 31 us; at 14 and above
// they lose (203 rows, 6144 x 1024: 13.4 -> 14.7 us). With up to 64 rows one row
// tile covers M, every weight is read once and the weight stream is the
// bound at any N: 64 rows, 128256 x 2048 162 -> 139 us, 28672 x 4096 55.9 ->
// 54.8 us; from 65 rows on a wide N would be read twice (77 rows, 28672 x 4096:
// 54 -> 61 us). The largest tile sums eight wavefronts' 20 blocks after a K loop
// that, up to K = 640, is shorter than that, and with one row tile of 65 to 80 rows
// up to 1024: the 64 x 128 tiles take those (77 rows, 9728 x 576 / x 896: 9.6 -> 8.1 /
// 11.6 -> 10.2 us; 150 rows, 6144 x 576 9.0 -> 8.1; 1100 rows, 1152 x 576 8.4 -> 7.5; but
// 300 rows, 4096 x 1024 10.5 -> 11.4, 77 rows, 14336 x 4096 31.8 -> 33.9).
constexpr int kLargestTile = kSliceTileCount - 1;

bool linear_slice_fits(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || K > (int64_t)1 << 21) return false;
    if (M <= 64) return true;
    int tile;
    const int64_t cost = best_tile(M, N, false, &tile);
    if (tile == kLargestTile && (K <= 640 || (K <= 1024 && M <= 80))) return false;
    return cost <= 13;
}

hipError_t launch_linear_slice(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                               const float* residual, void* y, int64_t M, int64_t K, int64_t N,
                               int out_mode, hipStream_t st) {
    SliceArgs a{};
    a.x = x; a.w = w; a.bias = bias; a.residual = residual; a.y = y;
    a.M = M; a.K = K; a.N = N;
    a.out_mode = out_mode;
    int tile = -1;
    best_tile(M, N, false, &tile);
    return launch_slice<kPlain>(tile, a, st);
}

hipError_t launch_linear_slice_swiglu(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                               uint16_t* y, int64_t M, int64_t K, int64_t N2, hipStream_t st) {
    SliceArgs a{};
    a.x = x; a.w = w; a.bias = bias; a.y = y;
    a.M = M; a.K = K; a.N = N2;
    int tile = -1;
    best_tile(M, N2, true, &tile);
    return launch_slice<kSwiGLU>(tile, a, st);
}

hipError_t launch_linear_slice_rope64(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                               uint16_t* y, int64_t M, int64_t K, int64_t N, int64_t rot_cols,
                               int64_t seq_len, const float* cosine, const float* sine,
                               hipStream_t st) {
    SliceArgs a{};
    a.x = x; a.w = w; a.bias = bias; a.y = y;
    a.M = M; a.K = K; a.N = N;
    a.cosine = cosine; a.sine = sine; a.seq_len = seq_len; a.rot_cols = rot_cols;
    int tile = -1;
    best_tile(M, N, true, &tile);
    return launch_slice<kRope>(tile, a, st);
}

// Against the better of the two other fp32 tiles; a tenth in favour of this
// kernel, whose fused epilogues save launches.
bool linear_slice_f32_fits(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || K > (int64_t)1 << 20) return false;
    int tile;
    const double us = slice_best_tile_f32(M, N, K, false, &tile);
    return us < f32_large_us(M, N, K) && us < 1.1 * f32_small_us(M, N, K);
}

hipError_t launch_linear_slice_f32(const LinearF32& l, hipStream_t st) {
    SliceArgs a{};
    a.x = l.x; a.w = l.w; a.bias32 = l.bias; a.residual = l.residual; a.y = l.y;
    a.M = l.M; a.K = l.K; a.N = l.N;
    a.y1 = l.y1; a.y2 = l.y2; a.n1 = l.n1; a.n2 = l.n2;
    a.cosine = l.cosine; a.sine = l.sine; a.seq_len = l.seq_len; a.rot_cols = l.rot_cols;
    const bool rope = l.cosine != nullptr;
    if (rope && (l.N % 64 || l.rot_cols % 64 || l.seq_len <= 0)) return hipErrorInvalidValue;
    int tile = -1;
    slice_best_tile_f32(l.M, l.N, l.K, rope, &tile);
    return rope ? launch_slice<kRope, true>(tile, a, st) : launch_slice<kPlain, true>(tile, a, st);
}

hipError_t launch_linear_slice_swiglu_f32(const float* x, const float* gate, const float* up,
                                          const float* gate_bias, const float* up_bias, float* y,
                                          int64_t M, int64_t K, int64_t N, hipStream_t st) {
    SliceArgs a{};
    a.x = x; a.w = gate; a.w2 = up; a.bias32 = gate_bias; a.bias2 = up_bias; a.y = y;
    a.M = M; a.K = K; a.N = N;
    int tile = -1;
    slice_best_tile_f32(M, 2 * N, K, true, &tile);
    return launch_slice<kSwiGLU, true>(tile, a, st);
}

}  // namespace ncm
