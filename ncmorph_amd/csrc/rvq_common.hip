// RVQ helpers shared by the encode and decode paths: shape checks, the
// level table, the fixed-order squared codebook norms and the decode.
#include "common.h"
#include "rvq.h"

#include <type_traits>

namespace ncm {

static bool pow2(int64_t s) { return s >= 1 && (s & (s - 1)) == 0; }

int rvq_check_shape(int64_t b, int64_t t, int64_t d, int64_t levels, const int32_t* strides,
                    int64_t v) {
    if (b < 1 || t < 1 || d < 64 || d % 64 != 0 || d > (int64_t(1) << 20)) return NCM_E_SHAPE;
    if (levels < 1 || levels > kMaxLevels) return NCM_E_SHAPE;
    if (v < 1 || v > 65536) return NCM_E_SHAPE;
    for (int64_t l = 0; l < levels; ++l) {
        if (!pow2(strides[l])) return NCM_E_SHAPE;
        if (l > 0 && strides[l] > strides[l - 1]) return NCM_E_SHAPE;
    }
    if (t % strides[0] != 0) return NCM_E_SHAPE;
    if (b > (int64_t(1) << 31) || t > (int64_t(1) << 31) || b * t > (int64_t(1) << 31))
        return NCM_E_SHAPE;
    return NCM_OK;
}

LevelTable make_level_table(int64_t t, int64_t levels, const int32_t* strides) {
    LevelTable L{};
    L.levels = (int32_t)levels;
    int64_t off = 0;
    for (int64_t l = 0; l < levels; ++l) {
        L.stride[l] = strides[l];
        L.offset[l] = off;
        off += t / strides[l];
    }
    L.total = off;
    return L;
}

// Fixed-order squared norm of a bf16 row (the oracle's ncmo_sumsq_bf16_fixed):
// lane j accumulates elements 256 m + 4 j + e with fmaf, then an xor
// butterfly, which every lane finishes with the same bits.
__device__ __forceinline__ float wave_sumsq_bf16(const uint16_t* c, int64_t d, int lane) {
    float acc = 0.0f;
    for (int64_t m = 0; m * 256 < d; ++m) {
        const int64_t i = m * 256 + 4 * lane;
        if (i < d) {
            const u32x2_t p = *(const u32x2_t*)(c + i);
            const float c0 = bf16_lo_to_f32(p[0]), c1 = bf16_hi_to_f32(p[0]);
            const float c2 = bf16_lo_to_f32(p[1]), c3 = bf16_hi_to_f32(p[1]);
            acc = __builtin_fmaf(c0, c0, acc);
            acc = __builtin_fmaf(c1, c1, acc);
            acc = __builtin_fmaf(c2, c2, acc);
            acc = __builtin_fmaf(c3, c3, acc);
        }
    }
    return wave_sum_xor(acc);  // xor butterfly 32, 16, ..., 1
}

__global__ void rvq_csq_kernel(const uint16_t* __restrict__ cb, int64_t rows, int64_t d,
                               float* __restrict__ csq) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const float s = wave_sumsq_bf16(cb + row * d, d, lane);
    if (lane == 0) csq[row] = s;
}

hipError_t launch_rvq_csq(const uint16_t* codebooks, int64_t rows, int64_t d, float* csq,
                          hipStream_t stream) {
    const int64_t blocks = (rows + 3) / 4;
    hipLaunchKernelGGL(rvq_csq_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, codebooks,
                       rows, d, csq);
    return hipGetLastError();
}

// recon[b, t, :] = sum over l (in order, from +0) of C_l[code_l[b, t / s_l]].
// A thread takes eight columns of R consecutive rows; a workgroup takes
// `chunks` such pieces of each of `groups` row groups, as many as fill its
// wavefronts. The codes of up to eight code rows are loaded together, then
// those rows, then they are added in level order; R = 4 (t a multiple of 4, so
// the rows share a sequence and every code of stride 4 or more) loads a level
// below n4 once for its four rows and one below n2 twice. Consecutive rows
// stay on one XCD, whose L2 then holds the coarse levels' rows that they share.
//
// Bound: writing recon and reading the finest levels' code rows. Against one
// thread per four columns, with 64-bit divisions for every level's position, us
// (1024 codes): 32768 rows of d 2048, strides 128 .. 1 217 -> 79, four levels of
// stride 1 131 -> 66, one level 55 -> 55; of d 576, four of stride 1 40 -> 22; 262144
// rows of d 64, strides 128 .. 1 55 -> 19, four of stride 1 33 -> 19, one 16.8 -> 15.8.
// (A wavefront per row or four rows, with its lanes past d idle and its loads
// always those of eight levels: 98, 104, 84, 55, 82, 109 and 103.)
template <int R>
__global__ __launch_bounds__(512) void rvq_decode_kernel(
    const int32_t* __restrict__ codes, uint32_t t, int64_t d, LevelTable L,
    const uint16_t* __restrict__ cb, int64_t v, float* __restrict__ recon, uint32_t rows,
    uint32_t chunks, uint32_t groups, int n4, int n2) {
    const uint32_t block = (uint32_t)xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const uint32_t g = threadIdx.x / chunks, c = threadIdx.x - g * chunks;
    const uint64_t first = ((uint64_t)block * groups + g) * R;
    const int64_t col = ((int64_t)blockIdx.y * chunks + c) * 8;
    if (g >= groups || first >= rows || col >= d) return;
    const uint32_t row = (uint32_t)first;
    const uint32_t bb = row / t, tt = row - bb * t;
    const int32_t* cr = codes + bb * L.total;
    float a[R][8];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < 8; ++e) a[r][e] = 0.0f;
    // N levels from l on, S code rows each (every R / S rows share one).
    auto batch = [&](auto n, auto s, int l) {
        constexpr int N = decltype(n)::value, S = decltype(s)::value;
        int32_t k[N][S];
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < S; ++j)
                k[i][j] = cr[L.offset[l + i] +
                             ((tt + j * (R / S)) >> __builtin_ctz((uint32_t)L.stride[l + i]))];
        u32x4_t p[N][S];
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < S; ++j) {
                const int32_t kk = k[i][j] < 0 ? 0 : (k[i][j] >= v ? (int32_t)(v - 1) : k[i][j]);
                p[i][j] = *(const u32x4_t*)(cb + ((int64_t)(l + i) * v + kk) * d + col);
            }
        // Every load in flight before the first sum (the compiler would fold
        // each row as it comes to save registers).
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t w = p[i][r / (R / S)][e];
                    a[r][2 * e] = a[r][2 * e] + bf16_lo_to_f32(w);
                    a[r][2 * e + 1] = a[r][2 * e + 1] + bf16_hi_to_f32(w);
                }
    };
    // Levels [l, end): eight code rows at a time, then what is left by halves.
    auto levels = [&](auto s, int l, int end) {
        constexpr int S = decltype(s)::value;
        for (; l + 8 / S <= end; l += 8 / S) batch(std::integral_constant<int, 8 / S>{}, s, l);
        if constexpr (S < 2)
            if (l + 4 <= end) {
                batch(std::integral_constant<int, 4>{}, s, l);
                l += 4;
            }
        if constexpr (S < 4)
            if (l + 2 <= end) {
                batch(std::integral_constant<int, 2>{}, s, l);
                l += 2;
            }
        if (l < end) batch(std::integral_constant<int, 1>{}, s, l);
    };
    if constexpr (R == 4) {
        levels(std::integral_constant<int, 1>{}, 0, n4);
        levels(std::integral_constant<int, 2>{}, n4, n2);
        levels(std::integral_constant<int, 4>{}, n2, L.levels);
    } else {
        levels(std::integral_constant<int, 1>{}, 0, L.levels);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float* o = recon + (int64_t)(row + r) * d + col;
        *(f32x4_t*)o = f32x4_t{a[r][0], a[r][1], a[r][2], a[r][3]};
        *(f32x4_t*)(o + 4) = f32x4_t{a[r][4], a[r][5], a[r][6], a[r][7]};
    }
}

// Elements of recon from which a thread takes four rows: an output of 256 MB,
// which the memory-side cache does not hold (one row -> four: 32768 x 2048, strides
// 128 .. 1 96 -> 79 us; 262144 x 512, one level 149 -> 103). Below, four rows leave too
// few loads in flight (32768 x 1024, one level 25.9 -> 28.9).
constexpr int64_t kDecodeFourRows = (int64_t)1 << 26;

hipError_t launch_rvq_decode(const int32_t* codes, int64_t b, int64_t t, int64_t d,
                             int64_t levels, const int32_t* strides, const uint16_t* codebooks,
                             int64_t v, float* recon, hipStream_t stream) {
    const LevelTable L = make_level_table(t, levels, strides);
    const int64_t rows = b * t;  // at most 2^31; strides are powers of two, d % 64 == 0
    int n4 = 0, n2 = 0;          // strides do not increase
    for (int l = 0; l < L.levels; ++l) {
        n4 += L.stride[l] >= 4;
        n2 += L.stride[l] >= 2;
    }
    const bool four = t % 4 == 0 && rows * d >= kDecodeFourRows;
    // 256 columns at a time, so that an XCD's L2 holds more of the codebooks' rows
    // (32768 x 2048, 1024 codes, four full-resolution levels 102 -> 66 us); four rows
    // and at most one such level read fewer rows than they write and take whole rows up to 4096
    // columns (strides 128 .. 1, 83 -> 79; with 4096 codes 112 -> 98).
    const int64_t most = four && L.levels - n2 < 2 ? 512 : 32;
    const int64_t shares = (d / 8 + most - 1) / most, chunks = (d / 8 + shares - 1) / shares;
    // Of the workgroup sizes the one that whole row pieces fill best.
    int64_t threads = (chunks + 63) / 64 * 64, groups = threads / chunks;
    for (int64_t n = threads + 64; n <= 512; n += 64)
        if (n / chunks * threads > groups * n) {
            threads = n;
            groups = n / chunks;
        }
    const int64_t per = groups * (four ? 4 : 1);
    const dim3 grid((unsigned)((rows + per - 1) / per), (unsigned)shares);
    hipLaunchKernelGGL(four ? rvq_decode_kernel<4> : rvq_decode_kernel<1>, grid,
                       dim3((unsigned)threads), 0, stream, codes, (uint32_t)t, d, L, codebooks, v,
                       recon, (uint32_t)rows, (uint32_t)chunks, (uint32_t)groups, n4, n2);
    return hipGetLastError();
}

}  // namespace ncm
