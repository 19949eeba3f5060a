// RVQ helpers shared by the encode and decode paths: shape checks, the
// level table, the fixed-order squared codebook norms and the decode.
#include "common.h"
#include "rvq.h"

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
// A wavefront takes R consecutive rows (so every code is one scalar load) and
// 64 VEC of their columns, VEC to a lane, and issues the code rows of eight
// levels together. R = 4 (t a multiple of 4, so the rows share a sequence and
// every code of stride 4 or more): such a level's row is loaded once for the
// four, a stride-2 level's twice. Consecutive rows stay on one XCD, whose L2
// then holds the coarse levels' rows that they share. Bound: writing recon and
// reading the finest levels' code rows (402 MB at 16 x 2048 x 2048, 8 levels).
// There: 283 us with one thread per four columns of a row and 64-bit divisions
// for every level's position (VALU), 172 us with R = 1, 131 us with R = 4.
template <int VEC, int R>
__global__ __launch_bounds__(256) void rvq_decode_kernel(const int32_t* __restrict__ codes,
                                                         uint32_t t, int64_t d, LevelTable L,
                                                         const uint16_t* __restrict__ cb,
                                                         int64_t v, float* __restrict__ recon,
                                                         uint32_t rows) {
    constexpr int W = VEC / 2;  // 32-bit words of VEC bf16 values
    typedef uint32_t words_t __attribute__((ext_vector_type(W)));
    const uint32_t group = (uint32_t)xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const uint32_t row = __builtin_amdgcn_readfirstlane((group * 4 + (threadIdx.x >> 6)) * R);
    if (row >= rows) return;
    const int64_t col = ((int64_t)blockIdx.y * 64 + (threadIdx.x & 63)) * VEC;
    if (col >= d) return;
    const uint32_t bb = row / t, tt = row - bb * t;
    const int32_t* cr = codes + bb * L.total;
    float a[R][VEC];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < VEC; ++e) a[r][e] = 0.0f;
    auto code_row = [&](int l, uint32_t pos) {
        int32_t k = cr[L.offset[l] + pos];
        k = k < 0 ? 0 : (k >= v ? (int32_t)(v - 1) : k);
        return *(const words_t*)(cb + ((int64_t)l * v + k) * d + col);
    };
    auto add = [&](int r, const words_t& p) {
#pragma unroll
        for (int e = 0; e < W; ++e) {
            a[r][2 * e] = a[r][2 * e] + bf16_lo_to_f32(p[e]);
            a[r][2 * e + 1] = a[r][2 * e + 1] + bf16_hi_to_f32(p[e]);
        }
    };
    for (int l0 = 0; l0 < L.levels; l0 += 8) {
        words_t p[8][R];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            // Past the last level: its row again, not added.
            const int l = l0 + i < L.levels ? l0 + i : L.levels - 1;
            const int sh = __builtin_ctz((uint32_t)L.stride[l]);
            p[i][0] = code_row(l, tt >> sh);
            if constexpr (R == 4) {
                if (sh < 2) p[i][2] = code_row(l, (tt + 2) >> sh);
                if (sh < 1) {
                    p[i][1] = code_row(l, tt + 1);
                    p[i][3] = code_row(l, tt + 3);
                }
            }
        }
        // Every load in flight before the first sum (the compiler would fold
        // each row as it comes to save registers).
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (l0 + i >= L.levels) break;
            add(0, p[i][0]);
            if constexpr (R == 4) {
                const int stride = L.stride[l0 + i];
                if (stride == 1) {
                    add(1, p[i][1]);
                    add(2, p[i][2]);
                    add(3, p[i][3]);
                } else {
                    add(1, p[i][0]);
                    if (stride == 2) {
                        add(2, p[i][2]);
                        add(3, p[i][2]);
                    } else {
                        add(2, p[i][0]);
                        add(3, p[i][0]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float* o = recon + (int64_t)(row + r) * d + col;
#pragma unroll
        for (int e = 0; e < VEC; e += 4)
            *(f32x4_t*)(o + e) = f32x4_t{a[r][e], a[r][e + 1], a[r][e + 2], a[r][e + 3]};
    }
}

constexpr int64_t kDecodeFourRows = 4096;

hipError_t launch_rvq_decode(const int32_t* codes, int64_t b, int64_t t, int64_t d,
                             int64_t levels, const int32_t* strides, const uint16_t* codebooks,
                             int64_t v, float* recon, hipStream_t stream) {
    const LevelTable L = make_level_table(t, levels, strides);
    const int64_t rows = b * t;  // at most 2^31; strides are powers of two, d % 64 == 0
    // Four rows a wavefront where there are enough of them to fill the chip.
    // Narrow rows: four columns to a lane fill the wavefront.
    const bool four = t % 4 == 0 && rows >= kDecodeFourRows;
    const int64_t per = four ? 16 : 4;
    const unsigned gx = (unsigned)((rows + per - 1) / per);
#define NCM_DEC(VEC, R)                                                                          \
    hipLaunchKernelGGL((rvq_decode_kernel<VEC, R>),                                              \
                       dim3(gx, (unsigned)((d + 64 * VEC - 1) / (64 * VEC))), dim3(256), 0,      \
                       stream, codes, (uint32_t)t, d, L, codebooks, v, recon, (uint32_t)rows)
    if (d >= 512) {
        if (four) NCM_DEC(8, 4);
        else NCM_DEC(8, 1);
    } else {
        if (four) NCM_DEC(4, 4);
        else NCM_DEC(4, 1);
    }
#undef NCM_DEC
    return hipGetLastError();
}

}  // namespace ncm
