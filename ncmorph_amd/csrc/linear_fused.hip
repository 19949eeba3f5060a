// The bf16 linear with epilogues that pair two 32-column MFMA tiles of one
// wave, fusing the elementwise op that follows the projection in the
// decoder (bf16 mode; the projection's own output is rounded to bf16 first,
// exactly as the unfused path writes it):
//   SwiGLU: weight rows are interleaved in groups of 32 (rows 64g .. 64g+31
//     are gate rows 32g .. 32g+31, rows 64g+32 .. 64g+63 the matching up
//     rows), so tiles 2p and 2p+1 of a wave hold gate and up of the same 32
//     features; the epilogue writes round(silu_bf16(gate) * up)
//     (src/decoder.zig:208-211) to y [M, N / 2].
//   RoPE (head_dim 64): tiles 2p and 2p+1 are the two halves of one head;
//     columns below rot_cols (the q and k heads) are rotated as rotate_head
//     does in bf16 mode (packages/kernels/root.zig:615-634) with table row
//     (row % seq_len), the rest (v) written as projected; y [M, N].
// Both write bf16 bits only.
#include "gemm_core.h"
#include "linear.h"

namespace ncm {

namespace {

constexpr int kEpiSwiGLU = 1;
constexpr int kEpiRope = 2;

struct PairArgs {
    const float* cosine;  // RoPE tables [seq_len, 64]
    const float* sine;
    int64_t seq_len;
    int64_t rot_cols;  // columns [0, rot_cols) are rotated
};

// The projections' output value of one accumulator is bf16(flush(acc +
// bias)), computed two values at a time with bf16x2_bits_rne (SwiGLU:
// swiglu_bits2 in common.h).

}  // namespace

template <class S, int EPI, bool HAS_BIAS>
__global__ __launch_bounds__(S::NT)
__attribute__((amdgpu_waves_per_eu(S::OCC, S::OCC))) void linear_pair_kernel(
    const void* __restrict__ x, const void* __restrict__ w, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, int tiles_n, int group_m,
    PairArgs pa) {
    static_assert(S::NB % 2 == 0 && S::WN % 64 == 0, "pairs of 32-column tiles per wave");
    extern __shared__ __attribute__((aligned(16))) char lds[];

    const int logical = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int per_group = group_m * tiles_n;
    const int g = logical / per_group;
    const int tiles_m = (int)((M + S::BM - 1) / S::BM);
    const int gm = min(group_m, tiles_m - g * group_m);
    const int in_g = logical % per_group;
    const int64_t m0 = (int64_t)(g * group_m + in_g % gm) * S::BM;
    const int64_t n0 = (int64_t)(in_g / gm) * S::BN;

    GemmAcc<S> acc;
    acc.zero();
    gemm_mainloop<S>((const char*)x + m0 * K * S::ESZ, K, operand_bytes(M, m0, K, S::ESZ),
                     (const char*)w + n0 * K * S::ESZ, K, operand_bytes(N, n0, K, S::ESZ), K, lds,
                     acc);

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    if (wave >= S::NWG) return;
    const int wm = wave % S::WGM;
    const int wn = wave / S::WGM;
    const int c = lane & 31;
    const int64_t ld = EPI == kEpiSwiGLU ? N / 2 : N;

    // Per group of 4 rows: a quad transpose leaves each lane with 4
    // consecutive columns of one row, so stores are 8 bytes and each RoPE
    // table half is one 16-byte load. Rows past M (a partial last row tile)
    // are computed on table row 0 and not stored.
    const int q = lane & 3;
    const int hrow = 4 * (lane >> 5) + q;
    const int c4 = c & ~3;
    // First column of pair p's first tile; N % 64 == 0: the pair is wholly in
    // or out (wave-uniform).
    auto col_of = [&](int p) { return n0 + wn * S::WN + 64 * p; };
    // bf16(flush(acc + bias)) is what the projection writes.
#pragma unroll
    for (int p = 0; p < S::NB / 2; ++p) {
        const int64_t col = col_of(p) + c;
        float ba = 0.0f, bb = 0.0f;
        if (HAS_BIAS && col < N) {
            ba = __uint_as_float((uint32_t)bias[col] << 16);
            bb = __uint_as_float((uint32_t)bias[col + 32] << 16);
        }
#pragma unroll
        for (int mb = 0; mb < S::MB; ++mb) {
            add_flush16(acc.v[mb][2 * p], ba);
            add_flush16(acc.v[mb][2 * p + 1], bb);
        }
    }

    if constexpr (EPI == kEpiSwiGLU) {
        // Elementwise first (gate and up of a column sit in the same lane and
        // element), then one transpose of the results.
#pragma unroll
        for (int p = 0; p < S::NB / 2; ++p) {
            if (col_of(p) >= N) break;
            const int64_t ca = (n0 + wn * S::WN) / 2 + 32 * p + c4;
#pragma unroll
            for (int mb = 0; mb < S::MB; ++mb)
#pragma unroll
                for (int blk = 0; blk < 4; ++blk) {
                    const int64_t m = m0 + wm * S::WM + mb * 32 + 8 * blk + hrow;
                    float r[4];
#pragma unroll
                    for (int j = 0; j < 4; j += 2) {
                        const int i = 4 * blk + j;
                        const uint32_t o = swiglu_bits2_flushed(
                            acc.v[mb][2 * p][i], acc.v[mb][2 * p + 1][i],
                            acc.v[mb][2 * p][i + 1], acc.v[mb][2 * p + 1][i + 1]);
                        r[j] = __uint_as_float(o & 0xFFFFu);
                        r[j + 1] = __uint_as_float(o >> 16);
                    }
                    quad_transpose4(r, q);
                    if (m < M) {
                        u32x2_t o;
                        o[0] = __float_as_uint(r[0]) | (__float_as_uint(r[1]) << 16);
                        o[1] = __float_as_uint(r[2]) | (__float_as_uint(r[3]) << 16);
                        __builtin_nontemporal_store(o, (u32x2_t*)(y + m * ld + ca));
                    }
                }
        }
        return;
    }

    // RoPE. The table row of a group of rows is loaded and rounded once for
    // all heads of the wavefront; its number is a 32-bit remainder from the
    // tile's first row's.
    const uint32_t seq = (uint32_t)pa.seq_len;
    const uint32_t t0 = (uint32_t)(m0 % pa.seq_len);
    const bool any_rot = col_of(0) < pa.rot_cols;
#pragma unroll
    for (int mb = 0; mb < S::MB; ++mb)
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
            const uint32_t dr = wm * S::WM + mb * 32 + 8 * blk + hrow;
            const int64_t m = m0 + dr;
            uint32_t tc[2], ts[2], tc2[2], ts2[2];
            if (any_rot) {
                const uint32_t t = m < M ? (t0 + dr) % seq : 0u;
                const float* ct = pa.cosine + (int64_t)t * 64 + c4;
                const float* st = pa.sine + (int64_t)t * 64 + c4;
                const f32x4_t cf = *(const f32x4_t*)ct, cs = *(const f32x4_t*)(ct + 32);
                const f32x4_t sf = *(const f32x4_t*)st, ss = *(const f32x4_t*)(st + 32);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    tc[h] = bf16x2_rne(cf[2 * h], cf[2 * h + 1]);
                    ts[h] = bf16x2_rne(sf[2 * h], sf[2 * h + 1]);
                    tc2[h] = bf16x2_rne(cs[2 * h], cs[2 * h + 1]);
                    ts2[h] = bf16x2_rne(ss[2 * h], ss[2 * h + 1]);
                }
            }
#pragma unroll
            for (int p = 0; p < S::NB / 2; ++p) {
                if (col_of(p) >= N) break;
                // The two tiles' bits of a row in one register through the
                // transpose, then two columns per register.
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    v[j] = __uint_as_float(bf16x2_bits_rne(acc.v[mb][2 * p][4 * blk + j],
                                                           acc.v[mb][2 * p + 1][4 * blk + j]));
                quad_transpose4(v, q);
                u32x2_t ra, rb;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t e = __float_as_uint(v[2 * h]), o = __float_as_uint(v[2 * h + 1]);
                    uint32_t lo = __builtin_amdgcn_perm(o, e, 0x05040100u);
                    uint32_t hi = __builtin_amdgcn_perm(o, e, 0x07060302u);
                    if (col_of(p) < pa.rot_cols) rope_bits2(lo, hi, tc[h], ts[h], tc2[h], ts2[h]);
                    ra[h] = lo;
                    rb[h] = hi;
                }
                if (m < M) {
                    uint16_t* dst = y + m * ld + col_of(p) + c4;
                    __builtin_nontemporal_store(ra, (u32x2_t*)dst);
                    __builtin_nontemporal_store(rb, (u32x2_t*)(dst + 32));
                }
            }
        }
}

template <class S, int EPI, bool HAS_BIAS>
static hipError_t launch_pair_t(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                                uint16_t* y, int64_t M, int64_t K, int64_t N, PairArgs pa,
                                hipStream_t stream) {
    auto kern = linear_pair_kernel<S, EPI, HAS_BIAS>;
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)kern,
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           S::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const int tiles_m = (int)((M + S::BM - 1) / S::BM);
    const int tiles_n = (int)((N + S::BN - 1) / S::BN);
    const int group_m = linear_band(tiles_m);
    hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n), dim3(S::NT), S::LDS_BYTES, stream, x, w,
                       bias, y, M, K, N, tiles_n, group_m, pa);
    return hipGetLastError();
}

template <int EPI>
static hipError_t launch_pair(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                              uint16_t* y, int64_t M, int64_t K, int64_t N, PairArgs pa,
                              hipStream_t st) {
    using L0 = GemmShape<256, 256, 64, 4, 2, 2, 8, true, 2, false, 1, 24, -1, true>;
    using L1 = GemmShape<128, 128, 64, 4, 2, 2, 8, true, 4, false, 1, -1, -1, true>;
    using L5 = GemmShape<256, 128, 64, 4, 2, 2, 8, true, 3, false, 1, -1, -1, true>;
    using L128x256 = GemmShape<128, 256, 64, 2, 4, 2, 8, true, 3, false, 1, -1, -1, true>;
    using L64x128 = GemmShape<64, 128, 64, 2, 2, 2, 8, true, 4, false, 1, -1, -1, true>;
    const bool hb = bias != nullptr;
    switch (linear_tile_config(M, N, -1)) {
        case 0:
            return hb ? launch_pair_t<L0, EPI, true>(x, w, bias, y, M, K, N, pa, st)
                      : launch_pair_t<L0, EPI, false>(x, w, bias, y, M, K, N, pa, st);
        case 1:
            return hb ? launch_pair_t<L1, EPI, true>(x, w, bias, y, M, K, N, pa, st)
                      : launch_pair_t<L1, EPI, false>(x, w, bias, y, M, K, N, pa, st);
        case 5:
            return hb ? launch_pair_t<L5, EPI, true>(x, w, bias, y, M, K, N, pa, st)
                      : launch_pair_t<L5, EPI, false>(x, w, bias, y, M, K, N, pa, st);
        case kTile128x256:
            return hb ? launch_pair_t<L128x256, EPI, true>(x, w, bias, y, M, K, N, pa, st)
                      : launch_pair_t<L128x256, EPI, false>(x, w, bias, y, M, K, N, pa, st);
        default:
            return hb ? launch_pair_t<L64x128, EPI, true>(x, w, bias, y, M, K, N, pa, st)
                      : launch_pair_t<L64x128, EPI, false>(x, w, bias, y, M, K, N, pa, st);
    }
}

hipError_t launch_linear_swiglu(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                                uint16_t* y, int64_t M, int64_t K, int64_t N2,
                                hipStream_t stream) {
    if (N2 % 64) return hipErrorInvalidValue;
    if (linear_slice_fits(M, N2, K))
        return launch_linear_slice_swiglu(x, w, bias, y, M, K, N2, stream);
    const int64_t r = linear_tail_rows(M, N2, K);
    if (r > 0) {
        const int64_t mm = M - r;
        hipError_t e = launch_pair<kEpiSwiGLU>(x, w, bias, y, mm, K, N2,
                                               PairArgs{nullptr, nullptr, 1, 0}, stream);
        if (e != hipSuccess) return e;
        return launch_linear_tail(x + mm * K, w, bias, nullptr, y + mm * (N2 / 2), r, K, N2 / 2,
                                  NCM_OUT_BF16, true, stream);
    }
    return launch_pair<kEpiSwiGLU>(x, w, bias, y, M, K, N2, PairArgs{nullptr, nullptr, 1, 0},
                                   stream);
}

hipError_t launch_linear_rope64(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                                uint16_t* y, int64_t M, int64_t K, int64_t N, int64_t rot_cols,
                                int64_t seq_len, const float* cosine, const float* sine,
                                hipStream_t stream) {
    if (N % 64 || rot_cols % 64 || seq_len <= 0) return hipErrorInvalidValue;
    if (linear_slice_fits(M, N, K))
        return launch_linear_slice_rope64(x, w, bias, y, M, K, N, rot_cols, seq_len, cosine, sine,
                                          stream);
    return launch_pair<kEpiRope>(x, w, bias, y, M, K, N,
                                 PairArgs{cosine, sine, seq_len, rot_cols}, stream);
}

}  // namespace ncm
