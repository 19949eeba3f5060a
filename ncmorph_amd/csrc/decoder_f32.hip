// The decoder prefill forward of src/decoder.zig:62-228 in its f32 mode
// (bf16_compute false: checkpoints that are not all BF16), with the
// per-stage trace of forward_with_trace. Per layer, all in fp32:
//   n    = rms_norm(h, input_norm)                          (root.zig:226-239)
//   q, k, v = n W^T (+ b)  -> [QK-norm] -> rotate_head      (root.zig:483-530, 615-634)
//   c    = softmax((q . k) / sqrt(hd) over allowed keys) v   (root.zig:536-578)
//   h    = h + (c W_o^T (+ b))
//   n    = rms_norm(h, post_attention_norm)
//   a    = silu(n W_gate^T (+ b)) * (n W_up^T (+ b))         (root.zig:255-261)
//   h    = h + (a W_down^T (+ b))
// then logits = rms_norm(h, final_norm) W_head^T. Where the few-row kernel
// (linear_slice.hip) takes a product, q|k|v run as one with the rotation of
// 64-wide heads, gate|up as one with the activation, and o and down with the
// residual add, the same values bit for bit (a traced stage runs apart).
// The projections run on the
// fp32 MFMA (launch_linear_f32: every product exact, the sums in the matrix
// core's order instead of the reference's increasing k); the bias is added
// after the product, as the reference's project does. The attention sums
// each dot product in dimension order, the softmax sum and every context
// element in key order, as the reference, so only exp differs (device expf
// against Zig's exp).
#include <hip/hip_runtime.h>

#include "common.h"
#include "decoder.h"
#include "linear.h"

namespace ncm {

namespace {

// hidden[r] = embed[ids[r]] (f32 table rows).
__global__ __launch_bounds__(256) void embed_rows_f32_kernel(const int64_t* __restrict__ ids,
                                                             const float* __restrict__ table,
                                                             float* __restrict__ hidden,
                                                             int64_t width) {
    const int64_t r = blockIdx.y;
    const float* src = table + ids[r] * width;
    float* dst = hidden + r * width;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < width;
         i += (int64_t)gridDim.x * 256)
        dst[i] = src[i];
}

// y[r, c] = y[r, c] + a[r, c] (a_rows = rows) or + a[c] (a_rows = 1, a bias).
__global__ __launch_bounds__(256) void add_f32_kernel(float* __restrict__ y,
                                                      const float* __restrict__ a, int64_t rows,
                                                      int64_t n, int64_t a_rows) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * n) return;
    const float av = a_rows == 1 ? a[i % n] : a[i];
    y[i] = y[i] + av;
}

// rotate_head in f32 mode (root.zig:615-634), in place: row r, head h at
// x[r * row_stride + h * hd ..]; table row r % seq_len. One thread per pair.
__global__ __launch_bounds__(256) void rope_rotate_f32_kernel(float* __restrict__ x, int64_t rows,
                                                              int64_t row_stride, int heads,
                                                              int hd, int64_t seq_len,
                                                              const float* __restrict__ cosine,
                                                              const float* __restrict__ sine) {
    const int half = hd >> 1;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * heads * half) return;
    const int i = (int)(idx % half);
    const int64_t rh = idx / half;
    const int h = (int)(rh % heads);
    const int64_t r = rh / heads;
    const int64_t pos = r % seq_len;
    float* e = x + r * row_stride + (int64_t)h * hd + i;
    const float first = e[0], second = e[half];
    const float* ct = cosine + pos * hd + i;
    const float* st = sine + pos * hd + i;
    const float left = first * ct[0];
    const float right = -second * st[0];
    const float right2 = first * st[half];
    const float left2 = second * ct[half];
    e[0] = left + right;
    e[half] = left2 + right2;
}

hipError_t launch_rope_rotate_f32(float* x, int64_t rows, int64_t row_stride, int heads, int hd,
                                  int64_t seq_len, const float* cosine, const float* sine,
                                  hipStream_t st) {
    const int64_t n = rows * heads * (hd / 2);
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(rope_rotate_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       st, x, rows, row_stride, heads, hd, seq_len, cosine, sine);
    return hipGetLastError();
}

constexpr int kAttnF32MaxHd = 256;
constexpr int kAttnQ = 8;          // queries (wavefronts) per workgroup
constexpr int kAttnPanel = 2048;   // keys whose scores a workgroup keeps in LDS

// f32-mode attention: a workgroup takes eight queries of one (sequence, head),
// one per wavefront, and stages KC keys (then their values) at a time in LDS
// for all of them, the next ones on their way in registers. A score is the dot product in dimension order (lane = key),
// then times 1 / sqrt(hd); the softmax sum runs in key order, and so does
// every context element (lane = dimension): the reference's orders, so only
// exp differs from it (device expf). The scores of up to kAttnPanel keys stay
// in LDS and are formed once; past that they are formed again, panel by
// panel, for the sum and for the context. Allowed keys, in increasing order:
// causal, [query - window + 1, query]; or with the level mask (seg_lo set),
// the prefix keys whose pad bit is clear, then [seg_lo[q], seg_hi[q]) (at or
// after the prefix). Masked keys (probability 0) add nothing, as in the
// reference unless V holds an infinity or NaN there; a query with no allowed
// key gets a zero context (root.zig:563-565).
//
// What bounds it at a 200-token prompt of 9 heads (225 workgroups): the chains
// of one wavefront (64 adds a score, one add a key in the sum and in the
// context), not memory. One wavefront per (query, head) that walked the keys
// three times, reading every K row from the caches by itself, took 90 us a
// layer there; this takes 17.

// Orders LDS accesses of one wavefront's lanes (its LDS operations run in
// program order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// HS: ceil(hd / 64); KC: 128, or 64 where 128 rows would not fit.
template <int HS, int KC>
__global__ __launch_bounds__(64 * kAttnQ) void attention_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    float* __restrict__ out, int64_t T, int group, int hd, int64_t q_stride, int64_t kv_stride,
    int64_t out_stride, int64_t window, float scale, int64_t prefix,
    const int32_t* __restrict__ seg_lo, const int32_t* __restrict__ seg_hi,
    const uint64_t* __restrict__ pad, int panel) {
    // [KC][hd + 4] staged K or V rows, [kAttnQ][hd] queries, then
    // [kAttnQ][panel + 4] scores.
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int ld = hd + 4, sld = panel + 4;
    float* rows = smem;
    float* qs = rows + KC * ld;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* sc = qs + kAttnQ * hd + wave * sld;
    const int h = blockIdx.y;
    const int64_t b = blockIdx.z;
    // The last queries (the most keys under a causal mask) first.
    const int64_t q0 = (int64_t)(gridDim.x - 1 - blockIdx.x) * kAttnQ;
    const int64_t qi = q0 + wave;
    const bool live = qi < T;
    const float* qrow = q + (b * T + (live ? qi : q0)) * q_stride + (int64_t)h * hd;
    const float* kbase = k + b * T * kv_stride + (int64_t)(h / group) * hd;
    const float* vbase = v + b * T * kv_stride + (int64_t)(h / group) * hd;
    for (int d = lane; d < hd; d += 64) qs[wave * hd + d] = qrow[d];

    // The walk of the workgroup: keys 0 .. P - 1, then base .. end - 1, the
    // union of its queries' ranges; this query's own range is [lo, hi).
    const int64_t P = seg_lo ? prefix : 0;
    int64_t base, end, lo, hi;
    if (seg_lo) {
        base = T;
        end = 0;
        lo = hi = 0;
        for (int i = 0; i < kAttnQ && q0 + i < T; ++i) {
            const int64_t l = seg_lo[b * T + q0 + i], e = seg_hi[b * T + q0 + i];
            if (i == wave) {
                lo = l;
                hi = e;
            }
            if (e > l) {
                base = l < base ? l : base;
                end = e > end ? e : end;
            }
        }
        if (end < base) base = end = P;
    } else {
        const int64_t last = q0 + kAttnQ < T ? q0 + kAttnQ : T;
        base = window > 0 && q0 - window + 1 > 0 ? q0 - window + 1 : 0;
        end = last;
        lo = window > 0 && qi - window + 1 > 0 ? qi - window + 1 : 0;
        hi = qi + 1;
    }
    const int64_t nkeys = P + end - base;
    auto key_of = [&](int64_t j) { return j < P ? j : base + (j - P); };
    auto allowed = [&](int64_t j) {
        if (!live || j >= nkeys) return false;
        if (j < P) return !pad || ((pad[j >> 6] >> (j & 63)) & 1ull) == 0ull;
        const int64_t key = key_of(j);
        return key >= lo && key < hi;
    };
    // Staging: TPR threads a row, thread t % TPR its 16-byte chunks t % TPR,
    // + TPR, ...
    constexpr int TPR = 64 * kAttnQ / KC;
    constexpr int NV = 16 * HS / TPR;
    const int srow = threadIdx.x / TPR, sch = threadIdx.x % TPR;
    f32x4_t pre[NV];
    auto fetch = [&](const float* src, int64_t c0) {
        const int64_t j = c0 + srow < nkeys ? c0 + srow : nkeys - 1;
        const float* r = src + key_of(j) * kv_stride;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (4 * (sch + TPR * i) < hd) pre[i] = *(const f32x4_t*)(r + 4 * (sch + TPR * i));
    };
    auto stage = [&]() {
        __syncthreads();  // every wavefront is past the rows staged before
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (4 * (sch + TPR * i) < hd)
                *(f32x4_t*)(rows + srow * ld + 4 * (sch + TPR * i)) = pre[i];
        __syncthreads();
    };
    // Scores of keys [p0, p1) into sc (masked: -inf); returns the maximum of
    // each lane's own keys. The first KC keys are already fetched; the first
    // values are fetched under the last keys' products.
    auto scores = [&](int64_t p0, int64_t p1) {
        float m = -INFINITY;
        for (int64_t c0 = p0; c0 < p1; c0 += KC) {
            stage();
            if (c0 + KC < p1)
                fetch(kbase, c0 + KC);
            else
                fetch(vbase, p0);
            bool ok[KC / 64];
            float s[KC / 64];
#pragma unroll
            for (int u = 0; u < KC / 64; ++u) {
                ok[u] = allowed(c0 + 64 * u + lane);
                s[u] = 0.0f;
            }
            const float* kr = rows + lane * ld;
            const float* qr = qs + wave * hd;
#pragma unroll 4
            for (int d = 0; d < hd; d += 4) {
                const f32x4_t q4 = *(const f32x4_t*)(qr + d);
#pragma unroll
                for (int u = 0; u < KC / 64; ++u) {
                    const f32x4_t k4 = *(const f32x4_t*)(kr + 64 * u * ld + d);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[u] = s[u] + q4[e] * k4[e];
                }
            }
#pragma unroll
            for (int u = 0; u < KC / 64; ++u) {
                const float t = ok[u] ? s[u] * scale : -INFINITY;
                sc[c0 - p0 + 64 * u + lane] = t;
                m = fmaxf(m, t);
            }
        }
        return m;
    };

    if (nkeys <= 0) {  // the whole workgroup
        if (live)
            for (int d = lane; d < hd; d += 64)
                out[(b * T + qi) * out_stride + (int64_t)h * hd + d] = 0.0f;
        return;
    }
    const bool once = nkeys <= panel;
    float m = -INFINITY;
    for (int64_t p0 = 0; p0 < nkeys; p0 += panel) {
        fetch(kbase, p0);
        m = fmaxf(m, scores(p0, p0 + panel < nkeys ? p0 + panel : nkeys));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    // The sum, in key order (a masked key adds 0, which changes no bit).
    float sum = 0.0f;
    for (int64_t p0 = 0; p0 < nkeys; p0 += panel) {
        const int64_t p1 = p0 + panel < nkeys ? p0 + panel : nkeys;
        if (!once) {
            fetch(kbase, p0);
            scores(p0, p1);
        }
        const int n = (int)(p1 - p0);
        wave_lds_fence();
        for (int j = lane; j < ((n + 63) & ~63); j += 64) {
            const float s = sc[j];
            sc[j] = allowed(p0 + j) ? expf(s - m) : 0.0f;
        }
        wave_lds_fence();
#pragma unroll 4
        for (int j = 0; j < n; j += 4) {  // past n: zeros
            const f32x4_t e = *(const f32x4_t*)(sc + j);
            sum = sum + e[0];
            sum = sum + e[1];
            sum = sum + e[2];
            sum = sum + e[3];
        }
    }
    // Probabilities and the context, lane = dimension.
    float acc[HS];
#pragma unroll
    for (int s = 0; s < HS; ++s) acc[s] = 0.0f;
    for (int64_t p0 = 0; p0 < nkeys; p0 += panel) {
        const int64_t p1 = p0 + panel < nkeys ? p0 + panel : nkeys;
        if (!once) {
            fetch(kbase, p0);
            scores(p0, p1);
        }
        const int n = (int)(p1 - p0);
        wave_lds_fence();
        for (int j = lane; j < ((n + 63) & ~63); j += 64) {
            const float s = sc[j];
            sc[j] = (once ? s : expf(s - m)) / sum;
        }
        for (int64_t c0 = p0; c0 < p1; c0 += 64) {
            const int half = (int)(c0 - p0) % KC;
            if (half == 0) {
                stage();
                if (c0 + KC < p1) fetch(vbase, c0 + KC);
            }
            // No finite maximum: every probability is 0 (root.zig:563-565).
            uint64_t okm = m == -INFINITY ? 0ull : __ballot(allowed(c0 + lane));
            const float* pr = sc + (c0 - p0);
            const float* vr = rows + half * ld + lane;
            if (okm == ~0ull) {
#pragma unroll 4
                for (int j = 0; j < 64; j += 4) {
                    const f32x4_t p4 = *(const f32x4_t*)(pr + j);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int s = 0; s < HS; ++s)
                            acc[s] = acc[s] + p4[e] * vr[(j + e) * ld + 64 * s];
                }
                continue;
            }
            // Some keys masked: four at a time, a masked one leaves acc alone.
            for (int j = 0; j < 64; j += 4) {
                const uint32_t ok4 = (uint32_t)(okm >> j) & 15u;
                if (!ok4) continue;
                const f32x4_t p4 = *(const f32x4_t*)(pr + j);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int s = 0; s < HS; ++s) {
                        const float t = acc[s] + p4[e] * vr[(j + e) * ld + 64 * s];
                        acc[s] = (ok4 >> e) & 1u ? t : acc[s];
                    }
            }
        }
    }
    if (!live) return;
    float* orow = out + (b * T + qi) * out_stride + (int64_t)h * hd;
#pragma unroll
    for (int s = 0; s < HS; ++s) {
        const int d = s * 64 + lane;
        if (d < hd) orow[d] = acc[s];
    }
}

template <int HS, int KC>
hipError_t launch_attention_f32_t(const float* q, const float* k, const float* v, float* out,
                                  int64_t batch, int64_t T, int q_heads, int kv_heads, int hd,
                                  int64_t q_stride, int64_t kv_stride, int64_t out_stride,
                                  int64_t window, int64_t prefix, const int32_t* seg_lo,
                                  const int32_t* seg_hi, const uint64_t* pad, hipStream_t st) {
    auto kern = attention_f32_kernel<HS, KC>;
    // A lane past hd reads up to 64 HS - hd floats beyond its row: the query
    // and score arrays that follow the staged rows hold them.
    constexpr int max_hd = 64 * HS;
    constexpr int max_lds =
        4 * (KC * (max_hd + 4) + kAttnQ * max_hd + kAttnQ * (kAttnPanel + 4));
    static_assert(max_lds <= 160 * 1024, "LDS budget of a gfx950 CU");
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
    if (attr != hipSuccess) return attr;
    const int64_t padded = (T + KC - 1) / KC * KC;
    const int panel = padded < kAttnPanel ? (int)padded : kAttnPanel;
    const size_t lds = 4 * (size_t)(KC * (hd + 4) + kAttnQ * hd + kAttnQ * (panel + 4));
    const dim3 grid((unsigned)((T + kAttnQ - 1) / kAttnQ), (unsigned)q_heads, (unsigned)batch);
    hipLaunchKernelGGL(kern, grid, dim3(64 * kAttnQ), lds, st, q, k, v, out, T,
                       q_heads / kv_heads, hd, q_stride, kv_stride, out_stride, window,
                       1.0f / sqrtf((float)hd), prefix, seg_lo, seg_hi, pad, panel);
    return hipGetLastError();
}

hipError_t launch_attention_f32(const float* q, const float* k, const float* v, float* out,
                                int64_t batch, int64_t T, int q_heads, int kv_heads, int hd,
                                int64_t q_stride, int64_t kv_stride, int64_t out_stride,
                                int64_t window, int64_t prefix, const int32_t* seg_lo,
                                const int32_t* seg_hi, const uint64_t* pad, hipStream_t st) {
    if (window >= T) window = 0;
#define NCM_ATTN(HS, KC)                                                                       \
    return launch_attention_f32_t<HS, KC>(q, k, v, out, batch, T, q_heads, kv_heads, hd, q_stride, \
                                      kv_stride, out_stride, window, prefix, seg_lo, seg_hi,   \
                                      pad, st)
    if (hd <= 64) NCM_ATTN(1, 128);
    if (hd <= 128) NCM_ATTN(2, 128);
    if (hd <= kAttnF32MaxHd) NCM_ATTN(4, 64);
#undef NCM_ATTN
    return hipErrorInvalidValue;
}

struct PlanF32 {
    int64_t T, q_w, kv_w;
    size_t o_hidden, o_normed, o_q, o_k, o_v, o_ctx, o_proj, o_gate, o_up, o_ids, total;
};

size_t up256(size_t v) { return (v + 255) & ~size_t(255); }

PlanF32 plan_f32(const ncm_decoder_shape_t& s, int64_t batch, int64_t seq) {
    PlanF32 p;
    p.T = batch * seq;
    p.q_w = (int64_t)s.q_heads * s.head_dim;
    p.kv_w = (int64_t)s.kv_heads * s.head_dim;
    size_t off = 0;
    auto carve = [&](size_t bytes) { const size_t o = off; off += up256(bytes); return o; };
    p.o_hidden = carve((size_t)p.T * s.hidden * 4);
    p.o_normed = carve((size_t)p.T * s.hidden * 4);
    p.o_q = carve((size_t)p.T * p.q_w * 4);
    p.o_k = carve((size_t)p.T * p.kv_w * 4);
    p.o_v = carve((size_t)p.T * p.kv_w * 4);
    p.o_ctx = carve((size_t)p.T * p.q_w * 4);
    p.o_proj = carve((size_t)p.T * s.hidden * 4);
    p.o_gate = carve((size_t)p.T * s.intermediate * 4);
    p.o_up = carve((size_t)p.T * s.intermediate * 4);
    p.o_ids = carve((size_t)p.T * 8);
    p.total = off;
    return p;
}

#define NCM_TRY(call)                                  \
    do {                                               \
        hipError_t e_ = (call);                        \
        if (e_ != hipSuccess) return e_;               \
    } while (0)

// Copies one stage [T, width] into trace layer `layer` (layer-major).
hipError_t trace_copy(float* dst, int layer, const float* src, int64_t T, int64_t width,
                      hipStream_t st) {
    if (!dst) return hipSuccess;
    const size_t bytes = (size_t)T * width * 4;
    return hipMemcpyAsync(dst + (int64_t)layer * T * width, src, bytes,
                          hipMemcpyDeviceToDevice, st);
}

}  // namespace

hipError_t launch_add_f32(float* y, const float* a, int64_t rows, int64_t n, int64_t a_rows,
                          hipStream_t st) {
    const int64_t total = rows * n;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(add_f32_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, y,
                       a, rows, n, a_rows);
    return hipGetLastError();
}

// y [rows, n] = x [rows, k] w^T (+ bias), f32.
hipError_t project_f32(const float* x, const float* w, const float* bias, float* y, int64_t rows,
                       int64_t k, int64_t n, hipStream_t st) {
    if (linear_slice_f32_fits(rows, n, k)) {
        LinearF32 l{};
        l.x = x; l.w = w; l.bias = bias; l.y = y;
        l.M = rows; l.K = k; l.N = n;
        return launch_linear_slice_f32(l, st);
    }
    NCM_TRY(launch_linear_f32(x, w, y, rows, k, n, st));
    if (bias) NCM_TRY(launch_add_f32(y, bias, rows, n, 1, st));
    return hipSuccess;
}

namespace {

// hidden [rows, n] += x [rows, k] w^T (+ bias). traced: the product itself is
// left in proj [rows, n] (scratch otherwise).
hipError_t project_residual_f32(const float* x, const float* w, const float* bias, float* hidden,
                                float* proj, bool traced, int64_t rows, int64_t k, int64_t n,
                                hipStream_t st) {
    if (!traced && linear_slice_f32_fits(rows, n, k)) {
        LinearF32 l{};
        l.x = x; l.w = w; l.bias = bias; l.residual = hidden; l.y = hidden;
        l.M = rows; l.K = k; l.N = n;
        return launch_linear_slice_f32(l, st);
    }
    NCM_TRY(project_f32(x, w, bias, proj, rows, k, n, st));
    return launch_add_f32(hidden, proj, rows, n, rows, st);
}

}  // namespace

hipError_t run_layers_f32(const LayerStackF32& a, hipStream_t st) {
    const ncm_decoder_shape_t& s = *a.shape;
    const int64_t T = a.batch * a.seq, H = s.hidden, I = s.intermediate;
    const int hd = s.head_dim;
    const int64_t q_w = (int64_t)s.q_heads * hd, kv_w = (int64_t)s.kv_heads * hd;
    const ncm_decoder_trace_t none{};
    const ncm_decoder_trace_t& tr = a.trace ? *a.trace : none;
    float *hidden = a.hidden, *normed = a.normed, *q = a.q, *k = a.k, *v = a.v, *ctx = a.ctx;
    float *proj = a.proj, *gate = a.gate, *up = a.up;
    for (int l = 0; l < s.layers; ++l) {
        const ncm_decoder_layer_f32_t& L = a.layers[l];
        NCM_TRY(launch_rms_norm_rows(hidden, L.input_norm, normed, T, H, s.rms_eps, NCM_OUT_F32,
                                     st));
        if (L.input_norm_bias) NCM_TRY(launch_add_f32(normed, L.input_norm_bias, T, H, 1, st));
        NCM_TRY(trace_copy(tr.input_norm, l, normed, T, H, st));
        const float* bq = L.qkv_bias;
        const int64_t rot = q_w + kv_w, qkv_w = rot + kv_w;
        if (linear_slice_f32_fits(T, qkv_w, H)) {
            // One product over the concatenated rows, split into q, k and v as
            // it is stored; 64-wide heads are rotated on the way.
            const bool rope = hd == 64 && !L.q_norm;
            LinearF32 m{};
            m.x = normed; m.w = L.qkv_weight; m.bias = bq; m.y = q;
            m.M = T; m.K = H; m.N = qkv_w;
            m.y1 = k; m.y2 = v; m.n1 = q_w; m.n2 = rot;
            if (rope) {
                m.cosine = a.cosine; m.sine = a.sine;
                m.seq_len = a.seq; m.rot_cols = rot;
            }
            NCM_TRY(launch_linear_slice_f32(m, st));
        } else {
            const float* wk = L.qkv_weight + q_w * H;
            const float* wv = wk + kv_w * H;
            NCM_TRY(project_f32(normed, L.qkv_weight, bq, q, T, H, q_w, st));
            NCM_TRY(project_f32(normed, wk, bq ? bq + q_w : nullptr, k, T, H, kv_w, st));
            NCM_TRY(project_f32(normed, wv, bq ? bq + rot : nullptr, v, T, H, kv_w, st));
        }
        if (L.q_norm) {  // QK-norm (f32 rms_norm of every head) before the rotation
            NCM_TRY(launch_rms_norm_rows(q, L.q_norm, q, T * s.q_heads, hd, s.rms_eps,
                                         NCM_OUT_F32, st));
            NCM_TRY(launch_rms_norm_rows(k, L.k_norm, k, T * s.kv_heads, hd, s.rms_eps,
                                         NCM_OUT_F32, st));
        }
        if (hd != 64 || L.q_norm || !linear_slice_f32_fits(T, qkv_w, H)) {
            NCM_TRY(launch_rope_rotate_f32(q, T, q_w, s.q_heads, hd, a.seq, a.cosine, a.sine, st));
            NCM_TRY(launch_rope_rotate_f32(k, T, kv_w, s.kv_heads, hd, a.seq, a.cosine, a.sine,
                                           st));
        }
        NCM_TRY(launch_attention_f32(q, k, v, ctx, a.batch, a.seq, s.q_heads, s.kv_heads, hd, q_w,
                                     kv_w, q_w, a.seg_lo ? 0 : s.window, a.prefix, a.seg_lo,
                                     a.seg_hi, a.pad, st));
        NCM_TRY(trace_copy(tr.attention_context, l, ctx, T, q_w, st));
        NCM_TRY(project_residual_f32(ctx, L.o_weight, L.o_bias, hidden, proj, tr.attention_output,
                                     T, q_w, H, st));
        NCM_TRY(trace_copy(tr.attention_output, l, proj, T, H, st));
        NCM_TRY(trace_copy(tr.attention_residual, l, hidden, T, H, st));
        NCM_TRY(launch_rms_norm_rows(hidden, L.post_attention_norm, normed, T, H, s.rms_eps,
                                     NCM_OUT_F32, st));
        if (L.post_attention_norm_bias)
            NCM_TRY(launch_add_f32(normed, L.post_attention_norm_bias, T, H, 1, st));
        NCM_TRY(trace_copy(tr.post_attention_norm, l, normed, T, H, st));
        if (!tr.gate_projection && !tr.up_projection && linear_slice_f32_fits(T, I, H)) {
            NCM_TRY(launch_linear_slice_swiglu_f32(normed, L.gate_weight, L.up_weight,
                                                   L.gate_bias, L.up_bias, gate, T, H, I, st));
        } else {
            NCM_TRY(project_f32(normed, L.gate_weight, L.gate_bias, gate, T, H, I, st));
            NCM_TRY(trace_copy(tr.gate_projection, l, gate, T, I, st));
            NCM_TRY(project_f32(normed, L.up_weight, L.up_bias, up, T, H, I, st));
            NCM_TRY(trace_copy(tr.up_projection, l, up, T, I, st));
            NCM_TRY(launch_silu_mul(gate, up, gate, T * I, NCM_OUT_F32, st));
        }
        NCM_TRY(trace_copy(tr.gate_up_product, l, gate, T, I, st));
        NCM_TRY(project_residual_f32(gate, L.down_weight, L.down_bias, hidden, proj,
                                     tr.mlp_output, T, I, H, st));
        NCM_TRY(trace_copy(tr.mlp_output, l, proj, T, H, st));
        NCM_TRY(trace_copy(tr.block_output, l, hidden, T, H, st));
    }
    return hipSuccess;
}

size_t decoder_f32_workspace_bytes(const ncm_decoder_shape_t& s, int64_t batch, int64_t seq) {
    return plan_f32(s, batch, seq).total;
}

hipError_t decoder_forward_f32(const ncm_decoder_shape_t& s, const ncm_decoder_layer_f32_t* layers,
                               const float* embed, const float* final_norm, const float* lm_head,
                               const float* cosine, const float* sine, const int64_t* host_ids,
                               int64_t batch, int64_t seq, float* logits,
                               const ncm_decoder_trace_t* trace, void* ws, hipStream_t st) {
    const PlanF32 p = plan_f32(s, batch, seq);
    char* w = (char*)ws;
    float* hidden = (float*)(w + p.o_hidden);
    float* normed = (float*)(w + p.o_normed);
    float* q = (float*)(w + p.o_q);
    float* k = (float*)(w + p.o_k);
    float* v = (float*)(w + p.o_v);
    float* ctx = (float*)(w + p.o_ctx);
    float* proj = (float*)(w + p.o_proj);
    float* gate = (float*)(w + p.o_gate);
    float* up = (float*)(w + p.o_up);
    int64_t* ids = (int64_t*)(w + p.o_ids);
    const int64_t T = p.T, H = s.hidden;
    const ncm_decoder_trace_t none{};
    const ncm_decoder_trace_t& tr = trace ? *trace : none;

    NCM_TRY(hipMemcpyAsync(ids, host_ids, (size_t)T * 8, hipMemcpyHostToDevice, st));
    {
        const dim3 grid((unsigned)((H + 255) / 256 < 64 ? (H + 255) / 256 : 64), (unsigned)T);
        hipLaunchKernelGGL(embed_rows_f32_kernel, grid, dim3(256), 0, st, ids, embed, hidden, H);
        NCM_TRY(hipGetLastError());
    }
    NCM_TRY(trace_copy(tr.block_input, 0, hidden, T, H, st));
    LayerStackF32 a{};
    a.shape = &s;
    a.layers = layers;
    a.batch = batch;
    a.seq = seq;
    a.cosine = cosine;
    a.sine = sine;
    a.hidden = hidden; a.normed = normed; a.q = q; a.k = k; a.v = v; a.ctx = ctx;
    a.proj = proj; a.gate = gate; a.up = up;
    a.trace = trace;
    NCM_TRY(run_layers_f32(a, st));
    NCM_TRY(launch_rms_norm_rows(hidden, final_norm, normed, T, H, s.rms_eps, NCM_OUT_F32, st));
    NCM_TRY(launch_linear_f32(normed, lm_head ? lm_head : embed, logits, T, H, s.vocab, st));
    return hipSuccess;
}

}  // namespace ncm
