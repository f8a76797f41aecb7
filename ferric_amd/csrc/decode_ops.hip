// The steps either side of the quantized matmuls in one decode layer, gfx950: RMSNorm (plain and fused with the residual
// add), rotary embedding, the per-head q/k norm + rotary + KV-cache append of a token's fused qkv row in one launch, the
// KV append on its own, and single-query attention over the cache (split over the keys, all query heads of a KV head
// sharing one pass over its keys and values).
//
// Replaces the reference's WGSL kernels RMSNORM / ADD_RMSNORM / ROPE / FUSED_ATTN / FUSED_ATTN_SPLIT / FUSED_ATTN_COMBINE
// (crates/ferric-tensor/src/lib.rs:2018-2074, 2118-2162, 2675-2726 ff.) and `append2` (lib.rs:1379-1398), as
// `Qwen3::attn` / `apply_layer` compose them (crates/ferric-llama/src/qwen3.rs:861-942, 979-1052).
//
// All of this is f32 arithmetic on small vectors: the kernels are launch- and latency-bound (a decode step has one row),
// except attention, which streams the layer's K and V rows once (HBM-bound: 2 * len * n_kv * head_dim * 4 bytes).
#include "common.hpp"

#include <type_traits>
#include "kvblock.hpp"
#include "prompt.hpp"

#include <hip/hip_fp16.h>

#include <math.h>

namespace {

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float v) {
    int t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xF, false);
    return v + __int_as_float(t);
}
// Sum over the 64 lanes of a wave, returned in every lane (through lane 63 and a scalar register).
__device__ __forceinline__ float wave_sum(float v) {
    v = dpp_add<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
    v = dpp_add<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
    v = dpp_add<0x141, 0xF>(v);  // row_half_mirror
    v = dpp_add<0x140, 0xF>(v);  // row_mirror: every lane of a 16-lane row holds the row sum
    v = dpp_add<0x142, 0xA>(v);  // row_bcast15 into rows 1 and 3
    v = dpp_add<0x143, 0xC>(v);  // row_bcast31 into rows 2 and 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// ---------------------------------------------------------------- RMSNorm, optionally of a + b
// out[r, j] = x[r, j] * (1 / sqrt(mean_j x^2 + eps)) * weight[j]   (lib.rs:2018-2033); with b: x = a + b, and the sum is
// written too (lib.rs:2057-2074). TPR threads share a row (a fixed-shape tree sum, so results do not depend on scheduling).
// Out = uint16_t: the normed rows as bf16, rounded as fhip_cvt_f32_bf16 rounds them -- what the matrix cores read, for a prompt: a
// launch and a trip of the f32 rows through memory less per matmul. count: a word that gets `by` more beside the rows, a decode step's position, whose own launch
// cost 2.5 us a token (null: none): eight layers behind 128 rows 634.4 -> 630.1 us a token, with the weights' trip under the row's.
// AHEAD: the weights are requested with the row and held, which takes their trip out of a workgroup's chain, and up to 32 registers (norm_ahead).
using fhip::pk_bf16;
__device__ __forceinline__ void store_norm(float* out, size_t j, float4 v) { ((float4*)out)[j] = v; }
__device__ __forceinline__ void store_norm(uint16_t* out, size_t j, float4 v) { ((uint2*)out)[j] = make_uint2(pk_bf16(v.x, v.y), pk_bf16(v.z, v.w)); }
__device__ __forceinline__ void store_norm(float* out, size_t j, float v) { out[j] = v; }
__device__ __forceinline__ void store_norm(uint16_t* out, size_t j, float v) { out[j] = (uint16_t)(pk_bf16(v, 0.f) & 0xFFFFu); }
template <int TPR, typename Out, bool AHEAD>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const float* a, const float* __restrict__ b,
                                                      const float* __restrict__ weight, size_t rows, int d, float eps,
                                                      float* sum_out, Out* __restrict__ norm_out, uint32_t* count, uint32_t by) {   // sum_out may be a
    if (count && blockIdx.x == 0 && threadIdx.x == 0) *count += by;
    constexpr int RPW = 256 / TPR;   // rows per workgroup
    constexpr int NV = 8;            // float4 per thread held in registers: rows up to 4 * NV * TPR values
    __shared__ float red[4];
    const int tid = threadIdx.x, sub = tid / TPR, t = tid % TPR;
    const size_t row = (size_t)blockIdx.x * RPW + sub;
    const bool live = row < rows;
    const size_t base = (live ? row : 0) * (size_t)d;
    const bool vec = (d & 3) == 0 && d <= 4 * NV * TPR && (((uintptr_t)a | (uintptr_t)b | (uintptr_t)weight | (uintptr_t)sum_out | (uintptr_t)norm_out) & 15) == 0;
    float ms = 0.f;
    if (vec) {
        // every load of the row is issued before the first use, so the row costs one memory round trip, not one per element (and, AHEAD, the weights none behind the sum)
        const int nv = d >> 2;
        float4 r[NV], w[AHEAD ? NV : 1];
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int j = t + i * TPR;
            r[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (j < nv) {
                r[i] = ((const float4*)(a + base))[j];
                if constexpr (AHEAD) w[i] = ((const float4*)weight)[j];
                if (b) { const float4 y = ((const float4*)(b + base))[j]; r[i].x += y.x; r[i].y += y.y; r[i].z += y.z; r[i].w += y.w; }
            }
        }
        if constexpr (AHEAD) asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < NV; i++) ms = fmaf(r[i].x, r[i].x, fmaf(r[i].y, r[i].y, fmaf(r[i].z, r[i].z, fmaf(r[i].w, r[i].w, ms))));
        ms = wave_sum(ms);
        if (TPR == 256) {
            if ((tid & 63) == 0) red[tid >> 6] = ms;
            __syncthreads();
            ms = (red[0] + red[1]) + (red[2] + red[3]);
        }
        const float inv = 1.0f / sqrtf(ms / (float)d + eps);
        if (!live) return;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int j = t + i * TPR;
            if (j < nv) {
                const float4 wi = AHEAD ? w[AHEAD ? i : 0] : ((const float4*)weight)[j];
                if (sum_out) ((float4*)(sum_out + base))[j] = r[i];
                store_norm(norm_out + base, (size_t)j, make_float4(r[i].x * inv * wi.x, r[i].y * inv * wi.y, r[i].z * inv * wi.z, r[i].w * inv * wi.w));
            }
        }
        return;
    }
    const float* xa = a + base;
    const float* xb = b ? b + base : nullptr;
    for (int j = t; j < d; j += TPR) {
        float v = xb ? xa[j] + xb[j] : xa[j];
        if (sum_out && live) sum_out[base + j] = v;
        ms = fmaf(v, v, ms);
    }
    ms = wave_sum(ms);
    if (TPR == 256) {
        if ((tid & 63) == 0) red[tid >> 6] = ms;
        __syncthreads();
        ms = (red[0] + red[1]) + (red[2] + red[3]);
    }
    const float inv = 1.0f / sqrtf(ms / (float)d + eps);
    if (!live) return;
    for (int j = t; j < d; j += TPR) {   // the same thread wrote sum_out[.., j] above, so reading it back is ordered
        float v = sum_out ? sum_out[base + j] : (xb ? xa[j] + xb[j] : xa[j]);
        store_norm(norm_out, base + j, v * inv * weight[j]);
    }
}

__global__ void u32_add_kernel(uint32_t* w, size_t n, uint32_t delta) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) w[i] += delta;
}

__global__ void add_kernel(const float* a, const float* __restrict__ b, size_t n, float* out, uint32_t* count, uint32_t by) {   // out may be a
    if (count && blockIdx.x == 0 && threadIdx.x == 0) *count += by;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] + b[i];
}

// out = a * sigmoid(g): the gate of a gated attention layer on the attention output (crates/ferric-llama/src/qwen3.rs:936-938;
// sigmoid as crates/ferric-tensor/src/lib.rs:1915, 1 / (1 + exp(-v)))
__global__ void mul_sigmoid_kernel(const float* a, const float* __restrict__ g, size_t n, float* out) {   // out may be a
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] * (1.0f / (1.0f + expf(-g[i])));
}

// out[r, j] = gelu_tanh(gu[r, j]) * gu[r, d + j] for rows [gate | up] of 2 d values: the GEGLU of qwen3.rs:953-958 with the
// tanh-approximated GELU of lib.rs:1926, 0.5 v (1 + tanh(clamp(0.79788456 (v + 0.044715 v^3), -15, 15)))
__global__ void geglu_kernel(const float* __restrict__ gu, size_t n, size_t d, float* __restrict__ out) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t r = i / d, j = i - r * d;
    const float v = gu[r * 2 * d + j], u = gu[r * 2 * d + d + j];
    float a = 0.7978845608028654f * (v + 0.044715f * v * v * v);
    a = fminf(fmaxf(a, -15.0f), 15.0f);
    out[i] = 0.5f * v * (1.0f + tanhf(a)) * u;
}

// ---------------------------------------------------------------- rotary embedding
// Pair c of a head rotates by angle pos * base^(-2c / n_rot) (times freq_scale[c]); partners are (c, c + n_rot/2) in the
// split-half layout and (2c, 2c + 1) interleaved; dims >= n_rot pass through (lib.rs:2118-2162, 2094-2116). The inverse
// frequency is evaluated in f64 and rounded to f32 once, the angle is the f32 product the reference forms.
// rate = -2 / n_rot * log(base) is the host's: the division and the logarithm in f64 were most of what a lane did for its pair.
__device__ __forceinline__ float rope_inv_freq(int c, double rate, const float* freq_scale) {
    const float inv = (float)exp((double)c * rate);
    return freq_scale ? inv * freq_scale[c] : inv;
}
// a pair after its rotation; which product is rounded is written out, so that every kernel that post-processes a head has the same bits
__device__ __forceinline__ float rot_lo(float x1, float x2, float cs, float sn) { return fmaf(x1, cs, -(x2 * sn)); }
__device__ __forceinline__ float rot_hi(float x1, float x2, float cs, float sn) { return fmaf(x1, sn, x2 * cs); }
inline double rope_rate(int n_rot, float base) { return n_rot > 0 ? -2.0 / (double)n_rot * log((double)base) : 0.0; }

__global__ void rope_kernel(const float* __restrict__ x, size_t src_row_stride, int t, int heads, int hd, int n_rot, double rate,
                            const uint32_t* __restrict__ pos, uint32_t pos_off, const float* __restrict__ freq_scale, int interleaved,
                            float* __restrict__ out) {
    const int half = n_rot / 2, per_head = hd - half;   // work items per head: the pairs, then the pass-through tail
    size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (size_t)t * heads * per_head) return;
    const int w = (int)(id % per_head), head = (int)((id / per_head) % heads), i = (int)(id / ((size_t)per_head * heads));
    const float* xi = x + (size_t)i * src_row_stride + (size_t)head * hd;
    float* oi = out + ((size_t)i * heads + head) * hd;
    if (w >= half) { const int c = n_rot + (w - half); oi[c] = xi[c]; return; }
    const int c = w;
    const float p = (float)(pos ? pos[i] : pos_off + (uint32_t)i);
    const float ang = p * rope_inv_freq(c, rate, freq_scale);
    float sn, cs;
    sincosf(ang, &sn, &cs);
    const int p0 = interleaved ? 2 * c : c, p1 = interleaved ? 2 * c + 1 : c + half;
    const float x1 = xi[p0], x2 = xi[p1];
    oi[p0] = x1 * cs - x2 * sn;
    oi[p1] = x2 * cs + x1 * sn;
}

// ---------------------------------------------------------------- qkv row -> q, K cache, V cache
// One wave per head of one token's fused qkv row (n_head query heads, n_kv key heads, n_kv value heads):
//   query / key head: + bias, RMSNorm over the head with q_norm / k_norm (when given), rotary embedding at the token's position;
//   the query goes to q_out[t, n_head * hd], the key to row pos of the K cache; a value head is copied (+ bias) to row pos of
//   the V cache. This is qwen3.rs:861-905 (qn, rope, append2) in one launch.
struct QkvPostParams {
    const float* qkv;        // [t, (n_head + 2 n_kv) * hd]
    const float* bias;       // same width, or null
    const float* q_norm;     // [hd] or null
    const float* k_norm;     // [hd] or null
    const uint32_t* pos;     // [t] absolute positions (device)
    const float* freq_scale; // [n_rot / 2] or null
    float* q_out;            // [t, n_head * hd]
    float* k_cache;          // [cap, n_kv * hd]
    float* v_cache;
    int t, n_head, n_kv, hd, n_rot, interleaved;
    uint32_t cap;
    float eps;
    double rate;             // rope_rate(n_rot, base)
    int kv_packed;           // != 0: k_cache / v_cache are packed [t, n_kv * hd] outputs, row i for token i (cap is not looked at)
};

__global__ __launch_bounds__(256) void qkv_post_kernel(QkvPostParams p) {
    const int lane = threadIdx.x & 63;
    const int per_tok = p.n_head + 2 * p.n_kv;
    const size_t wid = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wid >= (size_t)p.t * per_tok) return;
    const int i = (int)(wid / per_tok), h = (int)(wid % per_tok);
    const uint32_t pos = p.pos[i];
    const size_t col = (size_t)h * p.hd;
    const float* x = p.qkv + (size_t)i * per_tok * p.hd + col;
    const float* bias = p.bias ? p.bias + col : nullptr;
    const int kvw = p.n_kv * p.hd;
    float* dst;
    const float* nw;
    bool rotate = true;
    const size_t kv_row = p.kv_packed ? (size_t)i : (size_t)pos;
    if (h < p.n_head) { dst = p.q_out + ((size_t)i * p.n_head + h) * p.hd; nw = p.q_norm; }
    else if (h < p.n_head + p.n_kv) { dst = p.k_cache + kv_row * kvw + (size_t)(h - p.n_head) * p.hd; nw = p.k_norm; }
    else { dst = p.v_cache + kv_row * kvw + (size_t)(h - p.n_head - p.n_kv) * p.hd; nw = nullptr; rotate = false; }
    if (h >= p.n_head && !p.kv_packed && pos >= p.cap) return;   // a position past the cache is dropped, never written out of bounds
    if (!rotate) {
        for (int j = lane; j < p.hd; j += 64) dst[j] = bias ? x[j] + bias[j] : x[j];
        return;
    }
    float inv = 1.f;
    if (nw) {
        float ms = 0.f;
        for (int j = lane; j < p.hd; j += 64) { float v = bias ? x[j] + bias[j] : x[j]; ms = fmaf(v, v, ms); }
        ms = wave_sum(ms);
        inv = 1.0f / sqrtf(ms / (float)p.hd + p.eps);
    }
    auto val = [&](int j) { float v = bias ? x[j] + bias[j] : x[j]; return nw ? v * inv * nw[j] : v; };
    const int half = p.n_rot / 2;
    for (int c = lane; c < half; c += 64) {
        const float ang = (float)pos * rope_inv_freq(c, p.rate, p.freq_scale);
        float sn, cs;
        sincosf(ang, &sn, &cs);
        const int p0 = p.interleaved ? 2 * c : c, p1 = p.interleaved ? 2 * c + 1 : c + half;
        const float x1 = val(p0), x2 = val(p1);
        dst[p0] = rot_lo(x1, x2, cs, sn);
        dst[p1] = rot_hi(x1, x2, cs, sn);
    }
    for (int j = p.n_rot + lane; j < p.hd; j += 64) dst[j] = val(j);
}

// The same operations for heads of 64 or 128 dims rotated whole in the split-half layout, the common case. Of 128 a lane's two values are a pair, of 64 it has
// one, whose pair is 32 lanes away, so a head is read once and nothing is read again. A wave takes HPW consecutive heads of a token, requests them all before the
// first is worked on, and works the token's angles out once for them. The one-head form above paid, per head, three round trips in a row (the squares,
// the pair again, the weights) and the f64 exponential: 509 rows of 40 + 8 + 8 heads of 128 (29 MB) 19.2 us, here 7.6; 435 rows of 64 + 8 + 8 of 64 12.9 -> 8.3,
// 1016 of 8 + 8 + 8 8.9 -> 6.5.
template <int HD, int HPW>
__global__ __launch_bounds__(256) void qkv_post_heads_kernel(QkvPostParams p) {
    constexpr int E = HD / 64;
    const int lane = threadIdx.x & 63;
    const int per_tok = p.n_head + 2 * p.n_kv, waves_per_tok = (per_tok + HPW - 1) / HPW;
    const size_t wid = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wid >= (size_t)p.t * waves_per_tok) return;
    const int i = (int)(wid / waves_per_tok), h0 = (int)(wid % waves_per_tok) * HPW;
    const float* x = p.qkv + ((size_t)i * per_tok + h0) * HD + lane;
    float a[HPW][E];
#pragma unroll
    for (int j = 0; j < HPW; j++)
#pragma unroll
        for (int e = 0; e < E; e++) a[j][e] = x[(h0 + j < per_tok ? HD * j : 0) + 64 * e];
    const uint32_t pos = p.pos[i];
    float wq[E], wk[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        wq[e] = p.q_norm ? p.q_norm[lane + 64 * e] : 1.f;
        wk[e] = p.k_norm ? p.k_norm[lane + 64 * e] : 1.f;
    }
    if (p.bias) {
        const float* bias = p.bias + (size_t)h0 * HD + lane;
#pragma unroll
        for (int j = 0; j < HPW; j++)
#pragma unroll
            for (int e = 0; e < E; e++) a[j][e] += bias[(h0 + j < per_tok ? HD * j : 0) + 64 * e];
    }
    float sn = 0.f, cs = 1.f;
    if (h0 < p.n_head + p.n_kv) sincosf((float)pos * rope_inv_freq(lane & (HD / 2 - 1), p.rate, p.freq_scale), &sn, &cs);
    const bool stored = p.kv_packed || pos < p.cap;              // a position past the cache is dropped, never written out of bounds
    const size_t kv_row = (p.kv_packed ? (size_t)i : (size_t)pos) * p.n_kv;
#pragma unroll
    for (int j = 0; j < HPW; j++) {
        const int h = h0 + j;
        if (h >= per_tok || (h >= p.n_head && !stored)) return;
        const bool value = h >= p.n_head + p.n_kv, key = !value && h >= p.n_head;
        float* dst = value ? p.v_cache + (kv_row + (h - p.n_head - p.n_kv)) * HD
                           : key ? p.k_cache + (kv_row + (h - p.n_head)) * HD : p.q_out + ((size_t)i * p.n_head + h) * HD;
        float v[E];
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = a[j][e];
        if (!value) {
            if (key ? p.k_norm : p.q_norm) {
                const float sq = fmaf(v[E - 1], v[E - 1], E == 2 ? v[0] * v[0] : 0.f);
                const float inv = 1.0f / sqrtf(wave_sum(sq) / (float)HD + p.eps);
#pragma unroll
                for (int e = 0; e < E; e++) v[e] = v[e] * inv * (key ? wk[e] : wq[e]);
            }
            if constexpr (E == 2) {
                const float y1 = rot_lo(v[0], v[1], cs, sn), y2 = rot_hi(v[0], v[1], cs, sn);
                v[0] = y1;
                v[1] = y2;
            } else {
                const float other = __shfl_xor(v[0], 32);
                v[0] = lane < 32 ? rot_lo(v[0], other, cs, sn) : rot_hi(other, v[0], cs, sn);
            }
        }
#pragma unroll
        for (int e = 0; e < E; e++) dst[lane + 64 * e] = v[e];
    }
}

// ---------------------------------------------------------------- qkv row -> q, block-quantized K and V rows
// The post-processing of qkv_post_kernel and the stores of kvq_quant_kernel (kvquant.hip) in one launch, one wave per head: the finished
// key or value row stays in LDS, and the 32 lanes of a block find its scale by exchange and code a value each (the other kernel: one
// thread walks its block). Operation by operation the two launches' arithmetic, so the same bytes. A token of 40 + 8 + 8 heads of
// 128, Q8_0: 5.0 us against 4.7 + 4.4.
constexpr int POST_KVQ_HD = 256;   // head sizes it takes: multiples of 32 up to this
// Over the 32 lanes of a block, all of them active: in the 16 lanes of a row by rotations, then with the other row (in any order the same value).
template <typename Op>
__device__ __forceinline__ float half32(float v, Op op) {
    auto turned = [&](auto ctrl) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xF, 0xF, false)); };
    v = op(v, turned(std::integral_constant<int, 0x128>()));     // row_ror:8, 4, 2, 1
    v = op(v, turned(std::integral_constant<int, 0x124>()));
    v = op(v, turned(std::integral_constant<int, 0x122>()));
    v = op(v, turned(std::integral_constant<int, 0x121>()));
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
}
__device__ __forceinline__ float half32_max(float v) { return half32(v, [](float a, float b) { return fmaxf(a, b); }); }
__device__ __forceinline__ float half32_min(float v) { return half32(v, [](float a, float b) { return fminf(a, b); }); }
__device__ __forceinline__ uint16_t kv_f16_bits(float x) {   // a NaN keeps its sign and top payload bits and stays quiet, as kvquant.hip
    const uint32_t b = __float_as_uint(x);
    if ((b & 0x7F800000u) == 0x7F800000u && (b & 0x007FFFFFu) != 0)
        return (uint16_t)(((b >> 16) & 0x8000u) | 0x7C00u | 0x0200u | ((b & 0x007FFFFFu) >> 13));
    return __half_as_ushort(__float2half_rn(x));
}
__device__ __forceinline__ int kv_code(float r, float lo, float hi) { return r != r ? 0 : (int)fminf(fmaxf(r, lo), hi); }
// lane j of a half wave holds value j of block b (live: the same for the whole half); what its code stands for
template <int FMT>
__device__ __forceinline__ float quantize_lanes(float v, int j, bool live, uint32_t* __restrict__ codes, uint16_t* __restrict__ scales, size_t b) {
#pragma clang fp contract(off)
    if constexpr (FMT == FHIP_KVQ_Q8_0) {
        const float amax = half32_max(fmaxf(0.f, fabsf(v)));
        const float d = amax / 127.0f;
        const float inv = d > 0.f ? 1.0f / d : 0.f;
        const float t = v * inv;
        const float r = copysignf(floorf(fabsf(t) + 0.5f), t);
        const int c = kv_code(r, -127.0f, 127.0f);
        const uint16_t dbits = kv_f16_bits(d);
        if (live) {
            ((uint8_t*)codes)[b * 32 + j] = (uint8_t)c;
            if (j == 0) scales[b] = dbits;
        }
        return fhip::kvq_value<FMT>(c, fhip::kvq_scale(dbits), 0.f);
    } else {
        float d, q;
        uint16_t mbits = 0;
        if constexpr (FMT == FHIP_KVQ_Q4_0) {
            const float a = fabsf(v) > 0.f ? fabsf(v) : 0.f, amax = half32_max(a);          // the value of largest magnitude, the first of equals
            const int half = __lane_id() & 32;
            const uint32_t at = (uint32_t)(__builtin_amdgcn_ballot_w64(a == amax) >> half), neg = (uint32_t)(__builtin_amdgcn_ballot_w64(v < 0.f) >> half);
            const float mx = neg & (at & 0u - at) ? -amax : amax;
            d = mx / -8.0f;
            const float inv = d != 0.f ? 1.0f / d : 0.f;
            q = floorf(v * inv + 8.5f);
        } else {
            const float mn = half32_min(fminf(__builtin_inff(), v)), mx = half32_max(fmaxf(-__builtin_inff(), v));
            d = (mx - mn) / 15.0f;
            const float inv = d != 0.f ? 1.0f / d : 0.f;
            q = floorf((v - mn) * inv + 0.5f);
            mbits = kv_f16_bits(mn);
        }
        const int c = kv_code(q, 0.f, 15.f), c2 = __builtin_amdgcn_permlane16_swap((uint32_t)c, (uint32_t)c, false, false)[1];   // in the lower row the upper one's
        const uint16_t dbits = kv_f16_bits(d);
        if (live) {
            if (j < 16) ((uint8_t*)codes)[b * 16 + j] = (uint8_t)(c | (c2 << 4));
            if (j == 0) {
                if constexpr (FMT == FHIP_KVQ_Q4_0) scales[b] = dbits;
                else { scales[2 * b] = dbits; scales[2 * b + 1] = mbits; }
            }
        }
        return fhip::kvq_value<FMT>(c, fhip::kvq_scale(dbits), fhip::kvq_scale(mbits));
    }
}
struct KvqStore {
    uint32_t* k_codes; uint16_t* k_scales;
    uint32_t* v_codes; uint16_t* v_scales;
};
// The f32 rows that the stored blocks stand for, for an attention that reads those: a token's at its position, and rows 0 .. past - 1 of the caches, which
// `past_wgs` workgroups behind the others bring.
struct KvqRows {
    float *k, *v;            // [n, n_kv * hd]: a token whose position is n or more leaves no row
    uint32_t n, past;
    unsigned post_wgs;       // workgroups in front of those
};
template <int FMT>
__device__ __forceinline__ void past_rows(const KvqStore& st, const KvqRows& rows, int width) {
    const size_t w4 = width / 4, all = rows.past * w4;
    size_t id = (size_t)(blockIdx.x - rows.post_wgs) * 256 + threadIdx.x;
    const bool value = id >= all;
    id -= value ? all : 0;
    if (id >= all) return;
    const size_t i = id / w4;
    const int col = (int)(id - i * w4) * 4;
    const size_t b = i * (size_t)(width / 32) + col / 32;
    const float4 o = value ? fhip::kvq_values4<FMT>(st.v_codes, st.v_scales, b, col % 32) : fhip::kvq_values4<FMT>(st.k_codes, st.k_scales, b, col % 32);
    *(float4*)((value ? rows.v : rows.k) + 4 * id) = o;
}
template <int FMT, bool ROWS>
__global__ __launch_bounds__(256) void qkv_post_kvq_kernel(QkvPostParams p, KvqStore st, KvqRows out) {
    if (ROWS && blockIdx.x >= out.post_wgs) { past_rows<FMT>(st, out, p.n_kv * p.hd); return; }
    constexpr int EPL = POST_KVQ_HD / 64;
    __shared__ float rows[4][2][POST_KVQ_HD];                    // a wave's head: normed, then rotated
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per_tok = p.n_head + 2 * p.n_kv;
    const size_t wid = (size_t)blockIdx.x * 4 + wave;
    if (wid >= (size_t)p.t * per_tok) return;
    const int i = (int)(wid / per_tok), h = (int)(wid % per_tok);
    const float* x = p.qkv + ((size_t)i * per_tok + h) * p.hd;
    const float* bias = p.bias ? p.bias + (size_t)h * p.hd : nullptr;
    const bool is_q = h < p.n_head, is_k = !is_q && h < p.n_head + p.n_kv;
    const float* nw = is_q ? p.q_norm : is_k ? p.k_norm : nullptr;
    // the head, its bias and its norm's weights in one trip to memory
    float v[EPL], w[EPL];
#pragma unroll
    for (int e = 0; e < EPL; e++) {
        const int j = lane + 64 * e;
        v[e] = j < p.hd ? x[j] : 0.f;
        w[e] = nw && j < p.hd ? nw[j] : 1.f;
        if (bias && j < p.hd) v[e] += bias[j];
    }
    const uint32_t pos = p.pos[i];
    if (!is_q && pos >= p.cap) return;                           // a position past the cache is dropped, never written out of bounds
    if (nw) {
        float ms = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; e++)
            if (lane + 64 * e < p.hd) ms = fmaf(v[e], v[e], ms);
        ms = wave_sum(ms);
        const float inv = 1.0f / sqrtf(ms / (float)p.hd + p.eps);
#pragma unroll
        for (int e = 0; e < EPL; e++) v[e] = v[e] * inv * w[e];
    }
    float* const a = rows[wave][0];
    float* const y = rows[wave][1];
#pragma unroll
    for (int e = 0; e < EPL; e++)
        if (lane + 64 * e < p.hd) a[lane + 64 * e] = v[e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");       // the wave's own rows: its accesses complete in order
    if (is_q || is_k) {
        float* const dst = is_q ? p.q_out + ((size_t)i * p.n_head + h) * p.hd : y;
        const int half = p.n_rot / 2;
        for (int c = lane; c < half; c += 64) {
            const float ang = (float)pos * rope_inv_freq(c, p.rate, p.freq_scale);
            float sn, cs;
            sincosf(ang, &sn, &cs);
            const int p0 = p.interleaved ? 2 * c : c, p1 = p.interleaved ? 2 * c + 1 : c + half;
            const float x1 = a[p0], x2 = a[p1];
            dst[p0] = rot_lo(x1, x2, cs, sn);
            dst[p1] = rot_hi(x1, x2, cs, sn);
        }
        for (int j = p.n_rot + lane; j < p.hd; j += 64) dst[j] = a[j];
        if (is_q) return;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const float* const src = is_k ? y : a;
    const int head = h - p.n_head - (is_k ? 0 : p.n_kv);
    const size_t b0 = ((size_t)pos * p.n_kv + head) * (size_t)(p.hd / 32);
    for (int e = 0; e < p.hd; e += 64) {                         // uniform: both halves of the wave take part in the exchanges
        const int j = e + lane;
        const bool live = j < p.hd;
        const float stored = quantize_lanes<FMT>(live ? src[j] : 0.f, lane & 31, live, is_k ? st.k_codes : st.v_codes, is_k ? st.k_scales : st.v_scales, b0 + (size_t)(j >> 5));
        if (ROWS && live && pos < out.n) (is_k ? out.k : out.v)[((size_t)pos * p.n_kv + head) * p.hd + j] = stored;
    }
}

// The same with the rows for heads of 64 or 128 dims rotated whole in the split-half layout, in registers: HD = 128 as qkv_post_heads_kernel holds a head (a lane's two
// values are a pair), HD = 64 a value a lane, its pair's other one 32 lanes away. A wave takes HPW consecutive heads of a token. A prompt's layer on a quantized
// cache was four launches here (post-processing, stores, both caches' rows), 3 - 4 us each; stacks of 42 ... 191 rows, us: 42 x 3584, one layer behind 581 rows 209 -> 195,
// 86 x 3072 298 -> 281, 93 x 1280, four layers 460 -> 424, 139 x 2560, three 565 -> 543; 937 x 4608, four layers, 3081 -> 3071.
template <int FMT, int HD, int HPW>
__global__ __launch_bounds__(256) void qkv_post_rows_kernel(QkvPostParams p, KvqStore st, KvqRows out) {
    constexpr int E = HD / 64;
    if (blockIdx.x >= out.post_wgs) { past_rows<FMT>(st, out, p.n_kv * HD); return; }
    const int lane = threadIdx.x & 63;
    const int per_tok = p.n_head + 2 * p.n_kv, waves_per_tok = (per_tok + HPW - 1) / HPW;
    const size_t wid = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wid >= (size_t)p.t * waves_per_tok) return;
    const int i = (int)(wid / waves_per_tok), h0 = (int)(wid % waves_per_tok) * HPW;
    const float* x = p.qkv + ((size_t)i * per_tok + h0) * HD + lane;
    float a[HPW][E];
#pragma unroll
    for (int j = 0; j < HPW; j++)
#pragma unroll
        for (int e = 0; e < E; e++) a[j][e] = x[(h0 + j < per_tok ? HD * j : 0) + 64 * e];
    const uint32_t pos = p.pos[i];
    float wq[E], wk[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        wq[e] = p.q_norm ? p.q_norm[lane + 64 * e] : 1.f;
        wk[e] = p.k_norm ? p.k_norm[lane + 64 * e] : 1.f;
    }
    if (p.bias) {
        const float* bias = p.bias + (size_t)h0 * HD + lane;
#pragma unroll
        for (int j = 0; j < HPW; j++)
#pragma unroll
            for (int e = 0; e < E; e++) a[j][e] += bias[(h0 + j < per_tok ? HD * j : 0) + 64 * e];
    }
    float sn = 0.f, cs = 1.f;
    if (h0 < p.n_head + p.n_kv) sincosf((float)pos * rope_inv_freq(lane & (HD / 2 - 1), p.rate, p.freq_scale), &sn, &cs);
    const bool stored = pos < p.cap;                             // a position past the cache is dropped, never written out of bounds
#pragma unroll
    for (int j = 0; j < HPW; j++) {
        const int h = h0 + j;
        if (h >= per_tok || (h >= p.n_head && !stored)) return;  // (uniform: a wave has one token)
        const bool value = h >= p.n_head + p.n_kv, key = !value && h >= p.n_head;
        float v[E];
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = a[j][e];
        if (!value) {
            if (key ? p.k_norm : p.q_norm) {
                const float sq = fmaf(v[E - 1], v[E - 1], E == 2 ? v[0] * v[0] : 0.f);   // (a plain product would be fused with the sum's first addition)
                const float inv = 1.0f / sqrtf(wave_sum(sq) / (float)HD + p.eps);
#pragma unroll
                for (int e = 0; e < E; e++) v[e] = v[e] * inv * (key ? wk[e] : wq[e]);
            }
            if constexpr (E == 2) {
                const float y1 = rot_lo(v[0], v[1], cs, sn), y2 = rot_hi(v[0], v[1], cs, sn);
                v[0] = y1;
                v[1] = y2;
            } else {
                const float other = __shfl_xor(v[0], 32);
                v[0] = lane < 32 ? rot_lo(v[0], other, cs, sn) : rot_hi(other, v[0], cs, sn);
            }
        }
        if (h < p.n_head) {
#pragma unroll
            for (int e = 0; e < E; e++) p.q_out[((size_t)i * p.n_head + h) * HD + lane + 64 * e] = v[e];
            continue;
        }
        const size_t at = (size_t)pos * p.n_kv + (h - p.n_head - (value ? p.n_kv : 0));
#pragma unroll
        for (int e = 0; e < E; e++) {
            const float row = quantize_lanes<FMT>(v[e], lane & 31, true, value ? st.v_codes : st.k_codes, value ? st.v_scales : st.k_scales, at * (HD / 32) + 2 * e + (lane >> 5));
            if (pos < out.n) (value ? out.v : out.k)[at * HD + lane + 64 * e] = row;
        }
    }
}

// K and V rows of t tokens into their caches at the tokens' positions, one launch (lib.rs:1379-1398).
__global__ void kv_append_kernel(const float* __restrict__ k, const float* __restrict__ v, int t, int width, const uint32_t* __restrict__ pos,
                                 uint32_t pos_off, uint32_t cap, float* __restrict__ kc, float* __restrict__ vc) {
    size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (size_t)t * width) return;
    const int i = (int)(id / width), j = (int)(id % width);
    const uint32_t r = pos ? pos[i] : pos_off + (uint32_t)i;
    if (r >= cap) return;
    kc[(size_t)r * width + j] = k[id];
    vc[(size_t)r * width + j] = v[id];
}

// ---------------------------------------------------------------- single-query attention over the cache
// out[h] = softmax_j(q[h] . K[j, kv(h)] * scale) @ V[:, kv(h)]   for one query row (nn.rs:140-166, lib.rs:2675-2726).
// Workgroup (kv head, split). A key or value row is read by 16 lanes (DPL = hd / 16 consecutive dims each, 16-byte loads), so a
// wave works on 4 keys at a time and a workgroup is 16 independent key streams, each with its own running (max, sum,
// accumulator) per query head -- the reference's online softmax, lib.rs:2697-2722 -- over keys taken round-robin in pairs.
// Every row is read ONCE for all G = n_head / n_kv query heads of the group. A dot product is reduced inside its 16-lane
// row with 4 DPP adds. The 4 streams of a wave are merged by lane exchange, the 4 waves through LDS, the splits by
// attn_combine_kernel: always the same rescale, exp(m_part - m_all).
constexpr int ATT_KB = 2;         // keys in flight per stream

__device__ __forceinline__ float row16_sum(float v) {   // all 16 lanes of a DPP row get the row's sum
    v = dpp_add<0xB1, 0xF>(v);
    v = dpp_add<0x4E, 0xF>(v);
    v = dpp_add<0x141, 0xF>(v);
    v = dpp_add<0x140, 0xF>(v);
    return v;
}

template <int DPL>
__device__ __forceinline__ void load_dims(const float* p, float (&r)[DPL]) {   // p is 16-byte aligned
#pragma unroll
    for (int i = 0; i < DPL; i += 4) {
        float4 v = *(const float4*)(p + i);
        r[i] = v.x; r[i + 1] = v.y; r[i + 2] = v.z; r[i + 3] = v.w;
    }
}

// A block-quantized cache (kvquant.hip's layout) read in place: codes and f16 scales of the keys and of the values.
struct QCache {
    const uint32_t* k_codes; const uint16_t* k_scales;
    const uint32_t* v_codes; const uint16_t* v_scales;
};
// DPL (4 or 8) consecutive dims of one row, starting at column `col` (a multiple of DPL) of block row `key`: the values the
// dequantize kernel would write, by the same single operations (q * d; (q - 8) * d; q * d then + m, not fused), so attention
// over the codes is attention over the dequantized rows, bit for bit.
// What a lane holds of a row between the load and its use: the code words and scale halves as loaded (the next rows are
// requested while the current ones are worked on, and packed they cost a third of the registers of their f32 values).
template <int FMT, int DPL>
struct RawDims {
    uint32_t w[DPL / 4];
    uint16_t d, m;
};
template <int FMT, int DPL>
__device__ __forceinline__ RawDims<FMT, DPL> fetch_dims_q(const uint32_t* __restrict__ codes, const uint16_t* __restrict__ scales, size_t key,
                                                         int nblk, int col) {
    const size_t b = key * (size_t)nblk + (size_t)(col >> 5);
    const int j = col & 31;
    RawDims<FMT, DPL> r;
    r.m = 0;
    if constexpr (FMT == FHIP_KVQ_Q8_0) {
        r.d = scales[b];
#pragma unroll
        for (int w = 0; w < DPL / 4; w++) r.w[w] = codes[b * 8 + (j >> 2) + w];
    } else {
        if constexpr (FMT == FHIP_KVQ_Q4_0) r.d = scales[b];
        else { r.d = scales[2 * b]; r.m = scales[2 * b + 1]; }
#pragma unroll
        for (int w = 0; w < DPL / 4; w++) r.w[w] = codes[b * 4 + ((j & 15) >> 2) + w];
    }
    return r;
}
// one code word's four dims, scale and minimum as f32
template <int FMT>
__device__ __forceinline__ void expand_dims_f(uint32_t code, int shift, float d, float m, float (&r)[4]) {   // shift: 0 or 4, the 4-bit formats' half
#pragma clang fp contract(off)
    if constexpr (FMT == FHIP_KVQ_Q8_0) {
        r[0] = (float)(int8_t)(code & 255u) * d;
        r[1] = (float)(int8_t)((code >> 8) & 255u) * d;
        r[2] = (float)(int8_t)((code >> 16) & 255u) * d;
        r[3] = (float)(int8_t)(code >> 24) * d;
    } else {
        const uint32_t word = code >> shift;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float n = (float)((word >> (8 * i)) & 15u);
            if constexpr (FMT == FHIP_KVQ_Q4_0) r[i] = (n - 8.0f) * d;
            else { const float t = n * d; r[i] = t + m; }
        }
    }
}
template <int FMT, int DPL>
__device__ __forceinline__ void expand_dims_q(const RawDims<FMT, DPL>& raw, int col, float (&r)[DPL]) {
    const float d = __half2float(__ushort_as_half(raw.d)), m = __half2float(__ushort_as_half(raw.m));
#pragma unroll
    for (int w = 0; w < DPL / 4; w++) {
        float v[4];
        expand_dims_f<FMT>(raw.w[w], ((col + 4 * w) & 31) < 16 ? 0 : 4, d, m, v);
#pragma unroll
        for (int i = 0; i < 4; i++) r[4 * w + i] = v[i];
    }
}

// One head of the newest token's raw QKV row as a wave takes it through qkv_post_kernel's arithmetic: the values (+ bias) and the norm's
// weights in one trip to memory, lane + 64 i each ...
template <int HD>
struct PostHead {
    float x[HD / 64], w[HD / 64];
};
template <int HD>
__device__ __forceinline__ PostHead<HD> post_request(const QkvPostParams& fp, int src, const float* nw, int lane) {
    PostHead<HD> p;
    const float* x = fp.qkv + (size_t)src * HD;
    const float* bias = fp.bias ? fp.bias + (size_t)src * HD : nullptr;
#pragma unroll
    for (int i = 0; i < HD / 64; i++) {
        p.x[i] = bias ? x[lane + 64 * i] + bias[lane + 64 * i] : x[lane + 64 * i];
        p.w[i] = nw ? nw[lane + 64 * i] : 1.f;
    }
    return p;
}
// ... then normed (through `row`, the wave's own HD floats of LDS) and rotated by the lane's pair's angle into dst, LDS or memory.
template <int HD>
__device__ __forceinline__ void post_rotate(const QkvPostParams& fp, const PostHead<HD>& p, bool norm, float cs, float sn, int lane, float* row, float* dst) {
    static_assert(HD <= 128, "a lane rotates one pair");
    float inv = 1.f;
    if (norm) {
        float ms = 0.f;
#pragma unroll
        for (int i = 0; i < HD / 64; i++) ms = fmaf(p.x[i], p.x[i], ms);
        ms = wave_sum(ms);
        inv = 1.0f / sqrtf(ms / (float)HD + fp.eps);
    }
#pragma unroll
    for (int i = 0; i < HD / 64; i++) row[lane + 64 * i] = norm ? p.x[i] * inv * p.w[i] : p.x[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");      // the wave's own row: its accesses complete in order
    const int half = fp.n_rot / 2;
    if (lane < half) {
        const int p0 = fp.interleaved ? 2 * lane : lane, p1 = fp.interleaved ? 2 * lane + 1 : lane + half;
        const float x1 = row[p0], x2 = row[p1];
        dst[p0] = rot_lo(x1, x2, cs, sn);
        dst[p1] = rot_hi(x1, x2, cs, sn);
    }
    for (int e = fp.n_rot + lane; e < HD; e += 64) dst[e] = row[e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// FUSED: the query heads do not come from memory but are formed here from the raw QKV row of the newest token -- bias, per-head
// RMSNorm, rotation, exactly qkv_post_kernel's arithmetic -- by every workgroup for its own G heads, into LDS; and the
// workgroup whose key range holds the token's position also forms that token's K and V rows for its KV head and appends them
// to the cache before it starts on the keys (a store, a workgroup barrier, then the ordinary loop reads the row back like any
// other: no other workgroup's range holds that row). One launch less per layer than post-processing + attention. On a quantized cache (QF) the
// two rows go through LDS and quantize_lanes: 8.7 -> 5.8 us at 64 rows, 12.7 -> 9.9 at 1000, 24.7 -> 21.3 at 20000 (40 query and 8 KV heads of 128, Q8_0).
template <bool FUSED> struct CachePtr { typedef const float* __restrict__ type; };
template <> struct CachePtr<true> { typedef const float* type; };   // the fused kernel also writes the cache: no promise of no alias

// QF: -1 for an f32 cache (K, V), else the FHIP_KVQ_* format of the block-quantized cache in qc (K and V are null then).
// WV: waves of the workgroup. KvqStore (FUSED on a quantized cache): the cache of qc, to append to.
template <int G, int DPL, bool FUSED, int QF = -1, int WV = 4>
__device__ __forceinline__ void attn_split_body(const float* __restrict__ q, typename CachePtr<FUSED>::type K, typename CachePtr<FUSED>::type V,
                                                int n_kv, uint32_t len_host, const uint32_t* __restrict__ len_dev, float scale, int splits,
                                                uint32_t window, float softcap, float* __restrict__ part, float* __restrict__ out,
                                                const QkvPostParams& fp, int gq, const QCache& qc = QCache{}, const KvqStore& qst = KvqStore{}) {
    constexpr int HD = 16 * DPL, ATT_STREAMS = 4 * WV;
    __shared__ float sm_m[WV][G], sm_l[WV][G];
    __shared__ float sm_acc[WV][G][HD];
    __shared__ float sm_q[FUSED ? G : 1][FUSED ? HD : 1];
    __shared__ float sm_row[FUSED ? WV : 1][FUSED ? HD : 1], sm_kv[FUSED && QF >= 0 ? 2 : 1][FUSED && QF >= 0 ? HD : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane & 15;
    const int sid = wave * 4 + (lane >> 4);
    // Workgroup blockIdx.x takes the G query heads from head0 on; gq = query heads per KV head. gq == G: one workgroup per KV
    // head and split. gq > G (short caches, G = 1): one workgroup per query head, the KV head's rows read by each of them.
    // gq < 0 (G = 1, a one-dimensional grid): one workgroup per (query head, split) for -gq query heads per KV head, dealt so
    // that the workgroups of one KV head and split -- which read the same rows -- are consecutive slots of one XCD (workgroup
    // L runs on XCD L % 8): slot i = L / 8 of XCD x = L % 8 is query head i % g of group (i / g) * 8 + x.
    int head0 = blockIdx.x * G, kvh = gq > 0 ? head0 / gq : 0, split = blockIdx.y;
    if (gq < 0) {
        const int g = -gq, x = blockIdx.x & 7, i = blockIdx.x >> 3;
        const int grp = (i / g) * 8 + x;
        if (grp >= n_kv * splits) return;
        kvh = grp % n_kv; split = grp / n_kv; head0 = kvh * g + i % g;
    }
    // FUSED: the raw values of every head this wave will post-process (job j = wave + 4 r: query head j of the group, then
    // the key and the value row) are requested before anything else, the length word with them, so that one memory round
    // trip covers what used to be three in a row (the length, the first round's rows, the second round's).
    constexpr int ROUNDS = FUSED ? (G + 2 + WV - 1) / WV : 1;
    PostHead<HD> raw[ROUNDS];
    float freq = 0.f;
    if constexpr (FUSED) {
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {
            const int j = wave + WV * r;
            if (j < G + 2)
                raw[r] = post_request<HD>(fp, j < G ? head0 + j : (j == G ? fp.n_head + kvh : fp.n_head + n_kv + kvh),
                                          j < G ? fp.q_norm : (j == G ? fp.k_norm : nullptr), lane);
        }
        if (wave <= G && lane < fp.n_rot / 2) freq = rope_inv_freq(lane, fp.rate, fp.freq_scale);   // under the loads' latency
    }
    uint32_t len = len_dev ? *len_dev + 1u : len_host;   // the device word is the newest token's position
    asm volatile("" ::: "memory");                       // keeps the loads above in front of the arithmetic on the length
    if (len > len_host) len = len_host;
    // sliding window (nn.rs:92-111): only the last `window` keys count; 0 or >= len: all of them
    const uint32_t first = (window > 0 && window < len) ? len - window : 0u;
    const uint32_t per = (len - first + splits - 1) / splits;
    const uint32_t k0 = first + (uint32_t)split * per, k1 = min(len, k0 + per);
    const size_t stride = (size_t)n_kv * HD;
    const float* Kb = QF >= 0 ? nullptr : K + (size_t)kvh * HD + sub * DPL;
    const float* Vb = QF >= 0 ? nullptr : V + (size_t)kvh * HD + sub * DPL;

    // The rows of a step are requested one step ahead: a stream's steps depend on one another only through the running
    // maximum, so without this every step paid a memory round trip before its arithmetic (32 in a row for a split of 1024 keys).
    // A step past the split's end re-reads the split's last row (always a row of the cache) and is never used.
    constexpr int QFMT = QF >= 0 ? QF : 0;
    const int qcol = kvh * HD + sub * DPL, qnblk = n_kv * (HD / 32);
    RawDims<QFMT, DPL> kq[QF >= 0 ? ATT_KB : 1], vq[QF >= 0 ? ATT_KB : 1];
    float kf[QF >= 0 ? 1 : ATT_KB][DPL], vf[QF >= 0 ? 1 : ATT_KB][DPL];
    auto request = [&](uint32_t at) {
#pragma unroll
        for (int j = 0; j < ATT_KB; j++) {
            const uint32_t key = min(at + j, k1 - 1);   // a row past the split re-reads its last row and is masked below
            if constexpr (QF >= 0) {
                kq[j] = fetch_dims_q<QFMT, DPL>(qc.k_codes, qc.k_scales, key, qnblk, qcol);
                vq[j] = fetch_dims_q<QFMT, DPL>(qc.v_codes, qc.v_scales, key, qnblk, qcol);
            } else {
                load_dims<DPL>(Kb + key * stride, kf[j]);
                load_dims<DPL>(Vb + key * stride, vf[j]);
            }
        }
    };
    // FUSED: the first step's rows are requested in front of the post-processing, so that their memory round trip runs under it,
    // unless one of them could be the row this workgroup is about to append (then they are requested behind the barrier that
    // follows the store; a step past the split's end re-reads row k1 - 1, which is why that row counts too).
    bool requested = false;
    if constexpr (FUSED) {
        const uint32_t pos = *len_dev;
        if (k0 < k1 && (pos >= k0 + ATT_STREAMS * ATT_KB || pos >= k1)) {
            request(k0 + sid * ATT_KB);
            requested = true;
        }
    }
    if constexpr (FUSED) {
        const uint32_t pos = *len_dev;
        // the rows are appended by the workgroup whose keys include them; a position past the rows attention looks at (but
        // inside the cache) is still appended, by the last split, as the separate post-processing launch would
        const bool owner = pos < fp.cap && (pos < len ? (pos >= k0 && pos < k1) : split == splits - 1);
        const int njobs = G + (owner ? 2 : 0);
        const int kvw = n_kv * HD;
        float sn = 0.f, cs = 1.f;
        if (wave <= G) sincosf((float)pos * freq, &sn, &cs);
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {                 // job j < G: query head j of the group; G: the K row; G + 1: the V row
            const int j = wave + WV * r;
            if (j >= njobs) continue;
            if (j < G) {
                post_rotate<HD>(fp, raw[r], fp.q_norm != nullptr, cs, sn, lane, &sm_row[FUSED ? wave : 0][0], &sm_q[FUSED ? j : 0][0]);
                continue;
            }
            float* dst = QF >= 0 ? &sm_kv[FUSED && QF >= 0 ? j - G : 0][0] : (j == G ? fp.k_cache : fp.v_cache) + (size_t)pos * kvw + (size_t)kvh * HD;
            if (j == G) post_rotate<HD>(fp, raw[r], fp.k_norm != nullptr, cs, sn, lane, &sm_row[FUSED ? wave : 0][0], dst);
            else {
#pragma unroll
                for (int i = 0; i < HD / 64; i++) dst[lane + 64 * i] = raw[r].x[i];
            }
            if constexpr (QF >= 0) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                const size_t b0 = ((size_t)pos * n_kv + kvh) * (HD / 32);
#pragma unroll
                for (int e = lane; e < HD; e += 64)
                    quantize_lanes<QF>(dst[e], lane & 31, true, j == G ? qst.k_codes : qst.v_codes, j == G ? qst.k_scales : qst.v_scales, b0 + (size_t)(e >> 5));
            }
        }
        __syncthreads();
    }
    float qr[G][DPL], acc[G][DPL], m[G], l[G];
#pragma unroll
    for (int h = 0; h < G; h++) {
        m[h] = -3.0e38f; l[h] = 0.f;
        if constexpr (FUSED) {
#pragma unroll
            for (int i = 0; i < DPL; i++) qr[h][i] = sm_q[FUSED ? h : 0][sub * DPL + i];
        } else {
            load_dims<DPL>(q + ((size_t)head0 + h) * HD + sub * DPL, qr[h]);
        }
#pragma unroll
        for (int i = 0; i < DPL; i++) acc[h][i] = 0.f;
    }
    if (!requested) request(k0 + sid * ATT_KB);
    for (uint32_t kb = k0 + sid * ATT_KB; kb < k1; kb += ATT_STREAMS * ATT_KB) {
        float kr[ATT_KB][DPL], vr[ATT_KB][DPL];
#pragma unroll
        for (int j = 0; j < ATT_KB; j++) {
            if constexpr (QF >= 0) {
                expand_dims_q<QFMT, DPL>(kq[j], qcol, kr[j]);
                expand_dims_q<QFMT, DPL>(vq[j], qcol, vr[j]);
            } else {
#pragma unroll
                for (int i = 0; i < DPL; i++) { kr[j][i] = kf[j][i]; vr[j][i] = vf[j][i]; }
            }
        }
        request(kb + ATT_STREAMS * ATT_KB);
#pragma unroll
        for (int h = 0; h < G; h++) {
            float sc[ATT_KB];
#pragma unroll
            for (int j = 0; j < ATT_KB; j++) {
                float d = 0.f;
#pragma unroll
                for (int i = 0; i < DPL; i++) d = fmaf(qr[h][i], kr[j][i], d);
                d = row16_sum(d) * scale;
                if (softcap > 0.f) d = softcap * tanhf(d / softcap);   // cap * tanh(x / cap), crates/ferric-tensor/src/lib.rs:308
                sc[j] = (kb + j < k1) ? d : -3.0e38f;
            }
            float m_new = m[h];
#pragma unroll
            for (int j = 0; j < ATT_KB; j++) m_new = fmaxf(m_new, sc[j]);
            const float corr = __expf(m[h] - m_new);
            float e[ATT_KB], ps = 0.f;
#pragma unroll
            for (int j = 0; j < ATT_KB; j++) { e[j] = (kb + j < k1) ? __expf(sc[j] - m_new) : 0.f; ps += e[j]; }
            l[h] = fmaf(l[h], corr, ps);
#pragma unroll
            for (int i = 0; i < DPL; i++) {
                float a = acc[h][i] * corr;
#pragma unroll
                for (int j = 0; j < ATT_KB; j++) a = fmaf(e[j], vr[j][i], a);
                acc[h][i] = a;
            }
            m[h] = m_new;
        }
    }
    // merge the wave's four streams (rows of 16 lanes) by exchange with lanes ^16 and ^32
#pragma unroll
    for (int h = 0; h < G; h++) {
        float M = fmaxf(m[h], __shfl_xor(m[h], 16));
        M = fmaxf(M, __shfl_xor(M, 32));
        const float f = __expf(m[h] - M);
        float lv = l[h] * f;
        lv += __shfl_xor(lv, 16);
        lv += __shfl_xor(lv, 32);
#pragma unroll
        for (int i = 0; i < DPL; i++) {
            float a = acc[h][i] * f;
            a += __shfl_xor(a, 16);
            a += __shfl_xor(a, 32);
            if (lane < 16) sm_acc[wave][h][sub * DPL + i] = a;
        }
        if (lane == 0) { sm_m[wave][h] = M; sm_l[wave][h] = lv; }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * HD; idx += 64 * WV) {
        const int h = idx / HD, d = idx % HD;
        float M = sm_m[0][h];
#pragma unroll
        for (int w = 1; w < WV; w++) M = fmaxf(M, sm_m[w][h]);
        float L = 0.f, A = 0.f;
#pragma unroll
        for (int w = 0; w < WV; w++) {
            const float f = __expf(sm_m[w][h] - M);
            L = fmaf(sm_l[w][h], f, L);
            A = fmaf(sm_acc[w][h][d], f, A);
        }
        const int head = head0 + h;
        if (splits == 1) {
            out[(size_t)head * HD + d] = A / L;
        } else {
            float* pp = part + ((size_t)head * splits + split) * (HD + 2);
            pp[d] = A;
            if (d == 0) { pp[HD] = M; pp[HD + 1] = L; }
        }
    }
}

template <int G, int DPL, int WV>
__global__ __launch_bounds__(64 * WV) void attn_split_kernel(const float* __restrict__ q, const float* __restrict__ K, const float* __restrict__ V,
                                                             int n_kv, uint32_t len_host, const uint32_t* __restrict__ len_dev, float scale, int splits,
                                                             uint32_t window, float softcap, float* __restrict__ part, float* __restrict__ out, int gq) {
    attn_split_body<G, DPL, false, -1, WV>(q, K, V, n_kv, len_host, len_dev, scale, splits, window, softcap, part, out, QkvPostParams{}, gq);
}

template <int G, int DPL, int QF, int WV>
__global__ __launch_bounds__(64 * WV) void attn_split_kvq_kernel(const float* __restrict__ q, QCache qc, int n_kv, uint32_t len_host,
                                                                 const uint32_t* __restrict__ len_dev, float scale, int splits, uint32_t window,
                                                                 float softcap, float* __restrict__ part, float* __restrict__ out, int gq) {
    attn_split_body<G, DPL, false, QF, WV>(q, nullptr, nullptr, n_kv, len_host, len_dev, scale, splits, window, softcap, part, out, QkvPostParams{}, gq, qc);
}

template <int G, int DPL, int WV>
__global__ __launch_bounds__(64 * WV) void attn_split_fused_kernel(QkvPostParams fp, int n_kv, uint32_t len_host, const uint32_t* __restrict__ len_dev,
                                                                   float scale, int splits, uint32_t window, float softcap, float* __restrict__ part,
                                                                   float* __restrict__ out, int gq) {
    attn_split_body<G, DPL, true, -1, WV>(nullptr, fp.k_cache, fp.v_cache, n_kv, len_host, len_dev, scale, splits, window, softcap, part, out, fp, gq);
}

template <int G, int DPL, int QF, int WV>
__global__ __launch_bounds__(64 * WV) void attn_split_fused_kvq_kernel(QkvPostParams fp, KvqStore st, int n_kv, uint32_t len_host, const uint32_t* __restrict__ len_dev,
                                                                       float scale, int splits, uint32_t window, float softcap, float* __restrict__ part,
                                                                       float* __restrict__ out, int gq) {
    attn_split_body<G, DPL, true, QF, WV>(nullptr, nullptr, nullptr, n_kv, len_host, len_dev, scale, splits, window, softcap, part, out, fp, gq,
                                          QCache{st.k_codes, st.k_scales, st.v_codes, st.v_scales}, st);
}

// One workgroup per query head: weights exp(m_s - max m) of the splits once (each wave reduces them for itself; through LDS to
// the threads that need one), then every output dim is a weighted sum of the splits' accumulators over the weighted sum of their
// sums. splits <= 256. Thread (group, dim): group i of GROUPS takes splits i, i + GROUPS, ..., EARLY of them at once, the groups meet in LDS.
// Nothing but latency: with one thread a dim the splits came in six trips to memory one after the other, now in one (up to 64 splits;
// 128 in two): 40 heads of 128, 64 splits 5.0 us, 20 heads, 128 splits 8.4. A workgroup of sixteen waves takes longer to start and to meet, though, than a
// few splits take to add: one thread a dim | four | eight, us with the attention launch: 6 splits of 8 heads 6.3 | 6.6 | 7.2, 16 of 40 8.8 | 9.1 | 9.7, 24 of 8 without grouped
// heads 8.2 | 7.9 | 8.4, 41 of 8 heads 8.5 | 8.0 | 8.6, 52 10.4 (four) | 10.6, 64 of 40 24.7 | 23.6 | 23.6.
template <int GROUPS, int EARLY, int SPLITS>   // SPLITS: at most
__global__ __launch_bounds__(128 * GROUPS) void attn_combine_kernel(const float* __restrict__ part, int hd, int splits, float* __restrict__ out) {
    constexpr int NM = (SPLITS + 63) / 64;
    __shared__ float w[64 * NM];
    __shared__ float red[GROUPS][128];
    const int head = blockIdx.x, tid = threadIdx.x, lane = tid & 63, grp = GROUPS == 1 ? 0 : tid / hd, d = tid - grp * hd;   // (hd: 64 or 128)
    const float* pp = part + (size_t)head * splits * (hd + 2);
    // the first EARLY of the thread's splits are requested together with the splits' maxima and sums
    float pv[EARLY];
#pragma unroll
    for (int i = 0; i < EARLY; i++) {
        const int s = grp + GROUPS * i;
        pv[i] = s < splits ? pp[(size_t)s * (hd + 2) + d] : 0.f;
    }
    float mv[NM], lv[NM];
#pragma unroll
    for (int i = 0; i < NM; i++) {
        const int s = lane + 64 * i;
        mv[i] = -3.0e38f; lv[i] = 0.f;
        if (s < splits) { mv[i] = pp[(size_t)s * (hd + 2) + hd]; lv[i] = pp[(size_t)s * (hd + 2) + hd + 1]; }
    }
    float M = mv[0];
#pragma unroll
    for (int i = 1; i < NM; i++) M = fmaxf(M, mv[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
    float L = 0.f;
#pragma unroll
    for (int i = 0; i < NM; i++) {
        const int s = lane + 64 * i;
        const float f = s < splits ? __expf(mv[i] - M) : 0.f;
        L = fmaf(lv[i], f, L);
        if (tid < 64) w[s] = f;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) L += __shfl_xor(L, o);
    __syncthreads();
    float A = 0.f;
#pragma unroll
    for (int i = 0; i < EARLY; i++) A = fmaf(pv[i], w[grp + GROUPS * i], A);   // (0 past the last split)
    if constexpr (GROUPS * EARLY < SPLITS)
        for (int s0 = grp + GROUPS * EARLY; s0 < splits; s0 += GROUPS * EARLY) {
            float v[EARLY];
#pragma unroll
            for (int i = 0; i < EARLY; i++) {
                const int s = s0 + GROUPS * i;
                v[i] = s < splits ? pp[(size_t)s * (hd + 2) + d] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < EARLY; i++) A = fmaf(v[i], w[s0 + GROUPS * i], A);
        }
    if constexpr (GROUPS > 1) {
        red[grp][d] = A;
        __syncthreads();
        if (grp != 0) return;
#pragma unroll
        for (int i = 1; i < GROUPS; i++) A += red[i][d];
    }
    out[(size_t)head * hd + d] = A / L;
}
void launch_attn_combine(const float* part, int n_head, int hd, int splits, float* out, hipStream_t s) {
    const dim3 grid((unsigned)n_head);
    if (splits <= 16) hipLaunchKernelGGL((attn_combine_kernel<1, 16, 16>), grid, dim3((unsigned)hd), 0, s, part, hd, splits, out);
    else if (splits <= 64) hipLaunchKernelGGL((attn_combine_kernel<4, 8, 64>), grid, dim3((unsigned)(4 * hd)), 0, s, part, hd, splits, out);
    else hipLaunchKernelGGL((attn_combine_kernel<8, 8, 256>), grid, dim3((unsigned)(8 * hd)), 0, s, part, hd, splits, out);
}

// ---------------------------------------------------------------- the same over a long block-quantized cache, on the matrix cores
// All gq query heads of a KV head at once. A wave takes 32 keys at a time, in two tiles of 16, everything on v_mfma_f32_16x16x32_bf16 with
// the codes (whole numbers of at most eight bits, exact in bf16) as the A operand and an f32 cut into three bf16 values, whose sum it is, as
// the B operand: products are exact, sums f32.
//   Scores: A = one block of 32 dims of 16 keys, B = the query's 32 dims. Three instructions give the block's sum in f32; the block's scale
//   multiplies it. Lane n + 16 g ends up with keys 4 g .. 4 g + 3 of column n's query, so a query's maximum and sum are register operations
//   and two exchanges.
//   Values: A = 16 dims of one block of 32 keys, B = probability times the block's scale at that key (one rounding) of column n's query: the
//   eight keys of k-group g are the ones whose probabilities the lane holds. Two instructions a block and cut; the sums stay in the
//   accumulators, the running maximum's correction is skipped where no maximum moved.
// Up to five query heads a KV head (SPL): the 16 columns hold every query three times and column n takes cut n / gq of its query's products
// (the three sums meet at the end), a third of the values' instructions. Six to eight: a column a query, three instructions.
// Scales and key codes are requested as they lie, a row's bytes by neighbouring lanes, and go round through LDS (the wave's own part of it): a lane's own
// eight bytes of its key (row n) asked for directly cost the address unit a cycle a lane, 4 of the 7 thousand cycles of a round. Value codes come two blocks of a
// row by 16 lanes and are exchanged between halves of them (pair_up). A round's keys are requested when the round before has its own in LDS, its
// values when that round's are multiplied, the first round's keys in front of the post-processing; the raw heads before anything else, since loads return in
// order. Every wave cuts up its own head, so one barrier stands in front of the keys, and the three cuts of a sum meet in LDS.
// A workgroup a CU of eight waves, two a SIMD: 147 registers hold a round in flight, and the launch's fixed part (post-processing 4.5 us, the waves' sums 2)
// is paid once a CU. Workgroup L is split L % splits of KV head L / splits: with splits a multiple of eight an XCD's workgroups share the lines that hold all heads' scales
// of a row (KV head first, each of the eight XCDs fetched every one of them: 25.6 | 24.7 us).
// What bounds it: the rows' bytes (71 MB at 8 KV heads of 128, 32768 Q8_0 keys, at 5.5 - 6 TB/s behind the first request: 12 - 13 us of 23), close behind
// them instruction issue (640 vector instructions a round, a fifth each codes to bf16 and probabilities' cuts; 32 matrix instructions of 16 cycles, SPL).
// At that shape, kernel trace, 5 query heads a KV head: two workgroups a CU, keys by row, values a half word a load, none of it ahead of its round 28.1 us; now 23.2.
// With the combine launch, this kernel in that form -> now, us: head size 64, 8 KV heads, Q8_0 5200 / 16384 / 32768 keys 10.6 / 15.0 / 21.7 -> 8.8 / 11.0 / 14.8; 128, Q4_0,
// 4 KV heads of 8, 32768 keys 19.9 -> 16.3; 98 shapes 0.81 of the time (geometric mean). Two rounds ahead: 28.1 (the waves that post-process wait to issue).
// Before that, at that shape, us, values on f32 matrix instructions for six query heads and more, the dot-product kernel for fewer: 5 query
// heads a KV head 38.3, 8: 33.9; head size 64, 4: 23.0. Error against f64 (2-norm, relative, eighteen shapes) no larger in any:
// 2.2e-7 .. 2.5e-7 before, 1.4e-7 .. 1.8e-7 with the combine launch's present order.
// Q4_1: codes less the block's own code next to zero (an addition each) and, in place of the minimum, what that code stands for: at most half a step where the block has
// values on both sides of zero, and of the values' sign where it has not, so that neither term takes bits from the other. A score begins with those times the sums of the
// query's dims, a value's sum ends with their weighted sum. Error against f64 (2-norm) in that of the dot-product kernel, 120 products a kind of rows, geometric mean: about zero 0.95,
// every channel off zero by thrice the spread 0.98, one in sixteen by 12 times in keys 0.82, in values 1.01 (one code for all blocks, 7.5: 0.95, 0.99, 1.20 and 1.06; by 60 times 0.77 and
// 1.01, 1.57 and 1.10). us, the dot-product kernel -> this (less 7.5), with the combine launch: 8 query heads on each of 8 KV heads of 128, 14413 keys 34.8 -> 18.3 (17.3), 5 on 8 at 32768
// 41.5 -> 26.3 (25.4), 5 on 8 of 64 at 9000 15.9 -> 10.5 (10.3), 3 on 4 of 64 at 5200 10.1 -> 9.1 (9.0).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(8))) U4A8 { u32x4 v; };
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
union Frag { uint32_t w[4]; bf16x8 v; };
// the upper halves of two f32: two bf16 (exact where the lower halves are zero)
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); }

// Eight dims (8 g .. 8 g + 7 of a block of 32) of a key: its codes as bf16. 4-bit formats: less 8, and a sixteenth (Q4_1: `off` more) (v_cvt_off_f32_i4 makes that of a two's complement nibble in one
// instruction, where the byte, its conversion and the 8 were three; the scales carry the 16, so every bit is the same). 128 x 8 KV heads of 5, 32768 keys, with the combine launch 23.1 -> 21.2 us,
// 4 KV heads of 8 16.5 -> 15.6, heads of 64 16.4 -> 15.3: 804 -> 613 vector instructions a round beside its softmax.
template <int FMT>
__device__ __forceinline__ bf16x8 codes_bf16(const uint32_t (&w)[2], int shift, float off) {
    Frag f;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        float v[4];
        if constexpr (FMT == FHIP_KVQ_Q8_0) {
            v[0] = (float)(int8_t)(w[i] & 255u); v[1] = (float)(int8_t)((w[i] >> 8) & 255u);
            v[2] = (float)(int8_t)((w[i] >> 16) & 255u); v[3] = (float)(int8_t)(w[i] >> 24);
        } else {
            const uint32_t x = (w[i] ^ 0x88888888u) >> shift;
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = __builtin_amdgcn_cvt_off_f32_i4((int)(j % 3 ? (x >> (8 * j)) & 255u : x >> (8 * j))) + (FMT == FHIP_KVQ_Q4_1 ? off : 0.f);
        }
        f.w[2 * i] = upper_halves(v[0], v[1]);
        f.w[2 * i + 1] = upper_halves(v[2], v[3]);
    }
    return f.v;
}

constexpr int LONG_WAVES = 8, LONG_KEYS = 32;   // waves of a workgroup, keys a wave takes at a time
// FUSED: q is formed here from the raw QKV row and the workgroup whose keys hold the newest token appends it, as attn_split_body does (fp, st).
template <int HD, int FMT, bool SPL, bool FUSED>
__device__ __forceinline__ void attn_long_body(const float* __restrict__ q, const QCache& qc, int n_kv, uint32_t len_host, const uint32_t* __restrict__ len_dev,
                                               float scale, int splits, uint32_t window, float softcap, float* __restrict__ part, int gq,   // gq: query heads per KV head, at most 8 (SPL: 5)
                                               const QkvPostParams& fp, const KvqStore& st) {
    constexpr int NB = HD / 32, NT = LONG_KEYS / 16;                    // blocks of a row, tiles of 16 keys
    constexpr bool Q8 = FMT == FHIP_KVQ_Q8_0;
    constexpr int CW = Q8 ? 8 : 4;                                      // code words of a block
    constexpr int LR = NB * CW / 4, KL = LONG_KEYS * LR / 64;           // lanes that request a row's key codes, 16 bytes each; requests of a round
    constexpr int KROW = 16 * LR + 16;                                  // bytes of a row in LDS: sixteen rows' same 8 bytes lie in different banks
    constexpr bool MIN = FMT == FHIP_KVQ_Q4_1;
    constexpr int SW = MIN ? NB : NB / 2;                               // words of a row's scales (Q4_1: scale and minimum a word)
    __shared__ float sm_m[LONG_WAVES][8], sm_l[LONG_WAVES][8];
    constexpr int COLS = SPL ? 16 : 8;
    __shared__ __attribute__((aligned(16))) float sm_acc[LONG_WAVES][COLS][HD + 4];    // rows four banks apart
    __shared__ __attribute__((aligned(16))) float sm_d[LONG_WAVES][NB][64];   // rows 0 .. 31 the keys' scales, 32 .. 63 the values'
    __shared__ __attribute__((aligned(16))) float sm_min[MIN ? LONG_WAVES : 1][NB][64];   // MIN: what the block's code next to zero stands for, ...
    __shared__ __attribute__((aligned(16))) float sm_off[MIN ? LONG_WAVES : 1][NB][64];   // ... and 8 less that code, in sixteenths
    __shared__ float sm_qs[NB][16];                                     // MIN: the sum of block j's dims of column n's query
    __shared__ __attribute__((aligned(16))) uint8_t sm_k[LONG_WAVES][LONG_KEYS * KROW];   // a round's key codes, row by row
    __shared__ uint4 sm_q[NB][3][64];                                   // dims 32 j + 8 g .. + 7 of column n's query at lane n + 16 g, three bf16 each
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int cut = SPL ? n / gq : 0;                                   // the cut column n takes of its query (3: a column without one)
    const int kvh = blockIdx.y, split = blockIdx.x, head0 = kvh * gq;
    uint32_t len = len_dev ? *len_dev + 1u : len_host;
    if (len > len_host) len = len_host;
    const uint32_t first = (window > 0 && window < len) ? len - window : 0u;
    const uint32_t per = (len - first + splits - 1) / splits;
    const uint32_t k0 = first + (uint32_t)split * per, k1 = min(len, k0 + per);
    const int nblk = n_kv * NB;

    // What a round of 32 keys reads: key codes, scales (lanes 0 .. 31 the keys', 32 .. 63 the values'), and the value codes of block pair i at
    // key 16 t + 4 g + r: two units a lane (a unit is what a lane's A row of one block takes at a key: a half word, Q8_0, or a byte), units 2 n and 2 n + 1
    // of the pair's 32, so that lanes 0 .. 7 have the pair's first block and the others its second (pair_up).
    struct Round { u32x4 k[KL]; uint32_t sc[SW], v[NB / 2][NT][4]; } ra;
    constexpr uint32_t STEP = LONG_KEYS * LONG_WAVES;
    auto request_k = [&](Round& R, uint32_t kt) {
        kt = min(kt, k1 - 1u);
        const uint32_t last = k1 - 1u - kt;                             // rows past the split re-read its last row and count nothing
#pragma unroll
        for (int i = 0; i < KL; i++)
            R.k[i] = ((const U4A8*)(qc.k_codes + ((size_t)(kt + min((uint32_t)(i * (64 / LR) + lane / LR), last)) * nblk + (size_t)kvh * NB) * CW + 4 * (lane % LR)))->v;
        const size_t b = ((size_t)(kt + min((uint32_t)(lane & 31), last)) * nblk + (size_t)kvh * NB);
        const uint32_t* sp = (const uint32_t*)((lane < 32 ? qc.k_scales : qc.v_scales) + (MIN ? 2 * b : b));
#pragma unroll
        for (int i = 0; i < SW; i++) R.sc[i] = sp[i];
    };
    const uint32_t row_b = (uint32_t)nblk * (CW * 4);                   // bytes from a row's codes to the next row's
    auto load_units = [&](const char* p) -> uint32_t { return Q8 ? *(const uint32_t*)p : (uint32_t)*(const uint16_t*)p; };
    auto request_v = [&](Round& R, uint32_t kt) {
        kt = min(kt, k1 - 1u);
        const uint32_t last = k1 - 1u - kt;
        const char* vc = (const char*)(qc.v_codes + ((size_t)kt * nblk + (size_t)kvh * NB) * CW);
        const uint32_t at = (uint32_t)(Q8 ? 4 * n : 2 * n);
        if (last >= LONG_KEYS - 1u) {
            // a lane's own part of the address is the same for every row (and fits 32 bits); the rest is the wave's
            const uint32_t mine = (uint32_t)(4 * g) * row_b + at;
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int i = 0; i < NB / 2; i++) R.v[i][t][r] = load_units(vc + (size_t)(16 * t + r) * row_b + i * (2 * CW * 4) + mine);
        } else {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    uint32_t mine = (uint32_t)(4 * g);
                    asm volatile("" : "+v"(mine));                      // worked out here: kept from round to round these are eight more registers
                    const char* p = vc + (size_t)min(mine + (uint32_t)(16 * t + r), last) * row_b + at;
#pragma unroll
                    for (int i = 0; i < NB / 2; i++) R.v[i][t][r] = load_units(p + i * (2 * CW * 4));
                }
        }
    };
    uint32_t kt = k0 + (uint32_t)(LONG_KEYS * wave);
    // the heads' rows, the token's rows and the waves' scratch rows lie where the sums of the waves will
    float* const sq = FUSED ? &sm_acc[0][0][0] : nullptr;               // [8][HD] | [2][HD] | [LONG_WAVES][HD]
    static_assert(18 * HD <= LONG_WAVES * 8 * (HD + 4), "");
    bool owner = false;
    PostHead<HD> raw[2];                                                // up to ten jobs for eight waves: the query heads, the key head, the value head
    if constexpr (FUSED) {                                              // the first loads of all: behind the rows they would wait for them
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int j = wave + LONG_WAVES * r;
            if (j < gq + 2)
                raw[r] = post_request<HD>(fp, j < gq ? head0 + j : (j == gq ? fp.n_head + kvh : fp.n_head + n_kv + kvh), j < gq ? fp.q_norm : (j == gq ? fp.k_norm : nullptr), lane);
        }
        const uint32_t pos = *len_dev;
        owner = pos < fp.cap && (pos < len ? (pos >= k0 && pos < k1) : split == splits - 1);
    }
    if (!owner) request_k(ra, kt);                                      // their trip runs under the post-processing
    // A wave cuts its own query head up for all: lane 16 c + 4 j + g has dims 32 j + 8 g .. + 7 for the column of cut c (SPL; one column otherwise)
    auto cut_up = [&](int h, const float* row) {
        if (lane >= (SPL ? 48 : 16)) return;
        const int j = (lane >> 2) & 3, gg = lane & 3, col = SPL ? h + (lane >> 4) * gq : h;
        if (j >= NB) return;
        float x[8];
        load_dims<8>(row + 32 * j + 8 * gg, x);
        if constexpr (MIN) {
            float sum = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
            sum = dpp_add<0xB1, 0xF>(sum);      // over the quad, the block's four k-groups
            sum = dpp_add<0x4E, 0xF>(sum);
            if (gg == 0) sm_qs[j][col] = sum;
        }
#pragma unroll
        for (int t = 0; t < 3; t++) {
            sm_q[j][t][col + 16 * gg] = make_uint4(upper_halves(x[0], x[1]), upper_halves(x[2], x[3]), upper_halves(x[4], x[5]), upper_halves(x[6], x[7]));
#pragma unroll
            for (int i = 0; i < 8; i++) x[i] -= __uint_as_float(__float_as_uint(x[i]) & 0xFFFF0000u);   // exact
        }
    };
    if (wave < NB && n >= (SPL ? 3 * gq : gq)) {                        // columns without a query
#pragma unroll
        for (int t = 0; t < 3; t++) sm_q[wave][t][lane] = make_uint4(0u, 0u, 0u, 0u);
        if (MIN && g == 0) sm_qs[wave][n] = 0.f;
    }
    if constexpr (FUSED) {
        const int njobs = gq + (owner ? 2 : 0);
        const uint32_t pos = *len_dev;
        float sn = 0.f, cs = 1.f;
        if (wave < njobs && lane < fp.n_rot / 2) sincosf((float)pos * rope_inv_freq(lane, fp.rate, fp.freq_scale), &sn, &cs);
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int j = wave + LONG_WAVES * r;
            if (j >= njobs) continue;
            float* const dst = sq + j * HD + (j < gq ? 0 : (8 - gq) * HD);   // a query row, or rows 8 and 9
            if (j <= gq) post_rotate<HD>(fp, raw[r], (j < gq ? fp.q_norm : fp.k_norm) != nullptr, cs, sn, lane, sq + (10 + wave) * HD, dst);
            else {
#pragma unroll
                for (int i = 0; i < HD / 64; i++) dst[lane + 64 * i] = raw[r].x[i];
            }
            if (j < gq) cut_up(j, dst);
            else {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                const size_t b0 = ((size_t)pos * n_kv + kvh) * NB;
#pragma unroll
                for (int e = 0; e < HD; e += 64)
                    quantize_lanes<FMT>(dst[e + lane], lane & 31, true, j == gq ? st.k_codes : st.v_codes, j == gq ? st.k_scales : st.v_scales, b0 + (size_t)((e + lane) >> 5));
            }
        }
    } else if (wave < gq) cut_up(wave, q + ((size_t)head0 + wave) * HD);
    if (!owner) request_v(ra, kt);
    __syncthreads();
    if (owner) { request_k(ra, kt); request_v(ra, kt); }

    // Two keys' units of a block pair -> the lane's A rows of the first and of the second block, the later key's in the upper half: lanes 0 .. 7 of a row of 16
    // give their second units away for the first units of lanes 8 .. 15.
    auto pair_up = [&](uint32_t w0, uint32_t w1, uint32_t& first, uint32_t& second) {
        const uint32_t u0 = __builtin_amdgcn_perm(w1, w0, Q8 ? 0x05040100u : 0x0C040C00u), u1 = __builtin_amdgcn_perm(w1, w0, Q8 ? 0x07060302u : 0x0C050C01u);
        first = (uint32_t)__builtin_amdgcn_update_dpp((int)u0, (int)u1, 0x128, 0xF, 0xC, false);    // row_ror:8 into lanes 8 .. 15
        second = (uint32_t)__builtin_amdgcn_update_dpp((int)u1, (int)u0, 0x128, 0xF, 0x3, false);   // ... and 0 .. 7
    };
    const uint32_t cut1 = cut >= 1 ? 0xFFFF0000u : 0u, cut2 = cut >= 2 ? 0xFFFF0000u : 0u;

    f32x4 run[NB][2];                       // [block][tile]: A rows 4 g + r of column n
    float m = -3.0e38f, l = 0.f;            // of column n's query
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int i = 0; i < 2; i++) run[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    float qs[NB], floors[NB];               // MIN: sums of the query's dims; weighted sums of the values' minima over the lane's keys
#pragma unroll
    for (int j = 0; j < NB; j++) { qs[j] = MIN ? sm_qs[j][n] : 0.f; floors[j] = 0.f; }

    // a round; more: its registers take the wave's next one as they come free
    auto round = [&](Round& R, uint32_t kt, auto more) {
        const uint32_t last = k1 - 1u - kt;
#pragma unroll
        for (int i = 0; i < SW; i++) {
            const float lo = __half2float(__ushort_as_half((uint16_t)R.sc[i])), hi = __half2float(__ushort_as_half((uint16_t)(R.sc[i] >> 16)));
            if constexpr (MIN) {
                sm_d[wave][i][lane] = 16.0f * lo;
                const float zero = fminf(fmaxf(rintf(-hi * __builtin_amdgcn_rcpf(lo)), 0.f), 15.f);   // (any whole number does, the rest is exact for each)
                sm_min[wave][i][lane] = fmaf(zero, lo, hi);
                sm_off[wave][i][lane] = 0.0625f * (8.0f - zero);
            } else {
                sm_d[wave][2 * i][lane] = Q8 ? lo : 16.0f * lo;         // (4-bit codes are sixteenths)
                sm_d[wave][2 * i + 1][lane] = Q8 ? hi : 16.0f * hi;
            }
        }
#pragma unroll
        for (int i = 0; i < KL; i++) *(u32x4*)&sm_k[wave][(i * (64 / LR) + lane / LR) * KROW + 16 * (lane % LR)] = R.k[i];
        asm volatile("" ::: "memory");          // a wave's LDS accesses complete in order; this keeps the compiler's in order too
        if constexpr (decltype(more)::value) request_k(R, kt + STEP);

        float p[NT][4];                         // [tile][r]: key 16 t + 4 g + r of column n's query
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) p[t][r] = 0.f;
        if constexpr (MIN) {                    // before the products: the smaller terms first
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const f32x4 least = *(const f32x4*)&sm_min[wave][j][16 * t + 4 * g];
#pragma unroll
                    for (int r = 0; r < 4; r++) p[t][r] = fmaf(least[r], qs[j], p[t][r]);
                }
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
            Frag qf[3];
#pragma unroll
            for (int i = 0; i < 3; i++) { const uint4 w = sm_q[j][i][lane]; qf[i].w[0] = w.x; qf[i].w[1] = w.y; qf[i].w[2] = w.z; qf[i].w[3] = w.w; }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const uint2 w = *(const uint2*)&sm_k[wave][(16 * t + n) * KROW + 4 * CW * j + 8 * (g & (CW / 2 - 1))];
                const uint32_t kw[2] = {w.x, w.y};
                const bf16x8 c = codes_bf16<FMT>(kw, 4 * (g >> 1), MIN ? sm_off[wave][j][16 * t + n] : 0.f);
                f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 2; i >= 0; i--) a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c, qf[i].v, a, 0, 0, 0);
                const f32x4 d = *(const f32x4*)&sm_d[wave][j][16 * t + 4 * g];
#pragma unroll
                for (int r = 0; r < 4; r++) p[t][r] = fmaf(d[r], a[r], p[t][r]);
            }
            asm volatile("" ::: "memory");      // a block at a time: the operands of all of them do not fit the registers
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) p[t][r] *= scale;
        if (softcap > 0.f) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) p[t][r] = softcap * tanhf(p[t][r] / softcap);
        }
        const int lim = (int)min(last, (uint32_t)LONG_KEYS);
        const bool full = lim >= LONG_KEYS - 1;
        if (!full) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (4 * g > lim - (16 * t + r)) p[t][r] = -3.0e38f;
        }
        float top = -3.0e38f;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) top = fmaxf(top, p[t][r]);
        top = fmaxf(top, __shfl_xor(top, 16));
        top = fmaxf(top, __shfl_xor(top, 32));
        const float m_new = fmaxf(m, top), corr = __expf(m - m_new);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) p[t][r] = __expf(p[t][r] - m_new);
        if (!full) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (4 * g > lim - (16 * t + r)) p[t][r] = 0.f;
        }
        float ps[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) ps[t] = (p[t][0] + p[t][1]) + (p[t][2] + p[t][3]);
        l = fmaf(l, corr, ps[0] + ps[1]);
        if (__builtin_amdgcn_ballot_w64(m_new != m) != 0) {
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int i = 0; i < 2; i++) run[j][i] *= corr;
            if constexpr (MIN) {
#pragma unroll
                for (int j = 0; j < NB; j++) floors[j] *= corr;
            }
        }
        m = m_new;
        uint32_t vw[2][4];                      // [block of the pair]: the codes of keys 16 (e / 2) + 4 g + 2 (e % 2) and the next, a half word each
#pragma unroll
        for (int j = 0; j < NB; j++) {
            float x[2 * 4];                     // probability times the block's scale, key 16 t + 4 g + r at 4 t + r
            f32x4 off[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const f32x4 d = *(const f32x4*)&sm_d[wave][j][32 + 16 * t + 4 * g];
#pragma unroll
                for (int r = 0; r < 4; r++) x[4 * t + r] = p[t][r] * d[r];
                if constexpr (MIN) {
                    const f32x4 least = *(const f32x4*)&sm_min[wave][j][32 + 16 * t + 4 * g];
                    floors[j] += fmaf(p[t][0], least[0], p[t][1] * least[1]) + fmaf(p[t][2], least[2], p[t][3] * least[3]);
                    off[t] = *(const f32x4*)&sm_off[wave][j][32 + 16 * t + 4 * g];
                }
            }
            if (j % 2 == 0)
#pragma unroll
                for (int e = 0; e < 4; e++) pair_up(R.v[j / 2][e >> 1][2 * (e & 1)], R.v[j / 2][e >> 1][2 * (e & 1) + 1], vw[0][e], vw[1][e]);
            Frag a[2];                          // the codes of the block's two tiles of dims
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t w = vw[j & 1][e];
                    float lo, hi;
                    if constexpr (Q8) { lo = (float)(int8_t)(w >> (8 * i)); hi = (float)(int8_t)(w >> (16 + 8 * i)); }
                    else {
                        const uint32_t x = (w ^ 0x88888888u) >> (4 * i);
                        lo = __builtin_amdgcn_cvt_off_f32_i4((int)x); hi = __builtin_amdgcn_cvt_off_f32_i4((int)(x >> 16));
                        if constexpr (MIN) { lo += off[e >> 1][2 * (e & 1)]; hi += off[e >> 1][2 * (e & 1) + 1]; }
                    }
                    a[i].w[e] = upper_halves(lo, hi);
                }
            if constexpr (SPL) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    x[e] -= __uint_as_float(__float_as_uint(x[e]) & cut1);
                    x[e] -= __uint_as_float(__float_as_uint(x[e]) & cut2);
                }
                Frag f;
#pragma unroll
                for (int e = 0; e < 4; e++) f.w[e] = upper_halves(x[2 * e], x[2 * e + 1]);
#pragma unroll
                for (int i = 0; i < 2; i++) run[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, f.v, run[j][i], 0, 0, 0);
            } else {
                Frag f[3];
#pragma unroll
                for (int k = 0; k < 3; k++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        f[k].w[e] = upper_halves(x[2 * e], x[2 * e + 1]);
                        x[2 * e] -= __uint_as_float(__float_as_uint(x[2 * e]) & 0xFFFF0000u);
                        x[2 * e + 1] -= __uint_as_float(__float_as_uint(x[2 * e + 1]) & 0xFFFF0000u);
                    }
#pragma unroll
                for (int k = 2; k >= 0; k--)    // (smallest cut first)
#pragma unroll
                    for (int i = 0; i < 2; i++) run[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, f[k].v, run[j][i], 0, 0, 0);
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (decltype(more)::value) request_v(R, kt + STEP);
    };
    for (; kt + STEP < k1; kt += STEP) round(ra, kt, std::true_type{});
    if (kt < k1) round(ra, kt, std::false_type{});
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (lane < gq) { sm_m[wave][lane] = m; sm_l[wave][lane] = l; }
    if constexpr (MIN) {                    // to one of the query's columns
#pragma unroll
        for (int j = 0; j < NB; j++) {
            floors[j] += __shfl_xor(floors[j], 16);
            floors[j] += __shfl_xor(floors[j], 32);
#pragma unroll
            for (int i = 0; i < 2; i++) run[j][i] += n < gq ? floors[j] : 0.f;
        }
    }
    if (n < (SPL ? 3 * gq : gq)) {
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int mrow = 4 * g + r, unit = 2 * (mrow & 7) + (mrow >> 3);   // the A row's unit of the block: dims 2 u, 2 u + 1 (Q8_0), u, 16 + u
                sm_acc[wave][n][32 * j + (Q8 ? 2 * unit : unit)] = run[j][0][r];
                sm_acc[wave][n][32 * j + (Q8 ? 2 * unit + 1 : 16 + unit)] = run[j][1][r];
            }
    }
    __syncthreads();
    // four dims a thread; a query's three cuts meet here
    for (int idx = threadIdx.x; idx < gq * (HD / 4); idx += 64 * LONG_WAVES) {
        const int h = idx / (HD / 4), d = 4 * (idx % (HD / 4));
        float M = sm_m[0][h];
#pragma unroll
        for (int w = 1; w < LONG_WAVES; w++) M = fmaxf(M, sm_m[w][h]);
        float L = 0.f;
        f32x4 A = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < LONG_WAVES; w++) {
            const float f = __expf(sm_m[w][h] - M);
            L = fmaf(sm_l[w][h], f, L);
            f32x4 v = *(const f32x4*)&sm_acc[w][h][d];
            if constexpr (SPL) v += *(const f32x4*)&sm_acc[w][h + gq][d] + *(const f32x4*)&sm_acc[w][h + 2 * gq][d];
#pragma unroll
            for (int i = 0; i < 4; i++) A[i] = fmaf(v[i], f, A[i]);
        }
        float* pp = part + ((size_t)(head0 + h) * splits + split) * (HD + 2);
#pragma unroll
        for (int i = 0; i < 4; i++) pp[d + i] = A[i];
        if (d == 0) { pp[HD] = M; pp[HD + 1] = L; }
    }
}

template <int HD, int FMT, bool SPL>
__global__ __launch_bounds__(64 * LONG_WAVES, 2) void attn_long_kvq_kernel(const float* __restrict__ q, QCache qc, int n_kv, uint32_t len_host,
                                                                           const uint32_t* __restrict__ len_dev, float scale, int splits,
                                                                           uint32_t window, float softcap, float* __restrict__ part, int gq) {
    attn_long_body<HD, FMT, SPL, false>(q, qc, n_kv, len_host, len_dev, scale, splits, window, softcap, part, gq, QkvPostParams{}, KvqStore{});
}
template <int HD, int FMT, bool SPL>
__global__ __launch_bounds__(64 * LONG_WAVES, 2) void attn_long_fused_kvq_kernel(QkvPostParams fp, KvqStore st, int n_kv, uint32_t len_host,
                                                                                 const uint32_t* __restrict__ len_dev, float scale, int splits,
                                                                                 uint32_t window, float softcap, float* __restrict__ part, int gq) {
    attn_long_body<HD, FMT, SPL, true>(nullptr, QCache{st.k_codes, st.k_scales, st.v_codes, st.v_scales}, n_kv, len_host, len_dev, scale, splits, window, softcap, part, gq,
                                       fp, st);
}

// wide (G = 1): workgroups of ATT_WIDE waves
constexpr int ATT_WIDE = 16;
template <int G, class Kernel, class Wide, class... Args>
void attn_go(dim3 grid, hipStream_t s, bool wide, Kernel kernel, Wide kernel_wide, Args... args) {
    if (G == 1 && wide) hipLaunchKernelGGL(kernel_wide, grid, dim3(64 * ATT_WIDE), 0, s, args...);
    else hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, args...);
}

template <int G>
int launch_attn_g(int hd, dim3 grid, hipStream_t s, const float* q, const float* K, const float* V, int n_kv, uint32_t len, const uint32_t* d_len,
                  float scale, int splits, uint32_t window, float softcap, float* part, float* out, int gq = G, bool wide = false) {
    switch (hd) {
        case 64: attn_go<G>(grid, s, wide, attn_split_kernel<G, 4, 4>, attn_split_kernel<1, 4, ATT_WIDE>, q, K, V, n_kv, len, d_len, scale, splits, window, softcap, part, out, gq); break;
        case 128: attn_go<G>(grid, s, wide, attn_split_kernel<G, 8, 4>, attn_split_kernel<1, 8, ATT_WIDE>, q, K, V, n_kv, len, d_len, scale, splits, window, softcap, part, out, gq); break;
        default: return fhip::set_error(FHIP_ERR_SHAPE, "decode_attention: head_dim must be 64 or 128");
    }
    return FHIP_OK;
}

// What the launches over a quantized cache share; fp: the raw QKV row to post-process and append (null: q holds the queries).
struct KvqLaunch {
    hipStream_t s;
    const float* q;
    const QkvPostParams* fp;
    KvqStore cache;
    int n_kv;
    uint32_t len;
    const uint32_t* d_len;
    float scale;
    int splits;
    uint32_t window;
    float softcap;
    float *part, *out;
    QCache qc() const { return QCache{cache.k_codes, cache.k_scales, cache.v_codes, cache.v_scales}; }
};
template <int G, int DPL, int QF>
void launch_attn_kvq_hd(dim3 grid, const KvqLaunch& a, int gq, bool wide) {
    if (a.fp)
        attn_go<G>(grid, a.s, wide, attn_split_fused_kvq_kernel<G, DPL, QF, 4>, attn_split_fused_kvq_kernel<1, DPL, QF, ATT_WIDE>, *a.fp, a.cache, a.n_kv, a.len, a.d_len, a.scale,
                   a.splits, a.window, a.softcap, a.part, a.out, gq);
    else
        attn_go<G>(grid, a.s, wide, attn_split_kvq_kernel<G, DPL, QF, 4>, attn_split_kvq_kernel<1, DPL, QF, ATT_WIDE>, a.q, a.qc(), a.n_kv, a.len, a.d_len, a.scale, a.splits, a.window,
                   a.softcap, a.part, a.out, gq);
}
// gq: as attn_split_body's (G, -g, or query heads per KV head with G = 1)
template <int QF>
int launch_attn_kvq(int g, int hd, dim3 grid, const KvqLaunch& a, int gq, bool wide = false) {
    auto go = [&](auto Gc) {
        constexpr int G = decltype(Gc)::value;
        if (hd == 64) launch_attn_kvq_hd<G, 4, QF>(grid, a, gq, wide);
        else launch_attn_kvq_hd<G, 8, QF>(grid, a, gq, wide);
        return FHIP_OK;
    };
    switch (g) {
        case 1: return go(std::integral_constant<int, 1>{});
        case 2: return go(std::integral_constant<int, 2>{});
        case 3: return go(std::integral_constant<int, 3>{});
        case 4: return go(std::integral_constant<int, 4>{});
        case 5: return go(std::integral_constant<int, 5>{});
        case 6: return go(std::integral_constant<int, 6>{});
        case 7: return go(std::integral_constant<int, 7>{});
        case 8: return go(std::integral_constant<int, 8>{});
        default: return fhip::set_error(FHIP_ERR_SHAPE, "decode_attention: %d query heads per KV head (1..=8 supported)", g);
    }
}

// Which launches take it: its cost does not depend on the number of query heads a KV head, the kernel above costs less for one and two. us, this | that, both
// with the combine launch, on rows no cache holds. Three query heads a KV head, post-processed in the launch: heads of 128, Q8_0, 8 KV heads 5200 / 9000 / 32768 keys 13.8 | 14.4,
// 16.5 | 17.5, 30.2 | 31.6; 4 KV heads 13.3 | 13.1, 14.3 | 14.9, 20.2 | 22.2; 1 KV head 10.8 | 11.2, 11.7 | 12.7, 14.5 | 16.3; Q4_0 4 KV heads 14.2 | 13.3, 14.7 | 14.8, 20.5 | 23.0;
// heads of 64, 4 KV heads Q8_0 10.7 | 10.5, 11.1 | 11.6, 14.8 | 17.0. Post-processed before: Q8_0 8 KV heads 12.8 | 13.4, 15.8 | 15.7, 29.6 | 29.0; 16 KV heads 17.5 | 16.4, 20.9 | 20.3,
// 48.8 | 46.5 (in the launch 18.4 | 18.4, 21.4 | 22.7, 49.6 | 49.2). Four: 8 KV heads of 128, Q8_0 14.0 | 16.0, 16.6 | 19.1, 30.3 | 36.0; five 14.5 | 18.8, 17.2 | 21.3, 31.4 | 40.7.
// Key codes are read eight bytes at a time; a lane's offset inside a round's rows is kept in 32 bits (n_kv).
bool attn_long_takes(int fmt, int g, int n_kv, const uint32_t* k_codes) {
    if (g > 8 || n_kv > 65535 || ((uintptr_t)k_codes & 7) != 0) return false;
    return g >= 3;
}
// Half the splits of the kernels above, about one workgroup a CU, and never the one that needs no combine launch. 98 shapes of one to sixteen KV heads, 5200 .. 32768 keys: as many
// splits as above take 1.18 times as long (the fixed part twice a CU).
int attn_long_splits(int splits) { return splits <= 3 ? 2 : (splits + 1) / 2; }
template <int FMT>
void launch_attn_long_kvq(int g, int hd, dim3 grid, const KvqLaunch& a) {
    auto go = [&](auto kernel, auto fused) {
        if (a.fp) hipLaunchKernelGGL(fused, dim3(grid.y, grid.x), dim3(64 * LONG_WAVES), 0, a.s, *a.fp, a.cache, a.n_kv, a.len, a.d_len, a.scale, a.splits, a.window, a.softcap, a.part, g);
        else hipLaunchKernelGGL(kernel, dim3(grid.y, grid.x), dim3(64 * LONG_WAVES), 0, a.s, a.q, a.qc(), a.n_kv, a.len, a.d_len, a.scale, a.splits, a.window, a.softcap, a.part, g);
    };
    if (hd == 64) {
        if (g <= 5) go(attn_long_kvq_kernel<64, FMT, true>, attn_long_fused_kvq_kernel<64, FMT, true>);
        else go(attn_long_kvq_kernel<64, FMT, false>, attn_long_fused_kvq_kernel<64, FMT, false>);
    } else {
        if (g <= 5) go(attn_long_kvq_kernel<128, FMT, true>, attn_long_fused_kvq_kernel<128, FMT, true>);
        else go(attn_long_kvq_kernel<128, FMT, false>, attn_long_fused_kvq_kernel<128, FMT, false>);
    }
}

template <int G>
int launch_attn_fused_g(int hd, dim3 grid, hipStream_t s, const QkvPostParams& fp, int n_kv, uint32_t len, const uint32_t* d_len, float scale,
                        int splits, uint32_t window, float softcap, float* part, float* out, int gq = G, bool wide = false) {
    switch (hd) {
        case 64: attn_go<G>(grid, s, wide, attn_split_fused_kernel<G, 4, 4>, attn_split_fused_kernel<1, 4, ATT_WIDE>, fp, n_kv, len, d_len, scale, splits, window, softcap, part, out, gq); break;
        case 128: attn_go<G>(grid, s, wide, attn_split_fused_kernel<G, 8, 4>, attn_split_fused_kernel<1, 8, ATT_WIDE>, fp, n_kv, len, d_len, scale, splits, window, softcap, part, out, gq); break;
        default: return fhip::set_error(FHIP_ERR_SHAPE, "decode_attention: head_dim must be 64 or 128");
    }
    return FHIP_OK;
}

}  // namespace

namespace fhip {

// The weights with the row (AHEAD) while every CU has at most four workgroups; beyond, its registers leave fewer of them on a CU. us, behind the sum | with the row: rmsnorm, 64 rows
// of 4096 4.0 | 3.6, 256 of 2560 4.0 | 3.7, 1024 of 8192 11.6 | 10.7, 1500 of 1536 4.5 | 4.8, 2048 of 5120 12.9 | 13.7, 16384 of 768 16.4 | 19.4; sum, norm and bf16 rows, 1200 rows of
// 2560 7.3 | 7.3, 1500 of 1536 5.5 | 6.7, 2048 of 2048 9.5 | 11.0, 2048 of 5120 21.3 | 23.3, 65536 of 64 (four rows a workgroup) 17.6 | 20.6.
static bool norm_ahead(size_t grid) { return grid <= 4 * (size_t)(device_cus() > 0 ? device_cus() : 256); }
template <typename Out>
static int launch_rmsnorm_out(const float* a, const float* b, const float* weight, size_t rows, size_t d, float eps, float* sum_out, Out* norm_out,
                              hipStream_t s, uint32_t* count = nullptr, uint32_t by = 0) {
    if (rows == 0 || d == 0) return count ? launch_u32_add(count, 1, by, s) : FHIP_OK;
    if (d > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "rmsnorm: row length exceeds 2^31");
    const size_t grid = d <= 512 ? (rows + 3) / 4 : rows;
    if (grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "rmsnorm: too many rows for one launch");
    const bool ahead = norm_ahead(grid);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), 0, s, a, b, weight, rows, (int)d, eps, sum_out, norm_out, count, by); };
    if (d <= 512) ahead ? go(rmsnorm_kernel<64, Out, true>) : go(rmsnorm_kernel<64, Out, false>);
    else ahead ? go(rmsnorm_kernel<256, Out, true>) : go(rmsnorm_kernel<256, Out, false>);
    return check_hip(hipGetLastError(), "rmsnorm launch");
}

int launch_rmsnorm(const float* a, const float* b, const float* weight, size_t rows, size_t d, float eps, float* sum_out, float* norm_out,
                   hipStream_t s, uint32_t* count, uint32_t by) {
    return launch_rmsnorm_out(a, b, weight, rows, d, eps, sum_out, norm_out, s, count, by);
}
int launch_rmsnorm_bf16(const float* a, const float* b, const float* weight, size_t rows, size_t d, float eps, float* sum_out, uint16_t* norm_out,
                        hipStream_t s) {
    return launch_rmsnorm_out(a, b, weight, rows, d, eps, sum_out, norm_out, s);
}

int launch_u32_add(uint32_t* w, size_t n, uint32_t delta, hipStream_t s) {
    size_t grid = (n + 255) / 256;
    if (grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "u32_add: too many words for one launch");
    hipLaunchKernelGGL(u32_add_kernel, dim3((unsigned)grid), dim3(256), 0, s, w, n, delta);
    return check_hip(hipGetLastError(), "u32_add launch");
}

int launch_add(const float* a, const float* b, size_t n, float* out, hipStream_t s, uint32_t* count, uint32_t by) {
    if (n == 0) return count ? launch_u32_add(count, 1, by, s) : FHIP_OK;
    size_t grid = (n + 255) / 256;
    if (grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "add: too many elements for one launch");
    hipLaunchKernelGGL(add_kernel, dim3((unsigned)grid), dim3(256), 0, s, a, b, n, out, count, by);
    return check_hip(hipGetLastError(), "add launch");
}

int launch_mul_sigmoid(const float* a, const float* g, size_t n, float* out, hipStream_t s) {
    if (n == 0) return FHIP_OK;
    size_t grid = (n + 255) / 256;
    if (grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "mul_sigmoid: too many elements for one launch");
    hipLaunchKernelGGL(mul_sigmoid_kernel, dim3((unsigned)grid), dim3(256), 0, s, a, g, n, out);
    return check_hip(hipGetLastError(), "mul_sigmoid launch");
}

int launch_geglu(const float* gu, size_t t, size_t d, float* out, hipStream_t s) {
    const size_t n = t * d;
    if (n == 0) return FHIP_OK;
    size_t grid = (n + 255) / 256;
    if (grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "geglu: too many elements for one launch");
    hipLaunchKernelGGL(geglu_kernel, dim3((unsigned)grid), dim3(256), 0, s, gu, n, d, out);
    return check_hip(hipGetLastError(), "geglu launch");
}

int launch_rope(const float* x, size_t src_row_stride, size_t t, int heads, int hd, int n_rot, float base, const uint32_t* d_pos, uint32_t pos_off,
                const float* freq_scale, int interleaved, float* out, hipStream_t s) {
    if (t == 0 || heads == 0 || hd == 0) return FHIP_OK;
    size_t n = t * (size_t)heads * (size_t)(hd - n_rot / 2);
    size_t grid = (n + 255) / 256;
    if (t > 0x7FFFFFFFull || grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "rope: too many rows for one launch");
    hipLaunchKernelGGL(rope_kernel, dim3((unsigned)grid), dim3(256), 0, s, x, src_row_stride, (int)t, heads, hd, n_rot, rope_rate(n_rot, base), d_pos, pos_off,
                       freq_scale, interleaved, out);
    return check_hip(hipGetLastError(), "rope launch");
}

int launch_qkv_post(const float* qkv, const float* bias, const float* q_norm, const float* k_norm, const uint32_t* d_pos, const float* freq_scale,
                    size_t t, int n_head, int n_kv, int hd, int n_rot, int interleaved, float eps, float base, float* q_out, float* k_cache,
                    float* v_cache, size_t cap, hipStream_t s, bool kv_packed) {
    if (t == 0) return FHIP_OK;
    QkvPostParams p;
    p.qkv = qkv; p.bias = bias; p.q_norm = q_norm; p.k_norm = k_norm; p.pos = d_pos; p.freq_scale = freq_scale;
    p.q_out = q_out; p.k_cache = k_cache; p.v_cache = v_cache;
    p.t = (int)t; p.n_head = n_head; p.n_kv = n_kv; p.hd = hd; p.n_rot = n_rot; p.interleaved = interleaved;
    p.cap = (uint32_t)cap; p.eps = eps; p.rate = rope_rate(n_rot, base); p.kv_packed = kv_packed ? 1 : 0;
    const size_t per_tok = (size_t)(n_head + 2 * n_kv);
    if (t > 0x7FFFFFFFull || (t * per_tok + 3) / 4 > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "qkv_post: too many rows for one launch");
    // Four heads a wave once that leaves the CUs some four waves each; a token or two needs all the waves it can have. us, one | two | four | eight heads
    // of 128: 139 rows of 40 4.6 | 4.7 | 4.1 | 5.0; 276 of 32 5.1 | 4.8 | 4.5 | 5.7; 509 of 56 9.8 | 8.2 | 7.6 | 8.4; 699 of 80 16.9 | 12.6 | 12.0 | 12.9
    if ((hd == 64 || hd == 128) && n_rot == hd && !interleaved) {
        const size_t hpw = t * ((per_tok + 3) / 4) >= 4 * (size_t)device_cus() ? 4 : 1;
        const dim3 grid((unsigned)((t * ((per_tok + hpw - 1) / hpw) + 3) / 4));
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, p); };
        if (hd == 128) hpw == 4 ? go(qkv_post_heads_kernel<128, 4>) : go(qkv_post_heads_kernel<128, 1>);
        else hpw == 4 ? go(qkv_post_heads_kernel<64, 4>) : go(qkv_post_heads_kernel<64, 1>);
    } else {
        hipLaunchKernelGGL(qkv_post_kernel, dim3((unsigned)((t * per_tok + 3) / 4)), dim3(256), 0, s, p);
    }
    return check_hip(hipGetLastError(), "qkv_post launch");
}

bool qkv_post_kvq_takes(int hd) { return hd > 0 && hd % 32 == 0 && hd <= POST_KVQ_HD; }
template <int FMT>
static int post_kvq(const QkvPostParams& p, const KvqStore& st, KvqRows rows, hipStream_t s) {
    const size_t t = p.t, per_tok = (size_t)(p.n_head + 2 * p.n_kv), past = rows.past * ((size_t)p.n_kv * p.hd / 4) * 2, past_wgs = (past + 255) / 256;
    const bool whole = rows.k && (p.hd == 64 || p.hd == 128) && p.n_rot == p.hd && !p.interleaved;
    // Two heads a wave: us, one | two | four | eight on Q8_0 (Q4_0 and Q4_1 alike): 42 rows of 32 + 8 + 8 heads of 64 5.1 | 4.9 | 5.0 | 8.3, 276 of 16 + 8 + 8 of 128
    // 6.5 | 6.6 | 7.2 | 12.1, 509 of 40 + 8 + 8 of 128 11.8 | 10.8 | 11.1 | 16.1, 699 of 64 + 8 + 8 of 128 18.6 | 15.6 | 15.9 | 20.1 (a key or value head is a chain of a microsecond).
    const size_t hpw = whole ? 2 : 1, grid = (t * ((per_tok + hpw - 1) / hpw) + 3) / 4;
    if (t * per_tok > 0x7FFFFFFFull || grid + past_wgs > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "qkv_post_kvq: too many rows for one launch");
    rows.post_wgs = (unsigned)grid;
    const dim3 g((unsigned)(grid + past_wgs)), wg(256);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, wg, 0, s, p, st, rows); };
    if (!rows.k) go(qkv_post_kvq_kernel<FMT, false>);
    else if (!whole) go(qkv_post_kvq_kernel<FMT, true>);
    else p.hd == 128 ? go(qkv_post_rows_kernel<FMT, 128, 2>) : go(qkv_post_rows_kernel<FMT, 64, 2>);
    return check_hip(hipGetLastError(), "qkv_post_kvq launch");
}
int launch_qkv_post_kvq(int fmt, const float* qkv, const float* bias, const float* q_norm, const float* k_norm, const uint32_t* d_pos,
                        const float* freq_scale, size_t t, int n_head, int n_kv, int hd, int n_rot, int interleaved, float eps, float base, float* q_out,
                        uint32_t* k_codes, uint16_t* k_scales, uint32_t* v_codes, uint16_t* v_scales, size_t cap, hipStream_t s, float* k_rows, float* v_rows, size_t n_rows, size_t past) {
    if (t == 0) return FHIP_OK;
    if (t > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "qkv_post_kvq: too many rows for one launch");
    QkvPostParams p;
    p.qkv = qkv; p.bias = bias; p.q_norm = q_norm; p.k_norm = k_norm; p.pos = d_pos; p.freq_scale = freq_scale;
    p.q_out = q_out; p.k_cache = nullptr; p.v_cache = nullptr;
    p.t = (int)t; p.n_head = n_head; p.n_kv = n_kv; p.hd = hd; p.n_rot = n_rot; p.interleaved = interleaved;
    p.cap = (uint32_t)cap; p.eps = eps; p.rate = rope_rate(n_rot, base); p.kv_packed = 0;
    const KvqStore st{k_codes, k_scales, v_codes, v_scales};
    const KvqRows rows{k_rows, v_rows, (uint32_t)n_rows, (uint32_t)past, 0u};
    switch (fmt) {
        case FHIP_KVQ_Q8_0: return post_kvq<FHIP_KVQ_Q8_0>(p, st, rows, s);
        case FHIP_KVQ_Q4_0: return post_kvq<FHIP_KVQ_Q4_0>(p, st, rows, s);
        case FHIP_KVQ_Q4_1: return post_kvq<FHIP_KVQ_Q4_1>(p, st, rows, s);
        default: return set_error(FHIP_ERR_ARG, "qkv_post_kvq: unknown format %d", fmt);
    }
}

int launch_kv_append(const float* k, const float* v, size_t t, size_t width, const uint32_t* d_pos, uint32_t pos_off, size_t cap, float* kc,
                     float* vc, hipStream_t s) {
    if (t == 0 || width == 0) return FHIP_OK;
    size_t n = t * width, grid = (n + 255) / 256;
    if (t > 0x7FFFFFFFull || width > 0x7FFFFFFFull || grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "kv_append: too large for one launch");
    hipLaunchKernelGGL(kv_append_kernel, dim3((unsigned)grid), dim3(256), 0, s, k, v, (int)t, (int)width, d_pos, pos_off, (uint32_t)cap, kc, vc);
    return check_hip(hipGetLastError(), "kv_append launch");
}

// Caches of up to ATT_SHORT rows (a launch sized for that many): one workgroup per query head over the whole key range, no splits, no
// combine launch. The rows of a KV head are read by each of its query heads' workgroups (a few hundred KB out of the L2), which costs less
// than the second launch and the trip of the partial results through memory. A step of a workgroup's streams is a trip to memory (0.9 us on rows no
// cache holds), so from ATT_WIDE_FROM rows on it has sixteen waves, 128 keys a step, in place of four; fewer rows leave most of those without a key (48 rows
// 4.6 -> 5.6 us). Four waves -> sixteen, f32 cache, us: 130 / 200 / 256 rows 6.2 / 6.9 / 7.1 -> 5.8 / 6.2 / 6.5.
// Where it ends: heads of 128 dims on an f32 cache wait for memory in their one workgroup, where splits bring more of them: there it ends at ATT_SHORT_128 rows,
// and at ATT_SHORT_OWN for a head per KV head, whose rows no other workgroup reads. us with the post-processing, one workgroup a head | splits and combined, rows that
// no cache holds (over 700 MB) and, in brackets, that the Infinity Cache does: f32, 40 heads of 8 at 208 / 256 / 288 / 352 rows 8.8 | 9.5, 9.5 | 9.7, 10.2 | 9.1, 11.3 | 9.8 (256 / 288 / 352
// 7.8 | 8.3, 8.3 | 8.0, 9.2 | 8.5), 16 of 4 at 256 / 288 / 352 9.0 | 9.2, 9.9 | 9.0, 11.0 | 9.7, 2 of 1 at 288 / 352 7.3 | 6.9, 7.9 | 7.4; a KV head each, 8 heads at 128 / 192 / 256 / 352
// 7.7 | 8.1, 8.4 | 7.8, 9.8 | 8.1, 11.9 | 8.2 (192 / 256 / 352 6.8 | 6.9, 7.2 | 7.1, 8.4 | 7.3), 32 heads 7.9 | 8.3, 8.9 | 8.4, 9.9 | 8.7, 12.1 | 9.0. Heads of 64: 32 of 8 at 352 / 448
// 7.5 | 8.8, 8.4 | 8.8, a KV head each, 32 heads at 256 / 352 6.9 | 7.4, 8.0 | 7.5 (6.5 | 7.3). A quantized cache takes the f32 one's way, whose bits it promises, though it reads a
// quarter: Q8_0, 40 heads of 8 at 256 / 288 / 352 rows 7.6 | 8.8, 7.8 | 8.5, 8.8 | 9.6; a KV head each, 8 heads at 192 / 256 / 352 6.8 | 7.6, 7.4 | 7.7, 8.5 | 8.1.
constexpr size_t ATT_SHORT = 352, ATT_SHORT_128 = 256, ATT_SHORT_OWN = 192, ATT_WIDE_FROM = 97;
bool attn_per_query_head(size_t len, int n_head, int n_kv, int hd, bool ws = true) {   // ws: splits have a workspace to go to
    return len <= (!ws || hd != 128 ? ATT_SHORT : n_head == n_kv ? ATT_SHORT_OWN : ATT_SHORT_128);
}
bool attn_wide(size_t len) { return len >= ATT_WIDE_FROM; }

// Beyond that, up to ATT_MID rows under grouped query heads: one workgroup per (query head, split of at least ATT_MID_KEYS
// keys). The kernel that takes all query heads of a KV head at once holds 180 registers a lane (two waves per SIMD) and its
// waves spend their time in the dependent arithmetic of five softmax chains; with one head a workgroup (107 registers, four
// waves per SIMD) the same arithmetic is spread over five times the waves, and the rows they share come out of one XCD's L2
// (see the kernel's workgroup numbering). Chained 64-layer step, ms per token, this shape | all heads of a KV head per
// workgroup: 500 keys 3.99 | 4.24, 1000: 4.06 | 4.28, 2048: 4.22 | 4.56, 4096: 4.63 | 4.77, 6000: 4.97 | 4.90, 8000: 5.41 | 5.08.
constexpr size_t ATT_MID = 5120, ATT_MID_KEYS = 128;
bool attn_per_head_splits(size_t len, int n_head, int n_kv) { return n_kv > 0 && n_head > n_kv && len <= ATT_MID; }   // (asked behind attn_per_query_head)
// splits of at least ATT_MID_KEYS keys, at most about two and a half workgroups per CU over all query heads
int attn_mid_splits(size_t len, int n_head) {
    const int by_keys = (int)((len + ATT_MID_KEYS - 1) / ATT_MID_KEYS), cap = 5 * device_cus() / 2 / (n_head > 0 ? n_head : 1);
    const int s = by_keys < cap ? by_keys : cap;
    return s < 1 ? 1 : (s > 256 ? 256 : s);
}

// Splits of the key range otherwise: about two workgroups per CU over all KV heads, at least 64 keys each (two rounds of the
// workgroup's 16 streams x 2 keys), at most 256 (the combine kernel's LDS tables).
int attn_splits(size_t len, int n_kv) {
    if (n_kv <= 0) return 1;
    constexpr int keys = 64;
    int want = (2 * device_cus() + n_kv - 1) / n_kv;
    size_t by_keys = (len + (size_t)keys - 1) / (size_t)keys;
    int splits = (int)(by_keys < (size_t)want ? by_keys : (size_t)want);
    return splits < 1 ? 1 : (splits > 256 ? 256 : splits);
}

// the most splits any launch shape takes for this cache length: what the workspace has to hold
int attn_ws_splits(size_t len, int n_head, int n_kv, int hd) {
    if (attn_per_query_head(len, n_head, n_kv, hd)) return 1;
    const int a = attn_splits(len, n_kv);
    const int b = attn_per_head_splits(len, n_head, n_kv) ? attn_mid_splits(len, n_head) : 1;
    return a > b ? a : b;
}

int launch_decode_attention(const float* q, const float* K, const float* V, int n_head, int n_kv, int hd, size_t len, const uint32_t* d_len,
                            size_t window, float softcap, float* ws, float* out, hipStream_t s) {
    if (n_head == 0 || hd == 0) return FHIP_OK;
    if (len == 0) return set_error(FHIP_ERR_SHAPE, "decode_attention: empty cache");
    if (n_kv <= 0 || n_head % n_kv != 0) return set_error(FHIP_ERR_SHAPE, "decode_attention: n_heads must be a multiple of n_kv_heads");
    if (hd != 64 && hd != 128) return set_error(FHIP_ERR_SHAPE, "decode_attention: head_dim must be 64 or 128");
    if (len > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "decode_attention: cache length exceeds 2^31");
    const int g = n_head / n_kv;
    const float scale = 1.0f / sqrtf((float)hd);
    const uint32_t win = window > 0x7FFFFFFFull ? 0u : (uint32_t)window;   // a window that large is no window
    if (g > 8) return set_error(FHIP_ERR_SHAPE, "decode_attention: %d query heads per KV head (1..=8 supported)", g);
    if (attn_per_query_head(len, n_head, n_kv, hd, ws != nullptr)) {
        int rc = launch_attn_g<1>(hd, dim3((unsigned)n_head, 1), s, q, K, V, n_kv, (uint32_t)len, d_len, scale, 1, win, softcap, ws, out, g, attn_wide(len));
        return rc ? rc : check_hip(hipGetLastError(), "decode_attention launch");
    }
    const bool mid = attn_per_head_splits(len, n_head, n_kv);
    const int splits = mid ? attn_mid_splits(len, n_head) : attn_splits(len, n_kv);
    if (splits > 1 && !ws) return set_error(FHIP_ERR_ARG, "decode_attention: this cache length needs the workspace");
    dim3 grid((unsigned)n_kv, (unsigned)splits);
    int rc;
    if (mid) {
        const unsigned wgs = (unsigned)((n_kv * splits + 7) / 8 * 8 * g);
        rc = launch_attn_g<1>(hd, dim3(wgs, 1), s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out, -g);
    } else
    switch (g) {
        case 1: rc = launch_attn_g<1>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        case 2: rc = launch_attn_g<2>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        case 3: rc = launch_attn_g<3>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        case 4: rc = launch_attn_g<4>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        case 5: rc = launch_attn_g<5>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        case 6: rc = launch_attn_g<6>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        case 7: rc = launch_attn_g<7>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        case 8: rc = launch_attn_g<8>(hd, grid, s, q, K, V, n_kv, (uint32_t)len, d_len, scale, splits, win, softcap, ws, out); break;
        default: return set_error(FHIP_ERR_SHAPE, "decode_attention: %d query heads per KV head (1..=8 supported)", g);
    }
    if (rc) return rc;
    if ((rc = check_hip(hipGetLastError(), "decode_attention launch"))) return rc;
    if (splits > 1) {
        launch_attn_combine(ws, n_head, hd, splits, out, s);
        rc = check_hip(hipGetLastError(), "decode_attention combine launch");
    }
    return rc;
}

// One query row over a quantized cache: q, or, with fp, formed from the raw QKV row whose key and value are appended first.
static int launch_attention_over_kvq(const char* who, int fmt, const float* q, const QkvPostParams* fp, const KvqStore& cache, int n_head, int n_kv, int hd, size_t len,
                                     const uint32_t* d_len, size_t window, float softcap, float* ws, float* out, hipStream_t s) {
    if (n_head == 0 || hd == 0) return FHIP_OK;
    if (len == 0) return set_error(FHIP_ERR_SHAPE, "%s: empty cache", who);
    if (n_kv <= 0 || n_head % n_kv != 0) return set_error(FHIP_ERR_SHAPE, "%s: n_heads must be a multiple of n_kv_heads", who);
    if (hd != 64 && hd != 128) return set_error(FHIP_ERR_SHAPE, "%s: head_dim must be 64 or 128", who);
    if (len > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "%s: cache length exceeds 2^31", who);
    const int g = n_head / n_kv;
    const bool per_head = g >= 1 && g <= 8 && attn_per_query_head(len, n_head, n_kv, hd, ws != nullptr);   // as the f32 cache's launch: the same sums, the same bits
    const bool mid = g >= 1 && g <= 8 && attn_per_head_splits(len, n_head, n_kv);
    int splits = per_head ? 1 : mid ? attn_mid_splits(len, n_head) : attn_splits(len, n_kv);
    const bool lng = !per_head && !mid && splits > 1 && attn_long_takes(fmt, g, n_kv, cache.k_codes);
    if (lng) splits = attn_long_splits(splits);
    if (splits > 1 && !ws) return set_error(FHIP_ERR_ARG, "%s: this cache length needs the workspace", who);
    const KvqLaunch a{s, q, fp, cache, n_kv, (uint32_t)len, d_len, 1.0f / sqrtf((float)hd), splits, window > 0x7FFFFFFFull ? 0u : (uint32_t)window, softcap, ws, out};
    const dim3 grid = per_head ? dim3((unsigned)n_head, 1) : mid ? dim3((unsigned)((n_kv * splits + 7) / 8 * 8 * g), 1) : dim3((unsigned)n_kv, (unsigned)splits);
    const int G = per_head || mid ? 1 : g, gq = per_head ? g : mid ? -g : g;
    const bool wide = per_head && attn_wide(len);
    int rc = FHIP_OK;
    switch (fmt) {
        case FHIP_KVQ_Q8_0:
            if (lng) launch_attn_long_kvq<FHIP_KVQ_Q8_0>(g, hd, grid, a);
            else rc = launch_attn_kvq<FHIP_KVQ_Q8_0>(G, hd, grid, a, gq, wide);
            break;
        case FHIP_KVQ_Q4_0:
            if (lng) launch_attn_long_kvq<FHIP_KVQ_Q4_0>(g, hd, grid, a);
            else rc = launch_attn_kvq<FHIP_KVQ_Q4_0>(G, hd, grid, a, gq, wide);
            break;
        case FHIP_KVQ_Q4_1:
            if (lng) launch_attn_long_kvq<FHIP_KVQ_Q4_1>(g, hd, grid, a);
            else rc = launch_attn_kvq<FHIP_KVQ_Q4_1>(G, hd, grid, a, gq, wide);
            break;
        default: return set_error(FHIP_ERR_ARG, "%s: unknown KV format %d", who, fmt);
    }
    if (rc) return rc;
    if ((rc = check_hip(hipGetLastError(), "decode_attention launch"))) return rc;
    if (splits > 1) {
        launch_attn_combine(ws, n_head, hd, splits, out, s);
        rc = check_hip(hipGetLastError(), "decode_attention combine launch");
    }
    return rc;
}

int launch_decode_attention_kvq(int fmt, const float* q, const uint32_t* k_codes, const uint16_t* k_scales, const uint32_t* v_codes,
                                const uint16_t* v_scales, int n_head, int n_kv, int hd, size_t len, const uint32_t* d_len, size_t window,
                                float softcap, float* ws, float* out, hipStream_t s) {
    // (read only: without fp nothing is appended)
    const KvqStore cache{const_cast<uint32_t*>(k_codes), const_cast<uint16_t*>(k_scales), const_cast<uint32_t*>(v_codes), const_cast<uint16_t*>(v_scales)};
    return launch_attention_over_kvq("decode_attention", fmt, q, nullptr, cache, n_head, n_kv, hd, len, d_len, window, softcap, ws, out, s);
}

static QkvPostParams one_token_post(const float* qkv, const float* bias, const float* q_norm, const float* k_norm, const uint32_t* d_pos, const float* freq_scale, int n_head,
                                    int n_kv, int hd, int n_rot, bool interleaved, float eps, float base, size_t cap) {
    QkvPostParams fp;
    fp.qkv = qkv; fp.bias = bias; fp.q_norm = q_norm; fp.k_norm = k_norm; fp.pos = d_pos; fp.freq_scale = freq_scale;
    fp.q_out = nullptr; fp.k_cache = nullptr; fp.v_cache = nullptr;
    fp.t = 1; fp.n_head = n_head; fp.n_kv = n_kv; fp.hd = hd; fp.n_rot = n_rot; fp.interleaved = interleaved ? 1 : 0;
    fp.cap = (uint32_t)cap; fp.eps = eps; fp.rate = rope_rate(n_rot, base); fp.kv_packed = 0;
    return fp;
}

int launch_qkv_post_attention_kvq(int fmt, const float* qkv, const float* bias, const float* q_norm, const float* k_norm, const uint32_t* d_pos, const float* freq_scale,
                                  int n_head, int n_kv, int hd, int n_rot, bool interleaved, float eps, float base, uint32_t* k_codes, uint16_t* k_scales, uint32_t* v_codes,
                                  uint16_t* v_scales, size_t cap, size_t len, size_t window, float softcap, float* ws, float* out, hipStream_t s) {
    if (len > cap) return set_error(FHIP_ERR_SHAPE, "qkv_post_attention_kvq: length outside the cache");
    const QkvPostParams fp = one_token_post(qkv, bias, q_norm, k_norm, d_pos, freq_scale, n_head, n_kv, hd, n_rot, interleaved, eps, base, cap);
    return launch_attention_over_kvq("qkv_post_attention_kvq", fmt, nullptr, &fp, KvqStore{k_codes, k_scales, v_codes, v_scales}, n_head, n_kv, hd, len, d_pos, window, softcap, ws,
                                     out, s);
}

int launch_qkv_post_attention(const float* qkv, const float* bias, const float* q_norm, const float* k_norm, const uint32_t* d_pos,
                              const float* freq_scale, int n_head, int n_kv, int hd, int n_rot, bool interleaved, float eps, float base,
                              float* k_cache, float* v_cache, size_t cap, size_t len, size_t window, float softcap, float* ws, float* out,
                              hipStream_t s) {
    if (n_head == 0 || hd == 0) return FHIP_OK;
    if (len == 0) return set_error(FHIP_ERR_SHAPE, "qkv_post_attention: empty cache");
    if (n_kv <= 0 || n_head % n_kv != 0) return set_error(FHIP_ERR_SHAPE, "qkv_post_attention: n_heads must be a multiple of n_kv_heads");
    if (hd != 64 && hd != 128) return set_error(FHIP_ERR_SHAPE, "qkv_post_attention: head_dim must be 64 or 128");
    if (len > 0x7FFFFFFFull || len > cap) return set_error(FHIP_ERR_SHAPE, "qkv_post_attention: length outside the cache");
    const int g = n_head / n_kv;
    const bool mid = g <= 8 && attn_per_head_splits(len, n_head, n_kv);
    const bool per_head = attn_per_query_head(len, n_head, n_kv, hd, ws != nullptr);
    const int splits = per_head ? 1 : (mid ? attn_mid_splits(len, n_head) : attn_splits(len, n_kv));
    if (splits > 1 && !ws) return set_error(FHIP_ERR_ARG, "qkv_post_attention: this cache length needs the workspace");
    QkvPostParams fp = one_token_post(qkv, bias, q_norm, k_norm, d_pos, freq_scale, n_head, n_kv, hd, n_rot, interleaved, eps, base, cap);
    fp.k_cache = k_cache; fp.v_cache = v_cache;
    const float scale = 1.0f / sqrtf((float)hd);
    const uint32_t win = window > 0x7FFFFFFFull ? 0u : (uint32_t)window;
    if (g > 8) return set_error(FHIP_ERR_SHAPE, "qkv_post_attention: %d query heads per KV head (1..=8 supported)", g);
    if (per_head) {
        // every workgroup of a KV head forms the new token's K and V rows and stores them (the same bits from each) before
        // it reads them back with the other keys
        int rc = launch_attn_fused_g<1>(hd, dim3((unsigned)n_head, 1), s, fp, n_kv, (uint32_t)len, d_pos, scale, 1, win, softcap, ws, out, g, attn_wide(len));
        return rc ? rc : check_hip(hipGetLastError(), "qkv_post_attention launch");
    }
    dim3 grid((unsigned)n_kv, (unsigned)splits);
    int rc;
    if (mid) {
        const unsigned wgs = (unsigned)((n_kv * splits + 7) / 8 * 8 * g);
        rc = launch_attn_fused_g<1>(hd, dim3(wgs, 1), s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out, -g);
    } else
    switch (g) {
        case 1: rc = launch_attn_fused_g<1>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        case 2: rc = launch_attn_fused_g<2>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        case 3: rc = launch_attn_fused_g<3>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        case 4: rc = launch_attn_fused_g<4>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        case 5: rc = launch_attn_fused_g<5>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        case 6: rc = launch_attn_fused_g<6>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        case 7: rc = launch_attn_fused_g<7>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        case 8: rc = launch_attn_fused_g<8>(hd, grid, s, fp, n_kv, (uint32_t)len, d_pos, scale, splits, win, softcap, ws, out); break;
        default: return set_error(FHIP_ERR_SHAPE, "qkv_post_attention: %d query heads per KV head (1..=8 supported)", g);
    }
    if (rc) return rc;
    if ((rc = check_hip(hipGetLastError(), "qkv_post_attention launch"))) return rc;
    if (splits > 1) {
        launch_attn_combine(ws, n_head, hd, splits, out, s);
        rc = check_hip(hipGetLastError(), "qkv_post_attention combine launch");
    }
    return rc;
}

}  // namespace fhip
