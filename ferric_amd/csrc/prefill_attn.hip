// Causal attention for a block of query rows against the cache (prefill, chunked prefill, prefix-cached suffixes), gfx950.
//
//   out[i, h] = softmax_j(q[i, h] . K[j, kv(h)] / sqrt(dh)) @ V[:, kv(h)],   j <= off + i,   off = S - T
//
// One op for the reference's causal_attention (crates/ferric-tensor/src/nn.rs:40-57), causal_attention_win (:66-88, keys older
// than `window` masked), chunked_attention (:239-265, T query rows against S >= T cached rows, query i at position off + i)
// and flash_attention_prefill (crates/ferric-llama/src/qwen3.rs:925: "all three are the same math"), with the Gemma-2 score
// softcap (:59-61). The reference composes it from permutes, two batched matmuls and a masked softmax over a [nh, T, S] score
// tensor (or a WGSL flash kernel up to its shared-memory limit); here it is one flash-style launch on the matrix cores, at f32's grade.
//
// Two kernels: causal_attn_cut_kernel, on bf16 matrix instructions with every f32 operand cut into three bf16 values, is what a caller gets;
// causal_attn_kernel, on f32 matrix instructions, is what fhip_causal_attention_f32_products gives (prompts on a block-quantized cache,
// whose codes would be others and no better ones: the header). Measured, us, f32 -> cut, 40 query and 8 KV heads of 128: 509 rows x 809 keys 102.9 -> 72.6, 2048 x 2048 432 ->
// 274, 512 x 8192 1163 -> 789; few workgroups: 39 x 929, 8 heads 85.7 -> 70.3; heads of 64: 512 x 512, 32 heads 31.7 -> 27.7, 49 x 49 7.0 ->
// 6.8. Relative error against f64, same shapes: 5.6e-7 -> 4.5e-7, 4.5e-7 -> 3.7e-7, 1.65e-6 -> 1.41e-6, 6.8e-7 -> 5.6e-7, 2.7e-7 -> 2.0e-7,
// 1.7e-7 -> 1.2e-7. What bounds the cut kernel: the chain of a tile (cut and store 32 keys, products, statistics, products: 2.2 us a wave
// alone on its SIMD, of which 0.65 are MFMA) at one or two waves a SIMD, one tile after the other. So where the query blocks leave CUs idle, or one
// with two blocks working last, their keys are split between workgroups, whose sums a second launch joins (fhip_causal_attention_split): 509 x 809 rows 71.9 -> 56.8, 95 x 722, 8
// heads 54.4 -> 14.2 (causal_split). Error against f64 with ranges: no larger, sums are shorter.
//
// Why f32 matrix instructions (the second kernel, and the first one's tiling). v_mfma_f32_16x16x4_f32 multiplies f32 operands exactly and accumulates in f32: results have the
// grade of the reference's f32 arithmetic (the tests hold them to 1e-5 of the largest output against an f64 evaluation), where
// bf16 operands would leave three digits. It runs at the chip's f32 matrix rate (157 TFLOP/s), a sixteenth of bf16's.
//
// Tiling. A wave owns 16 query rows of one head; lane (c, ks) = (lane % 16, lane / 16). It keeps its query fragment in
// registers for the whole launch (query c, quarter ks of the dims: dh / 4 registers) and walks the key tiles of 32 rows that
// its queries may see. Per tile, with the two 16-key halves u = 0, 1:
//   S^T_u [16 keys x 16 queries] = K_u [16 x dh] . Q^T         (dh / 4 instructions each; an instruction's four k are one
//                                                               dim of every quarter)
//   online softmax down each column: a lane holds keys 16 u + 4 ks + i (i < 4) of ITS query, the other three lane groups the
//                                    rest, so a query's statistics are 8 register operations and two exchanges
//   O^T [dh x 16 queries] += V_tile^T [dh x 32 keys] . P^T     (dh / 16 output tiles x 8 instructions)
// Computing the transposes is what makes the second product free of data movement: register i of S^T_u in lane group ks is the
// probability of key 16 u + 4 ks + i for the lane's query, which is exactly the B operand of an instruction whose four k are
// the keys 16 u + 4 ks' + i (ks' = 0..3); the A operand reads those keys' value rows from LDS. The probabilities never leave
// their registers. Which dim an output row stands for is free as well: row m of output tile d is dim (dh / 16) m + d, so a
// lane's A operands of the dh / 16 instructions of a step are consecutive floats of one value row.
// Sixteen-row tiles rather than 32 x 32 ones keep a wave at 32 + 32 + 8 registers of fragments instead of 64 + 64 + 16, which
// is what leaves room to request the next K and V tile a tile ahead: with the larger tile the compiler had to move every
// prefetched piece out of the way as it arrived, one memory round trip after the other.
// The K and V tiles of a KV head go through LDS (K rows padded by 4 floats so that the 16-byte reads of a lane group start 4
// banks apart), shared by the 8 waves (128 queries) of a workgroup; workgroups of the same KV head read the same rows out of
// L2. Query blocks are issued longest first across all heads.
#include "common.hpp"
#include "prompt.hpp"

#include <math.h>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Output rows as f32, or as bf16 (rounded as fhip_cvt_f32_bf16 rounds them) for a matmul on the matrix cores.
using fhip::pk_bf16;
__device__ __forceinline__ void store_out(float* p, float4 v) { *(float4*)p = v; }
__device__ __forceinline__ void store_out(uint16_t* p, float4 v) { *(uint2*)p = make_uint2(pk_bf16(v.x, v.y), pk_bf16(v.z, v.w)); }

// Scores of a lane's query, at position qpos, against its keys j .. j + 3
__device__ __forceinline__ void scores(f32x4& s, int j, int qpos, bool whole, float scale, int window, float softcap) {
#pragma unroll
    for (int r = 0; r < 4; r++) s[r] *= scale;
    if (softcap > 0.f) {
#pragma unroll
        for (int r = 0; r < 4; r++) s[r] = softcap * tanhf(s[r] / softcap);    // cap * tanh(x / cap), crates/ferric-tensor/src/lib.rs:308
    }
    if (!whole) {
#pragma unroll
        for (int r = 0; r < 4; r++) s[r] = j + r <= qpos && (window == 0 || qpos - (j + r) < window) ? s[r] : -3.0e38f;   // nn.rs:128-133
    }
}
// A tile's scores into weights under the running statistics; returns what the sums so far are multiplied by.
__device__ __forceinline__ float weights(f32x4 (&s)[2], float& m, float& l) {
    float mt = -3.0e38f;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int r = 0; r < 4; r++) mt = fmaxf(mt, s[u][r]);
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
    mt = fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
    const float m_new = fmaxf(m, fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1])));
    const float corr = __expf(m - m_new);
    float ps = 0.f;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float p = s[u][r] > -2.9e38f ? __expf(s[u][r] - m_new) : 0.f;
            s[u][r] = p;
            ps += p;
        }
    l = fmaf(l, corr, ps);
    m = m_new;
    return corr;
}

// NW: waves (16 query rows each) per workgroup. STAGED: the workgroup's waves call it together and share the tiles in Ks [32][HD + 4] and Vs
// [32][HD]. Otherwise a wave comes alone, waits for no other and takes its operands from memory: the same instructions on the same
// values, the same bits, about three times the time.
template <int HD, int NW, bool STAGED, typename Out>
__device__ __forceinline__ void f32_body(float* Ks, float* Vs, const float* __restrict__ q, const float* __restrict__ K, const float* __restrict__ V, int T, int S, int n_head, int n_kv,
                                         float scale, int window, float softcap, Out* __restrict__ out) {
    constexpr int KS = HD + 4;              // floats per K row in LDS
    constexpr int QD = HD / 4;              // dims per quarter
    constexpr int NDT = HD / 16;            // output tiles of 16 rows
    constexpr int QROWS = 16 * NW;          // query rows per workgroup
    constexpr int NF = 32 * (HD / 4) / (64 * NW);   // 16-byte pieces of a K (and of a V) tile per thread
    static_assert(NF >= 1 && NF * 64 * NW == 32 * (HD / 4), "the tile divides over the threads");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, ks = lane >> 4;
    // Workgroups are handed out x first: all heads' last query blocks (which see the most keys), then all heads' second to
    // last, ... -- longest first over the whole launch, so the long ones do not start late and finish alone.
    const int head = blockIdx.x, kvh = head / (n_head / n_kv);
    const int qb = (int)gridDim.y - 1 - (int)blockIdx.y;
    const int off = S - T;
    const int wg_first = qb * QROWS, wg_last = min(T - 1, wg_first + QROWS - 1);
    const int i0 = wg_first + wave * 16;
    const bool wave_live = i0 < T;                              // a wave past the last query row only helps to load tiles
    const int i_last = min(i0 + 15, T - 1);
    const int i = min(i0 + c, T - 1), qpos = off + i;           // this lane's query row and its absolute position
    // key tiles the workgroup walks, and the ones this wave's queries can see
    const int kt_hi = (off + wg_last) / 32;
    const int kt_lo = window > 0 ? max(0, off + wg_first - window + 1) / 32 : 0;
    const int my_hi = wave_live ? (off + i_last) / 32 : -1;
    const int my_lo = window > 0 ? max(0, off + i0 - window + 1) / 32 : 0;

    float qf[QD];
    {
        const float* qp = q + ((size_t)i * n_head + head) * HD + ks * QD;
#pragma unroll
        for (int t = 0; t < QD; t += 4) {
            const float4 v = *(const float4*)(qp + t);
            qf[t] = v.x; qf[t + 1] = v.y; qf[t + 2] = v.z; qf[t + 3] = v.w;
        }
    }
    f32x4 oacc[NDT];
#pragma unroll
    for (int d = 0; d < NDT; d++) oacc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -3.0e38f, l = 0.f;
    const size_t kv_stride = (size_t)n_kv * HD;
    const float* Kh = K + (size_t)kvh * HD;
    const float* Vh = V + (size_t)kvh * HD;

    // The next tile's pieces wait in registers while the current tile is worked on (native vectors, indexed by unrolled
    // loops only: anything the compiler cannot keep in registers here lands in scratch memory, and every piece is then waited
    // for and stored as it arrives, one memory round trip after the other).
    f32x4 kreg[NF], vreg[NF];
    int prow[NF], pcol[NF];
#pragma unroll
    for (int n = 0; n < NF; n++) {
        const int f = tid + n * 64 * NW;
        prow[n] = f / (HD / 4);
        pcol[n] = (f % (HD / 4)) * 4;
    }
    auto request = [&](int kt) {
#pragma unroll
        for (int n = 0; n < NF; n++) {
            // rows past the cache repeat its last row; they are masked below
            const size_t src = (size_t)min(kt * 32 + prow[n], S - 1) * kv_stride + (size_t)pcol[n];
            kreg[n] = *(const f32x4*)(Kh + src);
            vreg[n] = *(const f32x4*)(Vh + src);
        }
    };
    if (STAGED) request(kt_lo);
    for (int kt = STAGED ? kt_lo : my_lo; kt <= (STAGED ? kt_hi : my_hi); kt++) {
        if constexpr (STAGED) {
            __syncthreads();                                    // every wave is done with the previous tile
#pragma unroll
            for (int n = 0; n < NF; n++) {
                *(f32x4*)(Ks + prow[n] * KS + pcol[n]) = kreg[n];
                *(f32x4*)(Vs + prow[n] * HD + pcol[n]) = vreg[n];
            }
            __syncthreads();
            request(min(kt + 1, kt_hi));                        // in flight under this tile's arithmetic
            if (kt < my_lo || kt > my_hi) continue;             // wave-uniform; the barriers above are reached by every wave
        }

        // the two halves' chains alternate, so an instruction does not wait for the result of the one before it
        f32x4 sacc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        const float* krow = STAGED ? Ks + c * KS + ks * QD : Kh + (size_t)min(kt * 32 + c, S - 1) * kv_stride + ks * QD;
        const float* krow16 = STAGED ? krow + 16 * KS : Kh + (size_t)min(kt * 32 + 16 + c, S - 1) * kv_stride + ks * QD;
#pragma unroll
        for (int t = 0; t < QD; t += 4) {
            const float4 k0 = *(const float4*)(krow + t), k1 = *(const float4*)(krow16 + t);
            sacc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k0.x, qf[t], sacc[0], 0, 0, 0);
            sacc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k1.x, qf[t], sacc[1], 0, 0, 0);
            sacc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k0.y, qf[t + 1], sacc[0], 0, 0, 0);
            sacc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k1.y, qf[t + 1], sacc[1], 0, 0, 0);
            sacc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k0.z, qf[t + 2], sacc[0], 0, 0, 0);
            sacc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k1.z, qf[t + 2], sacc[1], 0, 0, 0);
            sacc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k0.w, qf[t + 3], sacc[0], 0, 0, 0);
            sacc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k1.w, qf[t + 3], sacc[1], 0, 0, 0);
        }
        // a tile every query of the wave sees whole needs no mask
        const bool whole = kt * 32 + 31 <= off + i0 && (window == 0 || off + i_last - kt * 32 < window);
#pragma unroll
        for (int u = 0; u < 2; u++) scores(sacc[u], kt * 32 + 16 * u + 4 * ks, qpos, whole, scale, window, softcap);
        const float corr = weights(sacc, m, l);
#pragma unroll
        for (int d = 0; d < NDT; d++) oacc[d] *= corr;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int key = 16 * u + 4 * ks + r;
                const float* vrow = (STAGED ? Vs + key * HD : Vh + (size_t)min(kt * 32 + key, S - 1) * kv_stride) + NDT * c;
                float va[NDT];
#pragma unroll
                for (int d = 0; d < NDT; d += 4) {
                    const float4 t4 = *(const float4*)(vrow + d);
                    va[d] = t4.x; va[d + 1] = t4.y; va[d + 2] = t4.z; va[d + 3] = t4.w;
                }
#pragma unroll
                for (int d = 0; d < NDT; d++) oacc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[d], sacc[u][r], oacc[d], 0, 0, 0);
            }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (!wave_live || i0 + c >= T) return;
    const float inv = 1.0f / l;
    // register r of output tile d is row m = 4 ks + r, i.e. dim NDT m + d
    Out* op = out + ((size_t)i * n_head + head) * HD;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        Out* dst = op + NDT * (4 * ks + r);
#pragma unroll
        for (int d = 0; d < NDT; d += 4)
            store_out(dst + d, float4{oacc[d][r] * inv, oacc[d + 1][r] * inv, oacc[d + 2][r] * inv, oacc[d + 3][r] * inv});
    }
}

template <int HD, int NW, typename Out>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 4 : 2) void causal_attn_kernel(const float* __restrict__ q, const float* __restrict__ K, const float* __restrict__ V, int T,
                                                              int S, int n_head, int n_kv, float scale, int window, float softcap,
                                                              Out* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) float Ks[32 * (HD + 4)];    // floats per K row in LDS: four banks on from row to row
    __shared__ __attribute__((aligned(16))) float Vs[32 * HD];
    f32_body<HD, NW, true>(Ks, Vs, q, K, V, T, S, n_head, n_kv, scale, window, softcap, out);
}

// The key tiles that the query rows wg_first .. wg_last see, at least one.
struct KeyTiles {
    int lo, hi;
    __host__ __device__ int count() const { return hi - lo + 1; }
};
__host__ __device__ inline KeyTiles key_tiles(int off, int wg_first, int wg_last, int window) {
    const int first = off + wg_first - window + 1;
    return {window > 0 && first > 0 ? first / 32 : 0, (off + wg_last) / 32};
}

// 16 query rows of a head by a workgroup of four waves, for launches whose rows would leave SIMDs idle at a wave each (team_pays). A step is two key tiles:
// wave w takes the products of keys 16 w .. 16 w + 15 with the queries, the scores go to the others through LDS, every wave forms all weights and takes a
// quarter of the outputs' dims over all of the step's keys. Each sum is over the same products in the same order as where a wave has its rows to itself: the
// same bits. No two waves want the same K row or the same dims of V, so K goes through LDS only to be read coalesced, by the wave that multiplies it, and V not
// at all; one barrier a step, for the scores. The next step's products (one chain of dh / 4 instructions) run beside this step's weights, the next loads
// beside its outputs.
//
// What bounds it: 64 KB a step at head size 128 through one CU's L1, 28 bytes a ns, 1.9 us (1.2 us for 32 KB), of which the products are 0.9 at 2.4 GHz. Stages
// one after the other took 2.4 (issue of the loads 0.6, products 0.5, scores and their way through LDS 0.3, weights 0.2, outputs 0.8); K and V staged in
// LDS for all waves, three barriers, 2.6; eight waves and four tiles a step the same time a tile. us, a wave per 16 rows -> this (rows x keys, heads, KV
// heads, head size): 33 x 1057, 4, 4, 128 91.9 -> 34.2; 95 x 722, 8, 8, 128 63.5 -> 25.4; 152 x 152, 8, 4, 128 16.3 -> 8.9; 234 x 355, 32, 4, 128 36.2 -> 21.3;
// 509 x 809, 16, 8, 128 73.2 -> 40.5; 152 x 940, 8, 8, 64 48.3 -> 21.3; 512 x 512, 32, 8, 64 29.0 -> 21.9; 60 x 60, 16, 4, 64 6.0 -> 4.3.
template <int HD, typename Out>
__global__ __launch_bounds__(256, 2) void causal_attn_team_kernel(const float* __restrict__ q, const float* __restrict__ K, const float* __restrict__ V, int T,
                                                                  int S, int n_head, int n_kv, float scale, int window, float softcap,
                                                                  Out* __restrict__ out) {
    constexpr int KEYS = 64, QD = HD / 4;
    constexpr int NE = HD / 64;                 // output tiles of 16 dims a wave
    constexpr int KS = HD + 4;                  // floats a K row in LDS
    constexpr int NF = HD / 16;                 // 16-byte pieces of a wave's 16 K rows a lane
    constexpr int RL = HD / 4;                  // lanes a K row
    typedef float vec __attribute__((ext_vector_type(NE)));
    __shared__ __attribute__((aligned(16))) float Ks[KEYS * KS];        // each wave its own rows
    __shared__ __attribute__((aligned(16))) f32x4 Ss[2][256];           // scores [16 keys][lane], four keys of a query: a step's, the next one's
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, ks = lane >> 4;
    const int head = blockIdx.x, kvh = head / (n_head / n_kv);
    const int i0 = 16 * ((int)gridDim.y - 1 - (int)blockIdx.y);         // longest first
    const int off = S - T, i_last = min(i0 + 15, T - 1);
    const int i = min(i0 + c, T - 1), qpos = off + i;
    const KeyTiles seen = key_tiles(off, i0, i_last, window);
    const unsigned row_bytes = (unsigned)n_kv * HD * 4;                 // 64 rows of it stay under 2^32
    const int last_step = seen.lo + (seen.hi - seen.lo) / 2 * 2;

    float qf[QD];
    {
        const float* qp = q + ((size_t)i * n_head + head) * HD + ks * QD;
#pragma unroll
        for (int t = 0; t < QD; t += 4) {
            const f32x4 v = *(const f32x4*)(qp + t);
#pragma unroll
            for (int e = 0; e < 4; e++) qf[t + e] = v[e];
        }
    }
    f32x4 oacc[NE];
#pragma unroll
    for (int e = 0; e < NE; e++) oacc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -3.0e38f, l = 0.f;
    float* kmine = Ks + 16 * wave * KS;
    f32x4 kreg[NF], kf[NF];
    vec v[2][2][4];
    f32x4 sacc;
    // rows past the cache repeat its last row (masked below), steps past the last one that one
    const unsigned kcol = lane % RL * 16, vcol = (16 * wave + c) * NE * 4;
    unsigned krow[NF], vrow[2][2][4];
#pragma unroll
    for (int n = 0; n < NF; n++) krow[n] = (16 * wave + n * (64 / RL) + lane / RL) * row_bytes + kcol;
#pragma unroll
    for (int x = 0; x < 16; x++) vrow[x >> 3][x >> 2 & 1][x & 3] = (16 * (x >> 2) + 4 * ks + (x & 3)) * row_bytes + vcol;
    auto base = [&](const float* p, int kt) { return (const char*)(p + (size_t)kt * 32 * n_kv * HD + kvh * HD); };
    auto end = [&](int kt) { return (unsigned)min(S - 1 - kt * 32, KEYS) * row_bytes; };
    auto request_k = [&](int n, int kt) { kreg[n] = *(const f32x4*)(base(K, kt) + min(krow[n], end(kt) + kcol)); };
    auto request_v = [&](int x, int u, int r, int kt) { v[x][u][r] = *(const vec*)(base(V, kt) + min(vrow[x][u][r], end(kt) + vcol)); };
    auto store_k = [&](int n) { *(f32x4*)(kmine + (n * (64 / RL) + lane / RL) * KS + lane % RL * 4) = kreg[n]; };
    auto fragments = [&]() {
#pragma unroll
        for (int t = 0; t < NF; t++) kf[t] = *(const f32x4*)(kmine + c * KS + ks * QD + 4 * t);
    };
    auto own_rows = [&]() {                     // a wave's rows, written and read by different lanes of it
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto products = [&]() {
        sacc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < QD; t++) sacc = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t / 4][t % 4], qf[t], sacc, 0, 0, 0);
    };
    auto hand_over = [&](int kt, int buf) {
        const int my = kt + (wave >> 1);        // past the last tile: masked
        const bool whole = my * 32 + 31 <= off + i0 && (window == 0 || off + i_last - my * 32 < window);
        scores(sacc, kt * 32 + 16 * wave + 4 * ks, qpos, whole, scale, window, softcap);
        Ss[buf][64 * wave + lane] = sacc;
    };
    f32x4 p[2][2];
    float corr[2];
    auto take = [&](int buf) {
#pragma unroll
        for (int x = 0; x < 4; x++) p[x >> 1][x & 1] = Ss[buf][64 * x + lane];
    };
    auto step_weights = [&]() {
#pragma unroll
        for (int x = 0; x < 2; x++) corr[x] = weights(p[x], m, l);      // of a tile past the last: 1, and m and l stay
    };
    auto outputs = [&](int x, auto beside) {
#pragma unroll
        for (int e = 0; e < NE; e++) oacc[e] *= corr[x];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
#pragma unroll
                for (int e = 0; e < NE; e++) oacc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[x][u][r][e], p[x][u][r], oacc[e], 0, 0, 0);
                beside(x, u, r);
            }
    };

    auto at = [&](int kt) { return min(kt, last_step); };
#pragma unroll
    for (int n = 0; n < NF; n++) request_k(n, seen.lo);
#pragma unroll
    for (int n = 0; n < NF; n++) store_k(n);
#pragma unroll
    for (int n = 0; n < NF; n++) request_k(n, at(seen.lo + 2));
#pragma unroll
    for (int x = 0; x < 16; x++) request_v(x >> 3, x >> 2 & 1, x & 3, seen.lo);
    own_rows();
    fragments();
    products();
    own_rows();
#pragma unroll
    for (int n = 0; n < NF; n++) store_k(n);
#pragma unroll
    for (int n = 0; n < NF; n++) request_k(n, at(seen.lo + 4));
    own_rows();
    fragments();
    hand_over(seen.lo, 0);
    int buf = 0;
    for (int kt = seen.lo; kt < last_step; kt += 2) {
        __syncthreads();    // the only one: scores written next were read before it
        take(buf);
        buf ^= 1;
        products();                             // of the next step
        step_weights();
#pragma unroll
        for (int t = 0; t < QD; t++) {          // the weights beside the products: else these wait for each other first
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 128 / QD, 0);
        }
        own_rows();
        const int then = kt + 2;
        outputs(0, [&](int x, int u, int r) {
            request_v(x, u, r, then);
            if (4 * u + r < NF) store_k(4 * u + r);
        });
        outputs(1, [&](int x, int u, int r) {
            request_v(x, u, r, then);
            if (4 * u + r < NF) request_k(4 * u + r, at(kt + 6));
        });
        own_rows();
        fragments();
        hand_over(then, buf);
    }
    __syncthreads();
    take(buf);
    step_weights();
    outputs(0, [](int, int, int) {});
    if (last_step < seen.hi) outputs(1, [](int, int, int) {});
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (i0 + c >= T) return;
    const float inv = 1.0f / l;
    // register r of output tile e is row 4 ks + r of it, i.e. dim NE (16 wave + 4 ks + r) + e
    Out* op = out + ((size_t)i * n_head + head) * HD + NE * (16 * wave + 4 * ks);
#pragma unroll
    for (int y = 0; y < NE; y++) {
        auto value = [&](int n) { return oacc[n % NE][n / NE] * inv; };
        store_out(op + 4 * y, float4{value(4 * y), value(4 * y + 1), value(4 * y + 2), value(4 * y + 3)});
    }
}

// ------------------------------------------------------------------------------------------------------------------------------
// The same on bf16 matrix instructions. An f32 value is three bf16 values exactly (the nearest to it, the nearest to what is left, and
// what is left then), and a product of two f32 values is, to 2^-25, the six products of their cuts of which one factor at least is the
// first or both the second: six v_mfma_f32_16x16x32_bf16 of 16 cycles for 32 columns of k, where v_mfma_f32_16x16x4_f32 needs eight of 32.
// Sums are f32. Every operand keeps its 24 bits: a third cut is whole down to bf16's smallest value, 2^-133, which values V is multiplied by
// 2^40 for on the way (any f32 then has its last bit above that; exact, and taken off at the end). A query's or key's member under 2^-110
// and a probability under 2^-110 lose what lies below 2^-134: nothing to a score that goes into an exponential, nor to a row of a sum over 1.
//
// What three cuts cannot carry: an infinite member, or one that rounds to infinity, leaves infinity less infinity in the cuts behind, a NaN
// score has no weight in the f32 kernel, and sums near f32's limit can overflow in one cut and not in another. All of these leave a NaN or an
// infinity in a sum of the wave's, or no weight at all, so a wave looks over its sums once at the end, and one that finds such a value does
// its rows again on the f32 kernel's body: there the result is that kernel's, bit for bit. (A score one of whose partial sums passes f32's
// limit downwards counts as one of no weight, as any order of an f32 sum may have it.) What the look and V's factor cost, us: 509 x 809 rows 71.6 -> 72.6,
// 2048 x 2048 272 -> 274, 512 x 8192 777 -> 789, 49 x 49, heads of 64, 6.3 -> 6.8. The largest member kept tile by tile cost twice that (2048 x 2048 275,
// and thirty-two registers unless forced out before the barrier).
//
// Tiles, masks and statistics are the f32 kernel's: a wave owns 16 query rows of one head, lane (c, ks), key tiles of 32 rows. K and V are
// cut once a tile by the workgroup as they go to LDS, K as [plane][key][dim], V as [plane][dim][slot]: slot 8 ks + 4 u + i is key
// 16 u + 4 ks + i, the key whose probability register i of S^T_u holds in lane group ks, so the second product takes the probabilities
// from their registers and a lane's A operand, eight slots of one dim, is one 16-byte read. K rows are padded by 16 bytes and V rows
// (64 bytes) too: 16 lanes then cover the 64 banks once, in the reads and in the 8-byte writes of four keys x four dims a thread.
// ------------------------------------------------------------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// two values into their three cuts, packed in pairs
struct Cuts2 { uint32_t w[3]; };
__device__ __forceinline__ Cuts2 cut2(float a, float b) {
    Cuts2 r;
    r.w[0] = pk_bf16(a, b);
    a -= __uint_as_float(r.w[0] << 16);
    b -= __uint_as_float(r.w[0] & 0xFFFF0000u);
    r.w[1] = pk_bf16(a, b);
    a -= __uint_as_float(r.w[1] << 16);
    b -= __uint_as_float(r.w[1] & 0xFFFF0000u);
    r.w[2] = pk_bf16(a, b);
    return r;
}
// N accumulators' six products, the smallest first; the accumulators take turns, so that none waits for its last product
template <int N>
__device__ __forceinline__ void mfma_cuts(const bf16x8 (&a)[N][3], const bf16x8 (&b)[3], f32x4* acc) {
    constexpr int A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int x = 0; x < 6; x++)
#pragma unroll
        for (int n = 0; n < N; n++) acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n][A[x]], b[B[x]], acc[n], 0, 0, 0);
}

constexpr float V_UP = 0x1p40f;

// the largest magnitude of a lane's sums and of `top`; a NaN stays
template <int ND>
__device__ __forceinline__ float largest(float top, const f32x4 (&acc)[ND]) {
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int r = 0; r < 4; r++) top = __builtin_elementwise_maximum(top, fabsf(acc[d][r]));
    return top;
}

// Of `count` tiles, n ranges of per (the last one's may be fewer; none is empty, since (n - 1) per <= (n - 1) * most < the count).
struct KeyRanges { int n, per; };
__host__ __device__ inline KeyRanges key_ranges(int count, int most) {
    const int n = (count - 1) / most + 1;
    return {n, (count - 1) / n + 1};
}
// What a wave hands over of its 16 rows and one range of keys: [HD / 16][64] accumulators as its lanes hold them, [16] largest scores (NaN: these rows are
// the f32 body's), [16] sums of weights.
constexpr int part_floats(int hd) { return 16 * hd + 32; }
constexpr int CUT_WAVES = 4;                // of a workgroup whose keys are split

// SPLIT: blockIdx.z is a range of keys of at most `most` tiles, and the workgroup leaves what it has of them in `part`, [head][16 rows][ranges] slots, for
// causal_attn_join_kernel.
template <int HD, int NW, bool SPLIT, typename Out>
__global__ __launch_bounds__(64 * NW, 2) void causal_attn_cut_kernel(const float* __restrict__ q, const float* __restrict__ K, const float* __restrict__ V, int T,
                                                                     int S, int n_head, int n_kv, float scale, int window, float softcap,
                                                                     Out* __restrict__ out, float* __restrict__ part, int most) {
    constexpr int KROW = HD + 8;            // bf16 per K row and plane
    constexpr int VROW = 32 + 8;            // bf16 per V dim and plane
    constexpr int KP = 32 * KROW, VP = HD * VROW;   // bf16 per plane
    constexpr int NK = HD / 32;             // k-steps of the first product
    constexpr int ND = HD / 16;             // output tiles of 16 dims
    constexpr int UNITS = 8 * (HD / 4);     // blocks of four keys x four dims in a K (or V) tile
    constexpr int NU = (2 * UNITS + 64 * NW - 1) / (64 * NW);   // of those of K and V together, per thread
    __shared__ __attribute__((aligned(16))) uint16_t Ks[3 * KP];
    __shared__ __attribute__((aligned(16))) uint16_t Vs[3 * VP];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, ks = lane >> 4;
    const int head = blockIdx.x, kvh = head / (n_head / n_kv);
    const int qb = (int)gridDim.y - 1 - (int)blockIdx.y;        // longest first, as in the f32 kernel
    const int off = S - T;
    const int wg_first = qb * 16 * NW, wg_last = min(T - 1, wg_first + 16 * NW - 1);
    const int i0 = wg_first + wave * 16;
    const bool wave_live = i0 < T;
    const int i_last = min(i0 + 15, T - 1);
    const int i = min(i0 + c, T - 1), qpos = off + i;
    const KeyTiles seen = key_tiles(off, wg_first, wg_last, window);
    int kt_lo = seen.lo, kt_hi = seen.hi;
    if constexpr (SPLIT) {
        const KeyRanges kr = key_ranges(seen.count(), most);
        if ((int)blockIdx.z >= kr.n) return;
        kt_lo += (int)blockIdx.z * kr.per;
        kt_hi = min(kt_hi, kt_lo + kr.per - 1);
    }
    const int my_hi = wave_live ? (off + i_last) / 32 : -1;
    const int my_lo = window > 0 ? max(0, off + i0 - window + 1) / 32 : 0;

    bf16x8 qf[NK][3];                       // query c, dims 32 n + 8 ks + [0, 8)
    {
        const float* qp = q + ((size_t)i * n_head + head) * HD + 8 * ks;
#pragma unroll
        for (int n = 0; n < NK; n++) {
            const f32x4 a = *(const f32x4*)(qp + 32 * n), b = *(const f32x4*)(qp + 32 * n + 4);
            const Cuts2 w0 = cut2(a[0], a[1]), w1 = cut2(a[2], a[3]), w2 = cut2(b[0], b[1]), w3 = cut2(b[2], b[3]);
#pragma unroll
            for (int y = 0; y < 3; y++) qf[n][y] = __builtin_bit_cast(bf16x8, (u32x4){w0.w[y], w1.w[y], w2.w[y], w3.w[y]});
        }
    }
    f32x4 oacc[ND];
#pragma unroll
    for (int d = 0; d < ND; d++) oacc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -3.0e38f, l = 0.f;
    const size_t kv_stride = (size_t)n_kv * HD;

    // Unit x of a thread: number tid + 64 NW x, K's first (wave-uniform which). Keys 4 g .. 4 g + 3, dims 4 dq .. 4 dq + 3; of K a
    // wave takes whole rows (dq fastest), of V all eight key groups of eight dims' quads (g fastest).
    f32x4 piece[NU][4];
    int dst[NU];                            // of K: bf16 offset of (key 4 g, dim 4 dq); of V: of (dim 4 dq, slot of key 4 g)
    int key0[NU], dim0[NU];
#pragma unroll
    for (int x = 0; x < NU; x++) {
        const int n = tid + 64 * NW * x, v = n - UNITS;
        const int g = v < 0 ? n / (HD / 4) : v & 7, dq = v < 0 ? n % (HD / 4) : v >> 3;
        key0[x] = 4 * g;
        dim0[x] = 4 * dq;
        dst[x] = v < 0 ? 4 * g * KROW + 4 * dq : 4 * dq * VROW + 8 * (g & 3) + 4 * (g >> 2);
    }
    auto mine = [&](int x) { return 2 * UNITS % (64 * NW) == 0 || wave + NW * x < 2 * UNITS / 64; };
    auto is_k = [&](int x) { return UNITS % (64 * NW) == 0 ? x < UNITS / (64 * NW) : wave + NW * x < UNITS / 64; };
    auto load = [&](int kt) {
#pragma unroll
        for (int x = 0; x < NU; x++)
            if (mine(x)) {
                const float* src = (is_k(x) ? K : V) + (size_t)kvh * HD + dim0[x];
                // rows past the cache repeat its last row; they are masked below
#pragma unroll
                for (int r = 0; r < 4; r++) piece[x][r] = *(const f32x4*)(src + (size_t)min(kt * 32 + key0[x] + r, S - 1) * kv_stride);
            }
    };
    auto store = [&]() {
#pragma unroll
        for (int x = 0; x < NU; x++)
            if (mine(x)) {
                if (is_k(x)) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const Cuts2 w0 = cut2(piece[x][r][0], piece[x][r][1]), w1 = cut2(piece[x][r][2], piece[x][r][3]);
#pragma unroll
                        for (int y = 0; y < 3; y++) *(uint2*)(Ks + y * KP + dst[x] + r * KROW) = make_uint2(w0.w[y], w1.w[y]);
                    }
                } else {
#pragma unroll
                    for (int d = 0; d < 4; d++) {
                        const Cuts2 w0 = cut2(piece[x][0][d] * V_UP, piece[x][1][d] * V_UP), w1 = cut2(piece[x][2][d] * V_UP, piece[x][3][d] * V_UP);
#pragma unroll
                        for (int y = 0; y < 3; y++) *(uint2*)(Vs + y * VP + dst[x] + d * VROW) = make_uint2(w0.w[y], w1.w[y]);
                    }
                }
            }
    };
    load(kt_lo);
    for (int kt = kt_lo; kt <= kt_hi; kt++) {
        __syncthreads();                                        // every wave is done with the previous tile
        store();
        __syncthreads();
        load(min(kt + 1, kt_hi));                               // in flight under this tile's arithmetic
        if (kt < my_lo || kt > my_hi) continue;                 // wave-uniform; the barriers above are reached by every wave

        f32x4 sacc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        const uint16_t* krow = Ks + c * KROW + 8 * ks;
#pragma unroll
        for (int n = 0; n < NK; n++) {
            bf16x8 kf[2][3];
#pragma unroll
            for (int y = 0; y < 3; y++)
#pragma unroll
                for (int u = 0; u < 2; u++) kf[u][y] = *(const bf16x8*)(krow + y * KP + 16 * u * KROW + 32 * n);
            mfma_cuts(kf, qf[n], sacc);
        }
        const bool whole = kt * 32 + 31 <= off + i0 && (window == 0 || off + i_last - kt * 32 < window);
        float sc[8];                                            // of this lane's query against its 8 keys of the tile
#pragma unroll
        for (int x = 0; x < 8; x++) sc[x] = sacc[x >> 2][x & 3] * scale;
        if (softcap > 0.f) {
#pragma unroll
            for (int x = 0; x < 8; x++) sc[x] = softcap * tanhf(sc[x] / softcap);
        }
        if (!whole) {
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const int j = kt * 32 + 16 * (x >> 2) + 4 * ks + (x & 3);
                sc[x] = j <= qpos && (window == 0 || qpos - j < window) ? sc[x] : -INFINITY;   // nn.rs:128-133
            }
        }
        float mt = -3.0e38f;
#pragma unroll
        for (int x = 0; x < 8; x++) mt = fmaxf(mt, sc[x]);
        mt = fmaxf(mt, __shfl_xor(mt, 16));
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float m_new = fmaxf(m, mt);
        const float corr = __expf(m - m_new);
        float ps = 0.f;
#pragma unroll
        for (int x = 0; x < 8; x++) {
            sc[x] = __expf(sc[x] - m_new);                      // 0 of a masked key: m_new is finite
            ps += sc[x];
        }
        l = fmaf(l, corr, ps);
        m = m_new;
        const Cuts2 p0 = cut2(sc[0], sc[1]), p1 = cut2(sc[2], sc[3]), p2 = cut2(sc[4], sc[5]), p3 = cut2(sc[6], sc[7]);
        bf16x8 pf[3];
#pragma unroll
        for (int y = 0; y < 3; y++) pf[y] = __builtin_bit_cast(bf16x8, (u32x4){p0.w[y], p1.w[y], p2.w[y], p3.w[y]});
#pragma unroll
        for (int d = 0; d < ND; d++) oacc[d] *= corr;
        const uint16_t* vrow = Vs + c * VROW + 8 * ks;
#pragma unroll
        for (int d = 0; d < ND; d += 2) {
            bf16x8 vf[2][3];
#pragma unroll
            for (int y = 0; y < 3; y++)
#pragma unroll
                for (int e = 0; e < 2; e++) vf[e][y] = *(const bf16x8*)(vrow + y * VP + (16 * d + 16 * e) * VROW);
            mfma_cuts(vf, pf, oacc + d);
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (!wave_live) return;
    if constexpr (SPLIT) {
        if (my_hi < kt_lo || my_lo > kt_hi) return;             // the join does not ask for it
        const bool bad = !(largest<ND>(l, oacc) < INFINITY);    // rows that see none of these keys have l = 0 and a weight of 0 below
        if (__builtin_amdgcn_ballot_w64(bad) != 0) m = NAN;
        float* slot = part + (((size_t)head * ((T + 15) / 16) + i0 / 16) * gridDim.z + blockIdx.z) * part_floats(HD);
#pragma unroll
        for (int d = 0; d < ND; d++) *(f32x4*)(slot + (64 * d + lane) * 4) = oacc[d];
        if (ks == 0) { slot[16 * HD + c] = m; slot[16 * HD + 16 + c] = l; }
        return;
    }
    const float top = largest<ND>(l > 0.f ? l : INFINITY, oacc);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(top < INFINITY)) != 0, 0)) {
        f32_body<HD, NW, false>(nullptr, nullptr, q, K, V, T, S, n_head, n_kv, scale, window, softcap, out);
        return;
    }
    if (i0 + c >= T) return;
    const float inv = 1.0f / l * (1.0f / V_UP);                 // l <= 2^30: no rounding
    Out* op = out + ((size_t)i * n_head + head) * HD + 4 * ks;   // register r of output tile d is dim 16 d + 4 ks + r
#pragma unroll
    for (int d = 0; d < ND; d++) store_out(op + 16 * d, float4{oacc[d][0] * inv, oacc[d][1] * inv, oacc[d][2] * inv, oacc[d][3] * inv});
}

// The ranges of keys of 16 rows of a head, a wave: sum_j exp(m_j - max m) (acc_j, l_j) in the ranges' order. A wave that finds what the cuts do not carry, in a
// range or in the sum over them, does its rows on the f32 body, as it would have done without ranges.
template <int HD, typename Out>
__global__ __launch_bounds__(64) void causal_attn_join_kernel(const float* __restrict__ q, const float* __restrict__ K, const float* __restrict__ V, int T, int S,
                                                              int n_head, int n_kv, float scale, int window, float softcap, Out* __restrict__ out,
                                                              const float* __restrict__ part, int most, int slots) {
    constexpr int ND = HD / 16;
    const int lane = threadIdx.x, c = lane & 15, ks = lane >> 4;
    const int head = blockIdx.x, tile = (int)gridDim.y - 1 - (int)blockIdx.y, i0 = 16 * tile, off = S - T;   // the f32 body numbers its rows the same way
    const int wg_first = i0 / (16 * CUT_WAVES) * (16 * CUT_WAVES), wg_last = min(T - 1, wg_first + 16 * CUT_WAVES - 1);
    const KeyTiles seen = key_tiles(off, wg_first, wg_last, window);
    const KeyRanges kr = key_ranges(seen.count(), most);
    const int my_hi = (off + min(i0 + 15, T - 1)) / 32, my_lo = window > 0 ? max(0, off + i0 - window + 1) / 32 : 0;
    const int j_lo = (my_lo - seen.lo) / kr.per, j_hi = (my_hi - seen.lo) / kr.per;
    const float* slot = part + ((size_t)head * gridDim.y + tile) * slots * part_floats(HD);
    float m = -3.0e38f;
    bool bad = false;
#pragma unroll 4
    for (int j = j_lo; j <= j_hi; j++) {
        const float mj = slot[(size_t)j * part_floats(HD) + 16 * HD + c];
        bad |= mj != mj;
        m = fmaxf(m, mj);
    }
    f32x4 acc[ND];
#pragma unroll
    for (int d = 0; d < ND; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
#pragma unroll 2
    for (int j = j_lo; j <= j_hi; j++) {
        const float* p = slot + (size_t)j * part_floats(HD);
        const float w = __expf(p[16 * HD + c] - m);
        l = fmaf(w, p[16 * HD + 16 + c], l);
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const f32x4 o = *(const f32x4*)(p + (64 * d + lane) * 4);
#pragma unroll
            for (int r = 0; r < 4; r++) acc[d][r] = fmaf(w, o[r], acc[d][r]);
        }
    }
    const float top = largest<ND>(l > 0.f ? l : INFINITY, acc);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad || !(top < INFINITY)) != 0, 0)) {
        f32_body<HD, 1, false>(nullptr, nullptr, q, K, V, T, S, n_head, n_kv, scale, window, softcap, out);
        return;
    }
    if (i0 + c >= T) return;
    const float inv = 1.0f / l * (1.0f / V_UP);
    Out* op = out + ((size_t)(i0 + c) * n_head + head) * HD + 4 * ks;
#pragma unroll
    for (int d = 0; d < ND; d++) store_out(op + 16 * d, float4{acc[d][0] * inv, acc[d][1] * inv, acc[d][2] * inv, acc[d][3] * inv});
}

}  // namespace

namespace fhip {

static int waves_of(size_t t, size_t n_head) {
    // waves (16 query rows each) per workgroup: 8, or 4 while that leaves the chip fewer than two workgroups per CU
    const size_t cus = device_cus() > 0 ? device_cus() : 256;
    return ((t + 127) / 128) * n_head < 2 * cus ? 4 : 8;
}

// Whether 16 rows of a head get four waves of the f32 kernel's work (causal_attn_team_kernel) or one. A wave to itself takes 2.7 us a key tile at head size
// 128 and 1.55 at 64, and a launch that leaves CUs idle lasts as long as its longest row; four waves take 2.2 and 1.2 .. 1.45 us for two tiles, a CU's workgroups one after
// the other (they share its L1's bytes). So they are taken where the steps of a CU's share are at most 5/4 of the longest row's tiles. Over 150
// shapes (2 .. 1024 rows behind 0 .. 3000 keys, 4 .. 64 heads) 132 are: 0.41 .. 0.95 of the time and 4.0 | 4.1 at 3 x 4, 0.64 on average; the others would be 0.88 .. 1.31:
// 632 x 632, 32 heads of 64 39.2 | 34.4; 364 x 570, 40 of 128 54.8 | 52.7; 542 x 542, 64 of 128 74.5 | 82.4; 804 x 902, 64 of 64 89.5 | 117.3.
static bool team_pays(size_t t, size_t s, size_t n_head, int win) {
    const size_t cus = device_cus() > 0 ? device_cus() : 256, blocks = (t + 15) / 16;
    if (blocks > 65535) return false;
    const int off = (int)(s - t);
    auto tiles = [&](size_t b) { return (size_t)key_tiles(off, (int)(16 * b), (int)(16 * b + 16 < t ? 16 * b + 16 : t) - 1, win).count(); };
    const size_t most = 5 * tiles(blocks - 1) * cus / 4;
    size_t steps = 0;
    for (size_t b = 0; b < blocks && steps <= most; b++) steps += (tiles(b) + 1) / 2 * n_head;
    return steps <= most;
}

// Ranges of at most `most` key tiles, at most `slots` of them a query block; most = 0: the keys stay in one piece.
// A workgroup takes 2.15 us a tile of 64 rows at head size 128 and 1.3 at 64, and a CU's workgroups together 1.95 and 1.0, so a launch of one workgroup a CU or fewer
// lasts as long as the block with the most tiles, one of up to two a CU as long as that block and the shortest that lies beside it. Ranges cost 4 us (the
// join's launch) and a seventh, three tenths at head size 128 (their starts, the partial results' way through memory), and level the CUs' shares; where they are more
// than two a CU, a quarter of a range more, for the CUs that are left with one. The best size is 0.6 of a CU's share, two at least; it is flat around
// that and from 14 on, where the share, not the last workgroup, counts. us, one piece | ranges of 2, 3, 4, 6, 8, 14, 18 tiles (rows x keys, heads, KV heads, head size):
//   95 x 722, 8, 8, 128     54.4 | 14.2  15.4  16.8  20.7  25.3  32.2        377 x 954, 8, 4, 64     46.0 | 16.3  15.1  16.0  15.5  17.7  26.0  27.5
//   33 x 1057, 4, 4, 128    78.1 | 16.5  16.7  17.9  21.3  23.2  33.5  44.0  152 x 940, 8, 8, 64     44.9 | 13.5  12.4  12.9  14.7  17.5  25.8  27.0
//   234 x 355, 32, 4, 128   31.4 | 24.6  21.0  21.9  22.1  26.3              65 x 600, 64, 8, 64     31.5 | 19.6  18.4  17.9  17.2  18.5  20.6  20.7
//   1024 x 1024, 8, 4, 128  77.4 | 40.6  36.5  35.4  30.1  35.1  41.9  48.4  700 x 1200, 24, 8, 64   59.4 | 52.7  43.7  41.6  39.0  38.9  39.3  44.2
//   509 x 809, 40, 8, 128   71.9 | 82.3  68.8  63.5  63.0  58.8  59.8  56.8  1024 x 2048, 16, 4, 64  94.5 | 80.2  67.1  62.1  59.4  58.2  55.7  59.0
// Over 520 shapes (33 ... 1024 rows behind 0 ... 1024 keys, 4 ... 64 heads, with and without a window) 306 are split, to 0.63 of the time on average and at
// most to 1.00 (of 500 others 320, to 0.58, none slower); before the ranges' share at head size 128, the late ranges and blocks no longer than one range were counted, 319 were, up to 1.27 of the time:
// 390 x 451, 64 heads of 128 42.0 | 53.4; 655 x 655, 40 of 128 53.7 | 57.5; 834 x 870, 32 of 128, window 433 52.9 | 59.5. Not split before
// either: 77 x 77, 40 heads of 128 7.2 | 8.9  9.5, 205 x 205, 64 of 64 12.6 | 13.6  13.6  13.3  15.3, 1024 x 1024, 40 of 128 (640 workgroups) 85.6 | 139  119  110  101  97.8  95.6  97.6.
struct CausalSplit { int most = 0, slots = 0; };
static CausalSplit causal_split(size_t t, size_t s, size_t n_head, size_t hd, int win) {
    constexpr size_t ROWS = 16 * CUT_WAVES;
    constexpr int FEWEST = 5, RANGES = 32;       // tiles that are worth a join; what the join adds one after the other
    if (t == 0 || n_head == 0 || n_head > 65535 || s < t || s > 0x3FFFFFFFull || waves_of(t, n_head) != CUT_WAVES) return {};
    const size_t cus = device_cus() > 0 ? device_cus() : 256, blocks = (t + ROWS - 1) / ROWS, groups = blocks * n_head;
    if (groups > 2 * cus) return {};
    const int off = (int)(s - t);
    auto tiles = [&](size_t b) { return key_tiles(off, (int)(b * ROWS), (int)((b + 1) * ROWS < t ? (b + 1) * ROWS : t) - 1, win).count(); };
    size_t total = 0;
    int longest = 0;
    for (size_t b = 0; b < blocks; b++) {
        const int n = tiles(b);
        total += n * n_head;
        longest = n > longest ? n : longest;
    }
    if (longest < FEWEST) return {};
    const float one = hd == 128 ? 2.15f : 1.3f, both = hd == 128 ? 1.95f : 1.0f, share = (float)total / cus;
    int most = share <= 24.f ? (int)ceilf(0.6f * share) : (int)fmaxf(14.f, share / 4);
    most = most < 2 ? 2 : most;
    most = most * RANGES < longest ? (longest + RANGES - 1) / RANGES : most;
    auto units = [&](int m) {
        size_t n = 0;
        for (size_t b = 0; b < blocks; b++) n += (tiles(b) + m - 1) / m * n_head;
        return n;
    };
    for (int m = most; m <= most + most / 4; m++)        // a little longer where all of them then start at once (509 x 809: 15 tiles 62.5, 18 57)
        if (units(m) <= 2 * cus) { most = m; break; }
    if (most >= longest) return {};
    const float whole = groups <= cus ? one * longest : both * (longest + tiles(blocks - 1 - cus / n_head));   // blocks go out last first, all heads of each
    const float late = units(most) > 2 * cus ? 0.25f * one * most : 0.f;
    if (whole <= 4.f + fmaxf(one * most, (hd == 128 ? 1.3f : 1.15f) * both * share) + late) return {};
    return {most, (longest + most - 1) / most};
}

static int causal_window(size_t window, size_t s) { return window == 0 || window >= s ? 0 : (int)window; }   // a window that covers the cache is no window

static size_t split_bytes(const CausalSplit& sp, size_t t, size_t n_head, size_t hd) {
    return n_head * ((t + 15) / 16) * sp.slots * part_floats((int)hd) * sizeof(float);
}

size_t causal_attention_ws_bytes(size_t t, size_t s, size_t n_head, size_t hd, size_t window) {
    return split_bytes(causal_split(t, s, n_head, hd, causal_window(window, s)), t, n_head, hd);
}

template <typename Out>
static int launch_causal_out(const float* q, const float* K, const float* V, size_t t, size_t s, int n_head, int n_kv, int hd, size_t window,
                             float softcap, bool cuts, Out* out, float* ws, size_t ws_bytes, hipStream_t st) {
    if (t == 0 || n_head == 0 || hd == 0) return FHIP_OK;
    if (s < t) return set_error(FHIP_ERR_SHAPE, "cache (%zu) cannot be shorter than the query block (%zu)", s, t);   // nn.rs:73, :249
    if (n_kv <= 0 || n_head % n_kv != 0) return set_error(FHIP_ERR_SHAPE, "causal_attention: n_heads must be a multiple of n_kv_heads");
    if (hd != 64 && hd != 128) return set_error(FHIP_ERR_SHAPE, "causal_attention: head_dim must be 64 or 128");
    if (s > 0x3FFFFFFFull || n_head > 65535) return set_error(FHIP_ERR_SHAPE, "causal_attention: too large for one launch");
    const int nw = waves_of(t, n_head);
    const size_t qblocks = (t + (size_t)nw * 16 - 1) / ((size_t)nw * 16);
    if (qblocks > 65535) return set_error(FHIP_ERR_SHAPE, "causal_attention: too many query rows for one launch");
    dim3 grid((unsigned)n_head, (unsigned)qblocks);
    const dim3 wg(64 * nw);
    const float scale = 1.0f / sqrtf((float)hd);
    const int win = causal_window(window, s);
    auto cut = [&](auto kernel, auto to, int most) { hipLaunchKernelGGL(kernel, grid, wg, 0, st, q, K, V, (int)t, (int)s, n_head, n_kv, scale, win, softcap, to, ws, most); };
    auto f32 = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, wg, 0, st, q, K, V, (int)t, (int)s, n_head, n_kv, scale, win, softcap, out); };
    if (!cuts) {
        if (team_pays(t, s, n_head, win)) {
            grid.y = (unsigned)((t + 15) / 16);
            auto team = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, q, K, V, (int)t, (int)s, n_head, n_kv, scale, win, softcap, out); };
            hd == 128 ? team(causal_attn_team_kernel<128, Out>) : team(causal_attn_team_kernel<64, Out>);
            return check_hip(hipGetLastError(), "causal_attention launch");
        }
        if (hd == 128) nw == 8 ? f32(causal_attn_kernel<128, 8, Out>) : f32(causal_attn_kernel<128, 4, Out>);
        else nw == 8 ? f32(causal_attn_kernel<64, 8, Out>) : f32(causal_attn_kernel<64, 4, Out>);
        return check_hip(hipGetLastError(), "causal_attention launch");
    }
    const CausalSplit sp = ws ? causal_split(t, s, n_head, hd, win) : CausalSplit{};
    if (sp.most) {
        const size_t need = split_bytes(sp, t, n_head, hd);
        if (ws_bytes < need) return set_error(FHIP_ERR_ARG, "causal_attention: %zu bytes of workspace, %zu needed", ws_bytes, need);
        grid.z = (unsigned)sp.slots;
        hd == 128 ? cut(causal_attn_cut_kernel<128, CUT_WAVES, true, float>, ws, sp.most) : cut(causal_attn_cut_kernel<64, CUT_WAVES, true, float>, ws, sp.most);
        if (const int rc = check_hip(hipGetLastError(), "causal_attention launch")) return rc;
        auto join = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)n_head, (unsigned)((t + 15) / 16)), dim3(64), 0, st, q, K, V, (int)t, (int)s, n_head, n_kv, scale, win, softcap, out,
                               (const float*)ws, sp.most, sp.slots);
        };
        hd == 128 ? join(causal_attn_join_kernel<128, Out>) : join(causal_attn_join_kernel<64, Out>);
        return check_hip(hipGetLastError(), "causal_attention join launch");
    }
    if (hd == 128) nw == 8 ? cut(causal_attn_cut_kernel<128, 8, false, Out>, out, 0) : cut(causal_attn_cut_kernel<128, 4, false, Out>, out, 0);
    else nw == 8 ? cut(causal_attn_cut_kernel<64, 8, false, Out>, out, 0) : cut(causal_attn_cut_kernel<64, 4, false, Out>, out, 0);
    return check_hip(hipGetLastError(), "causal_attention launch");
}

int launch_causal_attention(const float* q, const float* K, const float* V, size_t t, size_t s, int n_head, int n_kv, int hd, size_t window,
                            float softcap, bool cuts, float* out, float* ws, size_t ws_bytes, hipStream_t st) {
    return launch_causal_out(q, K, V, t, s, n_head, n_kv, hd, window, softcap, cuts, out, ws, ws_bytes, st);
}
int launch_causal_attention_bf16(const float* q, const float* K, const float* V, size_t t, size_t s, int n_head, int n_kv, int hd, size_t window,
                                 float softcap, bool cuts, uint16_t* out, float* ws, size_t ws_bytes, hipStream_t st) {
    return launch_causal_out(q, K, V, t, s, n_head, n_kv, hd, window, softcap, cuts, out, ws, ws_bytes, st);
}

}  // namespace fhip
