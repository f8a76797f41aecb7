// Mat-vec for three to sixteen activation rows in one pass over a weight of the 32-value formats (Q4_0, Q4_1, Q5_0, Q5_1, Q8_0,
// IQ4_NL, IQ4_XS, MXFP4): the reference's matmul at small M (crates/ferric-tensor/src/dtype.rs:1838-1904, :3185-3420 and the CPU
// row loop crates/ferric-tensor/src/cpu_simd.rs:175-200, whose result for a row does not depend on the rows beside it).
//
// The arithmetic is the streaming mat-vec's (gemv.hip), bit for bit: activations as block fixed point (a scale per run of 32
// columns, two or three signed byte planes), exact integer dot products per block, the same f32 operations in the same order
// above them, the same trees for the sums over a row's blocks. What differs is who multiplies: v_mfma_i32_16x16x32_i8 takes one
// 32-column block of 16 weight rows (B operand) against every plane of four or eight activation rows (A operand), where the
// dot-product kernel spends eight instructions per plane, activation row and weight row, and reads the weight once per four rows.
//
// Layout. Lane (g4, c) = (lane / 16, lane % 16) of a wave holds weight row c of a tile of 16 rows; its accumulator registers are
// that row's plane sums with the activation rows g4, 4 + g4, ... The order of the 32 columns inside an instruction is free as long as
// both operands agree: k-group g4 takes the columns of dword g4 of a block's nibbles, 4 g4 + (0..3) out of the low and 16 + 4 g4 +
// (0..3) out of the high ones, so a lane needs one dword of every block. Four lanes load four neighbouring blocks of a row (16
// bytes of quants and the header each) and park them in the wave's LDS image, from where lane (g4, c) reads dword g4 of its
// row's blocks. (Loaded one row per lane of sixteen and exchanged with v_permlane32_swap and v_permlane16_swap instead,
// neighbouring lanes ask for different cache lines: 34816 x 5120 Q4_0 at 4 rows 40.8 us against 36.8.)
//
// A workgroup has R of the activation rows. Those of a pass of P groups (16 blocks, 512 columns each) are quantised once per workgroup into LDS, laid out as the A
// operands; an item of work is (tile of 16 weight rows, group) and the waves share the pass's items evenly. The group sums go
// to LDS and are added there in the row's group order, so neither the number of passes nor the dealing shows in the bits.
//
// What bounds it: instruction issue, twice. A block of a tile takes E matrix instructions (16 cycles each) and some 12 + 11 E
// vector instructions (four cycles each) at E pairs a lane; the quantiser takes about 16 per activation value and is repeated by
// every workgroup, 0.6 us an activation row of 4096 columns, which is what a batch of sixteen on a small weight spends its time on.
// us, cold, dot-product kernel -> this one, 24 bits: Q4_0 34816 x 5120 at 4 / 8 / 16 rows 42.3 / 84.1 / 169 -> 32.6 / 41.0 / 64.0 (the
// 100 MB of the weight: 18), 4096 x 4096 13.1 / 25.6 / 50.9 -> 9.6 / 12.3 / 20.9; MXFP4 9728 x 2560 15.1 / 28.3 / 55.9 -> 11.7 / 13.1 / 21.8;
// IQ4_NL 1467 x 1760 at 16 rows 37.1 -> 12.1.
//
// Built once per activation precision like gemv.hip (FHIP_GEMV_PLANES = 2 or 3).
#include "common.hpp"
#include "deq_at.hpp"
#include "fixed_point.hpp"
#include "lut16.hpp"

#include <algorithm>
#include <hip/hip_fp16.h>

#if FHIP_GEMV_PLANES == 2
#define WIDE_EXPORT(name) name##_p2
#else
#define WIDE_EXPORT(name) name##_p3
#endif
#define gemv_wide_kernel WIDE_EXPORT(gemv_wide_kernel)

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(1))) U4A1 { u32x4 v; };
struct __attribute__((packed, aligned(2))) U4A2 { u32x4 v; };
struct __attribute__((packed, aligned(8))) U4A8 { u32x4 v; };

__device__ __forceinline__ float f16_bits(uint32_t b) { return __half2float(__ushort_as_half((unsigned short)b)); }


// dword 0 of four 16-byte pieces that lie side by side
__device__ __forceinline__ u32x4 dwords4(const uint8_t* p) {
    return (u32x4){*(const uint32_t*)p, *(const uint32_t*)(p + 16), *(const uint32_t*)(p + 32), *(const uint32_t*)(p + 48)};
}

// ------------------------------------------------------------------------------------------------
// Per-format lane work. load(): one block of one weight row; park(): the lane's block, block b of four of row r, into the wave's
// LDS image (rows of 80 bytes: the sixteen rows of a dword read lie in different banks), its scale and offset as f32; fetch():
// dword g4 of row c's four blocks and the row's four scales. Then, per block j of the four, operand() makes the lane's eight
// weight bytes (four of the low half, four of the high half of the columns) and value() is gemv.hip's expression for the block,
// term for term.
// ------------------------------------------------------------------------------------------------
template <uint32_t TY, int BYTES, bool HAS_M, bool HAS_QH, int OFF>
struct Leg {
    static constexpr uint32_t TYPE = TY;
    static constexpr bool HAS_XQ = HAS_M || OFF != 0, BIG = false;
    static constexpr int QH = HAS_M ? 4 : 2, QS = QH + (HAS_QH ? 4 : 0);
    struct Data { u32x4 q; uint32_t dm, qh; };
    struct Four { u32x4 q, d, m, qh; };
    static __device__ __forceinline__ Data load(const uint8_t* row, int u) {
        const uint8_t* b = row + (uint32_t)(u * BYTES);
        const uint16_t* h = (const uint16_t*)b;
        Data d;
        d.dm = HAS_M ? ((uint32_t)h[0] | ((uint32_t)h[1] << 16)) : (uint32_t)h[0];
        d.qh = HAS_QH ? ((uint32_t)h[QH / 2] | ((uint32_t)h[QH / 2 + 1] << 16)) : 0u;
        d.q = ((const U4A2*)(b + QS))->v;
        return d;
    }
    static constexpr int ROW = 80, IMAGE = 16 * ROW + 256 * (1 + (HAS_M ? 1 : 0) + (HAS_QH ? 1 : 0));
    static __device__ __forceinline__ void park(uint8_t* wl, const Data& D, int, int r, int b) {
        *(u32x4*)(wl + r * ROW + 16 * b) = D.q;
        float* h = (float*)(wl + 16 * ROW) + 4 * r + b;
        h[0] = f16_bits(D.dm & 0xFFFFu);
        if constexpr (HAS_M) h[64] = f16_bits(D.dm >> 16);
        if constexpr (HAS_QH) ((uint32_t*)h)[HAS_M ? 128 : 64] = D.qh;
    }
    static __device__ __forceinline__ Four fetch(const uint8_t* wl, int c, int g4) {
        Four f;
        f.q = dwords4(wl + c * ROW + 4 * g4);
        const u32x4* h = (const u32x4*)(wl + 16 * ROW) + c;
        f.d = h[0];
        if constexpr (HAS_M) f.m = h[16];
        if constexpr (HAS_QH) f.qh = h[HAS_M ? 32 : 16];
        return f;
    }
    static __device__ __forceinline__ u32x2 operand(const Four& f, int j, int g4) {
        uint32_t lo = f.q[j] & 0x0F0F0F0Fu, hi = (f.q[j] >> 4) & 0x0F0F0F0Fu;
        if constexpr (HAS_QH) {   // bit k of a 4-bit field -> bit 4 of byte k
            const uint32_t h = f.qh[j] >> (4 * g4);
            lo |= (((h & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
            hi |= ((((h >> 16) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
        }
        return (u32x2){lo, hi};
    }
    // (a term that gemv.hip writes with a zero factor adds +-0 to a sum that is no -0: left out)
    static __device__ __forceinline__ float value(const Four& f, int j, float pf, float xs, float xq) {
        const float d = __uint_as_float(f.d[j]);
        const float t = OFF ? fmaf(-(float)OFF, xq, xs * pf) : xs * pf;
        if constexpr (HAS_M) return fmaf(d, t, __uint_as_float(f.m[j]) * xq);
        else return d * t;
    }
    static __device__ __forceinline__ bool big(const Four&, int) { return false; }
};
typedef Leg<FHIP_Q4_0, 18, false, false, 8> Q40;
typedef Leg<FHIP_Q4_1, 20, true, false, 0> Q41;
typedef Leg<FHIP_Q5_0, 22, false, true, 16> Q50;
typedef Leg<FHIP_Q5_1, 24, true, true, 0> Q51;


template <bool XS>
struct Iq4 {
    static constexpr uint32_t TYPE = XS ? FHIP_IQ4_XS : FHIP_IQ4_NL;
    static constexpr bool HAS_XQ = false, BIG = false;
    struct Data { u32x4 q; uint32_t h0, h1; };
    struct Four { u32x4 q, d; };
    static __device__ __forceinline__ Data load(const uint8_t* row, int u) {
        Data d;
        if constexpr (XS) {
            const uint8_t* b = row + (uint32_t)((u >> 3) * 136);
            d.h0 = *(const uint32_t*)b;
            d.h1 = *(const uint32_t*)(b + 4);
            d.q = ((const U4A8*)(b + 8 + 16 * (u & 7)))->v;
        } else {
            const uint8_t* b = row + (uint32_t)(u * 18);
            d.h0 = *(const uint16_t*)b;
            d.h1 = 0;
            d.q = ((const U4A2*)(b + 2))->v;
        }
        return d;
    }
    static constexpr int ROW = 80, IMAGE = 16 * ROW + 256;
    static __device__ __forceinline__ void park(uint8_t* wl, const Data& D, int u, int r, int b) {
        float dl = f16_bits(D.h0 & 0xFFFFu);
        if constexpr (XS) {
            const int ib = u & 7, ls = (int)(((D.h1 >> (4 * ib)) & 0xFu) | ((((D.h0 >> 16) >> (2 * ib)) & 3u) << 4));
            dl *= (float)(ls - 32);
        }
        *(u32x4*)(wl + r * ROW + 16 * b) = D.q;
        ((float*)(wl + 16 * ROW))[4 * r + b] = dl;
    }
    static __device__ __forceinline__ Four fetch(const uint8_t* wl, int c, int g4) {
        return Four{dwords4(wl + c * ROW + 4 * g4), ((const u32x4*)(wl + 16 * ROW))[c]};
    }
    static __device__ __forceinline__ u32x2 operand(const Four& f, int j, int) {
        // the codebook as int8 bytes, four levels per word (crates/ferric-gguf/src/lib.rs:751-791)
        constexpr fhip::Lut16 LUT = fhip::lut16(0xBFAD9881u, 0xF6EADDCFu, 0x26190D01u, 0x71594535u);
        return (u32x2){fhip::lut16x4(f.q[j] & 0x0F0F0F0Fu, LUT), fhip::lut16x4((f.q[j] >> 4) & 0x0F0F0F0Fu, LUT)};
    }
    static __device__ __forceinline__ float value(const Four& f, int j, float pf, float xs, float) { return (xs * pf) * __uint_as_float(f.d[j]); }
    static __device__ __forceinline__ bool big(const Four&, int) { return false; }
};

// MXFP4: weight = k * 2^(e - 128) with k the doubled E2M1 value; from e = 252 on a weight may be +-inf, which the reference
// forms before it meets the activation: such a block is summed element by element (big()), as in gemv.hip.
struct Mxf4 {
    static constexpr uint32_t TYPE = FHIP_MXFP4;
    static constexpr bool HAS_XQ = false, BIG = true;
    static constexpr fhip::Lut16 LUT = fhip::lut16(0x03020100u, 0x0C080604u, 0xFDFEFF00u, 0xF4F8FAFCu);
    struct Data { u32x4 q; uint32_t e; };
    struct Four { u32x4 q, d; };
    static __device__ __forceinline__ Data load(const uint8_t* row, int u) {
        const uint8_t* b = row + (uint32_t)(u * 17);
        Data d;
        d.e = b[0];
        d.q = ((const U4A1*)(b + 1))->v;
        return d;
    }
    static __device__ __forceinline__ uint32_t scale_bits(uint32_t e) { return e == 0 ? (1u << 21) : e == 1 ? (1u << 22) : (e - 1u) << 23; }
    static constexpr int ROW = 80, IMAGE = 16 * ROW + 256;
    static __device__ __forceinline__ void park(uint8_t* wl, const Data& D, int, int r, int b) {
        *(u32x4*)(wl + r * ROW + 16 * b) = D.q;
        ((uint32_t*)(wl + 16 * ROW))[4 * r + b] = scale_bits(D.e);
    }
    static __device__ __forceinline__ Four fetch(const uint8_t* wl, int c, int g4) {
        return Four{dwords4(wl + c * ROW + 4 * g4), ((const u32x4*)(wl + 16 * ROW))[c]};
    }
    static __device__ __forceinline__ u32x2 operand(const Four& f, int j, int) {
        return (u32x2){fhip::lut16x4(f.q[j] & 0x0F0F0F0Fu, LUT), fhip::lut16x4((f.q[j] >> 4) & 0x0F0F0F0Fu, LUT)};
    }
    static __device__ __forceinline__ float value(const Four& f, int j, float pf, float xs, float) { return (xs * pf) * __uint_as_float(f.d[j]); }
    static constexpr uint32_t BIG_BITS = 251u << 23;     // the scale of e = 252
    static __device__ __forceinline__ bool big(const Four& f, int j) { return f.d[j] >= BIG_BITS; }
};

// Q8_0: 34 B = [f16 d][32 int8]: two 16-byte pieces, k-group g4 takes dword g4 of each
struct Q80 {
    static constexpr uint32_t TYPE = FHIP_Q8_0;
    static constexpr bool HAS_XQ = false, BIG = false;
    struct Data { u32x4 q, q1; uint32_t d; };
    struct Four { u32x4 q, q1, d; };
    static __device__ __forceinline__ Data load(const uint8_t* row, int u) {
        const uint8_t* b = row + (uint32_t)(u * 34);
        Data d;
        d.d = *(const uint16_t*)b;
        d.q = ((const U4A2*)(b + 2))->v;
        d.q1 = ((const U4A2*)(b + 18))->v;
        return d;
    }
    static constexpr int ROW = 80, IMAGE = 32 * ROW + 256;   // the blocks' first 16 quants, then their last, as two images
    static __device__ __forceinline__ void park(uint8_t* wl, const Data& D, int, int r, int b) {
        *(u32x4*)(wl + r * ROW + 16 * b) = D.q;
        *(u32x4*)(wl + (16 + r) * ROW + 16 * b) = D.q1;
        ((float*)(wl + 32 * ROW))[4 * r + b] = f16_bits(D.d);
    }
    static __device__ __forceinline__ Four fetch(const uint8_t* wl, int c, int g4) {
        return Four{dwords4(wl + c * ROW + 4 * g4), dwords4(wl + (16 + c) * ROW + 4 * g4), ((const u32x4*)(wl + 32 * ROW))[c]};
    }
    static __device__ __forceinline__ u32x2 operand(const Four& f, int j, int) { return (u32x2){f.q[j], f.q1[j]}; }
    static __device__ __forceinline__ float value(const Four& f, int j, float pf, float xs, float) { return (xs * pf) * __uint_as_float(f.d[j]); }
    static __device__ __forceinline__ bool big(const Four&, int) { return false; }
};

struct WideParams {
    const uint8_t* W;
    const float* x;        // [T, cols]
    float* y;              // [T, N]
    int T, N, cols;
    int R;                 // activation rows per workgroup, blockIdx.y of them before its own
    size_t row_bytes;
    int units, NG;         // blocks of a row; 16-block groups of a row
    int P, passes;         // groups per pass
    int tiles;             // 16-row tiles per workgroup
    uint32_t scales_off, sums_off, flags_off, part_off, total_off, image_off;   // byte offsets in LDS
};

// waves of a workgroup at most, by the registers of E pairs a lane: 128, 168, or 256 where the element-by-element branch needs more
template <class F, int E> constexpr int max_waves() { return E == 1 ? 16 : E == 2 ? 12 : F::BIG ? 8 : 12; }

// An instruction's 16 A rows hold every plane of four activation rows (three planes: rows 4 g + p, the fourth idle) or of eight
// (two planes: rows 4 g + 2 k + p), so a lane's four accumulator registers are the plane sums of ONE or two (weight row, activation
// row) pairs and the f32 work of a lane follows the number of activation rows: E = 1, 2, 4 pairs a lane for up to 4, 8, 16 rows.
// Pair e of lane row g is activation row 4 e + g. (One plane of sixteen activation rows an instruction, the first layout, left
// the pairs of missing rows to be worked out all the same: 34816 x 5120 Q4_0 at 5 rows 61.9 us.)
//
// LDS. Planes of the pass's blocks: block ul at ul * US, in it [e][k-group 4][plane][g 4][8 bytes] (US: 8 bytes more than that, so
// that the sixteen blocks a wave's quantiser stores to lie in different banks); run scales and run sums [ul][g][E]; a flag per
// group whose runs block fixed point cannot all hold; group sums [group][rows][4 E + 4]; running sums [rows][4 E]; a wave's weights.
template <int E> constexpr int unit_stride() { return NP * 128 * E + 8; }
template <int E> constexpr int n_mma() { return NP == 3 ? E : (E + 1) / 2; }

template <class F, int E>
__global__ void __launch_bounds__((64 * max_waves<F, E>())) gemv_wide_kernel(WideParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int US = unit_stride<E>(), NM = n_mma<E>(), PS = 4 * E + 4;
    typedef float fE __attribute__((ext_vector_type(E)));
    const int tid = threadIdx.x, lane = tid & 63, W = (int)(blockDim.x >> 6);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g4 = lane >> 4, c = lane & 15;
    if constexpr (E < 4) {                                // the workgroup's activation rows (of more than eight a workgroup has all: these lines cost it 0.4 us)
        const int first = (int)blockIdx.y * p.R;
        p.T = p.T - first < p.R ? p.T - first : p.R;
        p.x += (size_t)first * p.cols;
        p.y += (size_t)first * p.N;
    }
    const int row0 = (int)blockIdx.x * p.tiles * 16;
    if (row0 >= p.N) return;                              // (the launcher sends no such workgroup)
    int nrows = p.N - row0;
    nrows = nrows < p.tiles * 16 ? nrows : p.tiles * 16;
    const int ntiles = (nrows + 15) >> 4;
    float* scales = (float*)(smem + p.scales_off);
    float* sums = (float*)(smem + p.sums_off);
    int* flags = (int*)(smem + p.flags_off);
    float* part = (float*)(smem + p.part_off);
    float* total = (float*)(smem + p.total_off);
    // the lane's A operand of instruction 0 in a block's planes: A row c is activation row c / 4 of a pair and, of c % 4, the plane
    // (three planes; the fourth row repeats the third) or pair and plane (two planes); instruction m is A_STEP bytes further
    constexpr int A_STEP = (NP == 3 ? 1 : 2) * NP * 128;
    const int rr = c & 3, a_off = (NP == 3 || E == 1 ? 0 : rr >> 1) * (NP * 128) + (g4 * NP + (NP == 3 ? (rr < 3 ? rr : 2) : rr & 1)) * 32 + (c >> 2) * 8;

    const uint8_t* const base = p.W + (size_t)row0 * p.row_bytes;
    auto row_of = [&](int tile) {
        const int r = tile * 16 + c;
        return base + (size_t)(r < nrows ? r : nrows - 1) * p.row_bytes;
    };
    const int lr = lane >> 2, lb = lane & 3;              // what the lane loads: block lb of four of row lr of a tile
    uint8_t* const wl = smem + p.image_off + wave * F::IMAGE;

    for (int pass = 0; pass < p.passes; pass++) {
        const int gbase = pass * p.P, P = p.NG - gbase < p.P ? p.NG - gbase : p.P;
        // the wave's items (tile, group of the pass): number wave, wave + W, ... of ntiles x P
        const int step_t = W / P, step_g = W - step_t * P;
        struct Item { int tile, gl; };
        auto after = [&](Item it) {
            it.tile += step_t; it.gl += step_g;
            if (it.gl >= P) { it.gl -= P; it.tile++; }
            return it;
        };
        // An item is four quads of blocks. Quad n of the wave's stream waits in buf[n % 4] from its request to its place in the
        // wave's LDS image, which is four quads later; from there it is read into registers while quad n - 1 is worked on.
        typename F::Data buf[4];
        auto block_of = [&](Item it, int i) {
            const int u = (gbase + it.gl) * 16 + 4 * i + lb;
            return u < p.units ? u : p.units - 1;
        };
        auto request = [&](Item it, int i) {
            const int r = it.tile * 16 + lr;              // (rows past the weight's end repeat the workgroup's last row)
            if (it.tile < ntiles) buf[i] = F::load(base + (size_t)(r < nrows ? r : nrows - 1) * p.row_bytes, block_of(it, i));
        };
        auto park = [&](Item it, int i) {
            if (it.tile < ntiles) F::park(wl, buf[i], block_of(it, i), lr, lb);
        };
        Item it0;
        it0.tile = __builtin_amdgcn_readfirstlane(wave / P);
        it0.gl = wave - it0.tile * P;
#pragma unroll
        for (int i = 0; i < 4; i++) request(it0, i);

        // ---- the pass's activations -> block fixed point: a wave takes one activation row of one group (64 lanes x 8 columns) at a time
        if (tid < p.P) flags[tid] = 0;
        __syncthreads();                                  // the flags are clear, and the planes of the pass before have been read
        // (the next two pieces are requested before the present two are worked on)
        struct Piece { float4 a, b; int t, g; } now[2], nxt[2];
        Item at{it0.tile, it0.gl};                        // (activation row, group) of the next piece to request: pieces are dealt like the items
        auto ask = [&](Piece& s) {
            s.t = at.tile; s.g = at.gl;
            at = after(at);
            s.a = float4{0.f, 0.f, 0.f, 0.f}; s.b = s.a;
            const int col = (gbase + s.g) * 512 + lane * 8;
            if (s.t < p.T && col < p.cols) {
                const float* src = p.x + (size_t)s.t * p.cols + col;
                s.a = *(const float4*)src; s.b = *(const float4*)(src + 4);
            }
        };
        ask(now[0]);
        ask(now[1]);
        while (now[0].t < p.T) {
            ask(nxt[0]);
            ask(nxt[1]);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (now[k].t < p.T) {
                    const Piece& s = now[k];
                    const float v[8] = {s.a.x, s.a.y, s.a.z, s.a.w, s.b.x, s.b.y, s.b.z, s.b.w};
                    uint32_t pl[NP][2];
                    float scale, qsum;
                    quantize8<32>(v, pl, scale, qsum);
                    const int ul = s.g * 16 + (lane >> 2), q4 = lane & 3, e = s.t >> 2, g = s.t & 3;
                    uint8_t* dst = smem + ul * US + e * (NP * 128) + g * 8 + 4 * (q4 >> 1);
#pragma unroll
                    for (int pp = 0; pp < NP; pp++) {
                        *(uint32_t*)(dst + (((2 * q4) & 3) * NP + pp) * 32) = pl[pp][0];
                        *(uint32_t*)(dst + (((2 * q4 + 1) & 3) * NP + pp) * 32) = pl[pp][1];
                    }
                    if (q4 == 0) {
                        scales[(ul * 4 + g) * E + e] = scale;
                        if constexpr (F::HAS_XQ) sums[(ul * 4 + g) * E + e] = qsum;
                        if (scale != scale) flags[s.g] = 1;
                    }
                }
            }
            now[0] = nxt[0]; now[1] = nxt[1];
        }
        __syncthreads();

        // ---- the items
        struct Ops { long a[NM]; };                       // a block's A operands
        // of block k of an item, from the addresses of its block 0
        auto read_ops = [&](const uint8_t* ap, int k) {
            Ops o;
#pragma unroll
            for (int m = 0; m < NM; m++) o.a[m] = *(const long*)(ap + k * US + m * A_STEP);
            return o;
        };
        // (the image is written by one set of lanes and read by another of the same wave, whose LDS operations keep their order;
        // the fence keeps the compiler's)
        auto image_fence = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
        Item it1 = after(it0);
        typename F::Four four;
        if (it0.tile < ntiles) {
            park(it0, 0);
            request(it1, 0);
            image_fence();
            four = F::fetch(wl, c, g4);
            image_fence();
        }
        while (it0.tile < ntiles) {
            const Item it2 = after(it1);
            const int tile = it0.tile, gl = it0.gl;
            {
                const int ul0 = gl * 16, u0 = (gbase + gl) * 16;
                const bool special_group = __builtin_amdgcn_readfirstlane(flags[gl]) != 0;
                const bool slow = special_group || u0 + 16 > p.units;
                float Q[4][E];                            // [quad of blocks][pair]
                const uint8_t* const ap = smem + ul0 * US + a_off;
                const float* const sp = scales + (ul0 * 4 + g4) * E;
                const float* const qp = sums + (ul0 * 4 + g4) * E;
                Ops cur = read_ops(ap, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int ub = u0 + 4 * i;            // wave-uniform
                    park(i < 3 ? it0 : it1, (i + 1) & 3);
                    request(i < 3 ? it1 : it2, (i + 1) & 3);
                    image_fence();
                    typename F::Four fnext;
                    float v[4][E];                        // [block of the quad][pair]
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        // the next block's operands are read a block ahead (left alone, the compiler reads all of an item's
                        // first and spills; without the read ahead a block waits for LDS, then for the matrix unit)
                        const fE xs = *(const fE*)(sp + (4 * i + j) * (4 * E));
                        fE xq = 0.f;
                        if constexpr (F::HAS_XQ) xq = *(const fE*)(qp + (4 * i + j) * (4 * E));
                        const Ops nxt = read_ops(ap, 4 * i + j < 15 ? 4 * i + j + 1 : 15);
                        const long wb = __builtin_bit_cast(long, F::operand(four, j, g4));
                        i32x4 acc[NM];
#pragma unroll
                        for (int m = 0; m < NM; m++) acc[m] = __builtin_amdgcn_mfma_i32_16x16x32_i8(cur.a[m], wb, i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < E; e++) {
                            int a[NP];
#pragma unroll
                            for (int pp = 0; pp < NP; pp++) a[pp] = NP == 3 ? acc[NP == 3 ? e : 0][pp] : acc[e >> 1 < NM ? e >> 1 : 0][2 * (e & 1) + pp];
                            v[j][e] = F::value(four, j, planes_f32(a), xs[e], xq[e]);
                        }
                        cur = nxt;
                        if (j == 2) { fnext = F::fetch(wl, c, g4); image_fence(); }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if constexpr (F::BIG) {
                        // a block of weights that may be +-inf: its products one by one on the activations as the planes hold them
                        const bool any_big = F::big(four, 0) || F::big(four, 1) || F::big(four, 2) || F::big(four, 3);
                        if (__builtin_amdgcn_ballot_w64(any_big) != 0) {
#pragma unroll 1
                            for (int je = 0; je < 4 * E; je++) {
                                const int j = je / E, e = je - j * E, ul = ul0 + 4 * i + j;
                                const uint32_t db = j == 0 ? four.d[0] : j == 1 ? four.d[1] : j == 2 ? four.d[2] : four.d[3];
                                if (db < Mxf4::BIG_BITS) continue;
                                const float d = __uint_as_float(db);
                                const uint8_t* qsb = row_of(tile) + (uint32_t)((ub + j < p.units ? ub + j : p.units - 1) * 17 + 1);
                                float a = 0.f;
#pragma unroll 1
                                for (int n = 0; n < 32; n++) {
                                    const uint32_t nib = n < 16 ? (uint32_t)qsb[n & 15] & 15u : (uint32_t)qsb[n & 15] >> 4;
                                    const uint32_t k = fhip::lut16x4(nib, Mxf4::LUT);
                                    int xv = 0;
#pragma unroll
                                    for (int pp = 0; pp < NP; pp++)
                                        xv = xv * 256 + (int)*(const int8_t*)(smem + ul * US + e * (NP * 128) + (((n & 15) >> 2) * NP + pp) * 32 + g4 * 8 + 4 * (n >> 4) + (n & 3));
                                    a = fmaf(scales[(ul * 4 + g4) * E + e] * (float)xv, (float)(int)(int8_t)k * d, a);
                                }
#pragma unroll
                                for (int jj = 0; jj < 4; jj++)
#pragma unroll
                                    for (int ee = 0; ee < E; ee++) v[jj][ee] = jj == j && ee == e ? a : v[jj][ee];
                            }
                        }
                    }
                    if (slow) {
                        // blocks past the row's end count as zero; a run block fixed point cannot hold is added element by element below
#pragma unroll
                        for (int j = 0; j < 4; j++)
#pragma unroll
                            for (int e = 0; e < E; e++) {
                                const float sc = scales[((ul0 + 4 * i + j) * 4 + g4) * E + e];
                                v[j][e] = ub + j < p.units && sc == sc ? v[j][e] : 0.f;
                            }
                    }
#pragma unroll
                    for (int e = 0; e < E; e++) Q[i][e] = (v[0][e] + v[1][e]) + (v[2][e] + v[3][e]);
                    four = fnext;
                }
                float tot[E];
#pragma unroll
                for (int e = 0; e < E; e++) tot[e] = (Q[0][e] + Q[3][e]) + (Q[2][e] + Q[1][e]);
                if (special_group) {
                    // the flagged runs from the raw activations and the exactly dequantised weights, summed over the group in the
                    // tree the streaming mat-vec uses there, (Q0 + Q1) + (Q3 + Q2)
                    const uint8_t* rowp = row_of(tile);
#pragma unroll 1
                    for (int e = 0; e < E; e++) {
                        const int t = 4 * e + g4;
                        float lo = 0.f, hi = 0.f;         // Q0 + Q1, Q3 + Q2
#pragma unroll 1
                        for (int i = 0; i < 4; i++) {
                            float e01 = 0.f, e23 = 0.f;
#pragma unroll 1
                            for (int j = 0; j < 4; j++) {
                                const int u = u0 + 4 * i + j;
                                const float sc = t < p.T ? scales[((ul0 + 4 * i + j) * 4 + g4) * E + e] : 0.f;
                                float a = 0.f;
                                if (u < p.units && sc != sc) {
#pragma unroll 1
                                    for (int k = 0; k < 32; k++) a += p.x[(size_t)t * p.cols + u * 32 + k] * fhip::deq_at<F::TYPE>(rowp, u * 32 + k);
                                }
                                if (j < 2) e01 = j == 0 ? a : e01 + a;
                                else e23 = j == 2 ? a : e23 + a;
                            }
                            const float S = e01 + e23;
                            if (i < 2) lo = i == 0 ? S : lo + S;
                            else hi = i == 2 ? S : S + hi;
                        }
                        const float a = lo + hi;
#pragma unroll
                        for (int ee = 0; ee < E; ee++) tot[ee] += ee == e ? a : 0.f;
                    }
                }
                fE out;
#pragma unroll
                for (int e = 0; e < E; e++) out[e] = tot[e];
                *(fE*)(part + ((size_t)gl * p.tiles * 16 + tile * 16 + c) * PS + g4 * E) = out;
            }
            it0 = it1; it1 = it2;
        }
        __syncthreads();

        // ---- the row's group sums in their order, on top of the passes before
        for (int q = tid; q < p.T * p.tiles * 16; q += (int)blockDim.x) {
            const int t = q / (p.tiles * 16), r = q - t * (p.tiles * 16);
            if (r >= nrows) continue;
            float a = pass ? total[q] : 0.f;
            for (int g = 0; g < P; g++) a += part[((size_t)g * p.tiles * 16 + r) * PS + (t & 3) * E + (t >> 2)];
            if (pass + 1 < p.passes) total[q] = a;
            else p.y[(size_t)t * p.N + row0 + r] = a;
        }
    }
}

size_t lds_of(int E, int P, int tiles, int passes, int W, int image, WideParams* p) {
    size_t o = (size_t)P * 16 * (NP * 128 * E + 8);
    o = (o + 15) & ~(size_t)15;
    const size_t scales = o; o += (size_t)P * 16 * 4 * E * 4;
    const size_t sums = o; o += (size_t)P * 16 * 4 * E * 4;
    const size_t flags = o; o += ((size_t)P * 4 + 15) & ~(size_t)15;
    const size_t part = o; o += (size_t)P * tiles * 16 * (4 * E + 4) * 4;
    const size_t total = o; o += passes > 1 ? (size_t)tiles * 16 * 4 * E * 4 : 0;
    const size_t img = o; o += (size_t)W * image;
    if (p) {
        p->scales_off = (uint32_t)scales; p->sums_off = (uint32_t)sums; p->flags_off = (uint32_t)flags;
        p->part_off = (uint32_t)part; p->total_off = (uint32_t)total; p->image_off = (uint32_t)img;
    }
    return o;
}

// How a launch of t rows is laid out with R of them a workgroup.
struct WidePlan { int R, E, tiles, P, passes, W; unsigned grid, row_groups; };
constexpr int pairs_of(int R) { return R <= 4 ? 1 : R <= 8 ? 2 : 4; }
static_assert(pairs_of((16 + 1) / 2) < 4, "four pairs a lane: one workgroup has all rows of a launch");
WidePlan wide_plan(int rows, int NG, int t, int R, int image, bool big, int cus, size_t lds_max) {
    WidePlan q;
    q.R = R; q.E = pairs_of(R);
    q.row_groups = (unsigned)((t + R - 1) / R);
    // one workgroup per CU, those of a row group each with the same number of 16-row tiles, at most sixteen (their sums lie in LDS beside the planes)
    const int share = cus > (int)q.row_groups ? cus / (int)q.row_groups : 1, all = (rows + 15) / 16, rounds = (all + share * 16 - 1) / (share * 16);
    q.tiles = (all + share * rounds - 1) / (share * rounds);
    q.grid = (unsigned)((all + q.tiles - 1) / q.tiles);
    // as many groups a pass as fit, the passes of equal size; a wave for every item of a pass, eight at least (they all quantise)
    const int most = q.E == 1 ? 16 : q.E == 4 && big ? 8 : 12;
    auto waves = [&](int P) { const int n = q.tiles * P; return n < 8 ? 8 : (n > most ? most : n); };
    q.passes = 0;
    const size_t fixed = lds_of(q.E, 0, q.tiles, 2, most, image, nullptr), each = lds_of(q.E, 1, q.tiles, 2, most, image, nullptr) - fixed;
    const int fit = lds_max > fixed ? (int)((unsigned)(lds_max - fixed) / (unsigned)each) : 0;       // of that many a pass all fit, and perhaps of some more
    for (int n = fit > 0 ? (NG + fit) / (fit + 1) : 1; n <= NG && !q.passes; n++) {
        q.P = (NG + n - 1) / n;
        if (lds_of(q.E, q.P, q.tiles, n, waves(q.P), image, nullptr) <= lds_max) q.passes = n;
    }
    if (!q.passes) return q;
    q.passes = (NG + q.P - 1) / q.P;
    q.W = waves(q.P);
    // More waves than items, as many as there may be, where each has two pieces to quantise and their images fit: the quantiser is what a workgroup of few tiles
    // does longest. us, a wave an item | all: Q5_1 993 x 4320 at 8 rows 13.6 | 12.1, Q4_0 1458 x 17248 at 7 41.8 | 37.2, 1312 x 13280 at 14 33.1 | 29.4. With
    // fewer pieces the barriers of more waves cost as much (IQ4_XS 1029 x 1792 at 4 rows 5.5 | 6.1), and where the images take a pass's room it has more of
    // them (Q5_1 949 x 2368 at 10 rows 12.6 | 15.7). Not for Q8_0, whose images are twice as large, at more than eight rows: 9238 x 512 at 16 7.9 | 8.7, 4914 x 1120 at 11 11.6 | 12.4; of 501
    // products 20 were longer by more than 3 %.
    const bool large = image > 2048 && q.E == 4;
    if (!large && q.W < most && R * q.P >= 2 * q.W && lds_of(q.E, q.P, q.tiles, q.passes, most, image, nullptr) <= lds_max) q.W = most;
    return q;
}

// us, on a weight of `mb` megabytes: a launch, per pass its barriers and first loads, the quantiser (rows x groups over the waves), the items (issue of the
// waves with items that share a SIMD), and the weight once for every row group. The constants are the best fit over 400 products of 3 .. 16 rows, 512 .. 34816 x
// 1024 .. 17408, seven formats, in every R: 11 % rms.
float wide_us(const WidePlan& q, float mb, int cus) {
    const float quantise = (NP == 3 ? 0.62f : 0.46f) * (q.R * q.P) / q.W, working = std::max(8, std::min(q.W, q.tiles * q.P)),
                item = (NP == 3 ? 1.19f : 1.f) * (q.E == 1 ? 0.056f : q.E == 2 ? 0.107f : 0.19f) * working;
    const unsigned rounds = (q.grid * q.row_groups + (unsigned)cus - 1) / (unsigned)cus;
    return 3.1f + rounds * q.passes * (2.6f + quantise + (q.tiles * q.P + q.W - 1) / q.W * item) + 0.16f * mb * q.row_groups;
}

template <class F, int E>
int launch_wide(const fhip_weight* w, const float* d_x, size_t t, const WidePlan& q, size_t lds_max, float* d_y, hipStream_t s) {
    WideParams p;
    p.W = w->d_raw; p.x = d_x; p.y = d_y;
    p.T = (int)t; p.R = q.R; p.N = (int)w->rows; p.cols = (int)w->cols; p.row_bytes = w->row_bytes;
    p.units = (int)(w->cols / 32);
    p.NG = (p.units + 15) / 16;
    p.tiles = q.tiles; p.P = q.P; p.passes = q.passes;
    const size_t lds = lds_of(E, p.P, p.tiles, p.passes, q.W, F::IMAGE, &p);
    static bool lds_raised = false;
    if (!lds_raised) {  // workgroups may use more than the default 64 KiB of the CU's 160 KiB
        (void)hipFuncSetAttribute((const void*)gemv_wide_kernel<F, E>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max);
        (void)hipGetLastError();
        lds_raised = true;
    }
    hipLaunchKernelGGL((gemv_wide_kernel<F, E>), dim3(q.grid, q.row_groups), dim3(64 * q.W), lds, s, p);
    return fhip::check_hip(hipGetLastError(), "gemv_wide launch");
}

// The rows of a batch by one workgroup or by up to four, each with its share of them and of the CUs: each then quantises fewer rows and holds fewer pairs a lane, and
// tiles too few for the CUs meet more of these, for the weight once more a group. Dealt out where the estimate is 8 % under that of one group. us, one | two | three |
// four groups, 24 bits: IQ4_XS 1636 x 13824 at 16 rows 55.2 | 32.7 | 31.6 | 25.0, MXFP4 1145 x 8160 at 8 20.3 | 13.7 | 13.2 | 16.2, 5433 x 14048 at 16 78.8 | 54.5 | 57.4 | 60.0,
// Q4_0 918 x 3680 at 5 9.6 | 8.2 | 7.7 | 7.7; not: Q4_1 29831 x 2688 at 16 41.0 | 45.6 | 60.7 | 56.2, MXFP4 22048 x 2592 at 7 (16 bits) 19.2 | 22.2 | 34.6 | 39.6. Over
// 1000 products of 3 .. 16 rows 0.77 of the time of one group with a wave an item (or of the dot-product kernel, where that had them), seven 3 .. 14 % slower, most where half the
// CUs for a group make two tiles of one (IQ4_XS 2642 x 15872 at 5 rows and 16 bits 20.2 | 24.0); the best of all layouts would give 0.98 of that. (At 5 % and a wave an item as good on average, but more are slower: Q4_0 2057 x 4096 at four rows 8.4 -> 9.9, whose 129
// tiles are one more than half the CUs.)
template <class F>
int launch_wide_fmt(const fhip_weight* w, const float* d_x, size_t t, float* d_y, hipStream_t s) {
    const int cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    const size_t lds_max = fhip::device_lds_bytes() > 0 ? fhip::device_lds_bytes() : 65536;
    const int NG = ((int)(w->cols / 32) + 15) / 16;
    const float mb = (float)w->rows * (float)w->row_bytes * 1e-6f;
    WidePlan best = wide_plan((int)w->rows, NG, (int)t, (int)t, F::IMAGE, F::BIG, cus, lds_max);
    if (!best.passes) return fhip::set_error(FHIP_ERR_SHAPE, "gemv_wide: a pass does not fit the workgroup's LDS");
    float us = wide_us(best, mb, cus) / 1.08f;
    for (int groups = 2; us > 7.f && groups <= 4 && groups <= (int)t; groups++) {   // (not the shortest, which the fit does not tell apart; 0.1 us of the host)
        const WidePlan q = wide_plan((int)w->rows, NG, (int)t, ((int)t + groups - 1) / groups, F::IMAGE, F::BIG, cus, lds_max);
        const float u = q.passes ? wide_us(q, mb, cus) : us;
        if (u < us) { us = u; best = q; }
    }
    switch (best.E) {
        case 1: return launch_wide<F, 1>(w, d_x, t, best, lds_max, d_y, s);
        case 2: return launch_wide<F, 2>(w, d_x, t, best, lds_max, d_y, s);
        default: return launch_wide<F, 4>(w, d_x, t, best, lds_max, d_y, s);
    }
}

}  // namespace

namespace fhip {

bool WIDE_EXPORT(gemv_wide_supports)(const fhip_weight* w, size_t t) {
    if (!w || t < 1 || t > 16 || w->rows == 0 || w->cols == 0 || w->cols % 32 != 0 || w->rows > 0x7FFFFF00ull) return false;
    switch (w->type) {
        case FHIP_Q4_0: case FHIP_Q4_1: case FHIP_Q5_0: case FHIP_Q5_1: case FHIP_Q8_0: case FHIP_IQ4_NL: case FHIP_IQ4_XS: case FHIP_MXFP4: break;
        default: return false;
    }
    // the streaming kernel's bits are what this kernel promises: only weights that take it (the longest rows go to the
    // shape-complete f32 kernel)
    return WIDE_EXPORT(gemv_streams)(w, 0);
}

// y [t, rows] = x [t, cols] W^T, t <= 16
int WIDE_EXPORT(launch_gemv_wide)(const fhip_weight* w, const float* d_x, size_t t, float* d_y, hipStream_t s) {
    switch (w->type) {
        case FHIP_Q4_0: return launch_wide_fmt<Q40>(w, d_x, t, d_y, s);
        case FHIP_Q4_1: return launch_wide_fmt<Q41>(w, d_x, t, d_y, s);
        case FHIP_Q5_0: return launch_wide_fmt<Q50>(w, d_x, t, d_y, s);
        case FHIP_Q5_1: return launch_wide_fmt<Q51>(w, d_x, t, d_y, s);
        case FHIP_Q8_0: return launch_wide_fmt<Q80>(w, d_x, t, d_y, s);
        case FHIP_IQ4_NL: return launch_wide_fmt<Iq4<false>>(w, d_x, t, d_y, s);
        case FHIP_IQ4_XS: return launch_wide_fmt<Iq4<true>>(w, d_x, t, d_y, s);
        case FHIP_MXFP4: return launch_wide_fmt<Mxf4>(w, d_x, t, d_y, s);
        default: return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "gemv_wide: no kernel for ggml type %u", w->type);
    }
}

}  // namespace fhip
