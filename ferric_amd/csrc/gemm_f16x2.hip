// Small-batch (1..32 activation rows) quantized matmul on the f16 matrix cores with f32-grade results, gfx950:
//     Y[t, n] = sum_k X[t, k] * dequant(W[n, k]),   X f32 [T, K], W raw GGUF blocks [N, K], Y f32 [T, N]
//
// Stands for Tensor::matmul_q with a few activation rows (crates/ferric-tensor/src/dtype.rs:935-944; kernels
// :2995-3051 Q4_K, :3423-3469 Q6_K), which the reference runs as one thread per output walking the weight row: the
// weights are re-read per activation row there. Here one pass over the weights serves every row.
//
// How the matrix cores give f32-grade results from 16-bit operands:
//   * Weights. A K-quant weight is (super-block scale d) x (small integer): d * (sc * q) - dmin * (m) for Q4_K with
//     sc, m < 64 and q < 16, d * (sc * (q - 32)) for Q6_K. The integer factor sc*q <= 945 is exact in f16, so the B
//     operand holds sc*q as f16 and the f32 factor d is applied to the f32 accumulator once per super-block. The Q4_K
//     minima are one more MFMA per super-block: sum_sb m[n, sb] * (sum of the activations of sub-block sb). (Q6_K:
//     |sc*(q-32)| can reach 4096; products above 2048 are rounded to even, a relative 2^-12 on those weights.)
//     Q8_0 (:2948-2990) is d * (int8): the B operand holds the quant, the f32 result of every 32-wide slice takes its
//     block's d.
//   * Activations. The 256 columns of a chunk of a row are scaled by a power of two so that their largest magnitude
//     lies in [2^14, 2^15), then split into hi = f16(x) and lo = f16(x - hi): two operand rows per activation row, 22
//     significant bits at the chunk's maximum. The 16 rows of a v_mfma_f32_16x16x32_f16 hold hi and lo of 8 activation
//     rows; a chunk's f32 result takes the chunk's scale out again as it joins the total, and the two partial results
//     are added in f32 at the end. (A scale per chunk, not per row: the preparation needs no pass over the whole row in
//     front of it -- one launch less per matmul -- and a chunk of small values keeps its bits beside a large one.)
//   * Unpack cost. A lane turns a dword of 8 nibbles into 8 f16 with 1 shift, 4 and-or (the nibble lands in the
//     mantissa of the f16 constant 1024 or, for the high nibble, 16 positions up) and 4 packed f16 fma that remove the
//     constant and apply the sub-block scale: 9 VALU for 8 weights, against ~30 for the bf16 path's f32 arithmetic.
//     The k order inside an MFMA is free as long as both operands agree, so the activations are laid out in the
//     order the nibbles come out (xsplit_f16_kernel does that once per call, or each workgroup for its own chunks).
//
// Lane (g4 = lane / 16, c = lane % 16) of a wave works on weight row c of a 16-row set and on k-group g4 of each
// 32-wide MFMA slice; a wave carries two row sets (32 weight rows), a workgroup four waves (128 rows; the row-streaming
// kernel for up to 8 activation rows: eight waves, 256 rows). The (row group, 256-column chunk) units are dealt to the workgroups in equal contiguous runs; a run that covers its
// group's whole K stores, any other adds atomically into a Y cleared beforehand. Where the sums are to be in an order, two kernels further down do the product: one keeps a
// weight row's whole K inside a workgroup, one the operand rows in LDS.
#include "f16x2.hpp"
#include <algorithm>
#include "loads.hpp"

#include <hip/hip_fp16.h>

#include <cmath>
#include <type_traits>

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float f16_bits(uint32_t b) { return __half2float(__ushort_as_half((unsigned short)b)); }
__device__ __forceinline__ uint32_t hfma2(uint32_t v, uint32_t s, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, v), __builtin_bit_cast(f16x2, s),
                                                                  __builtin_bit_cast(f16x2, c)));
}
__device__ __forceinline__ uint32_t hmul2(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, a) * __builtin_bit_cast(f16x2, b));
}
__device__ __forceinline__ uint32_t hadd2(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, a) + __builtin_bit_cast(f16x2, b));
}
__device__ __forceinline__ uint32_t splat_h(_Float16 h) { return __builtin_bit_cast(uint32_t, (f16x2){h, h}); }
// (a & m) | o in one instruction, its constants in registers: written out, the compiler takes two with a literal each, and these are
// a fifth of what a weight costs to unpack (8 rows: Q5_K 12000 x 5120 21.8 -> 20.2 us, Q4_K 34000 x 5120 34.9 -> 33.0, Q6_K 5120 x 17408 32.9 -> 32.2)
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t o) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(m), "v"(o));
    return r;
}

constexpr uint32_t H1024 = 0x64006400u;      // f16 pair (1024, 1024): mantissa step 1
constexpr uint32_t H64 = 0x54005400u;        // f16 pair (64, 64): mantissa step 1/16
constexpr uint32_t HNEG1024 = 0xE400E400u;   // (-1024, -1024)
constexpr uint32_t HNEG64 = 0xD400D400u;     // (-64, -64)
constexpr uint32_t HNEG96 = 0xD600D600u;     // (-96, -96)
constexpr uint32_t H16TH = 0x2C002C00u;      // (1/16, 1/16)

struct __attribute__((packed, aligned(2))) U4A2 { u32x4 v; };   // 16 bytes at an address that is only 2-byte aligned

constexpr int CHUNK = 256;   // columns per chunk: one K-quant super-block
// f16 per staged operand row of a chunk: 256 activations, 8 sub-block sums, 8 zeros, then the f32 factor that takes the
// chunk's scale out again (two f16 places) and 6 of padding (row stride 35 x 16 bytes: the 16 rows a 16-byte read
// instruction touches fall into different bank groups)
constexpr int XR = 280;
constexpr int XSCALE = 272;   // column of the f32 factor

__host__ __device__ constexpr int p4(int j) { return ((j & 1) << 1) | (j >> 1); }   // 0, 2, 1, 3: byte pairs (b0,b2), (b1,b3)

template <int I, int N, class Fn>
__device__ __forceinline__ void static_for(Fn&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// ------------------------------------------------------------------------------------------------
// Per-format weight streams. `Raw` is the register image of the bytes of one chunk of one weight row that lane
// k-group g4 unpacks; pre<I>() derives the scales slice I is the first to need; frag<I>() is the B operand of slice I (8 per chunk): the
// 8 weights this lane contributes, as integers times their sub-block scale; src_k(pos) is the column (inside the chunk)
// whose activation belongs at operand position pos = (I * 4 + g4) * 8 + j.
// ------------------------------------------------------------------------------------------------

struct Q4K {
    static constexpr int BLOCK = 144;
    static constexpr bool HAS_MIN = true;
    static __host__ __device__ constexpr int occupancy(int nt) { return nt == 1 ? 4 : (nt == 2 ? 3 : 2); }   // workgroups per CU the registers allow
    // lane g4 owns bytes qs[32 g4, +32): the low nibbles are sub-block 2 g4, the high nibbles 2 g4 + 1
    // (crates/ferric-gguf/src/lib.rs:805-823); slice I is dword I of those, j < 4 its low, j >= 4 its high nibbles.
    static __host__ __device__ constexpr int src_k(int pos) {
        const int j = pos & 7, g4 = (pos >> 3) & 3, i = pos >> 5;
        return 64 * g4 + 32 * (j >> 2) + 4 * i + p4(j & 3);
    }
    static __host__ __device__ constexpr int pos_of(int k) {   // inverse of src_k
        return (((k >> 2) & 7) * 4 + (k >> 6)) * 8 + 4 * ((k >> 5) & 1) + p4(k & 3);
    }
    struct Raw { u32x4 hd, q0, q1; };
    struct Head { u32x4 hd; };
    struct Ctx { uint32_t s0, c0, s1, c1; float d, dm; int sh; };   // sh: Q5_K's shift to its fifth-bit planes
    static __device__ __forceinline__ void prime(Raw& r, const uint8_t* row, int c, int g4) {
        const uint8_t* blk = row + (size_t)c * BLOCK;
        r.hd = *(const u32x4*)blk;
        r.q0 = *(const u32x4*)(blk + 16 + 32 * g4);
        r.q1 = *(const u32x4*)(blk + 32 + 32 * g4);
    }
    static __device__ __forceinline__ void head(Head& h, const uint8_t* row, int c) { h.hd = *(const u32x4*)(row + (size_t)c * BLOCK); }
    // row-streaming kernel: a block is PARTS 16-byte pieces in global memory and a row of LROW bytes in the wave's LDS image
    static constexpr int PARTS = 9, LROW = 144, TAILS = 0, ROWS_OCCUPANCY = 3;   // (workgroups of the four-wave row-streaming kernel per CU)
    static constexpr bool ROWS_AT_16 = false;   // 9..16 rows, cold weights: 44.9 us against 42.0 us for the one-row-per-lane kernel
    static constexpr bool ROW_PER_LANE = true, SLICE_SCALE = false;
    static __device__ __forceinline__ u32x4 ldg(const uint8_t* p) { return *(const u32x4*)p; }
    // where 16-byte piece `part` of chunk ck starts in the weight row / in the LDS row (tails: 2-byte pieces)
    static __device__ __forceinline__ uint32_t piece_off(int ck, int part, int) { return (uint32_t)(ck * BLOCK + 16 * part); }
    static __device__ __forceinline__ int piece_lds(int part) { return 16 * part; }
    static __device__ __forceinline__ uint32_t tail_off(int, int, int, bool& live) { live = false; return 0; }
    static __device__ __forceinline__ int tail_lds(int) { return 0; }
    static __device__ __forceinline__ void from_lds(Raw& r, const uint8_t* row, int g4) {
        r.hd = *(const u32x4*)row;
        r.q0 = *(const u32x4*)(row + 16 + 32 * g4);
        r.q1 = *(const u32x4*)(row + 32 + 32 * g4);
    }
    static __device__ __forceinline__ void take(Raw& r, const Head& h) { r.hd = h.hd; }
    // after slice I the registers it was the last to read are reloaded with the same bytes of chunk nc
    template <int I>
    static __device__ __forceinline__ void refill(Raw& r, const uint8_t* row, int nc, int g4) {
        const uint8_t* blk = row + (size_t)nc * BLOCK;
        if (I == 3) r.q0 = *(const u32x4*)(blk + 16 + 32 * g4);
        if (I == 7) r.q1 = *(const u32x4*)(blk + 32 + 32 * g4);
    }
    // get_sc_min (crates/ferric-gguf/src/lib.rs:795-804) as bytes: scales 0..3 / 4..7 and minima 0..3 / 4..7
    static __device__ __forceinline__ uint32_t sc_bytes(const u32x4& hd, bool upper) {
        return upper ? ((hd[3] & 0x0F0F0F0Fu) | ((hd[1] >> 2) & 0x30303030u)) : (hd[1] & 0x3F3F3F3Fu);
    }
    static __device__ __forceinline__ uint32_t min_bytes(const u32x4& hd, bool upper) {
        return upper ? (((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u)) : (hd[2] & 0x3F3F3F3Fu);
    }
    template <int I>
    static __device__ __forceinline__ void pre(const Raw& r, int g4, Ctx& x) {
        if (I != 0) return;
        const uint32_t scw = sc_bytes(r.hd, g4 >= 2) >> (16 * (g4 & 1));
        const uint32_t s0 = splat_h((_Float16)(unsigned short)(scw & 0xFFu)), s1 = splat_h((_Float16)(unsigned short)((scw >> 8) & 0xFFu));
        // low nibble: (1024 + q) * sc - 1024 sc; high nibble in place: (1024 + 16 q) * (sc / 16) - 64 sc. All exact in f16.
        x.s0 = s0; x.c0 = hmul2(s0, HNEG1024);
        x.s1 = hmul2(s1, H16TH); x.c1 = hmul2(s1, HNEG64);
        x.d = f16_bits(r.hd[0] & 0xFFFFu);
        x.dm = -64.0f * f16_bits(r.hd[0] >> 16);   // the sub-block sums are staged divided by 64
    }
    template <int I>
    static __device__ __forceinline__ f16x8 frag(const Raw& r, const Ctx& x) {
        const uint32_t w = I < 4 ? r.q0[I & 3] : r.q1[I & 3], w8 = w >> 8;
        u32x4 o;
        o[0] = hfma2(and_or(w, 0x000F000Fu, H1024), x.s0, x.c0);
        o[1] = hfma2(and_or(w8, 0x000F000Fu, H1024), x.s0, x.c0);
        o[2] = hfma2(and_or(w, 0x00F000F0u, H1024), x.s1, x.c1);
        o[3] = hfma2(and_or(w8, 0x00F000F0u, H1024), x.s1, x.c1);
        return __builtin_bit_cast(f16x8, o);
    }
    // B operand of the minima MFMA: m[0..7] of this row as f16 (in every k-group: the A operand holds zeros in all but group 0)
    static __device__ __forceinline__ f16x8 mins(const Raw& r, int) {
        const uint32_t lo = min_bytes(r.hd, false), hi = min_bytes(r.hd, true);
        u32x4 o;
        o[0] = hadd2(__builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u), HNEG1024);
        o[1] = hadd2(__builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u), HNEG1024);
        o[2] = hadd2(__builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u), HNEG1024);
        o[3] = hadd2(__builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u), HNEG1024);
        return __builtin_bit_cast(f16x8, o);
    }
};

// Q5_K (crates/ferric-gguf/src/lib.rs:687-716): Q4_K's header and nibbles with 32 bytes in between that hold a fifth bit
// for every weight: bit 2 g4 of qh[l] belongs to the low nibble of qs[32 g4 + l], bit 2 g4 + 1 to its high nibble. The
// operand order, the scales and the minima are Q4_K's; codes up to 31 times scales up to 63 are still exact in f16.
struct Q5K {
    static constexpr int BLOCK = 176;
    static constexpr bool HAS_MIN = true;
    static __host__ __device__ constexpr int occupancy(int nt) { return nt == 1 ? 3 : 2; }
    static __host__ __device__ constexpr int src_k(int pos) { return Q4K::src_k(pos); }
    static __host__ __device__ constexpr int pos_of(int k) { return Q4K::pos_of(k); }
    struct Raw { u32x4 hd, h0, h1, q0, q1; };
    struct Head { u32x4 hd; };
    typedef Q4K::Ctx Ctx;
    static __device__ __forceinline__ void prime(Raw& r, const uint8_t* row, int c, int g4) {
        const uint8_t* blk = row + (size_t)c * BLOCK;
        r.hd = *(const u32x4*)blk;
        r.h0 = *(const u32x4*)(blk + 16);
        r.h1 = *(const u32x4*)(blk + 32);
        r.q0 = *(const u32x4*)(blk + 48 + 32 * g4);
        r.q1 = *(const u32x4*)(blk + 64 + 32 * g4);
    }
    static __device__ __forceinline__ void head(Head& h, const uint8_t* row, int c) { h.hd = *(const u32x4*)(row + (size_t)c * BLOCK); }
    static constexpr int PARTS = 11, LROW = 176, TAILS = 0, ROWS_OCCUPANCY = 3;   // (workgroups of the four-wave row-streaming kernel per CU)
    static constexpr bool ROWS_AT_16 = false;
    static constexpr bool ROW_PER_LANE = true, SLICE_SCALE = false;
    static __device__ __forceinline__ u32x4 ldg(const uint8_t* p) { return *(const u32x4*)p; }
    static __device__ __forceinline__ uint32_t piece_off(int ck, int part, int) { return (uint32_t)(ck * BLOCK + 16 * part); }
    static __device__ __forceinline__ int piece_lds(int part) { return 16 * part; }
    static __device__ __forceinline__ uint32_t tail_off(int, int, int, bool& live) { live = false; return 0; }
    static __device__ __forceinline__ int tail_lds(int) { return 0; }
    static __device__ __forceinline__ void from_lds(Raw& r, const uint8_t* row, int g4) {
        r.hd = *(const u32x4*)row;
        r.h0 = *(const u32x4*)(row + 16);
        r.h1 = *(const u32x4*)(row + 32);
        r.q0 = *(const u32x4*)(row + 48 + 32 * g4);
        r.q1 = *(const u32x4*)(row + 64 + 32 * g4);
    }
    static __device__ __forceinline__ void take(Raw& r, const Head& h) { r.hd = h.hd; }
    template <int I>
    static __device__ __forceinline__ void refill(Raw& r, const uint8_t* row, int nc, int g4) {
        const uint8_t* blk = row + (size_t)nc * BLOCK;
        if (I == 3) { r.h0 = *(const u32x4*)(blk + 16); r.q0 = *(const u32x4*)(blk + 48 + 32 * g4); }
        if (I == 7) { r.h1 = *(const u32x4*)(blk + 32); r.q1 = *(const u32x4*)(blk + 64 + 32 * g4); }
    }
    template <int I>
    static __device__ __forceinline__ void pre(const Raw& r, int g4, Ctx& x) {
        if (I != 0) return;
        const uint32_t scw = Q4K::sc_bytes(r.hd, g4 >= 2) >> (16 * (g4 & 1));
        const uint32_t s0 = splat_h((_Float16)(unsigned short)(scw & 0xFFu)), s1 = splat_h((_Float16)(unsigned short)((scw >> 8) & 0xFFu));
        x.s0 = s0; x.c0 = hmul2(s0, HNEG1024);
        x.s1 = hmul2(s1, H16TH); x.c1 = hmul2(s1, HNEG64);
        x.d = f16_bits(r.hd[0] & 0xFFFFu);
        x.dm = -64.0f * f16_bits(r.hd[0] >> 16);
        // the two fifth-bit planes of this lane's sub-blocks, moved to bits 0 and 1 of every byte once for the chunk
        x.sh = 2 * g4;
    }
    // the fifth bit is worth 16: mantissa bit 4 beside a low nibble (step 1), bit 8 beside a high nibble in place (step 1/16)
    template <int I>
    static __device__ __forceinline__ f16x8 frag(const Raw& r, const Ctx& x) {
        const uint32_t w = I < 4 ? r.q0[I & 3] : r.q1[I & 3], w8 = w >> 8;
        const uint32_t hb = (I < 4 ? r.h0[I & 3] : r.h1[I & 3]) >> x.sh;
        u32x4 o;
        o[0] = hfma2(and_or(hb << 4, 0x00100010u, and_or(w, 0x000F000Fu, H1024)), x.s0, x.c0);
        o[1] = hfma2(and_or(hb >> 4, 0x00100010u, and_or(w8, 0x000F000Fu, H1024)), x.s0, x.c0);
        o[2] = hfma2(and_or(hb << 7, 0x01000100u, and_or(w, 0x00F000F0u, H1024)), x.s1, x.c1);
        o[3] = hfma2(and_or(hb >> 1, 0x01000100u, and_or(w8, 0x00F000F0u, H1024)), x.s1, x.c1);
        return __builtin_bit_cast(f16x8, o);
    }
    static __device__ __forceinline__ f16x8 mins(const Raw& r, int g4) {
        Q4K::Raw q;
        q.hd = r.hd;
        return Q4K::mins(q, g4);
    }
};

struct Q6K {
    static constexpr int BLOCK = 210;
    static constexpr bool HAS_MIN = false;
    static __host__ __device__ constexpr int occupancy(int nt) { return nt == 1 ? 3 : (nt == 2 ? 2 : 1); }
    // lane g4 = (hf, lh) owns l in [16 lh, 16 lh + 16) of half hf (crates/ferric-gguf/src/lib.rs:833-851): slice I = (par, dd) is
    // dword dd of ql[64 hf + 32 par + 16 lh ..] and of qh[32 hf + 16 lh ..]; j < 4 are the low nibbles (quarter par of the
    // half, high bits in field par of the qh byte), j >= 4 the high nibbles (quarter par + 2, field par + 2). All of a
    // lane's l share l / 16 = lh, so it needs four scales a chunk: sc[8 hf + 2 qt + lh].
    static __host__ __device__ constexpr int src_k(int pos) {
        const int j = pos & 7, g4 = (pos >> 3) & 3, i = pos >> 5;
        const int hf = g4 >> 1, lh = g4 & 1, par = i >> 2, dd = i & 3;
        return 128 * hf + 32 * (par + 2 * (j >> 2)) + 16 * lh + 4 * dd + p4(j & 3);
    }
    static __host__ __device__ constexpr int pos_of(int k) {   // inverse of src_k
        const int hf = k >> 7, qt = (k >> 5) & 3, lh = (k >> 4) & 1, dd = (k >> 2) & 3;
        return ((4 * (qt & 1) + dd) * 4 + 2 * hf + lh) * 8 + 4 * (qt >> 1) + p4(k & 3);
    }
    struct Raw { u32x4 ql[2], qh, sc; uint32_t d; };
    struct Head { u32x4 sc; uint32_t d; };
    struct Ctx { uint32_t s[4]; float d, dm; };
    static __device__ __forceinline__ u32x4 ld16(const uint8_t* p) { return fhip::load16_a2(p); }   // blocks of 210 bytes
    static __device__ __forceinline__ void head(Head& h, const uint8_t* row, int c) {
        const uint8_t* blk = row + (size_t)c * BLOCK;
        h.sc = ld16(blk + 192);
        h.d = *(const uint16_t*)(blk + 208);
    }
    static __device__ __forceinline__ void take(Raw& r, const Head& h) { r.sc = h.sc; r.d = h.d; }
    // row-streaming kernel: 13 16-byte pieces + the 2-byte d; LDS rows of 240 bytes (a multiple of 16 whose dword count,
    // 60, puts the 16 rows of a read instruction into different banks). Contiguous lanes read contiguous bytes here, which
    // the 2-byte alignment of the blocks does not slow down.
    static constexpr int PARTS = 13, LROW = 240, TAILS = 1, ROWS_OCCUPANCY = 3;   // (workgroups of the four-wave row-streaming kernel per CU)
    static constexpr bool ROWS_AT_16 = true;    // 9..16 rows, cold weights: 33.2 us against 41.2 us
    static constexpr bool ROW_PER_LANE = true, SLICE_SCALE = false;
    static __device__ __forceinline__ u32x4 ldg(const uint8_t* p) { return ((const U4A2*)p)->v; }
    static __device__ __forceinline__ uint32_t piece_off(int ck, int part, int) { return (uint32_t)(ck * BLOCK + 16 * part); }
    static __device__ __forceinline__ int piece_lds(int part) { return 16 * part; }
    static __device__ __forceinline__ uint32_t tail_off(int ck, int, int, bool& live) { live = true; return (uint32_t)(ck * BLOCK + 208); }
    static __device__ __forceinline__ int tail_lds(int) { return 208; }
    static __device__ __forceinline__ void from_lds(Raw& r, const uint8_t* row, int g4) {
        const int hf = g4 >> 1, lh = g4 & 1;
        r.ql[0] = *(const u32x4*)(row + 64 * hf + 16 * lh);
        r.ql[1] = *(const u32x4*)(row + 64 * hf + 32 + 16 * lh);
        r.qh = *(const u32x4*)(row + 128 + 32 * hf + 16 * lh);
        r.sc = *(const u32x4*)(row + 192);
        r.d = *(const uint16_t*)(row + 208);
    }
    static __device__ __forceinline__ void prime(Raw& r, const uint8_t* row, int c, int g4) {
        const uint8_t* blk = row + (size_t)c * BLOCK;
        const int hf = g4 >> 1, lh = g4 & 1;
        r.ql[0] = ld16(blk + 64 * hf + 16 * lh);
        r.ql[1] = ld16(blk + 64 * hf + 32 + 16 * lh);
        r.qh = ld16(blk + 128 + 32 * hf + 16 * lh);
        r.sc = ld16(blk + 192);
        r.d = *(const uint16_t*)(blk + 208);
    }
    // after slice I the registers it was the last to read are reloaded with the same bytes of chunk nc
    template <int I>
    static __device__ __forceinline__ void refill(Raw& r, const uint8_t* row, int nc, int g4) {
        const uint8_t* blk = row + (size_t)nc * BLOCK;
        const int hf = g4 >> 1, lh = g4 & 1;
        if (I == 3) r.ql[0] = ld16(blk + 64 * hf + 16 * lh);
        if (I == 7) {
            r.ql[1] = ld16(blk + 64 * hf + 32 + 16 * lh);
            r.qh = ld16(blk + 128 + 32 * hf + 16 * lh);
        }
    }
    template <int I>
    static __device__ __forceinline__ void pre(const Raw& r, int g4, Ctx& x) {
        if (I != 0) return;
        const int hf = g4 >> 1, lh = g4 & 1;
        const uint32_t w0 = (hf ? r.sc[2] : r.sc[0]) >> (8 * lh), w1 = (hf ? r.sc[3] : r.sc[1]) >> (8 * lh);
#pragma unroll
        for (int qt = 0; qt < 4; qt++) {
            const uint32_t w = qt < 2 ? w0 : w1;
            const int v = (int)(int8_t)((w >> (16 * (qt & 1))) & 0xFFu);
            const uint32_t sp = splat_h((_Float16)(short)v);
            x.s[qt] = sp;
        }
        x.d = f16_bits(r.d);
        x.dm = 0.f;
    }
    template <int I>
    static __device__ __forceinline__ f16x8 frag(const Raw& r, const Ctx& x) {
        constexpr int par = I >> 2, dd = I & 3, flo = par, fhi = par + 2;
        const uint32_t ql = r.ql[par][dd], qh = r.qh[dd];
        constexpr uint32_t NM = 0x00F000F0u, HM = 0x03000300u;
        // a 6-bit q lands in mantissa bits 4..9 of the f16 constant 64 (step 1/16): the value is 64 + q
        const uint32_t p0 = and_or(qh << (8 - 2 * flo), HM, and_or(ql << 4, NM, H64));
        const uint32_t p1 = and_or(qh >> (2 * flo), HM, and_or(ql >> 4, NM, H64));
        const uint32_t p2 = and_or(qh << (8 - 2 * fhi), HM, and_or(ql, NM, H64));
        const uint32_t p3 = and_or(qh >> (2 * fhi), HM, and_or(ql >> 8, NM, H64));
        u32x4 o;
        const uint32_t clo = hmul2(x.s[flo], HNEG96), chi = hmul2(x.s[fhi], HNEG96);   // (64 + q) * sc - 96 sc = (q - 32) * sc
        o[0] = hfma2(p0, x.s[flo], clo);
        o[1] = hfma2(p1, x.s[flo], clo);
        o[2] = hfma2(p2, x.s[fhi], chi);
        o[3] = hfma2(p3, x.s[fhi], chi);
        return __builtin_bit_cast(f16x8, o);
    }
    static __device__ __forceinline__ f16x8 mins(const Raw&, int) { return (f16x8){0, 0, 0, 0, 0, 0, 0, 0}; }
};


// Q8_0: 34-byte blocks of 32 int8 under one f16 scale (crates/ferric-gguf/src/lib.rs:855-872), eight blocks to a chunk.
// Only the row-streaming kernel reads it. A weight enters the B operand as the exact integer q; the block's scale is
// applied to the f32 result of each 32-wide slice, which is one block. The LDS row is the chunk's 256 quants followed
// by its 8 scales: 272 bytes, 68 dwords, so the 8-byte reads of a half wave (16 rows x 2 k-groups) cover all 64 banks.
struct Q80 {
    static constexpr int BLOCK = 34;
    static constexpr bool HAS_MIN = false;
    static __host__ __device__ constexpr int occupancy(int) { return 2; }
    static __host__ __device__ constexpr int src_k(int pos) { return pos; }   // slice I is block I, in order
    static __host__ __device__ constexpr int pos_of(int k) { return k; }
    static constexpr int PARTS = 16, LROW = 272, TAILS = 8, ROWS_OCCUPANCY = 3;   // (workgroups of the four-wave row-streaming kernel per CU)
    static constexpr bool ROWS_AT_16 = true;
    static constexpr bool ROW_PER_LANE = false, SLICE_SCALE = true;
    static __device__ __forceinline__ u32x4 ldg(const uint8_t* p) { return ((const U4A2*)p)->v; }
    // a row that ends inside its last chunk: the blocks past the end re-read the last real block and get scale 0
    static __device__ __forceinline__ uint32_t piece_off(int ck, int part, int nblk) {
        const int b = 8 * ck + (part >> 1);
        return (uint32_t)(BLOCK * (b < nblk ? b : nblk - 1) + 2 + 16 * (part & 1));
    }
    static __device__ __forceinline__ int piece_lds(int part) { return 16 * part; }
    static __device__ __forceinline__ uint32_t tail_off(int ck, int t, int nblk, bool& live) {
        const int b = 8 * ck + t;
        live = b < nblk;
        return (uint32_t)(BLOCK * (live ? b : nblk - 1));
    }
    static __device__ __forceinline__ int tail_lds(int t) { return 256 + 2 * t; }
    struct Raw { const uint8_t* row; };
    struct Ctx { float d, dm; };
    static __device__ __forceinline__ void from_lds(Raw& r, const uint8_t* row, int g4) { r.row = row + 8 * g4; }
    template <int I>
    static __device__ __forceinline__ void pre(const Raw& r, int g4, Ctx& x) {
        x.d = f16_bits(*(const uint16_t*)(r.row - 8 * g4 + 256 + 2 * I));
        x.dm = 0.f;
    }
    template <int I>
    static __device__ __forceinline__ f16x8 frag(const Raw& r, const Ctx&) {
        const u32x2 q = *(const u32x2*)(r.row + 32 * I);
        // int8 q -> the byte q + 128 in the mantissa of the f16 constant 1024 -> minus 1152
        const uint32_t a = q[0] ^ 0x80808080u, b = q[1] ^ 0x80808080u;
        constexpr uint32_t HNEG1152 = 0xE480E480u;
        u32x4 o;
        o[0] = hadd2(__builtin_amdgcn_perm(0x64646464u, a, 0x04010400u), HNEG1152);
        o[1] = hadd2(__builtin_amdgcn_perm(0x64646464u, a, 0x04030402u), HNEG1152);
        o[2] = hadd2(__builtin_amdgcn_perm(0x64646464u, b, 0x04010400u), HNEG1152);
        o[3] = hadd2(__builtin_amdgcn_perm(0x64646464u, b, 0x04030402u), HNEG1152);
        return __builtin_bit_cast(f16x8, o);
    }
    static __device__ __forceinline__ f16x8 mins(const Raw&, int) { return (f16x8){0, 0, 0, 0, 0, 0, 0, 0}; }
};

// ------------------------------------------------------------------------------------------------
// Activation preparation, one short kernel. Output per chunk: 16 NT operand rows of XR f16 (rows 16 q + i, i < 8: hi of
// activation row 8 q + i; rows 16 q + 8 + i: its lo), columns in operand order (F::pos_of), followed by the 8 sub-block
// sums / 64 (formats with minima), zeros, and the f32 factor that takes the chunk's power-of-two scale out again.
// SWIGLU: the row is silu(gate) * up of a [T, 2d] = [gate | up] matrix (crates/ferric-tensor/src/lib.rs:2603-2618).
// ------------------------------------------------------------------------------------------------
constexpr int MAXW = 64;   // rows of up to 65 536 columns

// element n of row t of the matrix the split reads: as stored, or, where the producing matmul left its partial outputs to this launch, their sum in sum_parts_kernel's order
__device__ __forceinline__ float x_at(const float* __restrict__ x, int t, size_t n, const fhip::F16Parts& src) {
    if (src.parts == 0) return x[n];
    const float* q = src.part + (size_t)t * src.ld + n;
    float a = q[0];
    for (int k0 = 1; k0 < src.parts; k0 += 4) {                 // (four requested at a time: one trip to memory for the usual two to five)
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = q[(size_t)(k0 + j < src.parts ? k0 + j : 0) * src.stride];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (k0 + j < src.parts) a += v[j];
    }
    return a;
}

template <bool SWIGLU>
__device__ __forceinline__ float act(const float* __restrict__ x, int t, int K, int k, const fhip::F16Parts& src) {
    if (SWIGLU) {
        const float g = x_at(x, t, k, src), u = x_at(x, t, (size_t)K + k, src);
        return (g / (1.0f + expf(-g))) * u;
    }
    return x_at(x, t, k, src);
}

// A chunk's scale out of the largest magnitude of its columns: the factor, and the one that takes it out again
__device__ __forceinline__ void chunk_scale(float m, float& sc, float& inv) {
    sc = 1.0f;
    inv = 1.0f;
    if (m > 0.f && m < INFINITY) {
        int ex;
        (void)frexpf(m, &ex);            // m < 2^ex
        ex = ex < -111 ? -111 : ex;      // the scale stays a finite f32; chunks below 2^-111 keep fewer bits
        sc = ldexpf(1.0f, 15 - ex);      // scaled maximum in [2^14, 2^15)
        inv = ldexpf(1.0f, ex - 15);
    }
}

// one workgroup per (chunk, operand row of a group of 8): thread k of it converts column k of the chunk
template <class F, bool SWIGLU>
__global__ void __launch_bounds__(256) xsplit_f16_kernel(const float* __restrict__ X, int T, int K, int NT, uint16_t* __restrict__ Xp,
                                                       float* __restrict__ zero, size_t zero_n, fhip::F16Parts src) {
    __shared__ float red[4];
    const int tid = threadIdx.x, lane = tid & 63;
    const size_t nwg = (size_t)gridDim.x * gridDim.y;
    for (size_t k = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + tid; k < zero_n; k += nwg * 256) zero[k] = 0.f;
    const int ck = blockIdx.x, t = blockIdx.y;
    const bool live = t < T;
    const int k = ck * CHUNK + tid;
    const float* x = X + (size_t)(live ? t : 0) * (SWIGLU ? 2 * (size_t)K : (size_t)K);
    const float raw = (live && k < K) ? act<SWIGLU>(x, live ? t : 0, K, k, src) : 0.f;
    // the chunk's largest magnitude (a NaN is not one: it reaches the operands as it is and makes the output row NaN)
    float m = fabsf(raw);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (lane == 0) red[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sc, inv;
    chunk_scale(m, sc, inv);
    const size_t row = ((size_t)(ck * NT + (t >> 3)) * 16 + (t & 7)) * XR;
    auto put = [&](int col, float v) {
        const _Float16 h = (_Float16)v;
        const _Float16 l = (_Float16)(v - (float)h);
        Xp[row + col] = __builtin_bit_cast(uint16_t, h);
        Xp[row + 8 * XR + col] = __builtin_bit_cast(uint16_t, l);
    };
    const float v = raw * sc;
    put(F::pos_of(tid), v);
    // columns 256..263: sub-block sums / 64 (|sum| <= 32 * 2^15, so the quotient stays below 2^14); 264..271: zeros
    float s = F::HAS_MIN ? v : 0.f;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((tid & 31) == 0) put(CHUNK + (tid >> 5), s * 0.015625f);
    if (tid < 8) put(CHUNK + 8 + tid, 0.f);
    // columns 272, 273 of the hi and the lo row: the factor as f32; 274..279: zeros
    if (tid >= 8 && tid < 16) {
        const uint32_t bits = __float_as_uint(inv);
        const uint16_t w = tid == 8 ? (uint16_t)(bits & 0xFFFFu) : tid == 9 ? (uint16_t)(bits >> 16) : (uint16_t)0;
        Xp[row + XSCALE + (tid - 8)] = w;
        Xp[row + 8 * XR + XSCALE + (tid - 8)] = w;
    }
}

template <int PERM>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), PERM, 0xF, 0xF, true));
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_TURNED = 0x141;

// A chunk of eight activation rows, four columns to a lane, as its sixteen operand rows in LDS (hi, then lo), by one wave: the bits of xsplit_f16_kernel. The rows are
// turned through the place the operands take (a lane then has a sub-block of a row: 32 columns, whose largest magnitude and sum are mostly its own).
template <class F>
__device__ __forceinline__ void split_chunk(const f32x4 (&x)[8], uint16_t* to, int lane) {
    constexpr int XROW = 4 * CHUNK + 16;
    static_assert(8 * XROW <= 16 * XR * 2, "eight activation rows fit their operand rows' place");
    uint8_t* const st = (uint8_t*)to;
    const int row = lane >> 3, sub = lane & 7;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int r = 0; r < 8; r++) *(f32x4*)(st + r * XROW + 16 * (lane ^ (lane >> 3))) = x[r];   // a row's 16-byte pieces, the eight of a sub-block turned by its number
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    f32x4 v[8];
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = *(const f32x4*)(st + row * XROW + 16 * (8 * sub + (j ^ sub)));
    // (a NaN is not the largest magnitude: it reaches the operands as it is)
#pragma unroll
    for (int j = 0; j < 8; j++) m = fmaxf(m, fmaxf(fmaxf(fabsf(v[j][0]), fabsf(v[j][1])), fmaxf(fabsf(v[j][2]), fabsf(v[j][3]))));
    m = fmaxf(m, dpp<DPP_XOR1>(m));
    m = fmaxf(m, dpp<DPP_XOR2>(m));
    m = fmaxf(m, dpp<DPP_HALF_TURNED>(m));
    float sc, inv;
    chunk_scale(m, sc, inv);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    uint16_t* const hi = to + row * XR;
    uint16_t* const lo = hi + 8 * XR;
#pragma unroll
    for (int j = 0; j < 8; j++) {                               // four columns' positions are one aligned run of eight bytes in every format's order
        f16x4 h, l;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[j][k] *= sc;
            const _Float16 a = (_Float16)v[j][k];
            h[F::pos_of(k)] = a;
            l[F::pos_of(k)] = (_Float16)(v[j][k] - (float)a);
        }
        const int pos = F::pos_of(32 * sub + 4 * j);
        *(f16x4*)(hi + pos) = h;
        *(f16x4*)(lo + pos) = l;
    }
    if constexpr (F::HAS_MIN) {
        // the sub-block's sum in the order of xsplit's exchanges: columns 16, 8, 4, 2, 1 apart
        f32x4 w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) w[j] = v[j] + v[j + 4];
        w[0] += w[2]; w[1] += w[3];
        w[0] += w[1];
        const float s = ((w[0][0] + w[0][2]) + (w[0][1] + w[0][3])) * 0.015625f;
        const _Float16 a = (_Float16)s;
        hi[CHUNK + sub] = __builtin_bit_cast(uint16_t, a);
        lo[CHUNK + sub] = __builtin_bit_cast(uint16_t, (_Float16)(s - (float)a));
        hi[CHUNK + 8 + sub] = 0;
        lo[CHUNK + 8 + sub] = 0;
    }
    const uint32_t ib = __float_as_uint(inv);
    const uint16_t part = (uint16_t)(sub == 0 ? ib & 0xFFFFu : sub == 1 ? ib >> 16 : 0u);
    hi[XSCALE + sub] = part;
    lo[XSCALE + sub] = part;
}

struct F16Params {
    const uint8_t* W;
    const uint16_t* Xp;   // prepared activations: [nchunks][16 NT][XR] f16
    const float* X;       // or the rows as they are, [T, K], for a kernel that prepares a chunk's operand rows itself
    int K;
    float* Y;             // [T, N]
    int T, N, nchunks;
    int nblk;             // Q8_0: blocks in a weight row (the last chunk may hold fewer than 8)
    size_t row_bytes;
    long long units;      // row groups * nchunks, chunk fastest
};

template <class F, int NT>
__global__ void __launch_bounds__(256, F::occupancy(NT)) gemm_q_f16x2_kernel(F16Params p) {
    constexpr int ROWS = 16 * NT, PIECES = ROWS * XR / 8, NP = (PIECES + 255) / 256;
    __shared__ __attribute__((aligned(16))) uint16_t Xs[2][ROWS * XR];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g4 = lane >> 4, c = lane & 15;
    const int nchunks = p.nchunks;
    // the units are dealt evenly: workgroup b takes [b U / G, (b + 1) U / G), so every CU carries the same number of them
    long long u = (long long)blockIdx.x * p.units / gridDim.x;
    const long long u_end = (long long)(blockIdx.x + 1) * p.units / gridDim.x;

    u32x4 stage[NP];
    auto load_x = [&](int ck) {
        const u32x4* src = (const u32x4*)(p.Xp + (size_t)ck * ROWS * XR);
#pragma unroll
        for (int q = 0; q < NP; q++)
            if (tid + 256 * q < PIECES) stage[q] = src[tid + 256 * q];
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int q = 0; q < NP; q++)
            if (tid + 256 * q < PIECES) ((u32x4*)Xs[buf])[tid + 256 * q] = stage[q];
    };
    const int a_rd = c * XR + 8 * g4;                     // + 16 q XR + 32 I
    const int m_rd = c * XR + CHUNK + (g4 ? 8 : 0);       // sub-block sums for k-group 0, zeros for the others

    for (int seg = 0; u < u_end; seg++) {
        const int grp = (int)(u / nchunks);
        const int c_begin = (int)(u - (long long)grp * nchunks);
        const int c_end = (long long)(nchunks - c_begin) < u_end - u ? nchunks : c_begin + (int)(u_end - u);
        u += c_end - c_begin;
        const bool whole = c_begin == 0 && c_end == nchunks;
        int n[2];
        const uint8_t* wrow[2];
#pragma unroll
        for (int s = 0; s < 2; s++) {
            n[s] = grp * 128 + wave * 32 + 16 * s + c;
            wrow[s] = p.W + (size_t)(n[s] < p.N ? n[s] : p.N - 1) * p.row_bytes;
        }
        f32x4 total[2][NT];
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int q = 0; q < NT; q++) total[s][q] = (f32x4){0.f, 0.f, 0.f, 0.f};
        // Weight bytes: the quant registers of a chunk are reloaded with the next chunk's bytes as soon as their last slice
        // has read them (half a chunk to a chunk ahead of their use); the few header bytes go through `hd` a chunk ahead.
        typename F::Raw raw[2];
        typename F::Head hd[2];
#pragma unroll
        for (int s = 0; s < 2; s++) F::prime(raw[s], wrow[s], c_begin, g4);
        load_x(c_begin);
        if (seg > 0) __syncthreads();   // the previous segment's last reads of buffer 0 are done
        store_x(0);
        __syncthreads();

        for (int ck = c_begin; ck < c_end; ck++) {
            const int buf = (ck - c_begin) & 1;
            const int cn = ck + 1 < c_end ? ck + 1 : ck;
#pragma unroll
            for (int s = 0; s < 2; s++) F::head(hd[s], wrow[s], cn);
            load_x(cn);
            typename F::Ctx x[2];
            f32x4 acc[2][NT];
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int q = 0; q < NT; q++) acc[s][q] = (f32x4){0.f, 0.f, 0.f, 0.f};
            static_for<0, 8>([&](auto Ic) {
                constexpr int I = decltype(Ic)::value;
                f16x8 a[NT];
#pragma unroll
                for (int q = 0; q < NT; q++) a[q] = *(const f16x8*)(&Xs[buf][a_rd + 16 * q * XR + 32 * I]);
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    F::template pre<I>(raw[s], g4, x[s]);
                    const f16x8 b = F::template frag<I>(raw[s], x[s]);
#pragma unroll
                    for (int q = 0; q < NT; q++) acc[s][q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[q], b, acc[s][q], 0, 0, 0);
                    F::template refill<I>(raw[s], wrow[s], cn, g4);
                }
            });
            // the chunk's f32 result: super-block scale times the integer-weight products (and the minima's term), then the
            // factor that takes the activation scale of the chunk's operand rows 4 g4 + r out again
            float e[NT][4];
#pragma unroll
            for (int q = 0; q < NT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) e[q][r] = *(const float*)(&Xs[buf][(16 * q + 4 * g4 + r) * XR + XSCALE]);
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int q = 0; q < NT; q++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[s][q][r] *= x[s].d;
            if constexpr (F::HAS_MIN) {
                f16x8 am[NT];
#pragma unroll
                for (int q = 0; q < NT; q++) am[q] = *(const f16x8*)(&Xs[buf][m_rd + 16 * q * XR]);
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const f16x8 bm = F::mins(raw[s], g4);
#pragma unroll
                    for (int q = 0; q < NT; q++) {
                        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                        const f32x4 accm = __builtin_amdgcn_mfma_f32_16x16x32_f16(am[q], bm, z, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[s][q][r] = fmaf(x[s].dm, accm[r], acc[s][q][r]);
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int q = 0; q < NT; q++)
#pragma unroll
                    for (int r = 0; r < 4; r++) total[s][q][r] = fmaf(e[q][r], acc[s][q][r], total[s][q][r]);
            store_x(buf ^ 1);
            __syncthreads();
#pragma unroll
            for (int s = 0; s < 2; s++) F::take(raw[s], hd[s]);
        }

        // D layout of the 16x16 MFMA: register r of lane (g4, c) is operand row 4 g4 + r, column c. Operand rows 0..7
        // are the hi parts of activation rows 8 q + [0, 8), rows 8..15 their lo parts: lanes g4 and g4 ^ 2 hold the
        // two parts of the same output.
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int q = 0; q < NT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int t = 8 * q + 4 * (g4 & 1) + r;
                    float v = total[s][q][r];
                    v += __shfl_xor(v, 32);
                    if (g4 < 2 && t < p.T && n[s] < p.N) {
                        float* y = p.Y + (size_t)t * p.N + n[s];
                        if (whole) *y = v;
                        else unsafeAtomicAdd(y, v);
                    }
                }
    }
}

// ------------------------------------------------------------------------------------------------
// Up to 8 activation rows, the same arithmetic with the weight bytes streamed the way the mat-vec kernel streams them: a
// wave fetches the chunk blocks of its 32 rows with contiguous lanes on contiguous bytes (9 lanes per 144-byte Q4_K block,
// 13 + a 2-byte tail per 210-byte Q6_K block), parks them in its own LDS image and reads them back one row per lane. A
// block is requested once, as one run of bytes, and the registers that wait for memory (the next chunk in flight) are not
// the registers in use, so loads are outstanding through all of a chunk's arithmetic. On weights no cache holds (each launch
// on bytes it has not seen) this takes 34 us for a 34816 x 5120 Q4_K weight and 27 us for 5120 x 17408 Q6_K, the kernel
// above 39 and 35.5 us: its one-row-per-lane loads ask for every cache line two or three times, 16 bytes at a time.
// ------------------------------------------------------------------------------------------------
// OWN_X: the workgroup makes the operand rows of its chunks itself out of the f32 rows, the bits of xsplit_f16_kernel's: a wave takes
// 8 NT / WAVES rows, a lane four columns (their four positions are one aligned run of eight bytes in every format's order).
template <class F, int NT, int WAVES, bool OWN_X>
__global__ void __launch_bounds__(64 * WAVES, WAVES == 8 ? 1 : (NT == 1 ? F::ROWS_OCCUPANCY : 2)) gemm_q_f16x2_rows_kernel(F16Params p) {
    // WAVES = 8 (up to 8 activation rows on the large K-split weights of the FFN block): ONE workgroup of eight waves (256 weight
    // rows) per CU. Three workgroups of four waves, each with its own staged activations, ended far apart -- the younger a workgroup on its CU the later (ends of the first / second / third
    // a CU received 24.2 / 26.0 / 28.8 us on the fused gate|up weight, 17.5 / 21.3 / 24.3 on the down projection), the last
    // one at 32.5 / 27.6 us; eight waves of one age share one staging and one barrier: whole calls 37.4 -> 35.2 and 31.6 -> 30.0 us
    // (twelve waves 35.7 - 36.8 / 30.7, ten 36.4 / 31.2, six 45.3 / 32.0, two workgroups of eight 36.2 / 35.0, of six 37.9 / 35.1).
    // Small weights and weights whose groups are not cut along K keep the four-wave workgroups (at 8 rows, ordered sums, eight waves
    // against four: 4096 x 4096 14.6 against 14.0 us, Q8_0 12288 x 4096 29.0 / 26.6, the vocabulary head 199 / 177).
    constexpr int NTHR = 64 * WAVES, GROUP = 32 * WAVES;
    constexpr int PIECES = 16 * NT * XR / 8, NP = (PIECES + NTHR - 1) / NTHR;
    constexpr int WP = 32 * F::PARTS, NW = (WP + 63) / 64;
    __shared__ __attribute__((aligned(16))) uint16_t Xs[2][16 * NT * XR];
    __shared__ __attribute__((aligned(16))) uint8_t Wl[WAVES][32 * F::LROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g4 = lane >> 4, c = lane & 15;
    const int nchunks = p.nchunks;
    // the units are dealt evenly: workgroup b takes [b U / G, (b + 1) U / G), so every CU carries the same number of them
    long long u = (long long)blockIdx.x * p.units / gridDim.x;
    const long long u_end = (long long)(blockIdx.x + 1) * p.units / gridDim.x;

    constexpr int RPW = 8 * NT / WAVES;      // OWN_X: activation rows per wave
    u32x4 stage[OWN_X ? 1 : NP];
    f32x4 xrow[OWN_X ? RPW : 1];
    auto load_x = [&](int ck) {
        if constexpr (OWN_X) {
            const int k = ck * CHUNK + 4 * lane;
#pragma unroll
            for (int r = 0; r < RPW; r++) {
                const int t = wave * RPW + r;
                xrow[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
                if (t < p.T && k < p.K) xrow[r] = *(const f32x4*)(p.X + (size_t)t * p.K + k);
            }
        } else {
            const u32x4* src = (const u32x4*)(p.Xp + (size_t)ck * 16 * NT * XR);
#pragma unroll
            for (int q = 0; q < NP; q++)
                if (tid + NTHR * q < PIECES) stage[q] = src[tid + NTHR * q];
        }
    };
    auto store_x = [&](int buf) {
        if constexpr (OWN_X) {
            const int pos = F::pos_of(4 * lane);
#pragma unroll
            for (int r = 0; r < RPW; r++) {
                const int t = wave * RPW + r;
                uint16_t* const hi = Xs[buf] + (16 * (t >> 3) + (t & 7)) * XR;
                uint16_t* const lo = hi + 8 * XR;
                // (a NaN is not the largest magnitude: it reaches the operands as it is)
                float m = fmaxf(fmaxf(fabsf(xrow[r][0]), fabsf(xrow[r][1])), fmaxf(fabsf(xrow[r][2]), fabsf(xrow[r][3])));
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
                float sc, inv;
                chunk_scale(m, sc, inv);
                uint32_t h[4], l[4];
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v[j] = xrow[r][j] * sc;
                    const _Float16 a = (_Float16)v[j];
                    h[F::pos_of(j)] = __builtin_bit_cast(uint16_t, a);
                    l[F::pos_of(j)] = __builtin_bit_cast(uint16_t, (_Float16)(v[j] - (float)a));
                }
                *(u32x2*)(hi + pos) = (u32x2){h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
                *(u32x2*)(lo + pos) = (u32x2){l[0] | (l[1] << 16), l[2] | (l[3] << 16)};
                if constexpr (F::HAS_MIN) {
                    // the sums of 32 columns in the order of xsplit's exchanges: columns 16, 8, 4, 2, 1 apart
#pragma unroll
                    for (int o = 4; o > 0; o >>= 1)
#pragma unroll
                        for (int j = 0; j < 4; j++) v[j] += __shfl_xor(v[j], o);
                    const float sum = ((v[0] + v[2]) + (v[1] + v[3])) * 0.015625f;
                    if ((lane & 7) == 0) {
                        const _Float16 a = (_Float16)sum;
                        hi[CHUNK + (lane >> 3)] = __builtin_bit_cast(uint16_t, a);
                        lo[CHUNK + (lane >> 3)] = __builtin_bit_cast(uint16_t, (_Float16)(sum - (float)a));
                    }
                    if (lane == 1) *(u32x4*)(hi + CHUNK + 8) = (u32x4){0u, 0u, 0u, 0u};
                    if (lane == 2) *(u32x4*)(lo + CHUNK + 8) = (u32x4){0u, 0u, 0u, 0u};
                }
                if (lane == 0) { *(float*)(hi + XSCALE) = inv; *(float*)(lo + XSCALE) = inv; }
            }
        } else {
#pragma unroll
            for (int q = 0; q < NP; q++)
                if (tid + NTHR * q < PIECES) ((u32x4*)Xs[buf])[tid + NTHR * q] = stage[q];
        }
    };
    const int a_rd = c * XR + 8 * g4;
    const int m_rd = c * XR + CHUNK + (g4 ? 8 : 0);

    // piece i * 64 + lane of the wave's chunk image is 16-byte part (piece % PARTS) of row (piece / PARTS)
    uint8_t* const wl = Wl[wave];
    u32x4 G[NW];
    constexpr int NTL = (32 * F::TAILS + 63) / 64;   // 2-byte tail pieces per lane
    uint32_t gt[NTL ? NTL : 1];
    // requests the bytes of unit (row group, chunk); rows past the end of the weight repeat its last row
    auto load_w = [&](int grp, int ck) {
        const int row0 = grp * GROUP + wave * 32 < p.N ? grp * GROUP + wave * 32 : p.N - 1;
        const int rmax = p.N - 1 - row0;
        const uint8_t* b = p.W + (size_t)row0 * p.row_bytes;
#pragma unroll
        for (int i = 0; i < NW; i++) {
            const int pc = i * 64 + lane, row = pc / F::PARTS;
            const uint32_t off = (uint32_t)(row < rmax ? row : rmax) * (uint32_t)p.row_bytes + F::piece_off(ck, pc - row * F::PARTS, p.nblk);
            if (pc < WP) G[i] = F::ldg(b + off);
        }
#pragma unroll
        for (int i = 0; i < NTL; i++) {
            const int tc = i * 64 + lane, row = tc / (F::TAILS ? F::TAILS : 1);
            bool live;
            const uint32_t off = (uint32_t)(row < rmax ? row : rmax) * (uint32_t)p.row_bytes + F::tail_off(ck, tc - row * F::TAILS, p.nblk, live);
            if (tc < 32 * F::TAILS) {
                gt[i] = *(const uint16_t*)(b + off);
                if (!live) gt[i] = 0;
            }
        }
    };
    auto park_w = [&]() {
#pragma unroll
        for (int i = 0; i < NW; i++) {
            const int pc = i * 64 + lane, row = pc / F::PARTS;
            if (pc < WP) *(u32x4*)(wl + row * F::LROW + F::piece_lds(pc - row * F::PARTS)) = G[i];
        }
#pragma unroll
        for (int i = 0; i < NTL; i++) {
            const int tc = i * 64 + lane, row = tc / (F::TAILS ? F::TAILS : 1);
            if (tc < 32 * F::TAILS) *(uint16_t*)(wl + row * F::LROW + F::tail_lds(tc - row * F::TAILS)) = (uint16_t)gt[i];
        }
    };
    if (u >= u_end) return;

    // The workgroup's run of units is one stream: the chunk after a group's last is the next group's first, fetched and
    // parked like any other, so a run that crosses a group boundary pays no second start-up.
    // (group, chunk) of the unit being worked on and of the next one to request: carried along by additions -- a 64-bit
    // division per unit is some hundred scalar instructions, as many cycles of a wave as the unit's arithmetic
    const long long u_begin = u;
    int grp = (int)(u / nchunks), ck = (int)(u - (long long)grp * nchunks);
    int lgrp = grp, lck = ck;
    auto request_next = [&]() {
        load_w(lgrp, lck);
        if (++lck == nchunks) { lck = 0; lgrp++; }
    };
    request_next();
    load_x(ck);
    store_x(0);
    park_w();
    if (u + 1 < u_end) request_next();
    __syncthreads();

    f32x4 total[2][NT];
    for (int it = 0; u < u_end; u++, it++) {
        const int buf = it & 1;
        const bool more = u + 1 < u_end;
        if (more) load_x(ck + 1 < nchunks ? ck + 1 : 0);
        if (u == u_begin || ck == 0) {
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int q = 0; q < NT; q++) total[s][q] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
        // the factor that takes the activation scale of this chunk's operand rows 4 g4 + r out again
        float e[NT][4];
#pragma unroll
        for (int q = 0; q < NT; q++)
#pragma unroll
            for (int r = 0; r < 4; r++) e[q][r] = *(const float*)(&Xs[buf][(16 * q + 4 * g4 + r) * XR + XSCALE]);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            typename F::Raw raw;
            F::from_lds(raw, wl + (16 * s + c) * F::LROW, g4);
            typename F::Ctx x;
            f32x4 acc[NT], ct[NT];     // the running MFMA result; the chunk's f32 result before the activation scale is taken out
            float dprev = 0.f;
#pragma unroll
            for (int q = 0; q < NT; q++) { acc[q] = (f32x4){0.f, 0.f, 0.f, 0.f}; ct[q] = (f32x4){0.f, 0.f, 0.f, 0.f}; }
            static_for<0, 8>([&](auto Ic) {
                constexpr int I = decltype(Ic)::value;
                F::template pre<I>(raw, g4, x);
                const f16x8 b = F::template frag<I>(raw, x);
                if constexpr (F::SLICE_SCALE) {
                    // every slice has a scale of its own: its product starts from zero, and joins the total while the next
                    // slice's MFMA runs
                    f32x4 cur[NT];
#pragma unroll
                    for (int q = 0; q < NT; q++) {
                        const f16x8 a = *(const f16x8*)(&Xs[buf][a_rd + 16 * q * XR + 32 * I]);
                        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                        cur[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, z, 0, 0, 0);
                        asm volatile("" : "+v"(cur[q]));
                    }
                    if constexpr (I > 0) {
#pragma unroll
                        for (int q = 0; q < NT; q++) {
#pragma unroll
                            for (int r = 0; r < 4; r++) ct[q][r] = fmaf(dprev, acc[q][r], ct[q][r]);
                            asm volatile("" : "+v"(ct[q]));
                        }
                    }
#pragma unroll
                    for (int q = 0; q < NT; q++) acc[q] = cur[q];
                    dprev = x.d;
                } else {
#pragma unroll
                    for (int q = 0; q < NT; q++) {
                        const f16x8 a = *(const f16x8*)(&Xs[buf][a_rd + 16 * q * XR + 32 * I]);
                        acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc[q], 0, 0, 0);
                        // keeps the MFMA here: left alone, the optimiser sinks the whole chain below the last fragment and holds
                        // all eight fragments and operand rows in registers meanwhile
                        asm volatile("" : "+v"(acc[q]));
                    }
                }
            });
            if constexpr (F::HAS_MIN) {
                const f16x8 bm = F::mins(raw, g4);
#pragma unroll
                for (int q = 0; q < NT; q++) {
                    const f16x8 am = *(const f16x8*)(&Xs[buf][m_rd + 16 * q * XR]);
                    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                    const f32x4 accm = __builtin_amdgcn_mfma_f32_16x16x32_f16(am, bm, z, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) ct[q][r] = fmaf(x.dm, accm[r], ct[q][r]);
                }
            }
            // the chunk's product (the last slice's, where every slice has its own scale), then out with the activation scale
#pragma unroll
            for (int q = 0; q < NT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) total[s][q][r] = fmaf(e[q][r], fmaf(x.d, acc[q][r], ct[q][r]), total[s][q][r]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more) {
            park_w();                             // unit u + 1 over unit u, which this wave has finished reading
            if (u + 2 < u_end) request_next();    // in flight through all of the next unit's arithmetic
            store_x(buf ^ 1);
        }
        if (!more || ck == nchunks - 1) {
            // this group's share is complete: whole iff the run held all of its chunks
            const bool whole = (long long)grp * nchunks >= u_begin && (long long)(grp + 1) * nchunks <= u_end;
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
              for (int q = 0; q < NT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int t = 8 * q + 4 * (g4 & 1) + r, n = grp * GROUP + wave * 32 + 16 * s + c;
                    float v = total[s][q][r];
                    v += __shfl_xor(v, 32);
                    if (g4 < 2 && t < p.T && n < p.N) {
                        float* y = p.Y + (size_t)t * p.N + n;
                        if (whole) *y = v;
                        else unsafeAtomicAdd(y, v);
                    }
                }
        }
        __syncthreads();
        if (++ck == nchunks) { ck = 0; grp++; }
    }
}

// ------------------------------------------------------------------------------------------------
// The same arithmetic with a weight row's whole K inside one workgroup: no operand rows prepared by a launch of their own, no partial sums
// in memory, no launch that adds them. Chunk ck belongs to wave ck % (waves of the workgroup), which makes the chunk's operand rows once
// (the bits are xsplit_f16_kernel's) and keeps them in registers for all the tiles of 16 weight rows the workgroup goes through; the waves' sums
// meet in LDS and are added in an order that the number of waves gives. A wave's weight bytes are fetched as in the row-streaming kernel, contiguous lanes on contiguous
// bytes into its own LDS image, its chunks of the next tile in flight through all of a tile's arithmetic. Activation rows come in sets of 8 NT,
// blockIdx.y their number: with few tiles the sets of a batch go to workgroups of their own, which read the weights again, from the caches.
//
// What bounds it: at few tiles a chain, the load of the rows, three trips through LDS and the first weights from HBM (4.5 us with one
// chunk a wave, 9 with 16 waves, 11 with two chunks, of which about 2 are the launch); at many the unpacking, as in the kernels above. Hence as many
// waves as there are chunks up to 16, and 12 with two chunks each where all are at work at once; and hence no branch and no conditional value among
// the loads: each one costs a wait for all loads before it (Q4_K 5120 x 2048 at 8 rows with such branches 12.4 us, without 7.6), and rows loaded in
// fragment order, 16 bytes to a lane from as many lines, cost the address unit 4 us more than rows loaded whole and turned in LDS.
// 8 rows, cold weights, us, before (two or three launches) | now: Q4_K 2000 x 1024 8.8 | 4.6, 4096 x 4096 13.3 | 8.9, 12000 x 3072 18.7 | 10.2,
// 34000 x 2048 24.4 | 15.8; Q6_K 4096 x 4096 13.4 | 8.9, 34000 x 3072 38.4 | 26.9; Q8_0 4096 x 4096 13.9 | 8.9, 34000 x 4096 58.1 | 41.8.
// 16 rows: Q4_K 2000 x 2048 12.9 | 6.1, 4096 x 4096 17.3 | 10.3, Q8_0 12000 x 3072 31.6 | 20.8. 32 rows: Q4_K 4096 x 4096 27.9 | 13.4.
// NT: sets of eight activation rows in one workgroup; C: chunks a wave holds (32 NT C registers of operands); WV: waves at most; EU: waves to a SIMD.
// ------------------------------------------------------------------------------------------------
struct HeldParams {
    const uint8_t* W;
    const float* X;       // [T, K]
    float* Y;             // [T, N]
    int T, N, K, nchunks, nblk, tiles, nw, like_rows;   // nw: waves of a workgroup
    size_t row_bytes;
};

template <class F, int NT, int C, int WV, int EU>
__global__ void __launch_bounds__(64 * WV, EU) gemm_q_f16x2_held_kernel(HeldParams p) {
    const bool like_rows = F::ROWS_AT_16 || p.like_rows;        // a chunk's expression is the row-streaming kernel's, or that of the kernel above it
    const int t0 = blockIdx.y * (8 * NT);                       // first activation row of the workgroup
    const float* const X = p.X + (size_t)t0 * p.K;
    float* const Y = p.Y + (size_t)t0 * p.N;
    const int T = p.T - t0;
    constexpr int WP = 16 * F::PARTS, NW = (WP + 63) / 64, NTL = (16 * F::TAILS + 63) / 64;
    constexpr int XROW = 4 * CHUNK + 16, AROW = 2 * CHUNK + 16; // bytes of a staged activation row and of an operand row: the 16 keep rows on different banks
    constexpr int IMAGE = 16 * F::LROW > 16 * AROW ? 16 * F::LROW : 16 * AROW;
    static_assert(8 * XROW <= IMAGE, "eight activation rows fit the image");
    __shared__ __attribute__((aligned(16))) uint8_t Wl[WV][IMAGE];
    __shared__ float Ps[2][WV][8 * NT][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = p.nw;                                        // (blockDim is a load from memory, whose wait would be one for all the loads before it)
    const int g4 = lane >> 4, c = lane & 15;
    uint8_t* const wl = Wl[wave];

    u32x4 G[C][NW];
    uint32_t gt[C][NTL ? NTL : 1];
    auto part = [&](int k) { const int pc = k * 64 + lane; return pc < WP ? pc : WP - 1; };
    auto tail = [&](int k) { const int tc = k * 64 + lane; return tc < 16 * F::TAILS ? tc : 16 * F::TAILS - 1; };
    auto load_w = [&](int tile, int i) {                       // rows past the end of the weight repeat its last row
        // (no branch: behind one, a wait would be for every load. What is past the end loads again what another lane or wave has loaded)
        const int mine = wave + nw * i, ck = mine < p.nchunks ? mine : p.nchunks - 1, row0 = tile * 16, rmax = p.N - 1 - row0;
        const uint8_t* b = p.W + (size_t)row0 * p.row_bytes;
#pragma unroll
        for (int k = 0; k < NW; k++) {
            const int pc = part(k), row = pc / F::PARTS;
            const uint32_t off = (uint32_t)(row < rmax ? row : rmax) * (uint32_t)p.row_bytes + F::piece_off(ck, pc - row * F::PARTS, p.nblk);
            G[i][k] = F::ldg(b + off);
        }
#pragma unroll
        for (int k = 0; k < NTL; k++) {
            const int tc = tail(k), row = tc / (F::TAILS ? F::TAILS : 1);
            bool live;
            const uint32_t off = (uint32_t)(row < rmax ? row : rmax) * (uint32_t)p.row_bytes + F::tail_off(ck, tc - row * F::TAILS, p.nblk, live);
            gt[i][k] = *(const uint16_t*)(b + off);
        }
    };
    auto park_w = [&](int i) {
#pragma unroll
        for (int k = 0; k < NW; k++) {
            const int pc = part(k), row = pc / F::PARTS;
            *(u32x4*)(wl + row * F::LROW + F::piece_lds(pc - row * F::PARTS)) = G[i][k];
        }
#pragma unroll
        for (int k = 0; k < NTL; k++) {
            const int tc = tail(k), row = tc / (F::TAILS ? F::TAILS : 1);
            bool live;
            F::tail_off(wave + nw * i, tc - row * F::TAILS, p.nblk, live);
            *(uint16_t*)(wl + row * F::LROW + F::tail_lds(tc - row * F::TAILS)) = live ? (uint16_t)gt[i][k] : (uint16_t)0;
        }
    };
    auto mine = [&](int i) { return wave + nw * i < p.nchunks; };   // wave-uniform
    f32x4 xr[C][NT][8];                                         // a chunk's 256 columns of a row, four to a lane
#pragma unroll
    for (int i = 0; i < C; i++)
#pragma unroll
        for (int q = 0; q < NT; q++)
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const int t = 8 * q + r, k = (wave + nw * i) * CHUNK + 4 * lane;
                xr[i][q][r] = *(const f32x4*)(X + (size_t)(t < T ? t : 0) * p.K + (k < p.K ? k : 0));   // (no branch: one would wait for every load)
            }
    constexpr bool LATE_W = WV == 12;                           // only once the first chunk's rows have left their registers (1500 x 6144 Q4_K at 16 rows 12.9 us, 13.8 before)
    asm volatile("" ::: "memory");                              // the rows are waited for first, the weights only once they are due
#pragma unroll
    for (int i = 0; i < C; i++)
        if (!LATE_W) load_w(blockIdx.x, i);
    asm volatile("" ::: "memory");

    // ---- operand rows of the wave's chunks: row c of a set is the hi (c < 8) or lo part of activation row c & 7
    f16x8 a[C][NT][8], am[C][NT];
    float e[C][NT][4];                                          // what takes the chunk's scale out of operand rows 4 g4 + r again
    const int row = lane >> 3, sub = lane & 7;                  // the 32 columns of an activation row that this lane cuts
#pragma unroll
    for (int i = 0; i < C; i++)
#pragma unroll
        for (int q = 0; q < NT; q++) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int r = 0; r < 8; r++) {                       // a row's 16-byte pieces, the eight of a sub-block turned by its number
                const bool in = 8 * q + r < T && (wave + nw * i) * CHUNK + 4 * lane < p.K;
                *(f32x4*)(wl + r * XROW + 16 * (lane ^ (lane >> 3))) = in ? xr[i][q][r] : (f32x4){0.f, 0.f, 0.f, 0.f};
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (LATE_W && i + q == 0) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < C; j++) load_w(blockIdx.x, j);
                asm volatile("" ::: "memory");
            }
            f32x4 v[8];
            float m = 0.f;
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = *(const f32x4*)(wl + row * XROW + 16 * (8 * sub + (j ^ sub)));
            // (a NaN is not the largest magnitude: it reaches the operands as it is)
#pragma unroll
            for (int j = 0; j < 8; j++) m = fmaxf(m, fmaxf(fmaxf(fabsf(v[j][0]), fabsf(v[j][1])), fmaxf(fabsf(v[j][2]), fabsf(v[j][3]))));
#pragma unroll
            for (int d = 1; d < 8; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
            float sc, inv;
            chunk_scale(m, sc, inv);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                f16x8 hi, low;
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float x = v[j + (k >> 2)][k & 3] *= sc;
                    hi[k] = (_Float16)x;
                    low[k] = (_Float16)(x - (float)hi[k]);
                }
                *(f16x8*)(wl + row * AROW + 64 * sub + 8 * j) = hi;
                *(f16x8*)(wl + (row + 8) * AROW + 64 * sub + 8 * j) = low;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const _Float16* ar = (const _Float16*)(wl + c * AROW);
#pragma unroll
            for (int I = 0; I < 8; I++) {                       // eight columns in the order of src_k: two fours, each in an order of its own
                const f16x4 l = *(const f16x4*)(ar + F::src_k((I * 4 + g4) * 8)), u = *(const f16x4*)(ar + F::src_k((I * 4 + g4) * 8 + 4));
                constexpr int O[8] = {F::src_k(0), F::src_k(1), F::src_k(2), F::src_k(3), F::src_k(4) - F::src_k(4) + 4, F::src_k(5) - F::src_k(4) + 4,
                                      F::src_k(6) - F::src_k(4) + 4, F::src_k(7) - F::src_k(4) + 4};
                a[i][q][I] = __builtin_shufflevector(l, u, O[0], O[1], O[2], O[3], O[4], O[5], O[6], O[7]);
            }
            if constexpr (F::HAS_MIN) {
                // the sub-block's sum in the order of xsplit's exchanges: columns 16, 8, 4, 2, 1 apart
                f32x4 w[4];
#pragma unroll
                for (int j = 0; j < 4; j++) w[j] = v[j] + v[j + 4];
                w[0] += w[2]; w[1] += w[3];
                w[0] += w[1];
                const float s = ((w[0][0] + w[0][2]) + (w[0][1] + w[0][3])) * 0.015625f;
                const _Float16 sh = (_Float16)s, sl = (_Float16)(s - (float)sh);
                const int both = __builtin_bit_cast(unsigned short, sh) | __builtin_bit_cast(unsigned short, sl) << 16;
#pragma unroll
                for (int k = 0; k < 8; k++) {                   // k-group 0 holds the eight sums, the others zeros
                    const unsigned w2 = (unsigned)__shfl(both, 8 * (c & 7) + k);
                    am[i][q][k] = g4 == 0 ? __builtin_bit_cast(_Float16, (unsigned short)(c >= 8 ? w2 >> 16 : w2)) : (_Float16)0.f;
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) e[i][q][r] = __shfl(inv, 8 * ((4 * g4 + r) & 7));
        }

    int buf = 0;
    auto one_tile = [&](int tile, auto Next) {                  // Next: there is another tile after this one
        f32x4 total[NT];
#pragma unroll
        for (int q = 0; q < NT; q++) total[q] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < C; i++) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the image is the wave's own: its accesses complete in order
            park_w(i);
            if constexpr (decltype(Next)::value) load_w(tile + gridDim.x, i);
            if (!mine(i)) continue;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            typename F::Raw raw;
            F::from_lds(raw, wl + c * F::LROW, g4);
            typename F::Ctx x;
            f32x4 acc[NT], ct[NT];
            float dprev = 0.f;
#pragma unroll
            for (int q = 0; q < NT; q++) { acc[q] = (f32x4){0.f, 0.f, 0.f, 0.f}; ct[q] = (f32x4){0.f, 0.f, 0.f, 0.f}; }
            static_for<0, 8>([&](auto Ic) {
                constexpr int I = decltype(Ic)::value;
                F::template pre<I>(raw, g4, x);
                const f16x8 b = F::template frag<I>(raw, x);
                if constexpr (F::SLICE_SCALE) {                 // as in the row-streaming kernel
                    f32x4 cur[NT];
#pragma unroll
                    for (int q = 0; q < NT; q++) cur[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][q][I], b, (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    if constexpr (I > 0) {
#pragma unroll
                        for (int q = 0; q < NT; q++)
#pragma unroll
                            for (int r = 0; r < 4; r++) ct[q][r] = fmaf(dprev, acc[q][r], ct[q][r]);
                    }
#pragma unroll
                    for (int q = 0; q < NT; q++) acc[q] = cur[q];
                    dprev = x.d;
                } else {
#pragma unroll
                    for (int q = 0; q < NT; q++) acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][q][I], b, acc[q], 0, 0, 0);
                }
            });
            if constexpr (F::HAS_MIN) {
                const f16x8 bm = F::mins(raw, g4);
#pragma unroll
                for (int q = 0; q < NT; q++) {
                    const f32x4 accm = __builtin_amdgcn_mfma_f32_16x16x32_f16(am[i][q], bm, (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) ct[q][r] = like_rows ? fmaf(x.dm, accm[r], ct[q][r]) : accm[r];
                }
            }
#pragma unroll
            for (int q = 0; q < NT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    total[q][r] = fmaf(e[i][q][r], like_rows ? fmaf(x.d, acc[q][r], ct[q][r]) : fmaf(x.dm, ct[q][r], acc[q][r] * x.d), total[q][r]);
        }
        // lanes g4 and g4 ^ 2 hold the hi and the lo part of the same output: two of a lane's four change sides, and every lane adds two
#pragma unroll
        for (int q = 0; q < NT; q++)
#pragma unroll
            for (int h = 0; h < 4; h += 2) {
                const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(total[q][h]), __float_as_uint(total[q][h + 1]), false, false);
                Ps[buf][wave][8 * q + 4 * (g4 & 1) + h + (g4 >> 1)][c] = __uint_as_float(v[0]) + __uint_as_float(v[1]);
            }
        __syncthreads();
        // four lanes to an output, every fourth wave's sum each, so that no wave is kept long from the next tile (8 rows, 12000 x 4096 Q4_K 12.9 us
        // with two waves adding for all, 12.0 so); of fewer than four waves, and where the registers are short, one lane
        if (NT * C < 4 && nw >= 4) {
            for (int o = tid >> 2; o < 8 * NT * 16; o += 16 * nw) {
                const int t = o >> 4, n = tile * 16 + (o & 15);
                float v = -0.f;                                 // (adds to any value without changing it)
                for (int w = tid & 3; w < nw; w += 4) v += Ps[buf][w][t][o & 15];
                v += dpp<DPP_XOR1>(v);
                v += dpp<DPP_XOR2>(v);
                if ((tid & 3) == 0 && t < T && n < p.N) Y[(size_t)t * p.N + n] = v;
            }
        } else {
            for (int o = tid; o < 8 * NT * 16; o += 64 * nw) {
                const int t = o >> 4, n = tile * 16 + (o & 15);
                float v = Ps[buf][0][t][o & 15];
                for (int w = 1; w < nw; w++) v += Ps[buf][w][t][o & 15];
                if (t < T && n < p.N) Y[(size_t)t * p.N + n] = v;
            }
        }
        buf ^= 1;
    };
    int tile = blockIdx.x;
    for (; tile + (int)gridDim.x < p.tiles; tile += gridDim.x) one_tile(tile, std::true_type{});
    one_tile(tile, std::false_type{});
}

// ------------------------------------------------------------------------------------------------
// The same arithmetic with the operand rows in LDS and no barrier among the products: a workgroup, one to a CU, makes the operand rows of its chunks (all of K, or one of
// `parts` ranges of it) once, and its sixteen waves then go through (tile of 16 weight rows, chunk) units on their own, each a run of them along K, the next unit's bytes in
// flight through all of a unit's arithmetic. A tile that two or more waves share is added in their order behind the loop; the ranges of K are partial outputs, which
// sum_parts_kernel or the reader of y adds in their order. blockIdx.z: sets of 8 NT activation rows.
//
// What bounds it (34816 x 5120 Q4_K, 8 rows, 27 us with its sums' 3): 6 until the operands lie in LDS, then 15 of instructions (117 vector, 9 matrix for 16 x 256 weights) beside 18 of
// HBM (5.5 TB/s), which hide each other but for 3. Four waves to a SIMD are what hides them: a kernel that held its chunks' operands in registers had two, a barrier a tile, and
// took 33.8. A second unit in flight costs 2 - 4 us (a burst in front of the operand rows), operand rows made four columns to a lane 1.5, unit addresses by lane 1.
// Us, sums in order, 8 rows, streaming or held kernel before | now: Q4_K 34816 x 5120 33.8 | 27.0, 4096 x 8192 15.2 | 11.1, 1000 x 17408 16.6 | 10.3; Q6_K 5120 x 17408 32.2 | 23.7; Q8_0
// 9429 x 9600 41.7 | 32.6; 16 rows Q4_K 34816 x 5120 53.3 | 34.5, Q6_K 5120 x 17408 41.3 | 26.9; 32 rows Q4_K 34816 x 5120 83.8 | 58.
// ------------------------------------------------------------------------------------------------
struct ResidentParams {
    const uint8_t* W;
    const uint16_t* Xp;   // prepared activations: [nchunks][16 NT][XR] f16
    const float* X;       // or the rows as they are, [T, K]
    float* Y;             // [T, N], or [parts][T, N] partial sums
    int part0;            // ADD: the range of K
    int T, N, K, nblk, chunks_each, chunks_over, tiles_each, tiles_over, xp_sets;   // xp_sets: sets of eight activation rows in Xp
    size_t row_bytes;
};
constexpr int RES_WAVES = 16;
// chunks whose operand rows fit beside the waves' images into the 160 KiB of LDS
template <class F, int NT>
constexpr int resident_chunks() { return (163840 - RES_WAVES * 16 * F::LROW) / (16 * NT * XR * 2); }

// ADD: one range of K, added to what is in Y (asked in the store of every launch, 12288 x 4608 Q4_K at 24 rows took 26.3 us in place of 25.5)
template <class F, int NT, bool OWN_X, bool ADD = false>
__global__ void __launch_bounds__(64 * RES_WAVES, RES_WAVES / 4) gemm_q_f16x2_resident_kernel(ResidentParams p) {
    constexpr int MAXC = resident_chunks<F, NT>(), WP = 16 * F::PARTS, NW = (WP + 63) / 64, NTL = (16 * F::TAILS + 63) / 64, WV = RES_WAVES;
    static_assert(16 * F::LROW >= 512 * NT, "a wave's share of a tile's sums fits its image");
    __shared__ __attribute__((aligned(16))) uint16_t Xs[MAXC * 16 * NT * XR];
    __shared__ __attribute__((aligned(16))) uint8_t Wl[WV][16 * F::LROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g4 = lane >> 4, c = lane & 15;
    uint8_t* const wl = Wl[wave];
    const int part = ADD ? p.part0 : blockIdx.x, j = blockIdx.y;   // the workgroup's chunks and tiles, shared out to within one
    const int c0 = part * p.chunks_each + (part < p.chunks_over ? part : p.chunks_over), cp = p.chunks_each + (part < p.chunks_over);
    const int tile0 = j * p.tiles_each + (j < p.tiles_over ? j : p.tiles_over), units = (p.tiles_each + (j < p.tiles_over)) * cp;
    auto run_of = [&](int w) { return (int)((uint32_t)(w * units) / WV); };
    const int lo = run_of(wave), hi = run_of(wave + 1);
    const int t0 = blockIdx.z * (8 * NT), T = p.T - t0;         // the first activation row of the workgroup's set, and how many are left

    // A lane's pieces of a unit lie at the same distance from the unit's first byte throughout (Q8_0: but for a last chunk that is not full). The last tile is the
    // weight's last sixteen rows: it reads, and does not store, rows of the tile before it where there are too few; rows past the end of a smaller weight repeat its last row.
    const int rmax = p.N < 16 ? p.N - 1 : 15;
    u32x4 G[NW];
    uint32_t gt[NTL ? NTL : 1], at[NW], tat[NTL ? NTL : 1];
    auto piece = [&](int k) { const int pc = k * 64 + lane; return pc < WP ? pc : WP - 1; };
    auto tail = [&](int k) { const int tc = k * 64 + lane; return tc < 16 * F::TAILS ? tc : 16 * F::TAILS - 1; };
#pragma unroll
    for (int k = 0; k < NW; k++) {
        const int row = piece(k) / F::PARTS;
        at[k] = (uint32_t)(row < rmax ? row : rmax) * (uint32_t)p.row_bytes + (F::SLICE_SCALE ? 0u : F::piece_off(0, piece(k) - row * F::PARTS, p.nblk));
    }
#pragma unroll
    for (int k = 0; k < NTL; k++) {
        const int row = tail(k) / (F::TAILS ? F::TAILS : 1);
        bool live;
        tat[k] = (uint32_t)(row < rmax ? row : rmax) * (uint32_t)p.row_bytes + (F::SLICE_SCALE ? 0u : F::tail_off(0, tail(k) - row * F::TAILS, p.nblk, live));
    }
    auto row0_of = [&](int tile) { const int r = (tile0 + tile) * 16; return r + 16 <= p.N ? r : p.N < 16 ? 0 : p.N - 16; };
    auto load_w = [&](int tile, int ck) {
        const uint8_t* b = p.W + (size_t)row0_of(tile) * p.row_bytes + (F::SLICE_SCALE ? 0u : (uint32_t)(c0 + ck) * F::BLOCK);
#pragma unroll
        for (int k = 0; k < NW; k++) G[k] = F::ldg(b + (at[k] + (F::SLICE_SCALE ? F::piece_off(c0 + ck, piece(k) % F::PARTS, p.nblk) : 0u)));
#pragma unroll
        for (int k = 0; k < NTL; k++) {
            bool live;
            gt[k] = *(const uint16_t*)(b + (tat[k] + (F::SLICE_SCALE ? F::tail_off(c0 + ck, tail(k) % (F::TAILS ? F::TAILS : 1), p.nblk, live) : 0u)));
        }
    };
    auto park_w = [&](int ck) {
#pragma unroll
        for (int k = 0; k < NW; k++) {
            const int pc = piece(k), row = pc / F::PARTS;
            *(u32x4*)(wl + row * F::LROW + F::piece_lds(pc - row * F::PARTS)) = G[k];
        }
#pragma unroll
        for (int k = 0; k < NTL; k++) {
            const int tc = tail(k), row = tc / (F::TAILS ? F::TAILS : 1);
            bool live;
            F::tail_off(c0 + ck, tc - row * F::TAILS, p.nblk, live);
            *(uint16_t*)(wl + row * F::LROW + F::tail_lds(tc - row * F::TAILS)) = live ? (uint16_t)gt[k] : (uint16_t)0;
        }
    };
    int tile = lo / cp, ck = lo - tile * cp;

    // ---- the operand rows of the workgroup's chunks (no branch among the loads; the rows are waited for first, the weights only once they are due)
    if constexpr (OWN_X) {
        static_assert(MAXC * NT <= WV, "a chunk of a set of eight rows to a wave");
        const int set = NT == 1 ? 0 : wave & 1, mine = NT == 1 ? wave : wave >> 1, k = (c0 + mine) * CHUNK + 4 * lane;
        f32x4 xr[8];
        if (mine < cp) {
#pragma unroll
            for (int r = 0; r < 8; r++) xr[r] = *(const f32x4*)(p.X + (size_t)(t0 + (8 * set + r < T ? 8 * set + r : 0)) * p.K + (k < p.K ? k : 0));
        }
        asm volatile("" ::: "memory");
        if (lo < hi) load_w(tile, ck);
        asm volatile("" ::: "memory");
        if (mine < cp) {
#pragma unroll
            for (int r = 0; r < 8; r++)
                if (8 * set + r >= T || k >= p.K) xr[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
            split_chunk<F>(xr, Xs + (mine * NT + set) * 16 * XR, lane);
        }
    } else {
        constexpr int EACH = 2 * NT * XR, NP = (MAXC * EACH + 64 * WV - 1) / (64 * WV);   // 16-byte pieces of a chunk
        const u32x4* src = (const u32x4*)p.Xp + ((size_t)c0 * p.xp_sets + blockIdx.z * NT) * (2 * XR);
        const int pieces = cp * EACH;
        u32x4 st[NP];
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int pc = i * 64 * WV + tid < pieces ? i * 64 * WV + tid : 0, k = pc / EACH;
            st[i] = src[(size_t)k * p.xp_sets * (2 * XR) + (pc - k * EACH)];
        }
        asm volatile("" ::: "memory");
        if (lo < hi) load_w(tile, ck);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (i * 64 * WV + tid < pieces) ((u32x4*)Xs)[i * 64 * WV + tid] = st[i];
    }
    __syncthreads();

    float* const Y = p.Y + ((size_t)(ADD ? 0 : part) * p.T + t0) * p.N;
    // what a lane holds of a tile's outputs: rows 8 q + 4 (g4 & 1) + 2 h + (g4 >> 1), column c
    auto store = [&](int tl, const float (&v)[NT][2]) {
        const int n = row0_of(tl) + c;
#pragma unroll
        for (int q = 0; q < NT; q++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int t = 8 * q + 4 * (g4 & 1) + 2 * h + (g4 >> 1);
                if (t < T && n < p.N && n >= (tile0 + tl) * 16) {
                    float* const y = Y + (size_t)t * p.N + n;
                    *y = ADD ? *y + v[q][h] : v[q][h];
                }
            }
    };
    f32x4 total[NT];
    float head[NT][2], last[NT][2];                             // sums of a tile that an earlier wave began; of one that a later wave ends
#pragma unroll
    for (int q = 0; q < NT; q++) {
        total[q] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; h++) head[q][h] = last[q][h] = 0.f;
    }
    bool open = false;                                          // the wave began its last tile and does not end it
    int first = ck;
    const int a_rd = c * XR + 8 * g4, m_rd = c * XR + CHUNK + (g4 ? 8 : 0);
    auto one_unit = [&](auto Next) {                            // Next: there is another unit after this one
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the image is the wave's own: its accesses complete in order
        park_w(ck);
        const int nt = ck + 1 == cp ? tile + 1 : tile, nck = ck + 1 == cp ? 0 : ck + 1;
        if constexpr (decltype(Next)::value) load_w(nt, nck);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint16_t* const xs = Xs + ck * 16 * NT * XR;
        typename F::Raw raw;
        F::from_lds(raw, wl + c * F::LROW, g4);
        typename F::Ctx x;
        f32x4 acc[NT], ct[NT];
        float dprev = 0.f;
#pragma unroll
        for (int q = 0; q < NT; q++) { acc[q] = (f32x4){0.f, 0.f, 0.f, 0.f}; ct[q] = (f32x4){0.f, 0.f, 0.f, 0.f}; }
        static_for<0, 8>([&](auto Ic) {
            constexpr int I = decltype(Ic)::value;
            F::template pre<I>(raw, g4, x);
            const f16x8 b = F::template frag<I>(raw, x);
            f32x4 cur[NT];
#pragma unroll
            for (int q = 0; q < NT; q++) {
                const f16x8 a = *(const f16x8*)(xs + a_rd + 16 * q * XR + 32 * I);
                cur[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, F::SLICE_SCALE ? (f32x4){0.f, 0.f, 0.f, 0.f} : acc[q], 0, 0, 0);
            }
            if constexpr (F::SLICE_SCALE && I > 0) {            // as in the row-streaming kernel
#pragma unroll
                for (int q = 0; q < NT; q++)
#pragma unroll
                    for (int r = 0; r < 4; r++) ct[q][r] = fmaf(dprev, acc[q][r], ct[q][r]);
            }
#pragma unroll
            for (int q = 0; q < NT; q++) acc[q] = cur[q];
            dprev = x.d;
        });
        if constexpr (F::HAS_MIN) {
            const f16x8 bm = F::mins(raw, g4);
#pragma unroll
            for (int q = 0; q < NT; q++) {
                const f32x4 accm = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const f16x8*)(xs + m_rd + 16 * q * XR), bm, (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) ct[q][r] = fmaf(x.dm, accm[r], ct[q][r]);
            }
        }
#pragma unroll
        for (int q = 0; q < NT; q++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                total[q][r] = fmaf(*(const float*)(xs + (16 * q + 4 * g4 + r) * XR + XSCALE), fmaf(x.d, acc[q][r], ct[q][r]), total[q][r]);
        if (!decltype(Next)::value || nck == 0) {
            float v[NT][2];
#pragma unroll
            for (int q = 0; q < NT; q++) {                      // lanes g4 and g4 ^ 2 hold the hi and the lo part of the same output
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(total[q][2 * h]), __float_as_uint(total[q][2 * h + 1]), false, false);
                    v[q][h] = __uint_as_float(w[0]) + __uint_as_float(w[1]);
                }
                total[q] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
            if (first == 0 && nck == 0) {
                store(tile, v);
            } else {
                open = first == 0;
#pragma unroll
                for (int q = 0; q < NT; q++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        if (open) last[q][h] = v[q][h];
                        else head[q][h] = v[q][h];
                    }
            }
            first = 0;
        }
        if (decltype(Next)::value) { tile = nt; ck = nck; }
    };
    if (lo < hi) {
        for (int u = lo; u + 1 < hi; u++) one_unit(std::true_type{});
        one_unit(std::false_type{});
    }
    // ---- the tiles that several waves share: by the wave that began it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int q = 0; q < NT; q++)
#pragma unroll
        for (int h = 0; h < 2; h++) ((float*)wl)[(2 * q + h) * 64 + lane] = head[q][h];
    __syncthreads();
    if (!open) return;
    const int end = (tile + 1) * cp;
    for (int w = wave + 1; w < WV && run_of(w) < end; w++) {
        if (run_of(w) == run_of(w + 1)) continue;
#pragma unroll
        for (int q = 0; q < NT; q++)
#pragma unroll
            for (int h = 0; h < 2; h++) last[q][h] += ((const float*)Wl[w])[(2 * q + h) * 64 + lane];
    }
    store(tile, last);
}

// Y = partial output 0 + partial output 1 + ... in that order
__global__ void __launch_bounds__(256) sum_parts_kernel(float* __restrict__ Y, const float* __restrict__ part, size_t n, int parts) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float a = part[i];
    for (int k0 = 1; k0 < parts; k0 += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = part[(size_t)(k0 + k < parts ? k0 + k : 0) * n + i];
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (k0 + k < parts) a += v[k];
    }
    Y[i] = a;
}

__global__ void zero_f32_kernel(float* __restrict__ out, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = 0.f;
}

struct Plan {
    int nt, nchunks;
    long long units, groups;
    long long wgs;        // workgroups that are resident together
    unsigned grid;
    bool split;
    int group;            // rows of a group: 256 for up to 8 activation rows (the eight-wave kernel), else 128
};

// workgroups of the kernel that serves `nt` operand row sets that fit on a CU together
template <class F>
constexpr int slots(int nt) { return nt == 1 ? F::ROWS_OCCUPANCY : (nt == 2 && F::ROWS_AT_16 ? 2 : F::occupancy(nt)); }

int prepared_sets(size_t t) { return t <= 8 ? 1 : t <= 16 ? 2 : 4; }   // sets of eight activation rows among the prepared operand rows

Plan make_plan(const fhip_weight* w, size_t t) {
    Plan q;
    q.nt = prepared_sets(t);
    q.nchunks = (int)((w->cols + CHUNK - 1) / CHUNK);
    const long long cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    // the eight-wave kernel (groups of 256 rows, one workgroup per CU): up to 8 rows on a K-quant weight of 48 MB and more whose
    // groups it cuts along K with every CU holding one share
    q.group = 128;
    if (q.nt == 1 && (w->type == FHIP_Q4_K || w->type == FHIP_Q5_K || w->type == FHIP_Q6_K) && w->nbytes >= ((size_t)48 << 20)) {
        const long long g8 = ((long long)w->rows + 255) / 256, u8 = g8 * q.nchunks, per8 = (u8 + cus - 1) / cus;
        if (u8 >= cus && per8 * 4 < (long long)q.nchunks * 3) q.group = 256;
    }
    const long long groups = ((long long)w->rows + q.group - 1) / q.group;
    q.units = groups * q.nchunks;
    const long long wgs = q.wgs = q.group == 256 ? cus : cus * (w->type == FHIP_Q6_K ? slots<Q6K>(q.nt) : w->type == FHIP_Q8_0 ? slots<Q80>(q.nt) :
                                 w->type == FHIP_Q5_K ? slots<Q5K>(q.nt) : slots<Q4K>(q.nt));
    // one workgroup per resident slot, each with the same share of the units (a grid of 2.66 workgroups per CU leaves
    // two thirds of the CUs with half as much again to do as the rest); shares of three quarters of a group's chunks or
    // more are rounded to whole groups, which store instead of adding
    const long long per = (q.units + wgs - 1) / wgs;
    if (per >= q.nchunks || per * 4 >= (long long)q.nchunks * 3) q.grid = (unsigned)groups;
    else q.grid = (unsigned)(q.units < wgs ? q.units : wgs);
    q.split = q.grid != (unsigned)groups;
    q.groups = groups;
    return q;
}

// Whether a launch that adds by atomics makes its operand rows itself: the same bits, a launch and a trip of the rows through memory less, but every workgroup that holds a chunk converts
// it (two rows of 256 values a wave, between a chunk's products and the next barrier). Rows of one chunk that the held kernel leaves (held_beats_streaming) only: us, itself | prepared, 8 rows,
// 20000 x 256 Q4_K 5.7 | 7.0, Q6_K 5.8 | 7.6, 60000 x 256 7.7 | 8.8, 8.3 | 9.8, Q8_0 9.8 | 11.2, 151936 x 256 14.1 | 12.8, 14.4 | 16.2, 18.5 | 19.0; 16 rows Q6_K 60000 x 256 10.8 | 11.5, 151936
// 23.1 | 21.7. Of two chunks 100000 x 512 Q4_K 18.3 | 15.8, Q6_K 21.5 | 20.9, 151936 x 512 22.3 | 20.2, 26.4 | 25.4. Of more, products that are not cut have too many.
bool own_x(const fhip_weight* w, const Plan& q, const float* d_x) {
    const bool rows_kernel = (q.nt == 1 && q.group == 128) || (q.nt == 2 && (w->type == FHIP_Q8_0 || w->type == FHIP_Q6_K));
    return rows_kernel && d_x && ((uintptr_t)d_x & 15) == 0 && q.nchunks == 1;
}

template <class F>
int launch_xsplit_fmt(const float* d_x, size_t t, size_t k, bool swiglu, uint16_t* d_xp, hipStream_t s, float* zero,
                      size_t zero_n, const fhip::F16Parts& src) {
    const int nt = prepared_sets(t);
    const dim3 grid((unsigned)((k + CHUNK - 1) / CHUNK), (unsigned)(8 * nt)), wg(256);
    if (swiglu) hipLaunchKernelGGL((xsplit_f16_kernel<F, true>), grid, wg, 0, s, d_x, (int)t, (int)k, nt, d_xp, zero, zero_n, src);
    else hipLaunchKernelGGL((xsplit_f16_kernel<F, false>), grid, wg, 0, s, d_x, (int)t, (int)k, nt, d_xp, zero, zero_n, src);
    return fhip::check_hip(hipGetLastError(), "xsplit_f16 launch");
}

template <class F>
int launch_fmt(const fhip_weight* w, const uint16_t* d_xp, const float* d_x, size_t t, float* d_y, hipStream_t s, bool y_cleared) {
    const Plan q = make_plan(w, t);
    F16Params p;
    p.W = w->d_raw; p.Xp = d_xp; p.X = d_x; p.K = (int)w->cols; p.Y = d_y;
    p.T = (int)t; p.N = (int)w->rows; p.nchunks = q.nchunks; p.row_bytes = w->row_bytes;
    p.nblk = (int)(w->cols / 32);
    p.units = q.units;
    if (q.split && !y_cleared) {
        const size_t n = t * w->rows;
        hipLaunchKernelGGL(zero_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d_y, n);
    }
    const bool own = d_x != nullptr;
    if (q.nt == 1 && q.group == 256) {
        if constexpr (F::ROW_PER_LANE) hipLaunchKernelGGL((gemm_q_f16x2_rows_kernel<F, 1, 8, false>), dim3(q.grid), dim3(512), 0, s, p);
    } else if (q.nt == 1) {
        if (own) hipLaunchKernelGGL((gemm_q_f16x2_rows_kernel<F, 1, 4, true>), dim3(q.grid), dim3(256), 0, s, p);
        else hipLaunchKernelGGL((gemm_q_f16x2_rows_kernel<F, 1, 4, false>), dim3(q.grid), dim3(256), 0, s, p);
    } else if (q.nt == 2 && F::ROWS_AT_16) {
        if constexpr (F::ROWS_AT_16) {
            if (own) hipLaunchKernelGGL((gemm_q_f16x2_rows_kernel<F, 2, 4, true>), dim3(q.grid), dim3(256), 0, s, p);
            else hipLaunchKernelGGL((gemm_q_f16x2_rows_kernel<F, 2, 4, false>), dim3(q.grid), dim3(256), 0, s, p);
        }
    }
    else if constexpr (F::ROW_PER_LANE) {
        if (q.nt == 2) hipLaunchKernelGGL((gemm_q_f16x2_kernel<F, 2>), dim3(q.grid), dim3(256), 0, s, p);
        else hipLaunchKernelGGL((gemm_q_f16x2_kernel<F, 4>), dim3(q.grid), dim3(256), 0, s, p);
    } else {
        return fhip::set_error(FHIP_ERR_SHAPE, "f16x2 matmul: this format takes at most 16 activation rows, got %zu", t);
    }
    return fhip::check_hip(hipGetLastError(), "gemm_q_f16x2 launch");
}

template <class F>
int launch_held_fmt(const fhip_weight* w, const float* d_x, size_t t, float* d_y, hipStream_t s) {
    HeldParams p;
    p.W = w->d_raw; p.X = d_x; p.Y = d_y;
    p.T = (int)t; p.N = (int)w->rows; p.K = (int)w->cols; p.nblk = (int)(w->cols / 32);
    p.nchunks = (int)((w->cols + CHUNK - 1) / CHUNK);
    p.tiles = (int)((w->rows + 15) / 16);
    p.row_bytes = w->row_bytes;
    const int cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    // Both sets of 9..16 rows in one workgroup where the tiles alone fill the chip several times over: 16 rows, us, apart | together:
    // 34000 x 4096 Q4_K 36.7 | 32.2, Q8_0 62.7 | 47.7, 12000 x 3072 Q6_K 18.1 | 18.3, Q4_K 15.3 | 18.0, 2000 x 4096 Q8_0 9.2 | 14.8
    const bool two = t > 8 && t <= 16 && p.nchunks <= 16 && p.tiles > 4 * cus;
    const int sets = two ? 1 : (int)((t + 7) / 8);
    // waves: one a chunk up to 16 (4096 x 4096 Q8_0 at 8 rows 9.1 us, 13.7 with eight of two chunks each); beyond, 12 with two chunks each, or eight with three
    // and no spill. Eight where workgroups go through several tiles of a format with minima (12 | 8 waves, 12000 x 5120 Q4_K 20.9 | 18.6, 2000 x 5120 11.9 | 12.2) and of rows
    // that leave the twelve no wave idle (12000 x 6144 Q8_0 27.2 | 26.1, 3000 x 5120 at 32 rows Q6_K 1.06 of the time with eight)
    const bool mins = w->type == FHIP_Q4_K || w->type == FHIP_Q5_K, several = p.tiles * sets > cus;
    const int most = two || p.nchunks <= 8 ? 8 : p.nchunks <= 16 ? 16 : several && (mins || p.nchunks > 22) ? 8 : 12;
    const int held = (p.nchunks + most - 1) / most;
    p.nw = (p.nchunks + held - 1) / held;
    p.like_rows = t <= 8;
    // one workgroup a CU; two of eight waves where there are many tiles for their chunks. Q4_K, 8 rows, one | two: 34000 x 512 10.3 | 9.0, 12000 x 512 5.7 | 5.5, 34000 x 2048
    // 15.9 | 15.8, 5120 x 2048 7.2 | 8.6; 32 rows: 5120 x 2048 1.18 of the time with two, 20000 x 2048 0.91, 5120 x 1024 1.04, 8000 x 1024 0.89
    int slots = cus * (!two && held == 1 && most == 8 && 2 * p.tiles * sets > 3 * p.nchunks * cus ? 2 : 1) / sets;
    if (slots < 1) slots = 1;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)(p.tiles < slots ? p.tiles : slots), (unsigned)sets), dim3(64 * p.nw), 0, s, p); };
    if (two) {
        if (held == 1) go(gemm_q_f16x2_held_kernel<F, 2, 1, 8, 2>);
        else go(gemm_q_f16x2_held_kernel<F, 2, 2, 8, 2>);
    } else if (most == 16) go(gemm_q_f16x2_held_kernel<F, 1, 1, 16, 4>);
    else if (most == 12) go(gemm_q_f16x2_held_kernel<F, 1, 2, 12, 3>);
    else if (held == 1) go(gemm_q_f16x2_held_kernel<F, 1, 1, 8, 4>);
    else go(gemm_q_f16x2_held_kernel<F, 1, 3, 8, 2>);
    return fhip::check_hip(hipGetLastError(), "gemm_q_f16x2 launch");
}

using ResPlan = fhip::F16Plan;
template <class F>
constexpr int resident_chunks_of(int nt) { return nt == 1 ? resident_chunks<F, 1>() : resident_chunks<F, 2>(); }
// How many ranges K is cut into: the fewest that fit, or more where the estimate below says so. In us, fitted to 676 products of three formats (100 .. 34816 x 512 .. 17408, 8 to
// 32 rows, every number of ranges): a round of four waves' operand rows 1, the longest run of units, the sums' launch 1.7 and 0.9 a megabyte of partial outputs, the
// rows an XCD fetches (workgroups go to the eight XCDs in turn: of 8 ranges each has one) 0.8 a megabyte; tiles that all sixteen waves share add a wave's sum at a time.
// What it picks takes 1.015 of the best number's time in the mean, 1.09 at the 95th percentile. Q5_K's unit stands between its neighbours': 96 products of it (300 .. 34816 x 2560 .. 17408) 1.029,
// Q4_K's of the same shapes 1.027, at most 1.12 (300 rows, either format).
ResPlan resident_plan(const fhip_weight* w, size_t t) {
    const int nchunks = (int)((w->cols + CHUNK - 1) / CHUNK), tiles = (int)((w->rows + 15) / 16), cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    const int nt = t <= 8 ? 1 : 2, sets = ((int)t + 8 * nt - 1) / (8 * nt);
    const int most = w->type == FHIP_Q6_K ? resident_chunks_of<Q6K>(nt) : w->type == FHIP_Q8_0 ? resident_chunks_of<Q80>(nt) : w->type == FHIP_Q5_K ? resident_chunks_of<Q5K>(nt) : resident_chunks_of<Q4K>(nt);
    const double unit = w->type == FHIP_Q6_K ? 2.4 : w->type == FHIP_Q8_0 ? 3.0 : w->type == FHIP_Q5_K ? 2.2 : 2.0, rows = 8.0 * nt * sets;
    ResPlan best{nt, sets, 0, 0};
    double least = 0;
    const int fewest = (nchunks + most - 1) / most;
    for (int parts = fewest; parts <= nchunks && parts <= (fewest > 13 ? fewest + 3 : 16); parts++) {
        const int per = std::max(1, std::min(cus / (parts * sets), tiles));
        const int held = (nchunks + parts - 1) / parts, units = (tiles + per - 1) / per * held, turn = parts % 8 == 0 ? 8 : parts % 4 == 0 ? 4 : parts % 2 == 0 ? 2 : 1;
        const double us = (held * nt + 3) / 4 + unit * ((units + RES_WAVES - 1) / RES_WAVES) + (parts > 1 ? 1.7 + 3.6e-6 * parts * rows * w->rows : 0.0) + 3.2e-6 * rows * w->cols / turn +
                          (units <= RES_WAVES ? 0.08 * held : 0.0);
        if (!best.parts || us < least) { best.parts = parts; best.per_part = per; least = us; }
    }
    return best;
}

const ResPlan& plan_of(const fhip_weight* w, size_t t) { return w->f16[t <= 8 ? 0 : t <= 16 ? 1 : 2]; }

template <class F>
int launch_resident_fmt(const fhip_weight* w, const uint16_t* d_xp, const float* d_x, size_t t, float* d_y, float* d_part, hipStream_t s, fhip::F16Parts* deferred) {
    const ResPlan q = plan_of(w, t);
    ResidentParams p;
    p.W = w->d_raw; p.Xp = d_xp; p.X = d_x; p.Y = q.parts > 1 ? d_part : d_y;
    p.T = (int)t; p.N = (int)w->rows; p.K = (int)w->cols; p.nblk = (int)(w->cols / 32); p.row_bytes = w->row_bytes; p.xp_sets = prepared_sets(t);
    const int tiles = (int)((w->rows + 15) / 16), nchunks = (int)((w->cols + CHUNK - 1) / CHUNK);
    p.chunks_each = nchunks / q.parts; p.chunks_over = nchunks % q.parts; p.tiles_each = tiles / q.per_part; p.tiles_over = tiles % q.per_part;
    const bool in_turn = q.parts > 1 && !d_part;     // the ranges one after the other, each added to y: the order and the bits of the sum of partial outputs
    p.part0 = 0;
    if (in_turn) p.Y = d_y;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(in_turn ? 1u : (unsigned)q.parts, (unsigned)q.per_part, (unsigned)q.sets), dim3(64 * RES_WAVES), 0, s, p); };
    if (q.nt == 1) {
        if (d_xp) go(gemm_q_f16x2_resident_kernel<F, 1, false>);
        else go(gemm_q_f16x2_resident_kernel<F, 1, true>);
    } else {
        if (d_xp) go(gemm_q_f16x2_resident_kernel<F, 2, false>);
        else go(gemm_q_f16x2_resident_kernel<F, 2, true>);
    }
    for (p.part0 = 1; in_turn && p.part0 < q.parts; p.part0++) {
        if (q.nt == 1) go(gemm_q_f16x2_resident_kernel<F, 1, true, true>);
        else go(gemm_q_f16x2_resident_kernel<F, 2, true, true>);
    }
    const size_t n = t * w->rows;
    if (deferred) *deferred = fhip::F16Parts{d_part, q.parts > 1 ? q.parts : 0, n, w->rows};
    else if (q.parts > 1 && !in_turn) hipLaunchKernelGGL(sum_parts_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d_y, (const float*)d_part, n, q.parts);
    return fhip::check_hip(hipGetLastError(), "gemm_q_f16x2 launch");
}

}  // namespace

namespace fhip {

// Where the held kernel is faster than the streaming ones that add by atomics (FHIP_BATCH_AUTO): their time over its own, cold weights. Tiles (of 16 weight rows) are counted
// in the chip's CUs.
// - One chunk (256 columns): up to three and a half tiles a CU; Q8_0 at 8 rows to twelve.
// - Up to eight rows: of 2 to 12 chunks always, but for two or three of a K-quant with more than 24 tiles; of 13 to 16 from half a tile on (Q4_K 4096 columns 0.2 tiles 0.89,
//   0.7 1.09), of more from one and a half (Q8_0 5120 columns 0.5 tiles 0.98, 2.0 1.31), with minima only over 20 chunks (Q4_K 20 chunks 2.2 tiles 0.89, 24 1.05).
// - Nine to sixteen: up to four tiles, with long rows always, with few chunks until the others cut nothing along K; beyond 16 chunks from a half to four (Q4_K 0.2 0.85, 0.5 1.03,
//   2.9 1.05, 6.6 0.89; not Q5_K, 2.2 0.87), and Q6_K and Q8_0 where the others' last round is mostly idle (17 tiles, 547 workgroups of 1024, 1.20 .. 1.36).
// - More: up to four tiles, to nine where the others cut (not of 9 chunks on: Q4_K 3072 columns at 32 rows 4.4 tiles 1.01, 6.6 0.82); beyond 16 chunks to 24 rows three, to 32 two (Q4_K
//   2.9 1.04, 4.4 0.90; 2.0 1.04, 2.9 0.90), Q6_K while tiles times sets of eight rows are two and a half (24 rows 0.7 1.07, 1.0 0.88), and where the last round is mostly idle.
int places_taken(const Plan& q) { return (int)(100 * q.groups / ((q.groups + q.wgs - 1) / q.wgs * q.wgs)); }   // percent of its rounds' workgroups
bool held_beats_streaming(const fhip_weight* w, size_t t) {
    const size_t chunks = (w->cols + CHUNK - 1) / CHUNK, tiles = (w->rows + 15) / 16, sets = (t + 7) / 8;
    const size_t cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    const bool q6 = w->type == FHIP_Q6_K, q8 = w->type == FHIP_Q8_0;
    if (chunks == 1) return 2 * tiles <= 7 * cus || (q8 && t <= 8 && tiles <= 12 * cus);
    if (t <= 8) {
        if (chunks <= 3) return q8 || tiles <= 24 * cus;
        if (chunks <= 16) return chunks <= 12 || 2 * tiles > cus;
        return (q6 || q8 || chunks > 20) && 2 * tiles > 3 * cus;
    }
    if (t <= 16) {
        if (chunks <= 16) return tiles <= 4 * cus || q8 || chunks >= (q6 && tiles <= 24 * cus ? 4 : 8) || make_plan(w, t).split;
        if ((q6 || q8) && tiles > 9 * cus) return places_taken(make_plan(w, t)) < 70;
        return w->type != FHIP_Q5_K && 2 * tiles >= cus && tiles <= 4 * cus;
    }
    const Plan q = make_plan(w, t);
    if (q6 && q.groups > q.wgs && places_taken(q) < (t <= 24 ? 70 : 60)) return true;
    if (chunks <= 16) return tiles <= 4 * cus || (tiles <= 9 * cus && q.split && chunks <= 8);
    return q6 ? 2 * tiles * sets <= 5 * cus : tiles <= (t <= 24 ? 3 : 2) * cus;
}
// And where it keeps a product whose sums are in order from the resident kernel: where tiles are few its one launch, with its sums in LDS, is the faster, and the longer so the fewer
// unpacking passes its sets of eight rows make (us, held | resident, cold weights, sums in order).
// - One chunk: only where the resident kernel's sixteen rows at a time are half empty (Q4_K 1300 x 256 at 8 rows 3.7 | 3.5, 16 3.7 | 3.9, 32 4.6 | 4.0; 34816 x 256 at 8 7.3 | 5.1).
// - Up to eight rows: a tile and a half a CU of the formats with minima, three of 8 to 12 chunks (Q4_K 4090 x 1280 5.5 | 5.6, 8200 x 1280 7.6 | 6.2, 12000 x 2304 9.7 | 9.3, 16400 12.1 |
//   11.3); Q6_K five, Q8_0 nine, and both whatever the tiles from 12 chunks on (Q6_K 16400 x 3072 16.6 | 18.3, 151936 x 4096 118.0 | 134.0, 128256 x 2560
//   76.0 | 68.9; Q8_0 34816 x 4064 45.9 | 47.6, 151936 x 3584 144.5 | 159.7).
// - Nine to sixteen: a tile and a half (Q4_K 4090 x 1024 5.4 | 7.0, 8200 x 1024 7.7 | 7.3, 34816 x 1280 22.8 | 13.4), three of eight chunks (12000 x 2048 11.4 | 12.7), five where there
//   are no minima either (Q6_K 20000 x 2048 16.6 | 18.4, Q8_0 20000 x 1760 17.4 | 19.6); two beyond (8200 x 2560 11.9 | 12.1). Vocabularies without minima are the held
//   one's again, from 12 chunks and 11 tiles on (Q6_K 41500 x 4096 at 16 42.6 | 44.9, 151936 x 3584 at 16 110.8 | 136.7, Q8_0 153.5 | 174.0).
// - More: eight tenths (Q4_K 3070 x 1024 at 24 rows 6.2 | 6.7, 4090 x 1024 7.0 | 6.7, 34816 x 1024 at 32 25.9 | 16.1), with 8 to 12 chunks a tile and a half to 24 rows (Q8_0 6100 x 2272 15.3 |
//   14.5, 8200 19.7 | 18.2), then one (4090 x 2272 at 32 12.7 | 14.0, 6100 17.2 | 14.9); with more chunks half of one (Q5_K 2050 x 3584 at 32 12.1 | 10.3).
// - Beyond 16 chunks: up to eight rows of a vocabulary without minima, Q6_K from ten tiles a CU on, Q8_0 from six (Q6_K 34816 x 5120 40.6 | 40.3, 60000 65.1 | 68.1, 151936 148.9 | 164.4; Q8_0
//   24600 x 5120 39.8 | 39.7, 60000 87.3 | 92.8, 151936 206.6 | 221.5; Q4_K 151936 x 5120 108.4 | 109.0). Elsewhere nowhere: 572 products (17, 20 and 24 chunks, 100 .. 8200 rows, 5 .. 32
//   activation rows) 0.61 .. 1.00 of its time, geometric mean 0.75.
// 2816 products of the four formats (1 .. 16 chunks, 515 .. 34816 rows, 8, 16, 24 and 32 activation rows): what this picks takes 1.006 of the faster one's time (geometric mean), 1.054 at the
// 95th percentile, 1.20 at most; of 2424 more (4 .. 24 chunks, 8200 .. 151936 rows, 5 .. 32 activation rows) 1.004, 1.036 and 1.20, 1.013 without the lines of vocabularies.
bool held_beats_resident(const fhip_weight* w, size_t t) {
    const size_t chunks = (w->cols + CHUNK - 1) / CHUNK, tiles = (w->rows + 15) / 16;
    const size_t cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    const bool q6 = w->type == FHIP_Q6_K, q8 = w->type == FHIP_Q8_0, mins = !q6 && !q8, middle = chunks >= (q8 ? 6 : 8) && chunks <= 12;
    auto halves = [&](size_t most) { return 2 * tiles <= most * cus; };   // half tiles a CU
    if (chunks > 16) return t <= 8 && !mins && tiles > (q6 ? 10 : 6) * cus;
    if (chunks == 1) return t > 8 && t <= 24 && halves(1);
    if (t <= 8) return halves(mins ? (middle ? 6 : 3) : q6 ? 10 : 18) || (!mins && chunks >= 12);
    if (t <= 16 && !mins && chunks >= 12 && tiles > 11 * cus) return true;
    if (chunks > 12) return halves(t <= 16 ? 4 : 1);
    if (t <= 16) return halves(!middle ? 3 : chunks > 8 ? 4 : mins ? 6 : 10);
    return middle ? halves(t <= 24 ? 3 : 2) : 5 * tiles <= 4 * cus;
}
// (all workgroups of a launch that stores y read the rows: none may have written over them)
bool apart(const fhip_weight* w, const float* d_x, size_t t, const float* d_y) {
    return (uintptr_t)d_y >= (uintptr_t)(d_x + t * w->cols) || (uintptr_t)d_x >= (uintptr_t)(d_y + t * w->rows);
}
bool gemm_f16x2_held_takes(const fhip_weight* w, const float* d_x, size_t t, const float* d_y) {
    return gemm_f16x2_takes(w, t) && d_x && ((uintptr_t)d_x & 15) == 0 && w->rows <= 0x7FFFFF00ull && (w->cols + CHUNK - 1) / CHUNK <= 24 && apart(w, d_x, t, d_y);
}
bool gemm_f16x2_held(const fhip_weight* w, const float* d_x, size_t t, const float* d_y) {
    return gemm_f16x2_held_takes(w, d_x, t, d_y) && (w->batch_policy == FHIP_BATCH_ORDERED ? held_beats_resident(w, t) : held_beats_streaming(w, t));
}
// The resident kernel makes its operand rows itself wherever it can: a launch in front that prepares them costs 2 - 10 us more, or as much where it is hidden (us, itself | prepared, Q4_K, 8 rows
// 2048 x 5120 8.1 | 10.7, 34816 x 5120 27.0 | 28.7; 32 rows 2048 x 5120 11.7 | 15.2, 34816 x 5120 61.2 | 64.1, 300 x 65536 17.8 | 27.5; 132 products of the four formats at 17, 24 and 32 rows
// 0.61 .. 1.02 of the time).
bool gemm_f16x2_resident_own_x(const fhip_weight* w, const float* d_x, size_t t, const float* d_y) {
    return d_x && ((uintptr_t)d_x & 15) == 0 && (gemm_f16x2_parts(w, t) > 1 || apart(w, d_x, t, d_y));
}

int launch_gemm_f16x2_held(const fhip_weight* w, const float* d_x, size_t t, float* d_y, hipStream_t s) {
    if (t == 0 || w->rows == 0) return FHIP_OK;
    switch (w->type) {
        case FHIP_Q4_K: return launch_held_fmt<Q4K>(w, d_x, t, d_y, s);
        case FHIP_Q5_K: return launch_held_fmt<Q5K>(w, d_x, t, d_y, s);
        case FHIP_Q6_K: return launch_held_fmt<Q6K>(w, d_x, t, d_y, s);
        case FHIP_Q8_0: return launch_held_fmt<Q80>(w, d_x, t, d_y, s);
        default: return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "f16x2 matmul: no kernel for ggml type %u", w->type);
    }
}

// (the entry points whose rows a caller prepares space for keep Q8_0 to 16 rows; where sums are in order it goes as far as the others)
bool gemm_f16x2_takes(const fhip_weight* w, size_t t) {
    return gemm_f16x2_supports(w, w && w->type == FHIP_Q8_0 && w->batch_policy == FHIP_BATCH_ORDERED && t > 16 && t <= 32 ? 16 : t);
}

bool gemm_f16x2_supports(const fhip_weight* w, size_t t) {
    if (!w || t < 1 || w->cols == 0 || w->cols > (size_t)MAXW * 1024) return false;
    if (w->type == FHIP_Q8_0) return t <= 16 && w->cols % 32 == 0;   // rows of any whole number of blocks
    return (w->type == FHIP_Q4_K || w->type == FHIP_Q5_K || w->type == FHIP_Q6_K) && t <= 32 && w->cols % CHUNK == 0;
}

void gemm_f16x2_lay_out(fhip_weight* w) {
    for (size_t t : {(size_t)8, (size_t)16, (size_t)32}) w->f16[t / 16] = gemm_f16x2_supports(w, 8) ? resident_plan(w, t) : ResPlan{1, 1, 1, 1};
}
int gemm_f16x2_parts(const fhip_weight* w, size_t t) { return plan_of(w, t).parts; }
// (the most any batch of up to t rows needs: a batch of fewer rows may be cut into more ranges)
size_t gemm_f16x2_parts_bytes(const fhip_weight* w, size_t t) {
    size_t m = 0;
    for (size_t u : {t, (size_t)8, (size_t)16}) {
        const int parts = u <= t ? gemm_f16x2_parts(w, u) : 1;
        if (parts > 1) m = std::max(m, (size_t)parts * u * w->rows * sizeof(float));
    }
    return m;
}
int launch_gemm_f16x2_resident(const fhip_weight* w, const uint16_t* d_xp, const float* d_x, size_t t, float* d_y, float* d_part, hipStream_t s, F16Parts* deferred) {
    switch (w->type) {
        case FHIP_Q4_K: return launch_resident_fmt<Q4K>(w, d_xp, d_x, t, d_y, d_part, s, deferred);
        case FHIP_Q5_K: return launch_resident_fmt<Q5K>(w, d_xp, d_x, t, d_y, d_part, s, deferred);
        case FHIP_Q6_K: return launch_resident_fmt<Q6K>(w, d_xp, d_x, t, d_y, d_part, s, deferred);
        case FHIP_Q8_0: return launch_resident_fmt<Q80>(w, d_xp, d_x, t, d_y, d_part, s, deferred);
        default: return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "f16x2 matmul: no kernel for ggml type %u", w->type);
    }
}

size_t gemm_f16x2_xp_bytes(const fhip_weight* w, size_t t) {
    return (w->cols + CHUNK - 1) / CHUNK * 16 * prepared_sets(t) * XR * sizeof(uint16_t);
}

bool gemm_f16x2_adds_into_y(const fhip_weight* w, size_t t) { return make_plan(w, t).split; }

int launch_xsplit_f16(const fhip_weight* w, const float* d_x, size_t t, bool swiglu, uint16_t* d_xp, hipStream_t s, float* zero, size_t zero_n,
                      const F16Parts* src_in) {
    const F16Parts src = src_in ? *src_in : F16Parts{nullptr, 0, 0, 0};
    switch (w->type) {
        case FHIP_Q4_K: return launch_xsplit_fmt<Q4K>(d_x, t, w->cols, swiglu, d_xp, s, zero, zero_n, src);
        case FHIP_Q5_K: return launch_xsplit_fmt<Q5K>(d_x, t, w->cols, swiglu, d_xp, s, zero, zero_n, src);
        case FHIP_Q6_K: return launch_xsplit_fmt<Q6K>(d_x, t, w->cols, swiglu, d_xp, s, zero, zero_n, src);
        case FHIP_Q8_0: return launch_xsplit_fmt<Q80>(d_x, t, w->cols, swiglu, d_xp, s, zero, zero_n, src);
        default: return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "f16x2 matmul: no kernel for ggml type %u", w->type);
    }
}

bool gemm_f16x2_own_x(const fhip_weight* w, const float* d_x, size_t t) { return own_x(w, make_plan(w, t), d_x); }

int launch_gemm_f16x2(const fhip_weight* w, const uint16_t* d_xp, size_t t, float* d_y, hipStream_t s, bool y_cleared, const float* d_x) {
    switch (w->type) {
        case FHIP_Q4_K: return launch_fmt<Q4K>(w, d_xp, d_x, t, d_y, s, y_cleared);
        case FHIP_Q5_K: return launch_fmt<Q5K>(w, d_xp, d_x, t, d_y, s, y_cleared);
        case FHIP_Q6_K: return launch_fmt<Q6K>(w, d_xp, d_x, t, d_y, s, y_cleared);
        case FHIP_Q8_0: return launch_fmt<Q80>(w, d_xp, d_x, t, d_y, s, y_cleared);
        default: return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "f16x2 matmul: no kernel for ggml type %u", w->type);
    }
}

}  // namespace fhip
