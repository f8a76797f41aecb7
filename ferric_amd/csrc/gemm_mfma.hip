// Prefill dequant-GEMM on the matrix cores, gfx950:  Y[t, n] = sum_k X[t, k] * dequant(W[n, k])
// X bf16 [T, K], W raw GGUF blocks [N, K], Y f32 [T, N], f32 accumulate.
//
// Stands for the reference's cooperative-matrix prefill kernels (crates/ferric-tensor/src/dtype.rs:2059-2096
// Q4_K, :1217-1257 Q6_K, :1333-1370 Q8_0, :1074-1131 Q5_K), which dequantize an 8x8 weight tile into shared memory and
// feed an 8x8 f32 matrix unit. Here the unit is v_mfma_f32_32x32x16_bf16.
//
// Shape of the kernel. The reference found this path bound by the unpack arithmetic, not the matrix
// unit (crates/ferric-core/src/lib.rs:90-101), and the same holds here: a weight costs ~3 VALU
// operations to turn into bf16, an MFMA retires 16K multiply-adds in 32 cycles. So
//   * each lane dequantizes 8 consecutive quants of one weight row, which is exactly the B fragment a lane
//     holds in a 32x32x16 MFMA: no transposition for the weights;
//   * a dequantized fragment is published once in LDS and used by every wave that multiplies those outputs, so unpack cost is amortised
//     over the workgroup's 256 activation rows -- or, on the tiles for shorter prompts, one wave unpacks for its own 64 or 128 rows and
//     LDS carries the activations alone;
//   * the next fragments are produced while the current MFMAs run, one MFMA alternating with its share of the unpack arithmetic, with
//     two waves per SIMD to fill each other's issue gaps;
//   * the activation tile, which all 8 waves of a workgroup share, is staged through LDS (padded rows,
//     16-byte reads);
//   * the 16 k of one MFMA are chosen inside ONE scale sub-block (the k order inside an MFMA is free as
//     long as both operands agree), so a fragment needs a single (scale, min) pair;
//   * weight bytes are fetched a whole 256-column chunk ahead into the registers the previous chunk has
//     just vacated (consume, then refill), so no weight load is waited for in the steady state.
// One k-step is 64 columns = 4 MFMA slices; a chunk is 4 steps = one K-quant super-block or 8 Q8_0 blocks.
// Dequantized values are exactly the f32 the CPU dequantizer produces, rounded to bf16 (RNE) by
// v_cvt_pk_bf16_f32.
// Four kernels: the tiled one (256 activation rows x 256 outputs per workgroup), its 160-column variant (256 or 128 rows) for output
// widths that 160 deals to the chip's workgroups exactly, one of 64 or 128 rows x 32 ... 256 outputs whose waves unpack for themselves
// (short prompts, small weights), and one for up to 32 rows; the launcher picks by a cost estimate. A launch that cuts output tiles along K sums the partial tiles in a fixed order: the same inputs give the
// same bits on every run.
#include "prompt.hpp"
#include "loads.hpp"

#include <hip/hip_fp16.h>

#include <numeric>
#include <type_traits>

// This file is compiled once per weight format (FHIP_GEMM_FORMAT: its struct below); the copy for Q4_K holds the entry points.
#define FHIP_GEMM_PASTE2(a, b) a##b
#define FHIP_GEMM_PASTE(a, b) FHIP_GEMM_PASTE2(a, b)
#define FHIP_GEMM_NAME(what) FHIP_GEMM_PASTE(FHIP_GEMM_PASTE(gemm_, FHIP_GEMM_FORMAT), what)
namespace fhip {
constexpr int GEMM_TILES = 13;
extern int g_gemm_tile;   // tests: 0 ... 12 pins a tile (BM_OF x BN_OF below), anything else: the estimate decides
#define FHIP_GEMM_DECLARE(F) \
    size_t gemm_##F##_ws_bytes(const fhip_weight* w, size_t columns, size_t t, bool run_sums); \
    int gemm_##F##_launch(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, float* d_ws, size_t ws_bytes, bool run_sums); \
    int gemm_##F##_launch_swiglu(const fhip_weight* w, const uint16_t* d_x, size_t t, uint16_t* d_h, hipStream_t s, float* d_ws, size_t ws_bytes);
FHIP_GEMM_DECLARE(Q4K) FHIP_GEMM_DECLARE(Q5K) FHIP_GEMM_DECLARE(Q6K) FHIP_GEMM_DECLARE(Q80)
}  // namespace fhip

namespace {

constexpr int NTILES = fhip::GEMM_TILES;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float f16_bits(uint32_t b) { return __half2float(__ushort_as_half((unsigned short)b)); }
__device__ __forceinline__ float ub(uint32_t v, int k) { return (float)((v >> (8 * k)) & 0xFFu); }
using fhip::pk_bf16;
// 8 weights w_i = fma(s, q_i, o) from the bytes of two dwords -> one MFMA operand (8 bf16). A byte in the low half of a 16-bit field is the
// f16 denormal q * 2^-24, which v_fma_mix_f32 takes as it stands (exact, with 2^24 in the scale: `s` is 2^24 times the weight's scale): two
// masks or byte shuffles a dword in place of four byte conversions.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
constexpr float Q_ULP = 16777216.f;   // 1 / the f16 denormal of the integer 1
__device__ __forceinline__ bf16x8 frag8(uint32_t e0, uint32_t o0, uint32_t e1, uint32_t o1, float s, float o) {   // even and odd bytes of each dword
    const f16x2 a = __builtin_bit_cast(f16x2, e0), b = __builtin_bit_cast(f16x2, o0), c = __builtin_bit_cast(f16x2, e1), d = __builtin_bit_cast(f16x2, o1);
    u32x4 r;
    r[0] = pk_bf16(fmaf((float)a[0], s, o), fmaf((float)b[0], s, o));
    r[1] = pk_bf16(fmaf((float)a[1], s, o), fmaf((float)b[1], s, o));
    r[2] = pk_bf16(fmaf((float)c[0], s, o), fmaf((float)d[0], s, o));
    r[3] = pk_bf16(fmaf((float)c[1], s, o), fmaf((float)d[1], s, o));
    return __builtin_bit_cast(bf16x8, r);
}
__device__ __forceinline__ bf16x8 frag8(uint32_t q0, uint32_t q1, float s, float o) {
    constexpr uint32_t ODD = 0x0C030C01u;   // bytes 1 and 3, each above a zero byte
    return frag8(q0 & 0x00FF00FFu, __builtin_amdgcn_perm(q0, q0, ODD), q1 & 0x00FF00FFu, __builtin_amdgcn_perm(q1, q1, ODD), s, o);
}
// the same from the nibbles of two dwords that `mask` (0x000F000F or 0x00F000F0) leaves
__device__ __forceinline__ bf16x8 frag8_nibbles(uint32_t q0, uint32_t q1, uint32_t mask, float s, float o) {
    return frag8(q0 & mask, (q0 >> 8) & mask, q1 & mask, (q1 >> 8) & mask, s, o);
}

constexpr int KSTEP = 64;            // columns per k-step: 4 MFMA slices of 16
constexpr int CHUNK = 256;           // columns per chunk: 4 steps
constexpr int LDS_ROW = KSTEP + 8;   // bf16 per staged activation row (+16 B pad: conflict-free 16-byte reads)

// Column of the 8 consecutive k that lane half h (= lane / 32) holds in slice t of a step, for both
// operands and every format: sub-block (t >> 1) of the step, elements 16h + 8(t & 1) + [0, 8).
__device__ __forceinline__ constexpr int kcol(int t, int h) { return 32 * (t >> 1) + 16 * h + 8 * (t & 1); }

// The elements of X (the launcher checks that T * K fits 31 bits) a thread stages: x_piece(t, T, K, col) + x_step(first, col, K) on, for columns first + col ... + 7 of
// row t. A row past T is row T - 1 (its outputs are not stored); columns past K (of a partial last chunk, staged as zeros) are read from earlier ones of the
// same row, whose end may be the end of mapped memory: nothing behind X is read.
__host__ __device__ constexpr uint32_t x_piece(int t, int T, int K, int col) { return (uint32_t)(t < T ? t : T - 1) * (uint32_t)K + (uint32_t)(col < K ? col : K - 8); }
__host__ __device__ constexpr int x_step(int first, int col, int K) { return first + col < K ? first : 0; }


// ------------------------------------------------------------------------------------------------
// Per-format weight streams. `Raw` is the per-lane register image of one chunk of one weight row (the
// half h of it this lane unpacks). prime() loads chunk c whole. For step G of a chunk, begin<G>() derives
// the step's scales into a `Ctx`, frag<G, T>() builds the B fragment of slice T, and refill<G>() reloads
// the registers step G has just read with the same bytes of chunk `nc` (the following chunk, clamped by
// the caller to one that exists).
// ------------------------------------------------------------------------------------------------

struct Q4K {
    static constexpr bool OWN_TURNS = false;
    using Eager = Q4K;
    static constexpr int BLOCK = 144;
    static constexpr float UNPACK_US = 1.4f;   // unpack of a 256 x 256 chunk by one workgroup
    // one chunk of a workgroup tile, in us, in the order of BM_OF x BN_OF (fitted, see plan_cost_us)
    static constexpr float CHUNK_US[NTILES] = {2.39f, 3.62f, 7.17f, 4.81f, 2.02f, 1.29f, 3.00f, 1.75f, 1.16f, 1.62f, 0.78f, 1.22f, 0.61f};
    static constexpr float RUN_CHUNK_US[7] = {3.43f, 4.76f, 8.15f, 5.19f, 2.84f, 2.00f, 3.29f};
    static constexpr bool PARTIAL = false;
    static __host__ __device__ int chunks(int K) { return K / 256; }
    struct Raw { u32x4 hd, hdn, q[4]; };
    struct Ctx { float d0, o0, d1, o1; };
    static __device__ __forceinline__ void prime(Raw& r, const uint8_t* row, int c, int h, int) {
        const uint8_t* blk = row + (size_t)c * BLOCK;
        r.hd = *(const u32x4*)blk;
        r.hdn = r.hd;
#pragma unroll
        for (int g = 0; g < 4; g++) r.q[g] = *(const u32x4*)(blk + 16 + 32 * g + 16 * h);
    }
    // get_sc_min (crates/ferric-gguf/src/lib.rs:795-804) for sub-block j (a compile-time constant after inlining)
    static __device__ __forceinline__ void sc_min(const u32x4& hd, int j, float& sc, float& mn) {
        const uint32_t a = hd[1], b = hd[2], c = hd[3];
        if (j < 4) {
            sc = (float)((a >> (8 * j)) & 63u);
            mn = (float)((b >> (8 * j)) & 63u);
        } else {
            const int i = j - 4;
            sc = (float)(((c >> (8 * i)) & 0xFu) | (((a >> (8 * i + 6)) & 3u) << 4));
            mn = (float)(((c >> (8 * i + 4)) & 0xFu) | (((b >> (8 * i + 6)) & 3u) << 4));
        }
    }
    template <int G>
    static __device__ __forceinline__ void begin(Raw& r, const uint8_t*, int, int, int, Ctx& x) {
        if (G == 0) r.hd = r.hdn;
        const float d = f16_bits(r.hd[0] & 0xFFFFu) * Q_ULP, dmin = f16_bits(r.hd[0] >> 16);
        float s0, m0, s1, m1;
        sc_min(r.hd, 2 * G, s0, m0);
        sc_min(r.hd, 2 * G + 1, s1, m1);
        // y = (d*sc)*q - (dmin*m): the product is exact in f32, so the fused form rounds identically.
        // The high nibbles stay in place (q * 16) and their scale carries the 1/16, an exact power of two.
        x.d0 = d * s0; x.o0 = -(dmin * m0); x.d1 = (d * s1) * 0.0625f; x.o1 = -(dmin * m1);
    }
    // slice T: sub-block 2G + (T >> 1) = low (T < 2) or high nibbles of bytes 32G + 16h + 8(T & 1) + [0, 8)
    template <int G, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        return frag8_nibbles(r.q[G][2 * (T & 1)], r.q[G][2 * (T & 1) + 1], T < 2 ? 0x000F000Fu : 0x00F000F0u, T < 2 ? x.d0 : x.d1, T < 2 ? x.o0 : x.o1);
    }
    template <int G>
    static __device__ __forceinline__ void refill(Raw& r, const uint8_t* row, int nc, int h, int) {
        const uint8_t* nb = row + (size_t)nc * BLOCK;
        r.q[G] = *(const u32x4*)(nb + 16 + 32 * G + 16 * h);
        if (G == 1) r.hdn = *(const u32x4*)nb;
    }
};

// Q5_K is Q4_K with a fifth bit per quant (the reference's matmul_q5_k_coop, crates/ferric-tensor/src/dtype.rs:1074-1131):
// 176 B = [f16 d][f16 dmin][scales 12 B][qh 32 B][qs 128 B]; bit s of qh[l] is the fifth bit of element l of sub-block s
// (crates/ferric-gguf/src/lib.rs:692-716), q = nibble + 16 * bit in 0..31, y = (d*sc)*q - dmin*m. A lane half h works on
// elements 16h + [0, 16) of every sub-block, so it holds the same 16 bytes qh[16h, 16h + 16) for the whole chunk; slice T of
// step G takes bit 2G + (T >> 1) of them. The high nibbles are shifted down (with the fifth bit on top they do not fit a
// byte in place), so both sub-block scales are plain d * sc.
struct Q5K {
    static constexpr bool OWN_TURNS = false;
    using Eager = Q5K;
    static constexpr int BLOCK = 176;
    static constexpr float UNPACK_US = 1.8f;
    static constexpr float CHUNK_US[NTILES] = {2.86f, 4.08f, 7.68f, 5.20f, 2.28f, 1.51f, 3.37f, 1.95f, 1.34f, 1.90f, 0.92f, 1.36f, 0.72f};
    static constexpr float RUN_CHUNK_US[7] = {3.83f, 5.16f, 9.41f, 6.12f, 3.17f, 2.26f, 3.78f};
    static constexpr bool PARTIAL = false;
    static __host__ __device__ int chunks(int K) { return K / 256; }
    struct Raw { u32x4 hd, hdn, qh, qhn, q[4]; };
    struct Ctx { float d0, o0, d1, o1; };
    static __device__ __forceinline__ void prime(Raw& r, const uint8_t* row, int c, int h, int) {
        const uint8_t* blk = row + (size_t)c * BLOCK;
        r.hd = *(const u32x4*)blk;
        r.hdn = r.hd;
        r.qh = *(const u32x4*)(blk + 16 + 16 * h);
        r.qhn = r.qh;
#pragma unroll
        for (int g = 0; g < 4; g++) r.q[g] = *(const u32x4*)(blk + 48 + 32 * g + 16 * h);
    }
    template <int G>
    static __device__ __forceinline__ void begin(Raw& r, const uint8_t*, int, int, int, Ctx& x) {
        if (G == 0) { r.hd = r.hdn; r.qh = r.qhn; }
        const float d = f16_bits(r.hd[0] & 0xFFFFu) * Q_ULP, dmin = f16_bits(r.hd[0] >> 16);
        float s0, m0, s1, m1;
        Q4K::sc_min(r.hd, 2 * G, s0, m0);
        Q4K::sc_min(r.hd, 2 * G + 1, s1, m1);
        // every product is exact in f32 (11-bit d, 6-bit scale, 5-bit quant), so the fused form rounds as the reference's
        x.d0 = d * s0; x.o0 = -(dmin * m0); x.d1 = d * s1; x.o1 = -(dmin * m1);
    }
    template <int G, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        constexpr int w = 2 * (T & 1), s = 2 * G + (T >> 1);
        uint32_t v[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t nib = T < 2 ? r.q[G][w + i] & 0x0F0F0F0Fu : (r.q[G][w + i] >> 4) & 0x0F0F0F0Fu;
            const uint32_t bit = (s >= 4 ? r.qh[w + i] >> (s - 4) : r.qh[w + i] << (4 - s)) & 0x10101010u;
            v[i] = nib | bit;
        }
        return frag8(v[0], v[1], T < 2 ? x.d0 : x.d1, T < 2 ? x.o0 : x.o1);
    }
    template <int G>
    static __device__ __forceinline__ void refill(Raw& r, const uint8_t* row, int nc, int h, int) {
        const uint8_t* nb = row + (size_t)nc * BLOCK;
        r.q[G] = *(const u32x4*)(nb + 48 + 32 * G + 16 * h);
        if (G == 1) { r.hdn = *(const u32x4*)nb; r.qhn = *(const u32x4*)(nb + 16 + 16 * h); }
    }
};

struct Q6K {
    static constexpr bool OWN_TURNS = true;
    using Eager = Q6K;
    // Step G covers half hf = G >> 1 of the super-block and its groups g0 = 2(G & 1), g0 + 1 (low nibbles of
    // ql for G even, high nibbles for G odd); slice T is group g = g0 + (T >> 1), l = 16h + 8(T & 1) + [0, 8),
    // whose scale is sc[8hf + 2g + h]  (crates/ferric-gguf/src/lib.rs:833-851).
    static constexpr int BLOCK = 210;
    static constexpr float UNPACK_US = 2.3f;
    static constexpr float CHUNK_US[NTILES] = {3.67f, 5.11f, 8.61f, 5.92f, 2.70f, 1.89f, 4.48f, 2.80f, 1.70f, 2.39f, 1.32f, 1.70f, 0.92f};
    static constexpr float RUN_CHUNK_US[7] = {5.93f, 6.83f, 9.84f, 6.27f, 4.68f, 3.95f, 4.35f};
    static constexpr bool PARTIAL = false;
    static __host__ __device__ int chunks(int K) { return K / 256; }
    struct Raw { u32x4 ql[2][2], qh[2], sc, scn; uint32_t d, dn; };
    struct Ctx { float d; };
    static __device__ __forceinline__ u32x4 ld16(const uint8_t* p) { return fhip::load16_a2(p); }   // 210-byte blocks: see loads.hpp
    static __device__ __forceinline__ void prime(Raw& r, const uint8_t* row, int c, int h, int) {
        const uint8_t* blk = row + (size_t)c * BLOCK;
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
            r.ql[hf][0] = ld16(blk + 64 * hf + 16 * h);
            r.ql[hf][1] = ld16(blk + 64 * hf + 32 + 16 * h);
            r.qh[hf] = ld16(blk + 128 + 32 * hf + 16 * h);
        }
        r.scn = ld16(blk + 192);
        r.dn = *(const uint16_t*)(blk + 208);
        r.sc = r.scn;
        r.d = r.dn;
    }
    template <int G>
    static __device__ __forceinline__ void begin(Raw& r, const uint8_t*, int, int h, int, Ctx& x) {
        if (G == 0) {
            // byte h of every 16-bit pair is this lane half's scale: shift it down once per chunk
#pragma unroll
            for (int w = 0; w < 4; w++) r.sc[w] = r.scn[w] >> (8 * h);
            r.d = r.dn;
        }
        x.d = f16_bits(r.d);
    }
    template <int G, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        constexpr int hf = G >> 1, g = 2 * (G & 1) + (T >> 1), par = T >> 1, w = 2 * (T & 1);
        const uint32_t l0 = r.ql[hf][par][w], l1 = r.ql[hf][par][w + 1];
        const uint32_t h0 = r.qh[hf][w], h1 = r.qh[hf][w + 1];
        uint32_t n0, n1, u0, u1;
        if (G & 1) { n0 = (l0 >> 4) & 0x0F0F0F0Fu; n1 = (l1 >> 4) & 0x0F0F0F0Fu; }
        else       { n0 = l0 & 0x0F0F0F0Fu;        n1 = l1 & 0x0F0F0F0Fu; }
        if (g < 2) { u0 = (h0 << (g < 2 ? 4 - 2 * g : 0)) & 0x30303030u; u1 = (h1 << (g < 2 ? 4 - 2 * g : 0)) & 0x30303030u; }
        else       { u0 = (h0 >> (g < 2 ? 0 : 2 * g - 4)) & 0x30303030u; u1 = (h1 >> (g < 2 ? 0 : 2 * g - 4)) & 0x30303030u; }
        const uint32_t scw = r.sc[2 * hf + (g >> 1)];
        const float ds = x.d * (float)(int8_t)((scw >> (16 * (g & 1))) & 0xFFu);
        // (d*sc)*(q-32) = ds*q - 32*ds, every term exact in f32
        return frag8(n0 | u0, n1 | u1, ds * Q_ULP, -32.0f * ds);
    }
    template <int G>
    static __device__ __forceinline__ void refill(Raw& r, const uint8_t* row, int nc, int h, int) {
        constexpr int hf = G >> 1;
        const uint8_t* nb = row + (size_t)nc * BLOCK;
        if (G & 1) {   // both nibble planes of this half are spent
            r.ql[hf][0] = ld16(nb + 64 * hf + 16 * h);
            r.ql[hf][1] = ld16(nb + 64 * hf + 32 + 16 * h);
            r.qh[hf] = ld16(nb + 128 + 32 * hf + 16 * h);
        }
        if (G == 1) {
            r.scn = ld16(nb + 192);
            r.dn = *(const uint16_t*)(nb + 208);
        }
    }
};

// LATE: a piece stays as it was loaded until the step that reads it shifts it into place (loads.hpp). Shifted beside its load it is
// waited for right there. In the 128 x 160 tile and the kernel of up to 32 rows a step is too short to hide that behind the other wave of a
// SIMD; at 256 rows it is not, and the registers of the unshifted pieces cost more (Eager). Measured, us, shifted at once -> late: 128 x 160 tiles of
// 5120 x 13824 at 64 / 128 / 256 rows 53.8 / 57.8 / 91.9 -> 47.4 / 50.7 / 80.2, of 4096 x 4096 at 128 29.4 -> 27.7; 256 x 256 at 2048 rows 379 -> 383,
// 256 x 160 on 17408 x 4096 387 -> 393. Q6_K, whose pieces are shifted once for four steps but unpacked by more arithmetic, lost 2 ... 7 % in every
// tile and shifts at once.
template <bool LATE>
struct Q80T {
    using Eager = Q80T<false>;
    static constexpr bool OWN_TURNS = true;
    // A chunk is 8 blocks of 34 bytes; step G covers blocks 2G, 2G+1; slice T is block 2G + (T >> 1),
    // elements 16h + 8(T & 1) + [0, 8). A trailing partial chunk is allowed: blocks past the row's end are
    // read from the last valid block's address and given scale 0 (their activations are staged as 0 too).
    static constexpr int BLOCK = 34;
    static constexpr float UNPACK_US = 5.1f;
    static constexpr float CHUNK_US[NTILES] = {4.66f, 5.96f, 11.44f, 6.65f, 3.15f, 2.23f, 4.62f, 2.91f, 1.98f, 2.76f, 1.22f, 1.76f, 0.93f};
    static constexpr float RUN_CHUNK_US[7] = {9.40f, 9.88f, 11.93f, 6.86f, 7.00f, 6.50f, 5.05f};
    static constexpr bool PARTIAL = true;   // a row may end inside a chunk
    static __host__ __device__ int chunks(int K) { return (K + 255) / 256; }
    struct Raw { fhip::Un16 q[4][2]; uint32_t d[4][2]; };
    struct Ctx { float d[2]; };
    static __device__ __forceinline__ const uint8_t* blk(const uint8_t* row, int c, int i, int nblk) {
        int bi = 8 * c + i;
        bi = bi < nblk ? bi : nblk - 1;
        return row + (size_t)bi * BLOCK;
    }
    static __device__ __forceinline__ void prime(Raw& r, const uint8_t* row, int c, int h, int nblk) {
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint8_t* p = blk(row, c, 2 * g + u, nblk);
                r.d[g][u] = *(const uint16_t*)p;
                r.q[g][u] = fhip::load16_un<LATE>(p + 2 + 16 * h);
            }
    }
    template <int G>
    static __device__ __forceinline__ void begin(Raw& r, const uint8_t* row, int c, int, int nblk, Ctx& x) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = 8 * c + 2 * G + u, bi = i < nblk ? i : nblk - 1;
            // the quants' address modulo 4: blocks are 34 bytes apart, the quants 2 behind the block's start
            if (LATE) fhip::shift_in_place(r.q[G][u], ((uint32_t)(uintptr_t)row + 2u * (uint32_t)(bi & 1) + 2u) & 2u);
            x.d[u] = i < nblk ? f16_bits(r.d[G][u]) : 0.0f;
        }
    }
    template <int G, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        // q = (q ^ 0x80) - 128 with the biased byte unsigned: d*q = d*u - 128*d, every term exact in f32
        const float d = x.d[T >> 1];
        return frag8(r.q[G][T >> 1].w[2 * (T & 1)] ^ 0x80808080u, r.q[G][T >> 1].w[2 * (T & 1) + 1] ^ 0x80808080u, d * Q_ULP, -128.0f * d);
    }
    template <int G>
    static __device__ __forceinline__ void refill(Raw& r, const uint8_t* row, int nc, int h, int nblk) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint8_t* p = blk(row, nc, 2 * G + u, nblk);
            r.d[G][u] = *(const uint16_t*)p;
            r.q[G][u] = fhip::load16_un<LATE>(p + 2 + 16 * h);
        }
    }
};

using Q80 = Q80T<true>;

struct GemmParams {
    const uint8_t* W;
    const uint16_t* X;   // bf16 bits [T, K]
    float* Y;            // [T, N]
    int T, N, K;
    int nblk;            // blocks per weight row
    size_t row_bytes;
    int tiles_n;         // workgroup tiles along N
    int nchunks;         // chunks per weight row
    int whole_rounds;    // rounds of whole tiles every workgroup computes first: tile = round * gridDim.x + blockIdx.x
    long long units;     // the remaining tiles' (tile, chunk) work units, chunk fastest
    int per;             // of those, units per workgroup
    float* ws;           // partial tiles of the left-over tiles that several runs share: [left-over tile][contributor][BM x 256]
    int kmax;            // contributor slots per left-over tile
    uint16_t* H;         // SwiGLU launches: bf16 [T, ff] in place of Y
    int ff;
};

// A SwiGLU launch computes H[t, n] = bf16(silu(gate) * up) with gate row n and up row ff + n of W. Its columns are dealt to the
// matrix instructions so that both meet in one lane: of every 32 columns the first 16 are gate rows, the other 16 the up rows of the
// same outputs (N counts these columns: 2 x ff rounded up to 16). The f32 pair of an output then lies 16 lanes apart, and one
// v_permlane16_swap of two accumulator registers (rows r and r + 1 of the tile) leaves every lane with gate and up of one output.
// Measured: the f32 gate|up matrix of 2048 x 34816 and the kernel that read it back took 100 us behind a 783 us GEMM.
__device__ __forceinline__ int swiglu_row(int v, int ff) {
    const int n = 16 * (v >> 5) + (v & 15);
    return (n < ff ? n : ff - 1) + (v & 16 ? ff : 0);
}
__device__ __forceinline__ float silu_mul(float g, float u) { return (g / (1.0f + expf(-g))) * u; }
// the 32 x 32 accumulator of rows t0 .. and columns v0 ..: outputs 16 * (v0 / 32) + (c & 15)
template <int R0 = 0, int NR = 16>
__device__ __forceinline__ void store_swiglu(const GemmParams& p, const f32x16& acc, int t0, int v0, int h, int c) {
    const int n = 16 * (v0 >> 5) + (c & 15);
#pragma unroll
    for (int r = R0; r < R0 + NR; r += 2) {
        const auto gu = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[r]), __float_as_uint(acc[r + 1]), false, false);
        const int t = t0 + 8 * (r >> 2) + 4 * h + (r & 3) + (c >> 4);
        if (t < p.T && n < p.ff)
            p.H[(size_t)t * p.ff + n] = (uint16_t)(pk_bf16(silu_mul(__uint_as_float(gu[0]), __uint_as_float(gu[1])), 0.f) & 0xFFFFu);
    }
}

template <int I, int N, class Fn>
__device__ __forceinline__ void static_for(Fn&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Workgroup = 8 waves, 2 along T x 4 along N; wave tile = 128 x 64; workgroup tile = 256 x 256.
// Two waves per SIMD: a wave issues one VALU instruction per ~6 cycles and one 16-byte LDS read per ~16, so
// a single wave cannot feed its own MFMAs and unpack at the same time; two can.
// The two waves of a T-pair need the same 64 weight rows. Each unpacks 32 of them (all four slices of a
// step) and publishes the fragments in LDS in MFMA operand order (lane L's 16 bytes at L*16), where both
// read them back: unpack work per MFMA halves, and a wave carries the raw bytes of one row only.
//
// Work distribution. One workgroup per CU. Every workgroup first computes `whole_rounds` whole tiles (tile =
// round * gridDim.x + blockIdx.x, so the workgroups running side by side share activation rows in L2). The
// tiles left over, fewer than one per workgroup, are cut along K: their (tile, chunk) units are dealt out in
// equal contiguous runs of `per`, so every CU does the same amount of MFMA work whatever the tile count (no
// partial last round). A run may start and end inside a tile: a segment that covers its tile's whole K stores
// the tile, any other stores its partial sums into the workspace slot (tile, contributor), contributor = the run's rank among
// the runs that touch the tile, and sum_split_tiles_kernel adds a tile's slots in that order afterwards: the result does not
// depend on which workgroup finishes first (f32 atomics into Y, which this replaced, gave run-to-run differences in the
// last bits wherever a tile had three contributors or more).
template <class F, bool SWIGLU>
__global__ void __launch_bounds__(512) gemm_q_bf16_kernel(GemmParams p) {
    constexpr int MI = 4, NI = 2, BM = 64 * MI, BN = 128 * NI;
    constexpr int FRAG = 512;                                   // bf16 per published fragment (64 lanes x 8)
    __shared__ __attribute__((aligned(16))) uint16_t As[2][BM * LDS_ROW];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][16 * NI * FRAG];   // [n-block 0..4 NI - 1][slice 0..3]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 3, wm = wave >> 2;
    const int h = lane >> 5, c = lane & 31;
    const int nchunks = p.nchunks;
    long long u = (long long)blockIdx.x * p.per;
    const long long u_end = u + p.per < p.units ? u + p.per : p.units;
  for (int round = 0;; round++) {
    int tile, c_begin, c_end;
    if (round < p.whole_rounds) {
        tile = round * gridDim.x + blockIdx.x;
        c_begin = 0;
        c_end = nchunks;
    } else {
        if (u >= u_end) break;
        const int rt = (int)(u / nchunks);
        tile = p.whole_rounds * gridDim.x + rt;
        c_begin = (int)(u - (long long)rt * nchunks);
        c_end = (long long)(nchunks - c_begin) < u_end - u ? nchunks : c_begin + (int)(u_end - u);
        u += c_end - c_begin;
    }
    const bool whole = c_begin == 0 && c_end == nchunks;
    const int tile_y = tile / p.tiles_n, tile_x = tile - tile_y * p.tiles_n;
    const int t0 = tile_y * BM + wm * (32 * MI);
    const int n0 = tile_x * BN + wn * (32 * NI);
    const int c_last = c_end - 1;

    // the weight row this lane unpacks: n-block 2*wn + wm of the workgroup tile; clamped: rows past N are computed but not stored
    const uint8_t* wrow;
    {
        int n = n0 + 32 * wm + c;
        n = n < p.N ? n : p.N - 1;
        wrow = p.W + (size_t)(SWIGLU ? swiglu_row(n, p.ff) : n) * p.row_bytes;
    }
    const int b_wr = ((2 * wn + wm) * 4) * FRAG + lane * 8;                     // + t * FRAG
    const int b_rd = ((NI * wn) * 4) * FRAG + lane * 8;                        // + (4 * j + t) * FRAG

    f32x16 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    // Activation staging: BM rows x 64 bf16 per step; thread `tid` moves the 16-byte piece (tid & 7) of rows
    // (tid >> 3) + 64q, q < MI. Rows past T are read from row T-1 (their outputs are never stored); columns
    // past K (a partial last chunk) are staged as zeros.
    const int a_col = (tid & 7) * 8;
    uint32_t a_src[MI];
#pragma unroll
    for (int q = 0; q < MI; q++) {
        int t = tile_y * BM + (tid >> 3) + 64 * q;
        a_src[q] = x_piece(t, p.T, p.K, a_col);
    }
    const int a_dst = (tid >> 3) * LDS_ROW + a_col;
    u32x4 stage[MI];
    auto load_a = [&](int s) {   // s = absolute step index (64 columns each)
        if constexpr (F::PARTIAL) {
            const bool ok = s * KSTEP + a_col < p.K;
            const int off = x_step(s * KSTEP, a_col, p.K);
            const uint32_t keep = ok ? 0xFFFFFFFFu : 0u;
#pragma unroll
            for (int q = 0; q < MI; q++) {
                u32x4 v = *(const u32x4*)(p.X + (a_src[q] + off));
                stage[q] = (u32x4){v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep};
            }
        } else {
            const int off = s * KSTEP < p.K ? s * KSTEP : 0;   // past the end: any valid address, the tile is never read
#pragma unroll
            for (int q = 0; q < MI; q++) stage[q] = *(const u32x4*)(p.X + (a_src[q] + off));
        }
    };
    auto store_a = [&](int buf) {
#pragma unroll
        for (int q = 0; q < MI; q++) *(u32x4*)(&As[buf][a_dst + 64 * q * LDS_ROW]) = stage[q];
    };
    const int a_rd = (wm * 32 * MI + c) * LDS_ROW + 16 * h;   // + 32*i rows, + kcol(t, 0)
    typename F::Raw raw;
    F::prime(raw, wrow, c_begin, h, p.nblk);
    load_a(4 * c_begin);
    {
        const int nc = c_begin + 1 < c_last ? c_begin + 1 : c_last;
        typename F::Ctx x;
        F::template begin<0>(raw, wrow, c_begin, h, p.nblk, x);
        static_for<0, 4>([&](auto T) {
            *(bf16x8*)(&Bs[0][b_wr + T.value * FRAG]) = F::template frag<0, T.value>(raw, x);
        });
        F::template refill<0>(raw, wrow, nc, h, p.nblk);
    }
    store_a(0);
    __syncthreads();

    // One k-step: the MFMAs of step (chunk ck, G) from LDS buffers G & 1, while this wave's fragments of the
    // following step are unpacked and published into the other B buffer and the following activations
    // travel global -> registers -> LDS. The step is cut into its four slices; each slice first reads the
    // next slice's operands from LDS, then alternates one MFMA with its share of the unpack arithmetic.
    // Nothing moves between slices.
    constexpr int VPM = (26 + MI * NI - 1) / (MI * NI);   // VALU instructions issued behind each MFMA
    auto step = [&](auto Gc, int ck) {
        constexpr int G = decltype(Gc)::value;
        constexpr int GN = (G + 1) & 3;
        constexpr int buf = G & 1;
        // fragments of step G+1 of this chunk, or of step 0 of the next one
        const int pc = G == 3 ? (ck + 1 < c_last ? ck + 1 : c_last) : ck;
        const int nc = pc + 1 < c_last ? pc + 1 : c_last;
        typename F::Ctx ctx;
        bf16x8 a[2][MI], b[2][NI];
        auto read_ops = [&](int t, bf16x8 (&da)[MI], bf16x8 (&db)[NI]) {
#pragma unroll
            for (int i = 0; i < MI; i++) da[i] = *(const bf16x8*)(&As[buf][a_rd + 32 * i * LDS_ROW + kcol(t, 0)]);
#pragma unroll
            for (int j = 0; j < NI; j++) db[j] = *(const bf16x8*)(&Bs[buf][b_rd + (4 * j + t) * FRAG]);
        };
        read_ops(0, a[0], b[0]);
        load_a(4 * ck + G + 1);
        F::template begin<GN>(raw, wrow, pc, h, p.nblk, ctx);
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, 4>([&](auto S) {
            constexpr int t = decltype(S)::value;
            if constexpr (t < 3) read_ops(t + 1, a[(t + 1) & 1], b[(t + 1) & 1]);
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NI; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[t & 1][i], b[t & 1][j], acc[i][j], 0, 0, 0);
            *(bf16x8*)(&Bs[buf ^ 1][b_wr + t * FRAG]) = F::template frag<GN, t>(raw, ctx);
            if constexpr (t < 3) __builtin_amdgcn_sched_group_barrier(0x100, MI + NI, 0);
#pragma unroll
            for (int u = 0; u < MI * NI; u++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
        F::template refill<GN>(raw, wrow, nc, h, p.nblk);
        store_a(buf ^ 1);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    for (int ck = c_begin; ck < c_end; ck++) {
        step(std::integral_constant<int, 0>{}, ck);
        step(std::integral_constant<int, 1>{}, ck);
        step(std::integral_constant<int, 2>{}, ck);
        step(std::integral_constant<int, 3>{}, ck);
    }

    // a partial tile goes to the slot of this run in the tile's contributor list: runs are numbered by blockIdx.x, and the
    // first run that touches left-over tile rt is the one that holds unit rt * nchunks
    float* part = nullptr;
    if (!whole) {
        const int rt = tile - p.whole_rounds * (int)gridDim.x;
        const int k = (int)blockIdx.x - (int)(((long long)rt * nchunks) / p.per);
        part = p.ws + ((size_t)rt * p.kmax + k) * (size_t)(BM * BN);
    }
    // D layout of the 32x32 MFMA: register r of lane (h, c) is row 8*(r/4) + 4*h + (r%4), column c
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++) {
            const int n = n0 + 32 * j + c;
            if (SWIGLU && whole) {
                store_swiglu(p, acc[i][j], t0 + 32 * i, n0 + 32 * j, h, c);
                continue;
            }
            if (n >= p.N) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int t = t0 + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
                if (t < p.T) {
                    if (whole) p.Y[(size_t)t * p.N + n] = acc[i][j][r];
                    else part[(size_t)(t - tile_y * BM) * BN + (n - tile_x * BN)] = acc[i][j][r];
                }
            }
        }
  }
}

// ------------------------------------------------------------------------------------------------
// The same kernel with a 256 x 160 workgroup tile. An output width of 5120 is 20 tiles of 256 columns but 32 of 160, and
// 32 x (T / 256) tile rows deal 2048, 1024 or 512 activation rows to the chip's 256 workgroups exactly: one whole tile
// each, or every tile cut along K in exactly two or four (no run that starts in one tile and ends in the next, so one
// partial tile per workgroup). Wave layout: 8 waves along T, 32 rows each, every wave holding all five 32-column blocks
// (MI = 1, NI = 5: 1.2 LDS operand reads per MFMA instead of 0.75). Waves 0..4 each unpack one 32-row weight block and
// publish its fragments; waves 5..7 only multiply (and, for the formats dear to unpack, move the activations: below). (The fifth block shared by waves
// 4..7, one slice each, so that every SIMD carries the same unpack arithmetic, was slower: 130 -> 141 us at T = 2048 --
// four more waves fetch raw bytes and derive scales every step.) Work distribution and K-split slots are the tall
// kernel's at MI = 4.
// MI = 2 is the tile at 128 rows, for prompts of 96 ... 256 rows, where the 256-row tile multiplies rows that do not exist
// or is cut along K more finely: four waves along T, and the five column blocks dealt to two wave groups, three to waves
// 0..3 and two to waves 4..7 -- wave w and wave w + 4 share a SIMD, so every SIMD still carries five blocks of MFMAs per
// slice. Measured against the best other tile, us: Q4_K 5120 x 5120 at 256 rows 36.1 -> 32.9, 34816 x 5120 at 128 rows
// 75.7 -> 68.9, Q6_K 5120 x 17408 at 128 rows 64.6 -> 59.0, Q8_0 12288 x 4096 at 128 rows 57.8 -> 52.3; at 512 rows of
// 5120 x 5120 (128 tiles cut in two instead of 64 cut in four) it is level, 49.2 against 48.0.
// ------------------------------------------------------------------------------------------------
template <class F, int MI, bool SWIGLU>
__global__ void __launch_bounds__(512) gemm_q_bf16_n160_kernel(GemmParams p) {
    constexpr int NB = 5;
    constexpr int BM = 64 * MI, BN = 32 * NB;
    constexpr int TW = BM / 32, NBW = TW == 8 ? NB : 3;         // waves along T; column blocks a wave holds at most
    constexpr int FRAG = 512;
    __shared__ __attribute__((aligned(16))) uint16_t As[2][BM * LDS_ROW];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][NB * 4 * FRAG];   // [n-block 0..4][slice 0..3]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c = lane & 31;
    const bool unpacker = wave < NB;                            // wave-uniform
    const int tw = TW == 8 ? wave : (wave & 3);                 // the wave's 32 activation rows of the tile
    const int j0 = TW == 8 ? 0 : (wave < 4 ? 0 : 3);            // its first column block ...
    const int nj = TW == 8 ? NB : (wave < 4 ? 3 : 2);           // ... and how many it holds (wave-uniform)
    const int nchunks = p.nchunks;
    long long u = (long long)blockIdx.x * p.per;
    const long long u_end = u + p.per < p.units ? u + p.per : p.units;
  for (int round = 0;; round++) {
    int tile, c_begin, c_end;
    if (round < p.whole_rounds) {
        tile = round * gridDim.x + blockIdx.x;
        c_begin = 0;
        c_end = nchunks;
    } else {
        if (u >= u_end) break;
        const int rt = (int)(u / nchunks);
        tile = p.whole_rounds * gridDim.x + rt;
        c_begin = (int)(u - (long long)rt * nchunks);
        c_end = (long long)(nchunks - c_begin) < u_end - u ? nchunks : c_begin + (int)(u_end - u);
        u += c_end - c_begin;
    }
    const bool whole = c_begin == 0 && c_end == nchunks;
    const int tile_y = tile / p.tiles_n, tile_x = tile - tile_y * p.tiles_n;
    const int t0 = tile_y * BM + 32 * tw;
    const int n0 = tile_x * BN;
    const int c_last = c_end - 1;

    // the weight row an unpacking lane works on: row c of n-block `wave` of the tile (clamped: rows past N are computed but
    // not stored); the other waves point at a valid row and never read it
    const uint8_t* wrow;
    {
        int n = n0 + 32 * (unpacker ? wave : 0) + c;
        n = n < p.N ? n : p.N - 1;
        wrow = p.W + (size_t)(SWIGLU ? swiglu_row(n, p.ff) : n) * p.row_bytes;
    }
    const int b_wr = (wave * 4) * FRAG + lane * 8;              // + t * FRAG (unpackers)
    const int b_rd = (4 * j0) * FRAG + lane * 8;                // + (4 * j + t) * FRAG

    f32x16 acc[NBW];
#pragma unroll
    for (int j = 0; j < NBW; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[j][r] = 0.f;

    // Activation staging, BM rows x 64 bf16 per step, global -> registers one step ahead -> padded LDS. Rows past T are read
    // from row T-1 (their outputs are never stored); columns past K (a partial last chunk) are staged as zeros. Who moves
    // them depends on what a weight costs to unpack. Q4_K: every thread, the 16-byte piece (tid & 7) of rows (tid >> 3) +
    // 64 q, as in the tall kernel. Q6_K and Q8_0: the three waves that unpack nothing -- lane sl of those 192 moves piece
    // (sl & 7) of rows (sl >> 3) + 24 q, q < 11 (the eleventh round holds 16 rows, for the first two of the three waves) --
    // which takes 20 of some 190 instructions a step off the waves that set the pace (Q8_0 5120 x 4096 at T = 2048 150 ->
    // 133 us, Q6_K 5120 x 17408 444 -> 432 us; Q4_K 5120 x 5120 131 -> 135 us, so it keeps the even split).
    // (at 128 rows: six rounds, the sixth holds 8 rows, for the first of the three waves)
    constexpr bool SPLIT = F::UNPACK_US > 2.f;
    constexpr int NQ = SPLIT ? (MI == 4 ? 11 : 6) : MI, RSTEP = SPLIT ? 24 : 64;
    const bool stager = SPLIT ? !unpacker : true;               // wave-uniform
    const bool qlast = SPLIT ? wave < NB + (MI == 4 ? 2 : 1) : true;   // wave-uniform: the wave has a piece in the last round
    const int sl = SPLIT ? (wave - NB) * 64 + lane : tid;
    const int a_col = (sl & 7) * 8;
    uint32_t a_src[NQ];
    u32x4 stage[NQ];
    if (stager) {
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int t = tile_y * BM + (sl >> 3) + RSTEP * q;
            a_src[q] = x_piece(t, p.T, p.K, a_col);
        }
    }
    const int a_dst = (sl >> 3) * LDS_ROW + a_col;              // + RSTEP q LDS_ROW
    auto load_a = [&](int s) {
        if constexpr (F::PARTIAL) {
            const bool ok = s * KSTEP + a_col < p.K;
            const int off = x_step(s * KSTEP, a_col, p.K);
            const uint32_t keep = ok ? 0xFFFFFFFFu : 0u;
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (q < NQ - 1 || qlast) {
                    u32x4 v = *(const u32x4*)(p.X + (a_src[q] + off));
                    stage[q] = (u32x4){v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep};
                }
        } else {
            const int off = s * KSTEP < p.K ? s * KSTEP : 0;   // past the end: any valid address, the tile is never read
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (q < NQ - 1 || qlast) stage[q] = *(const u32x4*)(p.X + (a_src[q] + off));
        }
    };
    auto store_a = [&](int buf) {
#pragma unroll
        for (int q = 0; q < NQ; q++)
            if (q < NQ - 1 || qlast) *(u32x4*)(&As[buf][a_dst + RSTEP * q * LDS_ROW]) = stage[q];
    };
    const int a_rd = (32 * tw + c) * LDS_ROW + 16 * h;          // + kcol(t, 0)
    typename F::Raw raw;
    if (stager) load_a(4 * c_begin);
    if (unpacker) {
        F::prime(raw, wrow, c_begin, h, p.nblk);
        const int nc = c_begin + 1 < c_last ? c_begin + 1 : c_last;
        typename F::Ctx x;
        F::template begin<0>(raw, wrow, c_begin, h, p.nblk, x);
        static_for<0, 4>([&](auto T) {
            *(bf16x8*)(&Bs[0][b_wr + T.value * FRAG]) = F::template frag<0, T.value>(raw, x);
        });
        F::template refill<0>(raw, wrow, nc, h, p.nblk);
    }
    if (stager) store_a(0);
    __syncthreads();

    // one k-step, as in the tall kernel; UNPACK: the wave produces its block's fragments, one behind each slice's MFMAs
    // (NJ: the column blocks the wave holds, a constant of the loop it runs)
    auto step = [&](auto Gc, auto Uc, auto Jc, int ck) {
        constexpr int G = decltype(Gc)::value;
        constexpr bool UNPACK = decltype(Uc)::value;
        constexpr int NJ = decltype(Jc)::value;
        constexpr int GN = (G + 1) & 3;
        constexpr int buf = G & 1;
        constexpr int VPM = (26 + NJ - 1) / NJ;
        const int pc = G == 3 ? (ck + 1 < c_last ? ck + 1 : c_last) : ck;
        const int nc = pc + 1 < c_last ? pc + 1 : c_last;
        typename F::Ctx ctx;
        bf16x8 a[2], b[2][NJ];
        auto read_ops = [&](int t, bf16x8& da, bf16x8 (&db)[NJ]) {
            da = *(const bf16x8*)(&As[buf][a_rd + kcol(t, 0)]);
#pragma unroll
            for (int j = 0; j < NJ; j++) db[j] = *(const bf16x8*)(&Bs[buf][b_rd + (4 * j + t) * FRAG]);
        };
        read_ops(0, a[0], b[0]);
        if constexpr (!(UNPACK && SPLIT)) load_a(4 * ck + G + 1);
        if constexpr (UNPACK) F::template begin<GN>(raw, wrow, pc, h, p.nblk, ctx);
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, 4>([&](auto S) {
            constexpr int t = decltype(S)::value;
            if constexpr (t < 3) read_ops(t + 1, a[(t + 1) & 1], b[(t + 1) & 1]);
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[t & 1], b[t & 1][j], acc[j], 0, 0, 0);
            if constexpr (UNPACK) *(bf16x8*)(&Bs[buf ^ 1][b_wr + t * FRAG]) = F::template frag<GN, t>(raw, ctx);
            if constexpr (t < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1 + NJ, 0);
#pragma unroll
            for (int m = 0; m < NJ; m++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if constexpr (UNPACK) __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
            }
            if constexpr (UNPACK) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (UNPACK) F::template refill<GN>(raw, wrow, nc, h, p.nblk);
        if constexpr (!(UNPACK && SPLIT)) store_a(buf ^ 1);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    auto run = [&](auto Uc, auto Jc) {
        for (int ck = c_begin; ck < c_end; ck++) {
            step(std::integral_constant<int, 0>{}, Uc, Jc, ck);
            step(std::integral_constant<int, 1>{}, Uc, Jc, ck);
            step(std::integral_constant<int, 2>{}, Uc, Jc, ck);
            step(std::integral_constant<int, 3>{}, Uc, Jc, ck);
        }
    };
    if constexpr (TW == 8) {
        if (unpacker) run(std::true_type{}, std::integral_constant<int, NB>{});
        else run(std::false_type{}, std::integral_constant<int, NB>{});
    } else {
        if (wave < 4) run(std::true_type{}, std::integral_constant<int, 3>{});
        else if (unpacker) run(std::true_type{}, std::integral_constant<int, 2>{});
        else run(std::false_type{}, std::integral_constant<int, 2>{});
    }

    float* part = nullptr;
    if (!whole) {
        const int rt = tile - p.whole_rounds * (int)gridDim.x;
        const int k = (int)blockIdx.x - (int)(((long long)rt * nchunks) / p.per);
        part = p.ws + ((size_t)rt * p.kmax + k) * (size_t)(BM * BN);
    }
    // D layout of the 32x32 MFMA: register r of lane (h, c) is row 8*(r/4) + 4*h + (r%4), column c
#pragma unroll
    for (int j = 0; j < NBW; j++) {
        const int n = n0 + 32 * (j0 + j) + c;
        if (j >= nj) continue;
        if (SWIGLU && whole) {
            store_swiglu(p, acc[j], t0, n0 + 32 * (j0 + j), h, c);
            continue;
        }
        if (n >= p.N) continue;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int t = t0 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (t < p.T) {
                if (whole) p.Y[(size_t)t * p.N + n] = acc[j][r];
                else part[(size_t)(t - tile_y * BM) * BN + (n - tile_x * BN)] = acc[j][r];
            }
        }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// The kernel for short prompts and small weights: a wave unpacks its own weights. A low tile of the kind above is bound by what a step
// moves through LDS (operands of both sides written once and read by every wave) and by its barrier every 64 columns: a 128 x 128 x 256
// chunk of Q4_K took 2.84 us there, 1.1 of it matrix instructions at the clock the chip holds. It takes 1.97 here (timing-only variants:
// 1.45 with no loads, 0.6 without the matrix instructions). Here a wave holds BM activation rows x 32 outputs, so a weight is
// unpacked by the one wave that multiplies it, straight into its B operand, and LDS carries the activations alone: a whole chunk of them
// at a time, double buffered, one barrier a chunk. The waves, mostly eight, are NW along N x KW along the chunk's four steps (a wave does
// S = 4 / KW of them), and the KW partial sums of an output meet in LDS when a run ends, added in order of the steps. Work distribution
// and slots of partial tiles are those of the tiled kernel. Measured with the tile the estimate picks, us, the tiled kernel alone before:
// Q4_K 5120 x 5120 at 64 / 128 / 512 rows 17.2 / 20.8 / 43.8 -> 14.3 / 20.4 / 37.6, 6112 x 2816 at 132 39.9 -> 15.9, 10176 x 2560 at 82 23.4 -> 15.2; Q6_K
// 5120 x 17408 at 128 57.0 -> 45.3; Q8_0 12152 x 1536 at 107 24.0 -> 14.9. Loading a chunk's activations and storing them to LDS at its end, where all
// waves wait, cost 2.45 us a chunk: a piece now goes to LDS behind each slice, a chunk after it was asked for.
// Per format: `Raw` holds what a lane half unpacks of S steps of one weight row, as it was loaded (pieces at 2-byte alignment are shifted
// into place by settle(), where they are first read); begin<I>() derives step I's scales, frag<I, T>() the operand of its slice T.
// ------------------------------------------------------------------------------------------------
template <int S>
struct OwnQ4K {
    static constexpr bool TURNS = false;
    static constexpr int SEGS = 2;
    struct Raw { u32x4 hd, q[S]; };
    struct Ctx { float d0, o0, d1, o1; };
    static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int c, int g0, int h, int) {
        const uint8_t* blk = row + (size_t)c * 144;
        r.hd = *(const u32x4*)blk;
#pragma unroll
        for (int i = 0; i < S; i++) r.q[i] = *(const u32x4*)(blk + 16 + 32 * (g0 + i) + 16 * h);
    }
    static __device__ __forceinline__ void settle(Raw&, const uint8_t*, int, int, int) {}
    // the scales (or minima) of sub-blocks 2G and 2G + 1 in the two low bytes, G = g0 + I
    static __device__ __forceinline__ uint32_t pair(uint32_t lo, uint32_t hi, uint32_t top, bool high, int sh) {
        return (high ? hi | ((top >> 2) & 0x30303030u) : lo & 0x3F3F3F3Fu) >> sh;
    }
    template <int I>
    static __device__ __forceinline__ void begin(const Raw& r, const uint8_t*, int, int g0, int, int, Ctx& x) {
        const int G = g0 + I, sh = 16 * (G & 1);
        const uint32_t a = r.hd[1], b = r.hd[2], cc = r.hd[3];
        const uint32_t sc = pair(a, cc & 0x0F0F0F0Fu, a, G >= 2, sh), mn = pair(b, (cc >> 4) & 0x0F0F0F0Fu, b, G >= 2, sh);
        const float d = f16_bits(r.hd[0] & 0xFFFFu) * Q_ULP, dmin = f16_bits(r.hd[0] >> 16);
        x.d0 = d * ub(sc, 0); x.o0 = -(dmin * ub(mn, 0)); x.d1 = (d * ub(sc, 1)) * 0.0625f; x.o1 = -(dmin * ub(mn, 1));
    }
    template <int I, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        return frag8_nibbles(r.q[I][2 * (T & 1)], r.q[I][2 * (T & 1) + 1], T < 2 ? 0x000F000Fu : 0x00F000F0u, T < 2 ? x.d0 : x.d1, T < 2 ? x.o0 : x.o1);
    }
};

template <int S>
struct OwnQ5K {
    static constexpr bool TURNS = false;
    static constexpr int SEGS = 2;
    struct Raw { u32x4 hd, qh, q[S]; };
    using Ctx = typename OwnQ4K<S>::Ctx;
    static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int c, int g0, int h, int) {
        const uint8_t* blk = row + (size_t)c * 176;
        r.hd = *(const u32x4*)blk;
        r.qh = *(const u32x4*)(blk + 16 + 16 * h);
#pragma unroll
        for (int i = 0; i < S; i++) r.q[i] = *(const u32x4*)(blk + 48 + 32 * (g0 + i) + 16 * h);
    }
    // bits 2 g0 ... of every qh byte to the bottom
    static __device__ __forceinline__ void settle(Raw& r, const uint8_t*, int, int g0, int) {
#pragma unroll
        for (int w = 0; w < 4; w++) r.qh[w] >>= 2 * g0;
    }
    template <int I>
    static __device__ __forceinline__ void begin(const Raw& r, const uint8_t*, int, int g0, int, int, Ctx& x) {
        const int G = g0 + I, sh = 16 * (G & 1);
        const uint32_t a = r.hd[1], b = r.hd[2], cc = r.hd[3];
        const uint32_t sc = OwnQ4K<S>::pair(a, cc & 0x0F0F0F0Fu, a, G >= 2, sh), mn = OwnQ4K<S>::pair(b, (cc >> 4) & 0x0F0F0F0Fu, b, G >= 2, sh);
        const float d = f16_bits(r.hd[0] & 0xFFFFu) * Q_ULP, dmin = f16_bits(r.hd[0] >> 16);
        x.d0 = d * ub(sc, 0); x.o0 = -(dmin * ub(mn, 0)); x.d1 = d * ub(sc, 1); x.o1 = -(dmin * ub(mn, 1));
    }
    template <int I, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        constexpr int w = 2 * (T & 1), s = 2 * I + (T >> 1);
        uint32_t v[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t nib = T < 2 ? r.q[I][w + i] & 0x0F0F0F0Fu : (r.q[I][w + i] >> 4) & 0x0F0F0F0Fu;
            const uint32_t bit = (s >= 4 ? r.qh[w + i] >> (s - 4) : r.qh[w + i] << (4 - s)) & 0x10101010u;
            v[i] = nib | bit;
        }
        return frag8(v[0], v[1], T < 2 ? x.d0 : x.d1, T < 2 ? x.o0 : x.o1);
    }
};

// Formats whose blocks are not whole 16-byte pieces (TURNS): their rows come in consecutive pieces and are turned through LDS (fetch, turn in the kernel). A segment is
// five pieces of each of the wave's 32 rows, the first from the dword at or below its first byte; piece_off() says where a piece lies in the row's chunk, take() reads
// segment G's part of a lane's Raw from its row's 80 bytes. 80 bytes apart, sixteen rows' 16-byte reads meet every bank once.
// Why: a load whose lanes each read a row of their own takes the address unit a cycle a lane, 0.2 us for the eight waves of a workgroup, and Q6_K needed 17
// such loads a chunk, Q8_0 24; of these, ten touch some twenty cache lines each. A chunk of 64 x 256 outputs: Q6_K 4.70 -> 4.15 us, Q8_0 6.25 -> 4.66, of 64 x 128 2.21 -> 2.03,
// 3.29 -> 2.23 (what is left over Q4_K's 2.39 and 1.29 is their unpacking, 307 and 294 vector
// instructions a wave for half a chunk of 32 outputs and 128 rows to Q4_K's 219, and the way through LDS, 0.6 and 2.3 cycles of bank conflicts an LDS
// instruction: the scales are read two bytes a lane). With the estimate fitted again, us: Q8_0 3160 x 3328 at 196 rows 26.0 -> 18.5, 2120 x 5632 at 206 28.9 -> 26.7; Q6_K 25736 x 11776 at 44 105 -> 90, 1712 x 13312 at 184 33.7 -> 29.8; FFN blocks of both, 1024 x 7680 at
// 271 53.8 -> 46.5. Q4_K's five loads a chunk turned the same way: 3 - 6 % slower.
constexpr int SEG_ROW = 80, SEG_BYTES = 32 * SEG_ROW;
__device__ __forceinline__ fhip::Un16 un16(const uint8_t* p) { return fhip::Un16{((const fhip::LdU4A4*)p)->v, *(const uint16_t*)(p + 16)}; }

template <int S>
struct OwnQ6K {
    static constexpr bool TURNS = true;
    static constexpr int SEGS = S == 4 ? 4 : 2, CHUNK_BYTES = 210;    // of each half: the nibbles; the bit pairs (three pieces), scales and d (two)
    static __device__ __forceinline__ int piece_off(int seg, int j, int g0) {
        const int hf = (g0 >> 1) + (seg >> 1);
        return (seg & 1) == 0 ? 64 * hf + 16 * j : j < 3 ? 128 + 32 * hf + 16 * j : 192 + 16 * (j - 3);
    }
    static constexpr int NH = S == 4 ? 2 : 1;                   // halves of the super-block the steps lie in
    struct Raw { fhip::Un16 ql[NH][2], qh[NH]; uint32_t sc[NH][3], d; };
    struct Ctx { float d; };
    // m: the block's address modulo 4
    template <int G>
    static __device__ __forceinline__ void take(Raw& r, const uint8_t* row, int g0, int h, uint32_t m) {
        constexpr int i = G >> 1;
        if constexpr ((G & 1) == 0) {
            r.ql[i][0] = un16(row + 16 * h);
            r.ql[i][1] = un16(row + 32 + 16 * h);
        } else {
            r.qh[i] = un16(row + 16 * h);
            const uint8_t* sc = row + 48 + 8 * ((g0 >> 1) + i);
            r.sc[i][0] = *(const uint32_t*)sc;
            r.sc[i][1] = *(const uint32_t*)(sc + 4);
            r.sc[i][2] = *(const uint16_t*)(sc + 8);
            if (G == SEGS - 1) r.d = *(const uint16_t*)(row + 64 + m);   // (the block before has taken its own from there)
        }
    }
    static __device__ __forceinline__ uint32_t parity(const uint8_t* row, int c) { return ((uint32_t)(uintptr_t)row + 2u * (uint32_t)(c & 1)) & 2u; }
    static __device__ __forceinline__ void settle(Raw& r, const uint8_t* row, int c, int g0, int h) {
        const uint32_t m = ((uint32_t)(uintptr_t)row + 2u * (uint32_t)(c & 1)) & 2u;     // every piece starts at a multiple of 4 of its block
#pragma unroll
        for (int i = 0; i < NH; i++) {
            fhip::shift_in_place(r.ql[i][0], m);
            fhip::shift_in_place(r.ql[i][1], m);
            fhip::shift_in_place(r.qh[i], m);
            // byte h of every 16-bit pair is this lane half's scale
            r.sc[i][0] = __builtin_amdgcn_alignbyte(r.sc[i][1], r.sc[i][0], m) >> (8 * h);
            r.sc[i][1] = __builtin_amdgcn_alignbyte(r.sc[i][2], r.sc[i][1], m) >> (8 * h);
        }
        if constexpr (S == 1) {                                 // an odd step's nibbles, bit pairs and scales to an even step's places
            const int sh = 4 * (g0 & 1);
#pragma unroll
            for (int w = 0; w < 4; w++) {
                r.ql[0][0].w[w] >>= sh;
                r.ql[0][1].w[w] >>= sh;
                r.qh[0].w[w] >>= sh;
            }
            r.sc[0][0] = g0 & 1 ? r.sc[0][1] : r.sc[0][0];
        }
    }
    template <int I>
    static __device__ __forceinline__ void begin(const Raw& r, const uint8_t*, int, int, int, int, Ctx& x) { x.d = f16_bits(r.d); }
    template <int I, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        constexpr int hf = I >> 1, odd = I & 1, g = 2 * odd + (T >> 1), par = T >> 1, w = 2 * (T & 1);
        const uint32_t l0 = r.ql[hf][par].w[w], l1 = r.ql[hf][par].w[w + 1];
        const uint32_t h0 = r.qh[hf].w[w], h1 = r.qh[hf].w[w + 1];
        const uint32_t n0 = (odd ? l0 >> 4 : l0) & 0x0F0F0F0Fu, n1 = (odd ? l1 >> 4 : l1) & 0x0F0F0F0Fu;
        const uint32_t u0 = (g < 2 ? h0 << (4 - 2 * (g & 1)) : h0 >> (2 * (g & 1))) & 0x30303030u;
        const uint32_t u1 = (g < 2 ? h1 << (4 - 2 * (g & 1)) : h1 >> (2 * (g & 1))) & 0x30303030u;
        const float ds = x.d * (float)(int8_t)((r.sc[hf][odd] >> (16 * (g & 1))) & 0xFFu);
        return frag8(n0 | u0, n1 | u1, ds * Q_ULP, -32.0f * ds);
    }
};

template <int S>
struct OwnQ80 {
    static constexpr bool TURNS = true;
    static constexpr int SEGS = S, CHUNK_BYTES = 272;                 // a step's two blocks; what lies behind a row's end has the scale 0
    static __device__ __forceinline__ int piece_off(int seg, int j, int g0) { return 68 * (g0 + seg) + 16 * j; }
    struct Raw { fhip::Un16 q[S][2]; uint32_t d[S][2]; };
    struct Ctx { float d[2]; };
    template <int G>
    static __device__ __forceinline__ void take(Raw& r, const uint8_t* row, int, int h, uint32_t m) {
        r.d[G][0] = *(const uint16_t*)(row + m);
        r.d[G][1] = *(const uint16_t*)(row + 34 + m);
        r.q[G][0] = un16(row + 16 * h + 2 * m);
        r.q[G][1] = un16(row + 36 + 16 * h);
    }
    static __device__ __forceinline__ uint32_t parity(const uint8_t* row, int) { return (uint32_t)(uintptr_t)row & 2u; }
    static __device__ __forceinline__ void settle(Raw&, const uint8_t*, int, int, int) {}
    template <int I>
    static __device__ __forceinline__ void begin(Raw& r, const uint8_t* row, int c, int g0, int, int nblk, Ctx& x) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = 8 * c + 2 * (g0 + I) + u, bi = i < nblk ? i : nblk - 1;
            fhip::shift_in_place(r.q[I][u], ((uint32_t)(uintptr_t)row + 2u * (uint32_t)(bi & 1) + 2u) & 2u);
            x.d[u] = i < nblk ? f16_bits(r.d[I][u]) : 0.0f;
        }
    }
    template <int I, int T>
    static __device__ __forceinline__ bf16x8 frag(const Raw& r, const Ctx& x) {
        const float d = x.d[T >> 1];
        return frag8(r.q[I][T >> 1].w[2 * (T & 1)] ^ 0x80808080u, r.q[I][T >> 1].w[2 * (T & 1) + 1] ^ 0x80808080u, d * Q_ULP, -128.0f * d);
    }
};

template <class F, int S> struct Own;
template <int S> struct Own<Q4K, S> { using type = OwnQ4K<S>; };
template <int S> struct Own<Q5K, S> { using type = OwnQ5K<S>; };
template <int S> struct Own<Q6K, S> { using type = OwnQ6K<S>; };
template <int S> struct Own<Q80, S> { using type = OwnQ80<S>; };

constexpr int XROW = CHUNK + 8;      // bf16 per staged activation row of a chunk (+16 B pad: conflict-free 16-byte reads)

template <class FMT, int MI, int NW, int KW, bool SWIGLU>
__global__ void __launch_bounds__(64 * NW * KW) gemm_q_bf16_own_kernel(GemmParams p) {
    constexpr int BM = 32 * MI, BN = 32 * NW, S = 4 / KW;
    constexpr int KEEP = 16 / KW;                               // of a fragment's 16 accumulator registers, those a wave stores in the end
    using F = typename Own<FMT, S>::type;
    __shared__ __attribute__((aligned(16))) uint16_t As[2][BM * XROW];
    __shared__ __attribute__((aligned(16))) uint8_t Seg[F::TURNS ? NW * KW * SEG_BYTES : 16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % NW, kg = wave / NW, g0 = S * kg;
    const int h = lane >> 5, c = lane & 31;
    const int nchunks = p.nchunks;
    long long u = (long long)blockIdx.x * p.per;
    const long long u_end = u + p.per < p.units ? u + p.per : p.units;
  for (int round = 0;; round++) {
    int tile, c_begin, c_end;
    if (round < p.whole_rounds) {
        tile = round * gridDim.x + blockIdx.x;
        c_begin = 0;
        c_end = nchunks;
    } else {
        if (u >= u_end) break;
        const int rt = (int)(u / nchunks);
        tile = p.whole_rounds * gridDim.x + rt;
        c_begin = (int)(u - (long long)rt * nchunks);
        c_end = (long long)(nchunks - c_begin) < u_end - u ? nchunks : c_begin + (int)(u_end - u);
        u += c_end - c_begin;
    }
    const bool whole = c_begin == 0 && c_end == nchunks;
    const int tile_y = tile / p.tiles_n, tile_x = tile - tile_y * p.tiles_n;
    const int t0 = tile_y * BM, n0 = tile_x * BN + 32 * wn;
    const int c_last = c_end - 1;
    const uint8_t* wrow;                                        // rows past N are computed but not stored
    {
        int n = n0 + c;
        n = n < p.N ? n : p.N - 1;
        wrow = p.W + (size_t)(SWIGLU ? swiglu_row(n, p.ff) : n) * p.row_bytes;
    }
    // Weights of a TURNS format. Of every two segments load k of five brings pieces 64 k + lane of their 2 x 160: row (64 k + lane) / 5 of the first, from
    // 160 on of the second.
    constexpr int PAIRS = (F::SEGS + 1) / 2, LOADS_A_PAIR = F::SEGS == 1 ? 3 : 5;
    u32x4 G[F::TURNS ? LOADS_A_PAIR : 1];
    uint32_t g_off[LOADS_A_PAIR];                               // from the wave's first row on (weights of 4 GB and more take other tiles: choose_plan)
    const int rows = SWIGLU ? p.ff : p.N, n_first = SWIGLU ? n0 / 2 : n0, first_row = n_first < rows ? n_first : rows - 1;
    uint8_t* const seg = Seg + (F::TURNS ? wave * SEG_BYTES : 0);
    auto piece = [&](int k) { const int q = 64 * k + lane; return q < 160 ? q : F::SEGS == 1 ? 159 : q - 160; };   // (past an only segment: its last again)
    auto second = [&](int k) { return F::SEGS > 1 && 64 * k + lane >= 160 ? 1 : 0; };
    if constexpr (F::TURNS) {
#pragma unroll
        for (int k = 0; k < LOADS_A_PAIR; k++) {
            const int q = piece(k), v = q / 5, r = SWIGLU ? v & 15 : v;
            g_off[k] = (uint32_t)((first_row + r < rows ? r : rows - 1 - first_row) + (SWIGLU && v > 15 ? p.ff : 0)) * (uint32_t)p.row_bytes + (uint32_t)F::piece_off(second(k), q % 5, g0);
        }
    }
    // the loads of segments 2 g and 2 g + 1 of chunk ck
    auto fetch = [&](auto Gc, u32x4 (&G)[F::TURNS ? LOADS_A_PAIR : 1], int ck) {
      if constexpr (F::TURNS) {
        constexpr int g = decltype(Gc)::value;
        const uint8_t* const from = p.W + ((size_t)first_row * p.row_bytes + (size_t)ck * F::CHUNK_BYTES);
        const uint32_t odd = (uint32_t)(uintptr_t)from & 3u;
#pragma unroll
        for (int k = 0; k < LOADS_A_PAIR; k++) {
            uint32_t off = g_off[k] + odd;
            if (g) off += F::piece_off(2 + second(k), piece(k) % 5, g0) - F::piece_off(second(k), piece(k) % 5, g0);
            G[k] = ((const fhip::LdU4A4*)(from - odd + (off & ~3u)))->v;
        }
      }
    };
    // ... to LDS and back, a row a lane. (One wave's LDS operations keep their order; the fence keeps the compiler's.)
    auto turn = [&](auto Gc, const u32x4 (&G)[F::TURNS ? LOADS_A_PAIR : 1], typename F::Raw& r, int ck) {
      if constexpr (F::TURNS) {
        constexpr int g = decltype(Gc)::value;
        const uint32_t m = F::parity(wrow, ck);
        auto fence = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
        fence();
        *(u32x4*)(seg + 16 * lane) = G[0];
        *(u32x4*)(seg + 1024 + 16 * lane) = G[1];
        if (lane < 32) *(u32x4*)(seg + 2048 + 16 * lane) = G[2];
        fence();
        F::template take<2 * g>(r, seg + c * SEG_ROW, g0, h, m);
        fence();
        if constexpr (F::SEGS > 1) {
            if (lane >= 32) *(u32x4*)(seg + 16 * (lane - 32)) = G[2];
            *(u32x4*)(seg + 512 + 16 * lane) = G[3];
            *(u32x4*)(seg + 1536 + 16 * lane) = G[4];
            fence();
            F::template take<2 * g + 1>(r, seg + c * SEG_ROW, g0, h, m);
            fence();
        }
      }
    };
    f32x16 acc[MI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.f;

    // Activation staging: thread `tid` moves the 16-byte piece (tid & 31) of rows (tid >> 5) + 16 q. Rows past T are read from row T-1,
    // columns past K (a partial last chunk) are staged as zeros.
    constexpr int RQ = 2 * NW * KW, NQ = (BM + RQ - 1) / RQ;    // rows a round of the threads moves, rounds
    const int a_col = (tid & 31) * 8;
    uint32_t a_src[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        int t = (tid >> 5) + RQ * q;
        t = t0 + (t < BM ? t : BM - 1);
        a_src[q] = x_piece(t, p.T, p.K, a_col);
    }
    const int a_dst = (tid >> 5) * XROW + a_col;
    // a last round of fewer rows: the threads past it write the tile's last row again, with what it holds
    const int a_dst_last = ((tid >> 5) + RQ * (NQ - 1) < BM ? (tid >> 5) + RQ * (NQ - 1) : BM - 1) * XROW + a_col;
    u32x4 stage[NQ];
    auto load_a = [&](int ck, int q) {
        const bool ok = !FMT::PARTIAL || ck * CHUNK + a_col < p.K;
        stage[q] = *(const u32x4*)(p.X + (a_src[q] + (FMT::PARTIAL ? x_step(ck * CHUNK, a_col, p.K) : ck * CHUNK)));
        if (FMT::PARTIAL) {
            const uint32_t keep = ok ? 0xFFFFFFFFu : 0u;
            stage[q] = (u32x4){stage[q][0] & keep, stage[q][1] & keep, stage[q][2] & keep, stage[q][3] & keep};
        }
    };
    auto store_a = [&](int buf, int q) { *(u32x4*)(&As[buf][q == NQ - 1 && BM % RQ != 0 ? a_dst_last : a_dst + RQ * q * XROW]) = stage[q]; };
    const int a_rd = c * XROW + 16 * h + KSTEP * g0;            // + 32 i rows, + KSTEP I + kcol(t, 0)

    // Chunk ck from activation buffer P and register set P. Slice by slice: the next slice's activations are read from LDS, then the
    // matrix instructions alternate with the unpacking of the next slice; behind them a piece of chunk ck + 1's activations, requested a
    // chunk ago, goes to the other buffer and its register asks for chunk ck + 2. The barrier stands in front of the last slice, whose
    // matrix instructions cover the first reads and the first unpacking of the next chunk.
    constexpr int NS = 4 * S, QS = (NQ + NS - 3) / (NS - 2);    // slices of a chunk; pieces moved behind each of the first NS - 2
    typename F::Raw raw[F::TURNS ? 1 : 2];                      // (a turned chunk lies in G until its predecessor has been unpacked)
    bf16x8 a[2][MI], b[2];
    typename F::Ctx ctx;
    auto read_a = [&](int buf, int s, bf16x8 (&d)[MI]) {
#pragma unroll
        for (int i = 0; i < MI; i++) d[i] = *(const bf16x8*)(&As[buf][a_rd + 32 * i * XROW + KSTEP * (s >> 2) + kcol(s & 3, 0)]);
    };
    auto chunk = [&](auto Pc, auto Lc, int ck) {
        constexpr int P = decltype(Pc)::value, R = F::TURNS ? 0 : P, RN = F::TURNS ? 0 : P ^ 1;   // Raw of this chunk and of the next
        constexpr bool LOADS = decltype(Lc)::value;
        const int c2 = ck + 2 < c_last ? ck + 2 : c_last;
        static_for<0, NS>([&](auto Sc) {
            constexpr int s = decltype(Sc)::value, n = s + 1;
            if constexpr (n < NS) read_a(P, n, a[n & 1]);
            else read_a(P ^ 1, 0, a[0]);
            if constexpr (n == NS) {
                F::settle(raw[RN], wrow, ck + 1, g0, h);
                F::template begin<0>(raw[RN], wrow, ck + 1, g0, h, p.nblk, ctx);
            } else if constexpr ((n & 3) == 0) F::template begin<(n >> 2)>(raw[R], wrow, ck, g0, h, p.nblk, ctx);
#pragma unroll
            for (int i = 0; i < MI; i++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s & 1][i], b[s & 1], acc[i], 0, 0, 0);
            if constexpr (n == NS) b[0] = F::template frag<0, 0>(raw[RN], ctx);
            else b[n & 1] = F::template frag<(n >> 2), (n & 3)>(raw[R], ctx);
            if constexpr (!F::TURNS) {
                if constexpr (LOADS && s == NS - 2) F::load(raw[R], wrow, c2, g0, h, p.nblk);
            } else if constexpr (s % (NS / PAIRS) == NS / PAIRS - 2) {   // behind the last frag() of a pair's registers: the next chunk's pair, then the loads of the pair behind it
                using std::integral_constant;
                constexpr int g = s / (NS / PAIRS);
                turn(integral_constant<int, g>{}, G, raw[0], ck + 1);
                if constexpr (g + 1 < PAIRS) fetch(integral_constant<int, g + 1>{}, G, ck + 1 < c_last ? ck + 1 : c_last);
                else if (LOADS) fetch(integral_constant<int, 0>{}, G, c2);
            }
#pragma unroll
            for (int q = QS * s; q < QS * (s + 1) && q < NQ; q++) {
                store_a(P ^ 1, q);
                if (LOADS) load_a(c2, q);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, MI, 0);
            constexpr int VPM = (24 + MI - 1) / MI;
#pragma unroll
            for (int m = 0; m < MI; m++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
            }
            if constexpr (s == NS - 2) __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    {
        const int c1 = c_begin < c_last ? c_begin + 1 : c_last;
#pragma unroll
        for (int q = 0; q < NQ; q++) load_a(c_begin, q);
        u32x4 G1[F::TURNS ? LOADS_A_PAIR : 1];                  // the first chunk's second pair
        using std::integral_constant;
        if constexpr (F::TURNS) {
            fetch(integral_constant<int, 0>{}, G, c_begin);
            if constexpr (PAIRS > 1) fetch(integral_constant<int, 1>{}, G1, c_begin);
        } else F::load(raw[0], wrow, c_begin, g0, h, p.nblk);
        if (round > 0) __syncthreads();                         // the last run's sums are read
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            store_a(0, q);
            load_a(c1, q);
        }
        if constexpr (F::TURNS) {
            turn(integral_constant<int, 0>{}, G, raw[0], c_begin);
            fetch(integral_constant<int, 0>{}, G, c1);
            if constexpr (PAIRS > 1) turn(integral_constant<int, 1>{}, G1, raw[0], c_begin);
        } else F::load(raw[1], wrow, c1, g0, h, p.nblk);
        __syncthreads();
        read_a(0, 0, a[0]);
        F::settle(raw[0], wrow, c_begin, g0, h);
        F::template begin<0>(raw[0], wrow, c_begin, g0, h, p.nblk, ctx);
        b[0] = F::template frag<0, 0>(raw[0], ctx);
        __builtin_amdgcn_sched_barrier(0);
    }
    using std::integral_constant;
    int ck = c_begin;
    for (; ck + 2 < c_end; ck += 2) {
        chunk(integral_constant<int, 0>{}, std::true_type{}, ck);
        chunk(integral_constant<int, 1>{}, std::true_type{}, ck + 1);
    }
    chunk(integral_constant<int, 0>{}, std::false_type{}, ck);
    if (ck + 1 < c_end) chunk(integral_constant<int, 1>{}, std::false_type{}, ck + 1);

    // the waves that share outputs meet: wave kg keeps registers [KEEP kg, KEEP kg + KEEP) of every fragment
    if constexpr (KW > 1) {
        float* sums = (float*)&As[0][0];
        // [wave][other steps][MI x KEEP registers][lane]
        auto slot = [&](int k_from, int k_to) { return ((k_from * NW + wn) * (KW - 1) + (k_to < k_from ? k_to : k_to - 1)) * (MI * KEEP * 64) + lane; };
        static_for<0, KW>([&](auto To) {
            constexpr int to = decltype(To)::value;
            if (to != kg) {
                float* q = sums + slot(kg, to);
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int r = 0; r < KEEP; r++) q[(i * KEEP + r) * 64] = acc[i][to * KEEP + r];
            }
        });
        __syncthreads();
        static_for<0, KW>([&](auto Kc) {
            constexpr int k = decltype(Kc)::value;
            if (k == kg) {
#pragma unroll
                for (int from = 0; from < KW; from++)
                    if (from != k) {
                        const float* q = sums + slot(from, k);
#pragma unroll
                        for (int i = 0; i < MI; i++)
#pragma unroll
                            for (int r = 0; r < KEEP; r++) acc[i][k * KEEP + r] += q[(i * KEEP + r) * 64];
                    }
            }
        });
    }
    float* part = nullptr;
    if (!whole) {
        const int rt = tile - p.whole_rounds * (int)gridDim.x;
        const int k = (int)blockIdx.x - (int)(((long long)rt * nchunks) / p.per);
        part = p.ws + ((size_t)rt * p.kmax + k) * (size_t)(BM * BN);
    }
    static_for<0, KW>([&](auto Kc) {
        constexpr int k = decltype(Kc)::value;
        if (k != kg) return;
        const int n = n0 + c;
#pragma unroll
        for (int i = 0; i < MI; i++) {
            if (SWIGLU && whole) {
                store_swiglu<k * KEEP, KEEP>(p, acc[i], t0 + 32 * i, n0, h, c);
                continue;
            }
            if (!whole) {                                       // a slot holds the whole tile, rows past T and columns past N included
#pragma unroll
                for (int r = k * KEEP; r < (k + 1) * KEEP; r++)
                    part[(32 * i + 8 * (r >> 2) + 4 * h + (r & 3)) * BN + 32 * wn + c] = acc[i][r];
                continue;
            }
            if (n >= p.N) continue;
            float* y = p.Y + (size_t)(t0 + 32 * i + 4 * h) * p.N + n;
            const int left = p.T - t0 - 32 * i - 4 * h;
#pragma unroll
            for (int r = k * KEEP; r < (k + 1) * KEEP; r++) {
                const int t = 8 * (r >> 2) + (r & 3);
                if (t < left) y[(size_t)t * p.N] = acc[i][r];
            }
        }
    });
  }
}

// Left-over tile `blockIdx.x` (BM x BN outputs, BN a multiple of 4), if more than one run contributed to it: Y = slot 0 +
// slot 1 + ... in that order. A thread owns four adjacent columns of one row (item blockIdx.y * 256 + threadIdx.x of the
// tile's BM * BN / 4) and asks for up to eight slots at once: the launch is a few dependent trips to memory long, so it
// is cut as finely as that allows (a thread per 16 rows took 7.6 us for the 40 tiles of 5120 x 5120 at T = 128).
__global__ void __launch_bounds__(256) sum_split_tiles_kernel(float* __restrict__ Y, const float* __restrict__ ws, int T, int N, int BM, int BN,
                                                            int tiles_n, int nchunks, int per, int kmax, int first_tile) {
    const int rt = blockIdx.x, tile = first_tile + rt;
    const long long u0 = (long long)rt * nchunks;
    const int nk = (int)((u0 + nchunks - 1) / per) - (int)(u0 / per) + 1;
    if (nk == 1) return;                          // one run covered the whole K of this tile and stored it
    const int tile_y = tile / tiles_n, tile_x = tile - tile_y * tiles_n;
    const int item = blockIdx.y * 256 + threadIdx.x, bn4 = BN >> 2;
    const int lt = item / bn4, c4 = (item - lt * bn4) * 4;
    const int t = tile_y * BM + lt, col = tile_x * BN + c4;
    if (lt >= BM || t >= T || col >= N) return;
    const size_t slot = (size_t)BM * BN;
    const float* q = ws + (size_t)rt * kmax * slot + (size_t)lt * BN + c4;
    float4 a = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < nk; k0 += 8) {
        float4 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = *(const float4*)(q + (size_t)(k0 + j < nk ? k0 + j : 0) * slot);
        if (k0 == 0) a = v[0];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (k0 + j > 0 && k0 + j < nk) { a.x += v[j].x; a.y += v[j].y; a.z += v[j].z; a.w += v[j].w; }
    }
    float* y = Y + (size_t)t * N + col;
    if ((N & 3) == 0) *(float4*)y = a;
    else {
        y[0] = a.x;
        if (col + 1 < N) y[1] = a.y;
        if (col + 2 < N) y[2] = a.z;
        if (col + 3 < N) y[3] = a.w;
    }
}

// The same for a SwiGLU launch: a thread adds the gate columns and the up columns of four adjacent outputs of one row.
__global__ void __launch_bounds__(256) sum_split_swiglu_kernel(uint16_t* __restrict__ H, const float* __restrict__ ws, int T, int ff, int BM, int BN,
                                                             int tiles_n, int nchunks, int per, int kmax, int first_tile) {
    const int rt = blockIdx.x, tile = first_tile + rt;
    const long long u0 = (long long)rt * nchunks;
    const int nk = (int)((u0 + nchunks - 1) / per) - (int)(u0 / per) + 1;
    if (nk == 1) return;
    const int tile_y = tile / tiles_n, tile_x = tile - tile_y * tiles_n;
    const int item = blockIdx.y * 256 + threadIdx.x, bn8 = BN >> 3;
    const int lt = item / bn8, c4 = (item - lt * bn8) * 4;         // output column of the tile
    const int t = tile_y * BM + lt, col = tile_x * (BN >> 1) + c4;
    if (lt >= BM || t >= T || col >= ff) return;
    const size_t slot = (size_t)BM * BN;
    const float* q = ws + (size_t)rt * kmax * slot + (size_t)lt * BN + 32 * (c4 >> 4) + (c4 & 15);
    float4 g = {0.f, 0.f, 0.f, 0.f}, u = g;
    for (int k0 = 0; k0 < nk; k0 += 4) {
        float4 vg[4], vu[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float* s = q + (size_t)(k0 + j < nk ? k0 + j : 0) * slot;
            vg[j] = *(const float4*)s;
            vu[j] = *(const float4*)(s + 16);
        }
        if (k0 == 0) { g = vg[0]; u = vu[0]; }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (k0 + j > 0 && k0 + j < nk) {
                g.x += vg[j].x; g.y += vg[j].y; g.z += vg[j].z; g.w += vg[j].w;
                u.x += vu[j].x; u.y += vu[j].y; u.z += vu[j].z; u.w += vu[j].w;
            }
    }
    const uint32_t lo = pk_bf16(silu_mul(g.x, u.x), silu_mul(g.y, u.y)), hi = pk_bf16(silu_mul(g.z, u.z), silu_mul(g.w, u.w));
    uint16_t* out = H + (size_t)t * ff + col;
    if ((ff & 3) == 0) *(uint2*)out = make_uint2(lo, hi);
    else {
        out[0] = (uint16_t)(lo & 0xFFFFu);
        if (col + 1 < ff) out[1] = (uint16_t)(lo >> 16);
        if (col + 2 < ff) out[2] = (uint16_t)(hi & 0xFFFFu);
        if (col + 3 < ff) out[3] = (uint16_t)(hi >> 16);
    }
}

// ------------------------------------------------------------------------------------------------
// T <= 32 (batched decode, short prompts): one 32-row MFMA slab of activations, so the kernel is bound by
// the weight stream and its unpack arithmetic, not by the matrix pipe. A workgroup is 4 waves on 4 adjacent
// 32-row weight blocks; each wave unpacks its own block straight into its B operand (no LDS for weights)
// with the weight bytes one chunk ahead, the same register image and refill order as the tiled kernel. The
// activations of a chunk (TP rows x 256 columns, TP = 8 or 32) are staged once per workgroup in LDS, double
// buffered, one barrier per chunk. The (128-row group, chunk) units, chunk fastest, are dealt to the
// workgroups in equal contiguous runs, two to four workgroups per CU; a segment that covers its group's whole K
// stores its tile, any other stores partial sums into the workspace slot (group, contributor) and sum_split_groups_kernel
// adds a group's slots in contributor order afterwards, as for the tiled kernel.
// ------------------------------------------------------------------------------------------------
struct SkinnyParams {
    const uint8_t* W;
    const uint16_t* X;
    float* Y;
    int T, N, K;
    int nblk;
    size_t row_bytes;
    int nchunks;
    long long units;   // 128-row groups * nchunks
    int per;           // units per workgroup
    float* ws;         // partial sums of groups that several runs share: [group][contributor][TP x 128]
    int kmax;          // contributor slots per group
};

template <class F, int TP>
__global__ void __launch_bounds__(256, TP == 8 ? 4 : 2) gemm_q_bf16_skinny_kernel(SkinnyParams p) {
    __shared__ __attribute__((aligned(16))) uint16_t Xs[2][TP * XROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c = lane & 31;
    const int nchunks = p.nchunks;
    long long u = (long long)blockIdx.x * p.per;
    const long long u_end = u + p.per < p.units ? u + p.per : p.units;
    // staging: thread `tid` moves the 16-byte piece (tid & 31) of rows (tid >> 5) + 8q, q < TP / 8; rows past T
    // repeat row T-1 (their outputs are never stored)
    constexpr int NQ = TP / 8;
    const int s_col = (tid & 31) * 8;
    uint32_t s_src[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        int t = (tid >> 5) + 8 * q;
        s_src[q] = (uint32_t)(t < p.T ? t : p.T - 1) * (uint32_t)p.K;
    }
    const int s_dst = (tid >> 5) * XROW + s_col;
    const int k_last = p.K - 8;   // a partial last chunk reads earlier columns of the same row (their weights are 0)
    u32x4 stage[NQ];
    auto load_x = [&](int ck) {
        int col = ck * CHUNK + s_col;
        col = col < k_last ? col : k_last;
#pragma unroll
        for (int q = 0; q < NQ; q++) stage[q] = *(const u32x4*)(p.X + (s_src[q] + col));
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int q = 0; q < NQ; q++) *(u32x4*)(&Xs[buf][s_dst + 8 * q * XROW]) = stage[q];
    };
    const int a_rd = (c & (TP - 1)) * XROW + 16 * h;   // + 64 * step + kcol(t, 0)

    for (int seg = 0; u < u_end; seg++) {
        const int grp = (int)(u / nchunks);
        const int c_begin = (int)(u - (long long)grp * nchunks);
        const int c_end = (long long)(nchunks - c_begin) < u_end - u ? nchunks : c_begin + (int)(u_end - u);
        u += c_end - c_begin;
        const bool whole = c_begin == 0 && c_end == nchunks;
        const int n = grp * 128 + wave * 32 + c;
        const uint8_t* wrow = p.W + (size_t)(n < p.N ? n : p.N - 1) * p.row_bytes;

        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.f;
        // Weight bytes: the whole next chunk is requested at the top of a chunk, all its loads back to back, so
        // the two or three cache lines a row's block spans are fetched from L2 once (loads of one block spread
        // over the chunk's steps would find the line evicted from L1 each time and refetch it).
        typename F::Raw raw, nxt;
        bf16x8 a[4], b[4];   // both operands of the step in flight; each slice is replaced as soon as its MFMA has issued
        F::prime(raw, wrow, c_begin, h, p.nblk);
        load_x(c_begin);
        if (seg > 0) __syncthreads();   // the previous segment's last reads of buffer 0 are done
        store_x(0);
        {
            typename F::Ctx x;
            F::template begin<0>(raw, wrow, c_begin, h, p.nblk, x);
            static_for<0, 4>([&](auto T) { b[T.value] = F::template frag<0, T.value>(raw, x); });
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; t++) a[t] = *(const bf16x8*)(&Xs[0][a_rd + kcol(t, 0)]);

        for (int ck = c_begin; ck < c_end; ck++) {
            const int buf = (ck - c_begin) & 1;
            const int cn = ck + 1 < c_end ? ck + 1 : ck;
            F::prime(nxt, wrow, cn, h, p.nblk);
            load_x(cn);
            static_for<0, 4>([&](auto Gc) {
                constexpr int G = decltype(Gc)::value;
                constexpr int GN = (G + 1) & 3;
                typename F::Ctx x;
                if constexpr (G == 3) {
                    F::template begin<0>(nxt, wrow, cn, h, p.nblk, x);
                    static_for<0, 4>([&](auto T) {
                        constexpr int t = decltype(T)::value;
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[t], b[t], acc, 0, 0, 0);
                        b[t] = F::template frag<0, t>(nxt, x);
                    });
                    store_x(buf ^ 1);
                    __syncthreads();
#pragma unroll
                    for (int t = 0; t < 4; t++) a[t] = *(const bf16x8*)(&Xs[buf ^ 1][a_rd + kcol(t, 0)]);
                } else {
                    F::template begin<GN>(raw, wrow, ck, h, p.nblk, x);
                    static_for<0, 4>([&](auto T) {
                        constexpr int t = decltype(T)::value;
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[t], b[t], acc, 0, 0, 0);
                        a[t] = *(const bf16x8*)(&Xs[buf][a_rd + KSTEP * (G + 1) + kcol(t, 0)]);
                        b[t] = F::template frag<GN, t>(raw, x);
                    });
                }
            });
            raw = nxt;
        }
        // runs are numbered by blockIdx.x; the first run that touches group grp is the one that holds unit grp * nchunks
        float* part = whole ? nullptr
                            : p.ws + ((size_t)grp * p.kmax + ((int)blockIdx.x - (int)(((long long)grp * nchunks) / p.per))) * (size_t)(TP * 128) + wave * 32 + c;
        if (n < p.N) {
#pragma unroll
            for (int r = 0; r < (TP == 8 ? 4 : 16); r++) {
                const int t = 8 * (r >> 2) + 4 * h + (r & 3);
                if (t < p.T) {
                    if (whole) p.Y[(size_t)t * p.N + n] = acc[r];
                    else part[t * 128] = acc[r];
                }
            }
        }
    }
}

// Group `blockIdx.x` of 128 outputs, if more than one run contributed to it: Y = slot 0 + slot 1 + ... in that order.
// Thread = output column (threadIdx.x & 127) of row 2 * blockIdx.y + (threadIdx.x >> 7); eight slots are requested at a time.
__global__ void __launch_bounds__(256) sum_split_groups_kernel(float* __restrict__ Y, const float* __restrict__ ws, int T, int N, int TP,
                                                             int nchunks, int per, int kmax) {
    const int grp = blockIdx.x;
    const long long u0 = (long long)grp * nchunks;
    const int nk = (int)((u0 + nchunks - 1) / per) - (int)(u0 / per) + 1;
    if (nk == 1) return;
    const int col = threadIdx.x & 127, n = grp * 128 + col, t = 2 * blockIdx.y + (threadIdx.x >> 7);
    if (n >= N || t >= T) return;
    const size_t slot = (size_t)TP * 128;
    const float* q = ws + (size_t)grp * kmax * slot + t * 128 + col;
    float a = q[0];
    for (int k0 = 1; k0 < nk; k0 += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = q[(size_t)(k0 + j < nk ? k0 + j : 0) * slot];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (k0 + j < nk) a += v[j];
    }
    Y[(size_t)t * N + n] = a;
}

struct SkinnyPlan { long long groups, units, per; unsigned grid; int kmax; int tp; bool split; };

static SkinnyPlan plan_skinny(size_t rows, int nchunks, size_t t, long long cus) {
    SkinnyPlan q;
    q.groups = ((long long)rows + 127) / 128;
    q.units = q.groups * nchunks;
    q.tp = t <= 8 ? 8 : 32;
    // workgroups per CU as the register budget allows: four with 8 activation rows staged, two with 32
    const long long wgs = cus * (t <= 8 ? 4 : 2);
    long long per = (q.units + wgs - 1) / wgs;
    if (per * 4 >= (long long)nchunks * 3 && per < nchunks) per = nchunks;   // nearly whole groups: make them whole
    if (per < 1) per = 1;
    q.per = per;
    q.grid = (unsigned)((q.units + per - 1) / per);
    q.split = per % nchunks != 0;
    // a group's nchunks units lie in at most this many runs of `per`
    q.kmax = q.split ? (int)((nchunks + per - 2) / per) + 1 : 1;
    return q;
}

static size_t skinny_ws_bytes(const SkinnyPlan& q) { return q.split ? (size_t)q.groups * q.kmax * q.tp * 128 * sizeof(float) : 0; }

template <class F>
int launch_skinny(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, float* d_ws, size_t ws_bytes) {
    SkinnyParams p;
    p.W = w->d_raw; p.X = d_x; p.Y = d_y;
    p.T = (int)t; p.N = (int)w->rows; p.K = (int)w->cols; p.row_bytes = w->row_bytes;
    p.nblk = (int)(w->row_bytes / F::BLOCK);
    p.nchunks = F::chunks(p.K);
    const long long cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    const SkinnyPlan q = plan_skinny(w->rows, p.nchunks, t, cus);
    p.units = q.units;
    p.per = (int)q.per;
    p.ws = d_ws; p.kmax = q.kmax;
    if (q.split && (!d_ws || ws_bytes < skinny_ws_bytes(q)))
        return fhip::set_error(FHIP_ERR_ARG, "gemm_q_bf16: the launch cuts row groups along K and needs %zu bytes of workspace", skinny_ws_bytes(q));
    if (t <= 8) hipLaunchKernelGGL((gemm_q_bf16_skinny_kernel<typename F::Eager, 8>), dim3(q.grid), dim3(256), 0, s, p);
    else hipLaunchKernelGGL((gemm_q_bf16_skinny_kernel<F, 32>), dim3(q.grid), dim3(256), 0, s, p);
    if (q.split)
        hipLaunchKernelGGL(sum_split_groups_kernel, dim3((unsigned)q.groups, (unsigned)((t + 1) / 2)), dim3(256), 0, s, d_y, (const float*)d_ws, p.T, p.N, q.tp, p.nchunks,
                           p.per, p.kmax);
    return fhip::check_hip(hipGetLastError(), "gemm_q_bf16 launch");
}

// The tiles: rows x outputs. 2, 3 and 6 share a weight's unpacking among the waves that multiply it, the others leave it to the one wave.
// The two behind the last are 4 and 5 with one wave along K (run sums, below).
constexpr int BM_OF[NTILES + 2] = {64, 128, 256, 256, 128, 64, 128, 128, 64, 64, 64, 128, 64, 128, 64}, BN_OF[NTILES + 2] = {256, 256, 256, 160, 128, 128, 160, 96, 96, 160, 64, 64, 32, 128, 128};

// How a launch is dealt to the chip: `whole_rounds` whole tiles per workgroup, then the left-over tiles cut along K into runs of `per` chunks.
struct TilePlan {
    int tile, bm, bn, nchunks;
    int whole_rounds, per;
    long long left, units, runs;        // left-over tiles, their chunks, the runs they are cut into
    bool split;                         // a run ends inside a tile
    int kmax;                           // most runs that touch one left-over tile
    unsigned grid;
};

static TilePlan plan_tiles(size_t columns, int nchunks, size_t t, int tile, long long cus) {
    TilePlan q;
    q.tile = tile; q.bm = BM_OF[tile]; q.bn = BN_OF[tile]; q.nchunks = nchunks;
    const long long tiles = (long long)((columns + q.bn - 1) / q.bn) * (long long)((t + q.bm - 1) / q.bm);
    q.whole_rounds = (int)(tiles / cus);
    q.left = tiles - q.whole_rounds * cus;
    q.units = q.left * nchunks;
    int per = (int)((q.units + cus - 1) / cus);
    // a run shorter than a tile's K that is close to it is rounded up to whole tiles: no partial tiles, no summing launch
    if (per * 4 >= nchunks * 3) per = nchunks;
    if (per < 1) per = 1;
    q.per = per;
    q.runs = (q.units + per - 1) / per;
    q.grid = q.whole_rounds > 0 ? (unsigned)cus : (unsigned)q.runs;
    q.split = q.left > 0 && per < nchunks;
    q.kmax = 1;
    // tile rt starts at unit rt * nchunks, `start` units into a run: the latest start meets the most runs
    for (long long rt = 0, start = 0; rt < q.left && q.split; rt++) {
        const int k = (int)(start + nchunks - 1) / per + 1;
        if (k > q.kmax) q.kmax = k;
        start = (start + nchunks) % per;
        if (start == 0) break;
    }
    return q;
}

// the partial tiles of a plan that cuts: runs meet one more tile for every tile boundary inside one
static long long plan_segments(const TilePlan& q) { return q.runs + (q.left - 1) - (q.left - 1) / (q.per / std::gcd(q.per, q.nchunks)); }

// Estimated duration of a plan in us: a start per tile or run a workgroup begins, chunks per workgroup x the cost of a chunk of that tile and format
// (F::CHUNK_US), and, where tiles are cut along K, 0.1 a chunk, the summing launch and the partial tiles, 4.2 per 256 of 128 x 128 written and read back.
// A linear model fitted (non-negative least squares on relative errors, 7 % rms) to 3700 launches: 357 weights of the four formats, 1024 ... 34816 rows
// of 1024 ... 17408 columns, 33 ... 2048 activation rows, every tile. On those the tile it picks is 1.4 % slower than the measured best on average
// (worst 25 %); the model it replaced, fitted to ten large weights, and the seven tiles it had were 20 % slower on average and up to 2.7 times
// (6112 x 2816 Q4_K at 132 rows 42.0 -> 16.6 us). Q6_K's and Q8_0's chunks were fitted again when their rows came to be turned, Q8_0's to 136
// launches a tile, Q6_K's to 350: fitted to 136 they priced 128 x 96 too low, and of 350 weights the pick was 3.0 % slower than the best on average and up to 1.30 times
// as slow as the model before (2480 x 9984 at 215 rows 34.8 -> 45.2 us); 1.8 % and 1.11 times now, where Q4_K, Q5_K and Q8_0 have 1.4, 1.8 and 1.3 % and at most 1.08 times. On
// those 1400 launches 64 x 256 is the pick of 3 %, which take 7 % longer without it, 64 x 160 of 4 % and 5 %, 64 x 64 of 22 % and 14 %; 128 x 96 of 3 %, to no gain.
// 64 x 32, four waves, came later and was fitted by itself, to 560 of its launches, the near ones weighted: where 64 x 64 leaves half the chip idle and has to be cut along K, it
// does not, and the summing launch is saved. It is the pick of 5 % of 480 drawn launches, to 0.77 of the time (at most 0.94): us, before -> now, Q4_K 6688 x 1024 at 54 rows 10.1 -> 7.2, Q5_K 7560 x 2560
// at 63 14.3 -> 12.1, Q6_K 2168 x 1024 at 134 11.6 -> 9.2, Q8_0 1856 x 1280 at 146 14.4 -> 10.2.
constexpr float START_US[NTILES] = {3.77f, 3.88f, 4.04f, 4.53f, 3.92f, 3.12f, 4.91f, 3.57f, 2.73f, 4.01f, 2.31f, 3.95f, 4.19f}, FIX_US = 3.29f, SLOT_US = 4.18f, CUT_US = 0.1f;
template <class F>
static float plan_cost_us(const TilePlan& q, long long cus) {
    const float chunks = (float)q.whole_rounds * (float)q.nchunks + (q.left > 0 ? (float)q.per : 0.f);
    const float starts = (float)q.whole_rounds + (q.left > 0 ? 1.f : 0.f);
    float fix = 0.f, again = 0.f;
    if (q.split) {
        const long long segs = plan_segments(q);
        fix = FIX_US + CUT_US * (float)q.per + SLOT_US * (float)(q.bm * q.bn) / 16384.f * (float)segs / (float)cus;
        again = (float)segs / (float)q.runs - 1.f;
    }
    return START_US[q.tile] * (starts + again) + chunks * F::CHUNK_US[q.tile] + fix;
}

static size_t plan_ws_bytes(const TilePlan& q) {
    return q.split ? (size_t)q.left * q.kmax * (size_t)(q.bm * q.bn) * sizeof(float) : 0;
}

// columns of a SwiGLU launch (see swiglu_row)
static size_t swiglu_columns(size_t ff) { return (ff + 15) / 16 * 32; }

static int fill_params(const fhip_weight* w, const uint16_t* d_x, size_t t, void* d_out, bool swiglu, int block, const TilePlan& q, float* d_ws, size_t ws_bytes,
                       GemmParams& p) {
    const size_t columns = swiglu ? swiglu_columns(w->rows / 2) : w->rows;
    p.W = w->d_raw; p.X = d_x; p.Y = swiglu ? nullptr : (float*)d_out; p.H = swiglu ? (uint16_t*)d_out : nullptr; p.ff = (int)(w->rows / 2);
    p.T = (int)t; p.N = (int)columns; p.K = (int)w->cols; p.row_bytes = w->row_bytes;
    p.nblk = (int)(w->row_bytes / block);
    p.nchunks = q.nchunks;
    p.tiles_n = (int)((columns + q.bn - 1) / q.bn);
    // one workgroup per CU (its LDS tiles take most of a CU's 160 KB)
    p.whole_rounds = q.whole_rounds;
    p.units = q.units;
    p.per = q.per;
    p.ws = d_ws; p.kmax = q.kmax;
    if (q.split && (!d_ws || ws_bytes < plan_ws_bytes(q)))
        return fhip::set_error(FHIP_ERR_ARG, "gemm_q_bf16: the launch cuts tiles along K and needs %zu bytes of workspace", plan_ws_bytes(q));
    return FHIP_OK;
}
static int launch_sums(const GemmParams& p, const TilePlan& q, bool swiglu, hipStream_t s) {
    const unsigned per_tile = (unsigned)(q.bm * q.bn / (swiglu ? 8 : 4) + 255) / 256;
    const int first = q.whole_rounds * (int)q.grid;
    if (q.split && swiglu)
        hipLaunchKernelGGL(sum_split_swiglu_kernel, dim3((unsigned)q.left, per_tile), dim3(256), 0, s, p.H, (const float*)p.ws, p.T, p.ff, q.bm, q.bn, p.tiles_n, p.nchunks, p.per,
                           p.kmax, first);
    else if (q.split)
        hipLaunchKernelGGL(sum_split_tiles_kernel, dim3((unsigned)q.left, per_tile), dim3(256), 0, s, p.Y, (const float*)p.ws, p.T, p.N, q.bm, q.bn, p.tiles_n, p.nchunks, p.per, p.kmax,
                           first);
    return fhip::check_hip(hipGetLastError(), "gemm_q_bf16 launch");
}
template <class F, int MI, int BN, bool SWIGLU>
int launch_shared(const fhip_weight* w, const uint16_t* d_x, size_t t, void* d_out, hipStream_t s, const TilePlan& q, float* d_ws, size_t ws_bytes) {
    GemmParams p;
    if (int rc = fill_params(w, d_x, t, d_out, SWIGLU, F::BLOCK, q, d_ws, ws_bytes, p)) return rc;
    using W = std::conditional_t<MI == 4, typename F::Eager, F>;
    if constexpr (BN == 256) hipLaunchKernelGGL((gemm_q_bf16_kernel<W, SWIGLU>), dim3(q.grid), dim3(512), 0, s, p);
    else hipLaunchKernelGGL((gemm_q_bf16_n160_kernel<W, MI, SWIGLU>), dim3(q.grid), dim3(512), 0, s, p);
    return launch_sums(p, q, SWIGLU, s);
}
template <class F, int MI, int NW, int KW, bool SWIGLU>
int launch_own(const fhip_weight* w, const uint16_t* d_x, size_t t, void* d_out, hipStream_t s, const TilePlan& q, float* d_ws, size_t ws_bytes) {
    GemmParams p;
    if (int rc = fill_params(w, d_x, t, d_out, SWIGLU, F::BLOCK, q, d_ws, ws_bytes, p)) return rc;
    hipLaunchKernelGGL((gemm_q_bf16_own_kernel<F, MI, NW, KW, SWIGLU>), dim3(q.grid), dim3(64 * NW * KW), 0, s, p);
    return launch_sums(p, q, SWIGLU, s);
}


// A launch of run sums: one wave adds all products of a run for an output, and the runs are those of seven tiles and this estimate, which
// therefore stand as they are. For rows whose every last bit is stored further on, as the codes of a block-quantized cache: in four layers of a
// prompt block on one, sums in another order make 38 % of the codes others (none is nearer f64), and a cache that was stored before would not
// be met again. The tiles of short prompts run on the kernel whose waves unpack for themselves, one along K, which adds in the same order.
// The figures below are no times of today's kernels, four of the seven tiles' kernels are gone: they say where runs end, on a chip of as many CUs, and are kept for that.
constexpr int RUN_TILE_OF[7] = {0, 1, 2, 3, NTILES, NTILES + 1, 6};
constexpr float RUN_FIXUP_US[7] = {0.9f, -2.3f, -13.2f, -5.2f, -1.0f, 1.5f, 0.4f};
template <class F>
static float run_sums_cost_us(const TilePlan& q, int i, long long cus) {
    const float chunks = (float)q.whole_rounds * (float)q.nchunks + (q.left > 0 ? (float)q.per : 0.f);
    const float starts = (float)q.whole_rounds + (q.left > 0 ? 1.f : 0.f);
    float fix = 0.f, extra_starts = 0.f;
    if (q.split) {
        const long long segs = plan_segments(q);
        fix = RUN_FIXUP_US[i] + 7.77f * (float)(q.bm / 64) * ((float)q.bn / 256.f) * (float)segs / (float)cus;
        fix = fix > 0.f ? fix : 0.f;
        extra_starts = (float)segs / (float)q.runs - 1.f;
    }
    return 4.29f + 1.5f * starts + 3.96f * extra_starts + chunks * F::RUN_CHUNK_US[i] + fix;
}

// the tile the estimate picks for this launch
template <class F>
static void choose_plan(const fhip_weight* w, size_t columns, size_t t, bool run_sums, TilePlan& out) {
    const long long cus = fhip::device_cus() > 0 ? fhip::device_cus() : 256;
    const int nchunks = F::chunks((int)w->cols);
    float best_cost = 0.f;
    if (run_sums) {
        for (int i = 0; i < 7; i++) {
            const TilePlan q = plan_tiles(columns, nchunks, t, RUN_TILE_OF[i], cus);
            const float c = run_sums_cost_us<F>(q, i, cus);
            if (best_cost == 0.f || c < 0.98f * best_cost) { best_cost = c; out = q; }
        }
        return;
    }
    for (int i = 0; i < NTILES; i++) {
        if (fhip::g_gemm_tile >= 0 && fhip::g_gemm_tile < NTILES && i != fhip::g_gemm_tile) continue;
        if (F::OWN_TURNS && i != 2 && i != 3 && i != 6 && w->nbytes > 0xFFF00000u) continue;   // offsets of 32 bits within the weight
        const TilePlan q = plan_tiles(columns, nchunks, t, i, cus);
        const float c = plan_cost_us<F>(q, cus);
        if (best_cost == 0.f || c < best_cost) { best_cost = c; out = q; }
    }
    if (best_cost == 0.f) out = plan_tiles(columns, nchunks, t, 3, cus);     // (a pinned tile that the weight is too large for)
}

template <class F>
static size_t ws_bytes_fmt(const fhip_weight* w, size_t columns, size_t t, bool run_sums) {
    if (t <= 32) return skinny_ws_bytes(plan_skinny(w->rows, F::chunks((int)w->cols), t, fhip::device_cus() > 0 ? fhip::device_cus() : 256));
    TilePlan q;
    choose_plan<F>(w, columns, t, run_sums, q);
    return plan_ws_bytes(q);
}

template <class F, bool SWIGLU>
int launch_tiled(const fhip_weight* w, const uint16_t* d_x, size_t t, void* d_y, hipStream_t s, float* d_ws, size_t ws_bytes, bool run_sums = false) {
    TilePlan q;
    choose_plan<F>(w, SWIGLU ? swiglu_columns(w->rows / 2) : w->rows, t, run_sums, q);
    switch (q.tile) {
        case 0: return launch_own<F, 2, 8, 1, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 1: return launch_own<F, 4, 8, 1, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 2: return launch_shared<F, 4, 256, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 3: return launch_shared<F, 4, 160, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 4: return launch_own<F, 4, 4, 2, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 5: return launch_own<F, 2, 4, 2, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 6: return launch_shared<F, 2, 160, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 7: return launch_own<F, 4, 3, 2, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 8: return launch_own<F, 2, 3, 2, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 9: return launch_own<F, 2, 5, 2, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 10: return launch_own<F, 2, 2, 4, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 11: return launch_own<F, 4, 2, 4, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        case 12: return launch_own<F, 2, 1, 4, SWIGLU>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
    }
    if constexpr (!SWIGLU) {
        if (q.tile == NTILES) return launch_own<F, 4, 4, 1, false>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
        if (q.tile == NTILES + 1) return launch_own<F, 2, 4, 1, false>(w, d_x, t, d_y, s, q, d_ws, ws_bytes);
    }
    return fhip::set_error(FHIP_ERR_ARG, "gemm_q_bf16: no tile %d", q.tile);
}

template <class F>
int launch_fmt(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, float* d_ws, size_t ws_bytes, bool run_sums) {
    if (t <= 32) return launch_skinny<F>(w, d_x, t, d_y, s, d_ws, ws_bytes);
    return launch_tiled<F, false>(w, d_x, t, d_y, s, d_ws, ws_bytes, run_sums);
}

}  // namespace

namespace fhip {
size_t FHIP_GEMM_NAME(_ws_bytes)(const fhip_weight* w, size_t columns, size_t t, bool run_sums) { return ws_bytes_fmt<FHIP_GEMM_FORMAT>(w, columns, t, run_sums); }
int FHIP_GEMM_NAME(_launch)(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, float* d_ws, size_t ws_bytes, bool run_sums) {
    return launch_fmt<FHIP_GEMM_FORMAT>(w, d_x, t, d_y, s, d_ws, ws_bytes, run_sums);
}
int FHIP_GEMM_NAME(_launch_swiglu)(const fhip_weight* w, const uint16_t* d_x, size_t t, uint16_t* d_h, hipStream_t s, float* d_ws, size_t ws_bytes) {
    return launch_tiled<FHIP_GEMM_FORMAT, true>(w, d_x, t, d_h, s, d_ws, ws_bytes);
}
}  // namespace fhip

#ifdef FHIP_GEMM_ENTRY
namespace {

// f32 -> bf16 (round to nearest even), 8 values per thread, the tail one by one
__global__ void __launch_bounds__(256) cvt_f32_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ out, size_t n) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= n) return;
    if (i + 8 <= n) {
        const float4 a = *(const float4*)(x + i), b = *(const float4*)(x + i + 4);
        u32x4 r = {pk_bf16(a.x, a.y), pk_bf16(a.z, a.w), pk_bf16(b.x, b.y), pk_bf16(b.z, b.w)};
        *(u32x4*)(out + i) = r;
    } else {
        for (size_t k = i; k < n; k++) out[k] = (uint16_t)(pk_bf16(x[k], 0.f) & 0xFFFFu);
    }
}

// SwiGLU of a [t, 2d] = [gate | up] f32 matrix, written as bf16 [t, d] for the down projection's A operand.
// Same arithmetic as the un-fused f32 op (crates/ferric-tensor/src/lib.rs:2603-2618), then one RNE rounding.
__global__ void __launch_bounds__(256) swiglu_bf16_kernel(const float* __restrict__ gu, size_t n, size_t d, uint16_t* __restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t row = i / d, col = i % d;
    const float g = gu[row * 2 * d + col], u = gu[row * 2 * d + d + col];
    out[i] = (uint16_t)(pk_bf16(silu_mul(g, u), 0.f) & 0xFFFFu);
}

}  // namespace

namespace fhip {

int launch_swiglu_bf16(const float* d_gu, size_t t, size_t d, uint16_t* d_out, hipStream_t s) {
    const size_t n = t * d;
    if (n == 0) return FHIP_OK;
    hipLaunchKernelGGL(swiglu_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d_gu, n, d, d_out);
    return check_hip(hipGetLastError(), "swiglu_bf16 launch");
}

int launch_cvt_bf16(const float* d_x, size_t n, uint16_t* d_out, hipStream_t s) {
    if (n == 0) return FHIP_OK;
    if ((((uintptr_t)d_x | (uintptr_t)d_out) & 15) != 0) return set_error(FHIP_ERR_ARG, "cvt_f32_bf16: pointers must be 16-byte aligned");
    hipLaunchKernelGGL(cvt_f32_bf16_kernel, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, s, d_x, d_out, n);
    return check_hip(hipGetLastError(), "cvt_f32_bf16 launch");
}

int g_gemm_tile = -1;
int gemm_bf16_force_tile(int tile) {
    const int before = g_gemm_tile;
    g_gemm_tile = tile;
    return before;
}

size_t gemm_bf16_ws_bytes(const fhip_weight* w, size_t t, bool run_sums) {
    if (!w || t == 0 || w->rows == 0) return 0;
    switch (w->type) {
        case FHIP_Q4_K: return gemm_Q4K_ws_bytes(w, w->rows, t, run_sums);
        case FHIP_Q6_K: return gemm_Q6K_ws_bytes(w, w->rows, t, run_sums);
        case FHIP_Q8_0: return gemm_Q80_ws_bytes(w, w->rows, t, run_sums);
        case FHIP_Q5_K: return gemm_Q5K_ws_bytes(w, w->rows, t, run_sums);
        default: return 0;
    }
}

int launch_gemm_bf16(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, float* d_ws, size_t ws_bytes, bool run_sums) {
    if (t == 0 || w->rows == 0) return FHIP_OK;
    if (((uintptr_t)d_x & 15) != 0) return set_error(FHIP_ERR_ARG, "gemm_q_bf16: x must be 16-byte aligned");
    if ((unsigned long long)t * w->cols >= (1ull << 31))
        return set_error(FHIP_ERR_SHAPE, "gemm_q_bf16: t * cols must be below 2^31 (got %zu x %zu)", t, w->cols);
    switch (w->type) {
        case FHIP_Q4_K: return gemm_Q4K_launch(w, d_x, t, d_y, s, d_ws, ws_bytes, run_sums);
        case FHIP_Q6_K: return gemm_Q6K_launch(w, d_x, t, d_y, s, d_ws, ws_bytes, run_sums);
        case FHIP_Q8_0: return gemm_Q80_launch(w, d_x, t, d_y, s, d_ws, ws_bytes, run_sums);
        case FHIP_Q5_K: return gemm_Q5K_launch(w, d_x, t, d_y, s, d_ws, ws_bytes, run_sums);
        default: return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "QMatrix: no native matmul for ggml type %u", w->type);
    }
}

size_t gemm_bf16_ws_bytes(const fhip_weight* w, size_t t) { return gemm_bf16_ws_bytes(w, t, false); }
int launch_gemm_bf16(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, float* d_ws, size_t ws_bytes) {
    return launch_gemm_bf16(w, d_x, t, d_y, s, d_ws, ws_bytes, false);
}

// H [t, rows / 2] = bf16(silu(gate) * up) of the stacked [gate | up] weight, for more than 32 rows (fewer: launch_gemm_bf16 and
// launch_swiglu_bf16)
size_t gemm_bf16_swiglu_ws_bytes(const fhip_weight* w, size_t t) {
    if (!w || t <= 32 || w->rows == 0 || w->rows % 2 != 0) return 0;
    const size_t columns = swiglu_columns(w->rows / 2);
    switch (w->type) {
        case FHIP_Q4_K: return gemm_Q4K_ws_bytes(w, columns, t, false);
        case FHIP_Q6_K: return gemm_Q6K_ws_bytes(w, columns, t, false);
        case FHIP_Q8_0: return gemm_Q80_ws_bytes(w, columns, t, false);
        case FHIP_Q5_K: return gemm_Q5K_ws_bytes(w, columns, t, false);
        default: return 0;
    }
}

int launch_gemm_bf16_swiglu(const fhip_weight* w, const uint16_t* d_x, size_t t, uint16_t* d_h, hipStream_t s, float* d_ws, size_t ws_bytes) {
    if (((uintptr_t)d_x & 15) != 0) return set_error(FHIP_ERR_ARG, "gemm_q_bf16: x must be 16-byte aligned");
    if ((unsigned long long)t * w->cols >= (1ull << 31))
        return set_error(FHIP_ERR_SHAPE, "gemm_q_bf16: t * cols must be below 2^31 (got %zu x %zu)", t, w->cols);
    switch (w->type) {
        case FHIP_Q4_K: return gemm_Q4K_launch_swiglu(w, d_x, t, d_h, s, d_ws, ws_bytes);
        case FHIP_Q6_K: return gemm_Q6K_launch_swiglu(w, d_x, t, d_h, s, d_ws, ws_bytes);
        case FHIP_Q8_0: return gemm_Q80_launch_swiglu(w, d_x, t, d_h, s, d_ws, ws_bytes);
        case FHIP_Q5_K: return gemm_Q5K_launch_swiglu(w, d_x, t, d_h, s, d_ws, ws_bytes);
        default: return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "QMatrix: no native matmul for ggml type %u", w->type);
    }
}

}  // namespace fhip
#endif
