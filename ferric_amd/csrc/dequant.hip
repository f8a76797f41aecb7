// Bit-exact block unpackers for Q8_0 / Q4_K / Q6_K (and Q4_0 / Q4_1 / Q5_0 / Q5_1 / Q5_K) on gfx950.
//
// The reference CPU dequantizers round every f32 operation separately (Rust never fuses a*b+c):
//   Q8_0  y = f32(q) * d                       crates/ferric-gguf/src/lib.rs:608-615
//   Q4_K  y = (d*sc)*q - (dmin*m)              crates/ferric-gguf/src/lib.rs:793-825
//   Q6_K  y = (d*sc)*q                         crates/ferric-gguf/src/lib.rs:721-746
// so this file is compiled with -ffp-contract=off AND spells every operation with the
// round-to-nearest intrinsics, which the compiler never contracts.
//
// These kernels are write-bound (4 B out per 0.53-1.06 B in): one lane produces 4 consecutive
// outputs and stores them as one 16-byte vector, so a wave writes 1 KiB contiguous per store.
#include "hostmem.hpp"
#include "through.hpp"

#include <hip/hip_fp16.h>

namespace {

using fhip::store_through;
using fhip::u32x4;

__device__ __forceinline__ float f16_bits(uint32_t b) {
    // v_cvt_f32_f16: exact for every finite / subnormal / infinite pattern.
    return __half2float(__ushort_as_half((unsigned short)b));
}

// 4 bytes from a 2-byte-aligned address (Q8_0 and Q6_K blocks are only 2-byte aligned).
__device__ __forceinline__ uint32_t ld4_a2(const uint8_t* p) {
    const uint16_t* h = (const uint16_t*)p;
    return (uint32_t)h[0] | ((uint32_t)h[1] << 16);
}

__global__ void f16_to_f32_kernel(const uint16_t* __restrict__ in, size_t n, float* __restrict__ out) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f16_bits(in[i]);
}

// crates/ferric-gguf/src/lib.rs:501: a bf16 pattern is the top half of the f32 pattern
__global__ void bf16_to_f32_kernel(const uint16_t* __restrict__ in, size_t n, float* __restrict__ out) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = __uint_as_float((uint32_t)in[i] << 16);
}

// ---- Q8_0: 34 B = [f16 d][i8 q[32]] ------------------------------------------------------------
__device__ __forceinline__ float4 deq_q8_0(const uint8_t* b, int j) {
    float d = f16_bits(*(const uint16_t*)b);
    uint32_t q = ld4_a2(b + 2 + j);
    float4 o;
    o.x = __fmul_rn((float)(int8_t)(q & 0xFF), d);
    o.y = __fmul_rn((float)(int8_t)((q >> 8) & 0xFF), d);
    o.z = __fmul_rn((float)(int8_t)((q >> 16) & 0xFF), d);
    o.w = __fmul_rn((float)(int8_t)(q >> 24), d);
    return o;
}

// ---- Q4_K: 144 B = [f16 d][f16 dmin][u8 s[12]][u8 qs[128]] --------------------------------------
// 6-bit (scale, min) of sub-block j -- get_sc_min, crates/ferric-gguf/src/lib.rs:795-804.
__device__ __forceinline__ void q4k_sc_min(const uint8_t* s, int j, uint32_t& sc, uint32_t& m) {
    if (j < 4) {
        sc = s[j] & 63u;
        m = s[j + 4] & 63u;
    } else {
        sc = (s[j + 4] & 0x0Fu) | ((uint32_t)(s[j - 4] >> 6) << 4);
        m = (uint32_t)(s[j + 4] >> 4) | ((uint32_t)(s[j] >> 6) << 4);
    }
}

__device__ __forceinline__ float4 deq_q4_k(const uint8_t* b, int v) {   // b 16-byte aligned
    int sb = v >> 5, l = v & 31;
    uint32_t hd = *(const uint32_t*)b;
    float d = f16_bits(hd & 0xFFFFu), dmin = f16_bits(hd >> 16);
    uint32_t sc, m;
    q4k_sc_min(b + 4, sb, sc, m);
    uint32_t q = *(const uint32_t*)(b + 16 + 32 * (sb >> 1) + l);
    if (sb & 1) q >>= 4;
    q &= 0x0F0F0F0Fu;
    float d1 = __fmul_rn(d, (float)sc), mm = __fmul_rn(dmin, (float)m);
    float4 o;
    o.x = __fsub_rn(__fmul_rn(d1, (float)(q & 0xFF)), mm);
    o.y = __fsub_rn(__fmul_rn(d1, (float)((q >> 8) & 0xFF)), mm);
    o.z = __fsub_rn(__fmul_rn(d1, (float)((q >> 16) & 0xFF)), mm);
    o.w = __fsub_rn(__fmul_rn(d1, (float)(q >> 24)), mm);
    return o;
}

// ---- Q6_K: 210 B = [u8 ql[128]][u8 qh[64]][i8 sc[16]][f16 d] ------------------------------------
__device__ __forceinline__ float4 deq_q6_k(const uint8_t* b, int v) {   // b 2-byte aligned
    int hf = v >> 7, w = v & 127, g = w >> 5, l = w & 31, is = l >> 4;
    float d = f16_bits(*(const uint16_t*)(b + 208));
    float sc = (float)(int8_t)b[192 + 8 * hf + is + 2 * g];
    uint32_t ql = ld4_a2(b + 64 * hf + 32 * (g & 1) + l);
    uint32_t qh = ld4_a2(b + 128 + 32 * hf + l);
    uint32_t nib = (g >= 2 ? (ql >> 4) : ql) & 0x0F0F0F0Fu;
    uint32_t q = nib | (((qh >> (2 * g)) & 0x03030303u) << 4);
    float ds = __fmul_rn(d, sc);
    float4 o;
    o.x = __fmul_rn(ds, (float)((int)(q & 0xFF) - 32));
    o.y = __fmul_rn(ds, (float)((int)((q >> 8) & 0xFF) - 32));
    o.z = __fmul_rn(ds, (float)((int)((q >> 16) & 0xFF) - 32));
    o.w = __fmul_rn(ds, (float)((int)(q >> 24) - 32));
    return o;
}

// ---- the 32-value formats: [f16 d][f16 m]?[u32 qh]?[u8 qs[16]], blocks 2-byte aligned ----------------------
// value i < 16 is the low nibble of qs[i], value 16 + i the high one; the fifth bit of value v is bit v of qh.
//   Q4_0 y = f32(n - 8) * d            lib.rs:618-629      Q4_1 y = f32(n) * d + m            lib.rs:633-645
//   Q5_0 y = f32((n | b<<4) - 16) * d  lib.rs:650-665      Q5_1 y = f32(n | b<<4) * d + m     lib.rs:669-684
template <bool HAS_M, bool HAS_QH, int OFF>
__device__ __forceinline__ float4 deq_legacy(const uint8_t* b, int v) {
    constexpr int QH = HAS_M ? 4 : 2, QS = QH + (HAS_QH ? 4 : 0);
    float d = f16_bits(*(const uint16_t*)b);
    float m = HAS_M ? f16_bits(*(const uint16_t*)(b + 2)) : 0.f;
    uint32_t q = ld4_a2(b + QS + (v & 15));
    if (v >= 16) q >>= 4;
    q &= 0x0F0F0F0Fu;
    if (HAS_QH) {
        uint32_t hb = (ld4_a2(b + QH) >> v) & 0xFu;
        q |= ((hb * 0x00204081u) & 0x01010101u) << 4;   // bit j of hb -> bit 4 of byte j
    }
    float o[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        float f = (float)((int)((q >> (8 * k)) & 0xFF) - OFF);
        o[k] = HAS_M ? __fadd_rn(__fmul_rn(f, d), m) : __fmul_rn(f, d);
    }
    return make_float4(o[0], o[1], o[2], o[3]);
}

// ---- Q5_K: 176 B = [f16 d][f16 dmin][u8 s[12]][u8 qh[32]][u8 qs[128]]; y = (d*sc)*(n + 16*bit) - dmin*m, lib.rs:692-716
__device__ __forceinline__ float4 deq_q5_k(const uint8_t* b, int v) {   // b 16-byte aligned
    int sb = v >> 5, l = v & 31;
    uint32_t hd = *(const uint32_t*)b;
    float d = f16_bits(hd & 0xFFFFu), dmin = f16_bits(hd >> 16);
    uint32_t sc, m;
    q4k_sc_min(b + 4, sb, sc, m);
    uint32_t q = *(const uint32_t*)(b + 48 + 32 * (sb >> 1) + l);
    if (sb & 1) q >>= 4;
    q &= 0x0F0F0F0Fu;
    q |= ((*(const uint32_t*)(b + 16 + l) >> sb) & 0x01010101u) << 4;   // bit sb of qh[l + k]
    float d1 = __fmul_rn(d, (float)sc), mm = __fmul_rn(dmin, (float)m);
    float4 o;
    o.x = __fsub_rn(__fmul_rn(d1, (float)(q & 0xFF)), mm);
    o.y = __fsub_rn(__fmul_rn(d1, (float)((q >> 8) & 0xFF)), mm);
    o.z = __fsub_rn(__fmul_rn(d1, (float)((q >> 16) & 0xFF)), mm);
    o.w = __fsub_rn(__fmul_rn(d1, (float)(q >> 24)), mm);
    return o;
}

// ---- IQ4_NL / IQ4_XS: 4-bit indices into a 16-level non-linear codebook (lib.rs:751), value = scale * level.
//   IQ4_NL 18 B = [f16 d][qs[16]]                                  y = d * kv[idx]                  lib.rs:755-767
//   IQ4_XS 136 B = [f16 d][u16 scales_h][scales_l[4]][qs[128]]     y = (d * (ls - 32)) * kv[idx]    lib.rs:772-791
// element j of a 32-value (sub-)block is the low nibble of its qs[j], element 16 + j the high nibble. Every product is exact
// in f32 (11-bit d x 6-bit ls x 7-bit level), so the order of the two multiplies cannot change a bit.
__device__ const float KV_IQ4NL[16] = {-127.f, -104.f, -83.f, -65.f, -49.f, -35.f, -22.f, -10.f, 1.f, 13.f, 25.f, 38.f, 53.f, 69.f, 89.f, 113.f};

template <bool XS>
__device__ __forceinline__ float4 deq_iq4(const uint8_t* b, int v) {
    uint32_t q;
    float dl;
    bool high;
    if (XS) {
        int ib = v >> 5, l = v & 31;             // b 8-byte aligned
        uint32_t hd = *(const uint32_t*)b, sl = *(const uint32_t*)(b + 4);
        int ls = (int)(((sl >> (4 * ib)) & 0xFu) | ((((hd >> 16) >> (2 * ib)) & 3u) << 4));
        dl = __fmul_rn(f16_bits(hd & 0xFFFFu), (float)(ls - 32));
        q = *(const uint32_t*)(b + 8 + 16 * ib + (l & 15));
        high = l >= 16;
    } else {
        dl = f16_bits(*(const uint16_t*)b);
        q = ld4_a2(b + 2 + (v & 15));
        high = v >= 16;
    }
    if (high) q >>= 4;
    float o[4];
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = __fmul_rn(dl, KV_IQ4NL[(q >> (8 * k)) & 0xFu]);
    return make_float4(o[0], o[1], o[2], o[3]);
}

// ---- MXFP4: 17 B = [u8 e][qs[16]]; y = (2 * E2M1[code]) * 2^(e - 128), lib.rs:857-908. The doubled table with the halved
// scale keeps (e = 255, code = 1) at the finite 2^127; e = 0 and 1 give subnormal scales, built from their bit patterns.
// One IEEE multiply per value: it rounds only where the result is subnormal or overflows, exactly as the reference's does.
__device__ const float KV_MXFP4_2X[16] = {0.f, 1.f, 2.f, 3.f, 4.f, 6.f, 8.f, 12.f, 0.f, -1.f, -2.f, -3.f, -4.f, -6.f, -8.f, -12.f};

__device__ __forceinline__ float4 deq_mxfp4(const uint8_t* b, int v) {   // b has no alignment at all: byte loads
    uint32_t e = b[0];
    float d = __uint_as_float(e == 0 ? (1u << 21) : e == 1 ? (1u << 22) : (e - 1u) << 23);
    const uint8_t* qs = b + 1 + (v & 15);
    int sh = v >= 16 ? 4 : 0;
    float o[4];
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = __fmul_rn(KV_MXFP4_2X[(qs[k] >> sh) & 0xFu], d);
    return make_float4(o[0], o[1], o[2], o[3]);
}

// values v .. v + 3 of the block at b
template <uint32_t TYPE>
__device__ __forceinline__ float4 deq4(const uint8_t* b, int v) {
    if constexpr (TYPE == FHIP_Q8_0) return deq_q8_0(b, v);
    else if constexpr (TYPE == FHIP_Q4_K) return deq_q4_k(b, v);
    else if constexpr (TYPE == FHIP_Q5_K) return deq_q5_k(b, v);
    else if constexpr (TYPE == FHIP_Q6_K) return deq_q6_k(b, v);
    else if constexpr (TYPE == FHIP_Q4_0) return deq_legacy<false, false, 8>(b, v);
    else if constexpr (TYPE == FHIP_Q4_1) return deq_legacy<true, false, 0>(b, v);
    else if constexpr (TYPE == FHIP_Q5_0) return deq_legacy<false, true, 16>(b, v);
    else if constexpr (TYPE == FHIP_Q5_1) return deq_legacy<true, true, 0>(b, v);
    else if constexpr (TYPE == FHIP_IQ4_NL) return deq_iq4<false>(b, v);
    else if constexpr (TYPE == FHIP_IQ4_XS) return deq_iq4<true>(b, v);
    else return deq_mxfp4(b, v);
}

template <uint32_t TYPE, int VALS, int BYTES>
__global__ void deq_kernel(const uint8_t* __restrict__ raw, size_t nquads, float* __restrict__ out) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;  // one lane = 4 values
    if (t >= nquads) return;
    *(float4*)(out + t * 4) = deq4<TYPE>(raw + t / (VALS / 4) * BYTES, (int)(t % (VALS / 4)) * 4);
}

// Blocks in pinned host memory to floats in pinned host memory, a workgroup DEQ_TILE values: its bytes come over the bus in 16-byte pieces, all at
// once, and are unpacked out of LDS (a load of a narrower piece is a request on the bus of its own); the floats go back as the copy kernels' do, and
// so does the confirmation. The trip over the bus bounds it: one launch in the place of a copy up, an unpacking and a copy down, of which each
// waited for the one before. us a call, three launches -> one: 8928 values Q5_0 21.2 -> 15.3, 17056 Q4_0 23.1 -> 16.0, 96192 Q5_1 39.3 -> 30.3; in
// chunks 1352704 Q5_K 205 -> 187, 4283648 IQ4_XS 472 -> 418, 20971520 Q6_K 2463 -> 2348.
constexpr int DEQ_TILE = 4096, DEQ_THREADS = 512;

template <uint32_t TYPE, int VALS, int BYTES>
__global__ __launch_bounds__(DEQ_THREADS) void deq_through_kernel(const uint8_t* __restrict__ raw, uint32_t nblocks, float* __restrict__ out, uint32_t* __restrict__ done, uint32_t seq) {
    constexpr uint32_t TILE_BLOCKS = DEQ_TILE / VALS, PIECES = TILE_BLOCKS * BYTES / 16;
    static_assert(TILE_BLOCKS * BYTES % 16 == 0, "a tile's bytes start on a piece");
    __shared__ u32x4 lds[PIECES];
    const uint32_t first = blockIdx.x * TILE_BLOCKS, blocks = min(TILE_BLOCKS, nblocks - first);
    const u32x4* src = (const u32x4*)(raw + (size_t)first * BYTES);
    for (uint32_t i = threadIdx.x; i < (blocks * BYTES + 15) / 16; i += DEQ_THREADS) lds[i] = src[i];
    __syncthreads();
    u32x4* dst = (u32x4*)(out + (size_t)first * VALS);
    for (uint32_t i = threadIdx.x; i < blocks * (VALS / 4); i += DEQ_THREADS)
        store_through(dst + i, __builtin_bit_cast(u32x4, deq4<TYPE>((const uint8_t*)lds + i / (VALS / 4) * BYTES, (int)(i % (VALS / 4)) * 4)));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) store_through(done + blockIdx.x, seq);
}

// go(kernel of the type)
template <class Go>
int of_type(uint32_t type, Go go) {
    switch (type) {
        case FHIP_Q8_0: go.template operator()<FHIP_Q8_0, 32, 34>(); break;
        case FHIP_Q4_K: go.template operator()<FHIP_Q4_K, 256, 144>(); break;
        case FHIP_Q6_K: go.template operator()<FHIP_Q6_K, 256, 210>(); break;
        case FHIP_Q5_K: go.template operator()<FHIP_Q5_K, 256, 176>(); break;
        case FHIP_Q4_0: go.template operator()<FHIP_Q4_0, 32, 18>(); break;
        case FHIP_Q4_1: go.template operator()<FHIP_Q4_1, 32, 20>(); break;
        case FHIP_Q5_0: go.template operator()<FHIP_Q5_0, 32, 22>(); break;
        case FHIP_Q5_1: go.template operator()<FHIP_Q5_1, 32, 24>(); break;
        case FHIP_IQ4_NL: go.template operator()<FHIP_IQ4_NL, 32, 18>(); break;
        case FHIP_IQ4_XS: go.template operator()<FHIP_IQ4_XS, 256, 136>(); break;
        case FHIP_MXFP4: go.template operator()<FHIP_MXFP4, 32, 17>(); break;
        default: return fhip::set_error(FHIP_ERR_UNSUPPORTED_TYPE, "unsupported ggml type %u", type);
    }
    return fhip::check_hip(hipGetLastError(), "dequant launch");
}
struct ToDevice {
    const uint8_t* raw; size_t nquads; float* out; hipStream_t s;
    template <uint32_t TYPE, int VALS, int BYTES> void operator()() const {
        hipLaunchKernelGGL((deq_kernel<TYPE, VALS, BYTES>), dim3((unsigned)((nquads + 255) / 256)), dim3(256), 0, s, raw, nquads, out);
    }
};
struct ToHost {
    const uint8_t* raw; uint32_t nblocks; float* out; uint32_t *done, seq; hipStream_t s; int* wgs;
    template <uint32_t TYPE, int VALS, int BYTES> void operator()() const {
        *wgs = (int)((nblocks + DEQ_TILE / VALS - 1) / (DEQ_TILE / VALS));
        hipLaunchKernelGGL((deq_through_kernel<TYPE, VALS, BYTES>), dim3((unsigned)*wgs), dim3(DEQ_THREADS), 0, s, raw, nblocks, out, done, seq);
    }
};

}  // namespace

namespace fhip {

int launch_f16_to_f32(const uint16_t* d_bits, size_t n, float* d_out, hipStream_t s) {
    if (n == 0) return FHIP_OK;
    unsigned grid = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(f16_to_f32_kernel, dim3(grid), dim3(256), 0, s, d_bits, n, d_out);
    return check_hip(hipGetLastError(), "f16_to_f32 launch");
}

int launch_bf16_to_f32(const uint16_t* d_bits, size_t n, float* d_out, hipStream_t s) {
    if (n == 0) return FHIP_OK;
    unsigned grid = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(bf16_to_f32_kernel, dim3(grid), dim3(256), 0, s, d_bits, n, d_out);
    return check_hip(hipGetLastError(), "bf16_to_f32 launch");
}

int launch_dequant(uint32_t type, const uint8_t* d_raw, size_t nblocks, float* d_out, hipStream_t s) {
    if (nblocks == 0) return FHIP_OK;
    size_t vals = (type == FHIP_Q4_K || type == FHIP_Q5_K || type == FHIP_Q6_K || type == FHIP_IQ4_XS) ? 256 : 32;
    size_t nquads = nblocks * vals / 4;
    size_t grid = (nquads + 255) / 256;
    if (grid > 0x7FFFFFFFull) return set_error(FHIP_ERR_ARG, "dequant: %zu blocks exceed one launch", nblocks);
    return of_type(type, ToDevice{d_raw, nquads, d_out, s});
}

int launch_dequant_through(uint32_t type, const uint8_t* pinned_raw, size_t nblocks, float* pinned_out, uint32_t* done, uint32_t seq, hipStream_t s, int* wgs) {
    return of_type(type, ToHost{pinned_raw, (uint32_t)nblocks, pinned_out, done, seq, s, wgs});
}

}  // namespace fhip
