// Wide loads from addresses that are only 2-byte aligned (Q6_K blocks are 210 bytes, Q8_0 blocks 34, the legacy 4/5-bit
// blocks 18..24). The memory pipeline splits a dwordx2 / dwordx4 load whose address is not a multiple of 4 and runs it
// at about 60 % of the aligned rate (measured on the Q6_K down projection: 47 us with such loads, 31 us aligned). So
// the load is made from the dword boundary at or below the address and the bytes are shifted into place: one
// v_alignbyte_b32 per dword. The last two bytes come from their own 2-byte load, so nothing outside [p, p + n) is read
// beyond the two bytes below p that lie in the same dword.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace fhip {

typedef uint32_t ld_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t ld_u32x2 __attribute__((ext_vector_type(2)));
struct __attribute__((packed, aligned(4))) LdU4A4 { ld_u32x4 v; };
struct __attribute__((packed, aligned(4))) LdU2A4 { ld_u32x2 v; };

__device__ __forceinline__ ld_u32x4 load16_a2(const uint8_t* p) {
    const uint32_t m = (uint32_t)(uintptr_t)p & 2u;
    const ld_u32x4 w = ((const LdU4A4*)(p - m))->v;
    const uint32_t e = *(const uint16_t*)(p + 14);
    return (ld_u32x4){__builtin_amdgcn_alignbyte(w[1], w[0], m), __builtin_amdgcn_alignbyte(w[2], w[1], m),
                      __builtin_amdgcn_alignbyte(w[3], w[2], m), __builtin_amdgcn_alignbyte(e, w[3], m)};
}

__device__ __forceinline__ ld_u32x2 load8_a2(const uint8_t* p) {
    const uint32_t m = (uint32_t)(uintptr_t)p & 2u;
    const ld_u32x2 w = ((const LdU2A4*)(p - m))->v;
    const uint32_t e = *(const uint16_t*)(p + 6);
    return (ld_u32x2){__builtin_amdgcn_alignbyte(w[1], w[0], m), __builtin_amdgcn_alignbyte(e, w[1], m)};
}

// The same in two halves, for loops that ask for a piece long before they read it. The shift needs the loaded dwords: beside the load
// it is a wait for memory however far the first use is, since the compiler does not carry it over a barrier. So the piece is kept as
// it came and shifted where it is read, by the address modulo 4 (0 or 2). LATE = false shifts at once,
// in registers of the plain size.
struct Un16 { ld_u32x4 w; uint32_t e; };
template <bool LATE>
__device__ __forceinline__ Un16 load16_un(const uint8_t* p) {
    if (!LATE) return Un16{load16_a2(p), 0u};
    return Un16{((const LdU4A4*)(p - ((uint32_t)(uintptr_t)p & 2u)))->v, *(const uint16_t*)(p + 14)};
}
__device__ __forceinline__ void shift_in_place(Un16& u, uint32_t m) {
    u.w = (ld_u32x4){__builtin_amdgcn_alignbyte(u.w[1], u.w[0], m), __builtin_amdgcn_alignbyte(u.w[2], u.w[1], m),
                     __builtin_amdgcn_alignbyte(u.w[3], u.w[2], m), __builtin_amdgcn_alignbyte(u.e, u.w[3], m)};
}

}  // namespace fhip
