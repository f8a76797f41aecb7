// Four 4-bit indices (one per byte, the upper nibbles clear) looked up in a table of sixteen bytes by two byte permutes and two exclusive ors.
//
// v_perm_b32 takes selectors 0 .. 7 as bytes of its two words; 8 .. 11 give the sign of bytes 1, 3, 5, 7 over the byte, 12 gives 0 and 13 .. 15 give 255. So the
// permute of the table's lower half by an index from 8 on is a constant, that of its upper half by (index ^ 8) one for an index below 8, and with
// each half's bytes stored less the other's constant the exclusive or of the two permutes is the entry: no mask, no selection. (Both halves by the
// index modulo 8 and a selection by bit 3, before: eight instructions and a multiplication, now four.) The kernels that look codes up are bound by
// instruction issue; us, before -> now, 24 bits: MXFP4 9728 x 2560, 2 rows 8.7 -> 8.4, 4 rows 9.9 -> 9.6, 12288 x 8192, 1 / 2 / 4 / 8 / 16 rows 15.4 -> 14.2, 30.4 -> 28.1, 23.3 ->
// 22.3, 32.0 -> 30.8, 52.7 -> 52.1; IQ4_XS 14.5 -> 13.5, 28.7 -> 26.6, 21.5 -> 20.5, 30.0 -> 29.0, 46.4 -> 45.5; IQ4_NL 14.6 -> 13.7, 28.9 -> 27.1.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fhip {

struct Lut16 { uint32_t lo[2], hi[2]; };
// t: the sixteen bytes in order, four a word
constexpr Lut16 lut16(uint32_t t0, uint32_t t1, uint32_t t2, uint32_t t3) {
    const uint32_t w[4] = {t0, t1, t2, t3};
    uint32_t t[16] = {}, p[8] = {}, n[8] = {};
    for (int i = 0; i < 16; i++) t[i] = (w[i / 4] >> (8 * (i % 4))) & 0xFF;
    auto sign = [](uint32_t b) { return b & 0x80u ? 0xFFu : 0u; };
    for (int i = 4; i < 8; i++) {           // the other half's selectors 12 .. 15
        const uint32_t other = i == 4 ? 0u : 0xFFu;
        p[i] = t[i] ^ other;
        n[i] = t[8 + i] ^ other;
    }
    constexpr int order[4] = {2, 3, 1, 0};  // selector 8 + i: the sign of byte 2 i + 1, which is known by then
    for (int k = 0; k < 4; k++) {
        const int i = order[k];
        p[i] = t[i] ^ sign(n[2 * i + 1]);
        n[i] = t[8 + i] ^ sign(p[2 * i + 1]);
    }
    Lut16 r = {};
    for (int i = 0; i < 8; i++) {
        r.lo[i / 4] |= p[i] << (8 * (i % 4));
        r.hi[i / 4] |= n[i] << (8 * (i % 4));
    }
    return r;
}

__device__ __forceinline__ uint32_t lut16x4(uint32_t idx, const Lut16& t) {
    return __builtin_amdgcn_perm(t.lo[1], t.lo[0], idx) ^ __builtin_amdgcn_perm(t.hi[1], t.hi[0], idx ^ 0x08080808u);
}

}  // namespace fhip
