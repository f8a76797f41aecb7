// What a block of a quantized KV cache dequantizes to (kvquant.hip, decode_ops.hip): the reference's separately rounded f32 operations
// (crates/ferric-tensor/src/kvquant.rs:1100-1186), so no multiply-add is fused here whatever the file's default.
#pragma once
#include "common.hpp"

#include <hip/hip_fp16.h>

namespace fhip {

__device__ __forceinline__ float kvq_scale(uint16_t h) { return __half2float(__ushort_as_half(h)); }
// value of a code: q in [-127, 127] of a Q8_0 block, [0, 15] of a four-bit one; m: Q4_1's minimum
template <int FMT>
__device__ __forceinline__ float kvq_value(int q, float d, float m) {
#pragma clang fp contract(off)
    if constexpr (FMT == FHIP_KVQ_Q8_0) return (float)q * d;
    else if constexpr (FMT == FHIP_KVQ_Q4_0) return ((float)q - 8.0f) * d;
    else return (float)q * d + m;
}
// values j .. j + 3 of block b, j a multiple of 4
template <int FMT>
__device__ __forceinline__ float4 kvq_values4(const uint32_t* __restrict__ codes, const uint16_t* __restrict__ scales, size_t b, int j) {
    const float d = kvq_scale(scales[FMT == FHIP_KVQ_Q4_1 ? 2 * b : b]), m = FMT == FHIP_KVQ_Q4_1 ? kvq_scale(scales[2 * b + 1]) : 0.f;
    if constexpr (FMT == FHIP_KVQ_Q8_0) {
        const uint32_t w = codes[b * 8 + j / 4];
        return make_float4(kvq_value<FMT>((int8_t)(w & 255u), d, m), kvq_value<FMT>((int8_t)((w >> 8) & 255u), d, m),
                           kvq_value<FMT>((int8_t)((w >> 16) & 255u), d, m), kvq_value<FMT>((int8_t)(w >> 24), d, m));
    } else {
        const uint32_t w = codes[b * 4 + (j % 16) / 4] >> (j < 16 ? 0 : 4);
        return make_float4(kvq_value<FMT>(w & 15u, d, m), kvq_value<FMT>((w >> 8) & 15u, d, m), kvq_value<FMT>((w >> 16) & 15u, d, m),
                           kvq_value<FMT>((w >> 24) & 15u, d, m));
    }
}

}  // namespace fhip
