// What the prompt path's translation units offer each other beside common.hpp.
#pragma once
#include "common.hpp"

namespace fhip {

// gemm_mfma.hip
int launch_gemm_bf16_swiglu(const fhip_weight* w, const uint16_t* d_x, size_t t, uint16_t* d_h, hipStream_t s, float* d_ws, size_t ws_bytes);
size_t gemm_bf16_swiglu_ws_bytes(const fhip_weight* w, size_t t);

}  // namespace fhip
