// What the prompt path's translation units offer each other beside common.hpp.
#pragma once
#include "common.hpp"

namespace fhip {

// two floats rounded to bf16 (to nearest, ties to even): v_cvt_pk_bf16_f32, a in the low half
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2)); }

// gemm_mfma.hip
int launch_gemm_bf16_swiglu(const fhip_weight* w, const uint16_t* d_x, size_t t, uint16_t* d_h, hipStream_t s, float* d_ws, size_t ws_bytes);
size_t gemm_bf16_swiglu_ws_bytes(const fhip_weight* w, size_t t);
// common.hpp's, with every output's products added in the order that stays (fhip_gemm_q_bf16_run_sums) if run_sums says so
int launch_gemm_bf16(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, float* d_ws, size_t ws_bytes, bool run_sums);
size_t gemm_bf16_ws_bytes(const fhip_weight* w, size_t t, bool run_sums);

// decode_ops.hip, prefill_attn.hip: the f32 launches with their result rounded to bf16, as launch_cvt_bf16 rounds it
int launch_rmsnorm_bf16(const float* a, const float* b, const float* weight, size_t rows, size_t d, float eps, float* sum_out, uint16_t* norm_out,
                        hipStream_t s);
int launch_causal_attention_bf16(const float* q, const float* K, const float* V, size_t t, size_t s, int n_head, int n_kv, int hd, size_t window,
                                 float softcap, bool cuts, uint16_t* out, float* ws, size_t ws_bytes, hipStream_t st);

}  // namespace fhip
