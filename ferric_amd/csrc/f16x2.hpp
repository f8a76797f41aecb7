// gemm_f16x2.hip: up to 32 activation rows in one pass over the weights, f16 matrix cores, f32-grade results
#pragma once
#include "common.hpp"

namespace fhip {

bool gemm_f16x2_supports(const fhip_weight* w, size_t t);
size_t gemm_f16x2_xp_bytes(const fhip_weight* w, size_t t);       // prepared-activation buffer for t rows
bool gemm_f16x2_adds_into_y(const fhip_weight* w, size_t t);      // true: the launch adds into y, a cleared y saves it a launch
// Where a matmul's output still lies as partial outputs, one for each range of K: their sum in that order (parts == 0: as it is)
struct F16Parts {
    const float* part;
    int parts;
    size_t stride, ld;    // from one to the next, and from row to row
};

// splits the rows of x [t, cols] (swiglu: of silu(gate) * up of x [t, 2 cols]) chunk by chunk into scaled f16 hi / lo
// operand rows, each carrying the factor that takes its scale out again
// src: x is the output of a matmul whose ordered sum was left to this launch (launch_gemm_f16x2_resident with `deferred`)
int launch_xsplit_f16(const fhip_weight* w, const float* d_x, size_t t, bool swiglu, uint16_t* d_xp, hipStream_t s, float* zero = nullptr,
                      size_t zero_n = 0, const F16Parts* src = nullptr);
// y_cleared: y is zero where the launch adds into it
int launch_gemm_f16x2(const fhip_weight* w, const uint16_t* d_xp, size_t t, float* d_y, hipStream_t s, bool y_cleared = false, const float* d_x = nullptr);
// true: launch_gemm_f16x2 given d_x (the f32 rows) makes its operand rows itself, without launch_xsplit_f16 in front of it (d_xp is not read)
bool gemm_f16x2_own_x(const fhip_weight* w, const float* d_x, size_t t);

// Sums in order (FHIP_BATCH_ORDERED), up to 32 rows of every format.
bool gemm_f16x2_takes(const fhip_weight* w, size_t t);
// the whole product, y = x W^T, in one launch without a workspace: whether it can, whether it is the faster one (of any policy), and the launch
bool gemm_f16x2_held_takes(const fhip_weight* w, const float* d_x, size_t t, const float* d_y);
bool gemm_f16x2_held(const fhip_weight* w, const float* d_x, size_t t, const float* d_y);
int launch_gemm_f16x2_held(const fhip_weight* w, const float* d_x, size_t t, float* d_y, hipStream_t s);
// the product from prepared rows (d_xp) or, where gemm_f16x2_resident_own_x says so, from the rows as they are (d_xp null): one launch and, where it cuts K into more than
// one part, one that adds the partial outputs (d_part: gemm_f16x2_parts_bytes) or leaves them to the reader of y (deferred). d_part null: a launch a part, each adding to y,
// which has the same bits (the rows as they are, apart from y, and not deferred)
void gemm_f16x2_lay_out(fhip_weight* w);     // a new handle's plans, which the others read
int gemm_f16x2_parts(const fhip_weight* w, size_t t);
size_t gemm_f16x2_parts_bytes(const fhip_weight* w, size_t t);
bool gemm_f16x2_resident_own_x(const fhip_weight* w, const float* d_x, size_t t, const float* d_y);
int launch_gemm_f16x2_resident(const fhip_weight* w, const uint16_t* d_xp, const float* d_x, size_t t, float* d_y, float* d_part, hipStream_t s, F16Parts* deferred);

}  // namespace fhip
