// gemv_wide.hip's host side, for test_launch_rules.py.
#include "../ferric_amd/csrc/gemv_wide.hip"
#include "launch_rules.hpp"

extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipErrorNoDevice; }
namespace fhip {
size_t device_lds_bytes() { return 163840; }
bool gemv_streams_p3(const fhip_weight*, size_t) { return true; }
}  // namespace fhip

// t activation rows, `each` of them a workgroup: pairs of rows a lane holds, tiles, groups a pass, passes, waves, workgroups of a group of activation rows, these groups
template <class F>
static void plan(size_t rows, size_t cols, size_t t, size_t each, int64_t out[7]) {
    const WidePlan q = wide_plan((int)rows, (int)(cols / 32 + 15) / 16, (int)t, (int)each, F::IMAGE, F::BIG, 256, 163840);
    const int64_t v[7] = {q.E, q.tiles, q.P, q.passes, q.W, q.grid, q.row_groups};
    for (int i = 0; i < 7; i++) out[i] = v[i];
}
extern "C" void h_wide_plan(uint32_t type, size_t rows, size_t cols, size_t t, size_t each, int64_t out[7]) {
    type == FHIP_Q8_0 ? plan<Q80>(rows, cols, t, each, out) : type == FHIP_MXFP4 ? plan<Mxf4>(rows, cols, t, each, out) : plan<Q50>(rows, cols, t, each, out);
}
