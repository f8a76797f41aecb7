// gemm_f16x2.hip's host side, for test_launch_rules.py.
#include "../ferric_amd/csrc/gemm_f16x2.hip"
#include "launch_rules.hpp"

namespace {
fhip_weight shaped(uint32_t type, size_t rows, size_t cols) {
    fhip_weight w{};
    w.type = type; w.rows = rows; w.cols = cols; w.batch_policy = FHIP_BATCH_ORDERED;
    fhip::gemm_f16x2_lay_out(&w);
    return w;
}
}  // namespace
extern "C" {
// rows outputs x cols columns x t activation rows, sums in order: whether the held kernel is taken where both can do it
int h_held(uint32_t type, size_t rows, size_t cols, size_t t) {
    const fhip_weight w = shaped(type, rows, cols);
    return fhip::held_beats_resident(&w, t);
}
// the resident kernel's launch: sets of eight rows a workgroup and workgroups' sets, ranges of K, workgroups of a range, the most chunks of a range that fit, bytes of partial outputs
void h_resident(uint32_t type, size_t rows, size_t cols, size_t t, int64_t out[6]) {
    const fhip_weight w = shaped(type, rows, cols);
    const ResPlan q = plan_of(&w, t);
    const int most = type == FHIP_Q4_K ? resident_chunks_of<Q4K>(q.nt) : type == FHIP_Q5_K ? resident_chunks_of<Q5K>(q.nt) : type == FHIP_Q6_K ? resident_chunks_of<Q6K>(q.nt) : resident_chunks_of<Q80>(q.nt);
    const int64_t v[6] = {q.nt, q.sets, q.parts, q.per_part, most, (int64_t)fhip::gemm_f16x2_parts_bytes(&w, t)};
    for (int i = 0; i < 6; i++) out[i] = v[i];
}
}
