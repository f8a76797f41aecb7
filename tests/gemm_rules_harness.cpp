// gemm_mfma.hip's host side, for test_launch_rules.py.
#include "../ferric_amd/csrc/gemm_mfma.hip"
#include "launch_rules.hpp"

int fhip::g_gemm_tile = -1;
extern "C" {
// the first of eight elements of X that a thread stages for columns first + col ... + 7 of row t
uint32_t h_x_at(int t, int T, int K, int first, int col) { return x_piece(t, T, K, col) + x_step(first, col, K); }

// the launch of `rows` outputs x `cols` columns x t activation rows: tile, its rows, its outputs, whole rounds, chunks a run, workgroups
void h_plan(uint32_t type, size_t rows, size_t cols, size_t t, int run_sums, int64_t out[6]) {
    fhip_weight w{};
    w.type = type; w.rows = rows; w.cols = cols;
    TilePlan q{};
    switch (type) {
        case FHIP_Q4_K: choose_plan<Q4K>(&w, rows, t, run_sums != 0, q); break;
        case FHIP_Q5_K: choose_plan<Q5K>(&w, rows, t, run_sums != 0, q); break;
        case FHIP_Q6_K: choose_plan<Q6K>(&w, rows, t, run_sums != 0, q); break;
        default: choose_plan<Q80>(&w, rows, t, run_sums != 0, q);
    }
    const int64_t v[6] = {q.tile, q.bm, q.bn, q.whole_rounds, q.per, (int64_t)q.grid};
    for (int i = 0; i < 6; i++) out[i] = v[i];
}
}
