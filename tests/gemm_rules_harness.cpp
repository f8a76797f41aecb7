// gemm_mfma.hip's host side, for test_launch_rules.py.
#include "../ferric_amd/csrc/gemm_mfma.hip"
#include "launch_rules.hpp"

int fhip::g_gemm_tile = -1;
extern "C" {
// the first of eight elements of X that a thread stages for columns first + col ... + 7 of row t
uint32_t h_x_at(int t, int T, int K, int first, int col) { return x_piece(t, T, K, col) + x_step(first, col, K); }
}
