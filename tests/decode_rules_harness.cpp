// decode_ops.hip's host side, for test_launch_rules.py.
#include "../ferric_amd/csrc/decode_ops.hip"
#include "launch_rules.hpp"

extern "C" int h_norm_ahead(size_t grid) { return fhip::norm_ahead(grid); }
