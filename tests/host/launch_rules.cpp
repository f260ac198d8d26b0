// The rules of csrc/launch_rules.h as C functions, for tests/test_launch_rules.py.
#include "../../p40-kernel_amd/csrc/launch_rules.h"

extern "C" {
int rms_per_block(int64_t n_tok, int64_t nhb, int64_t cus) { return pq2::rms_per_block(n_tok, nhb, cus); }
}
