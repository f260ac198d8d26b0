// The rules of csrc/launch_rules.h as C functions, for tests/test_launch_rules.py.
#include "../../p40-kernel_amd/csrc/launch_rules.h"

extern "C" {
int rms_per_block(int64_t n_tok, int64_t nhb, int64_t cus) { return pq2::rms_per_block(n_tok, nhb, cus); }
int small_shape(int64_t n_out, int nb, int64_t cus) {
    const pq2::SmallShape s = pq2::small_shape(n_out, nb, cus);
    return 16 * s.rt * 100 + s.ks;
}
int mid_pick(int64_t n_out, int64_t n_tok, int nb, int cus) {
    float us = 0.0f;
    const pq2::MidShape & s = pq2::mid_shapes[pq2::mid_pick(n_out, n_tok, nb, cus, &us)];
    return 16 * s.mi * 1000 + 16 * s.ni;
}
float mid_us(int64_t n_out, int64_t n_tok, int nb, int cus) {
    float us = 0.0f;
    pq2::mid_pick(n_out, n_tok, nb, cus, &us);
    return us;
}
void prefill_plan(int wide, int small, int64_t n_out, int64_t n_tok, int nb, int cus, int64_t * plan) {
    int mi = 8;
    plan[0] = n_tok;
    plan[1] = wide ? pq2::wide_rows(n_out, n_tok, nb, cus, &mi) : 0;
    pq2::prefill_plan(wide != 0, small != 0, n_out, n_tok, nb, cus, &plan[0], &plan[1], &mi);
    plan[2] = plan[1] > 0 ? 32 * mi : 0;
}
}
