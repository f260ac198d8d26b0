// launch_rules.h -- rules that choose a kernel or a shape from sizes alone:
// plain host C++, so that they are tested without a GPU.
#ifndef PQ2_LAUNCH_RULES_H
#define PQ2_LAUNCH_RULES_H

#include <stdint.h>

namespace pq2 {

// RMSNorm -> FWHT -> Q8_1 of n_tok rows of nhb blocks of 1024: a workgroup per
// block, which reads its whole row for the sum of squares (true), or one per
// token, which reads the row once where its waves hold it (up to 32 blocks) and
// else twice.  The first spreads few tokens over the CUs and its repeated reads
// cost more with every further round of workgroups; the second takes about as
// long for one token as for one on each CU, the longer the more blocks a wave
// has.  So the line is a number of workgroups per block and CU that grows with
// the row.  Measured on MI355X (256 CUs, us, per block / per token):
//   up to 14 blocks, 1 a CU: 52 x 5120 5.11 / 4.84, 33 x 8192 5.35 / 4.75
//   15 to 17, 2: 24 x 15360 6.68 / 6.69, 40 x 16384 7.70 / 6.94, 16 x 17408 6.84 /
//     7.39, 28 x 17408 7.28 / 7.71, 32 x 17408 7.98 / 7.77
//   18 and more, 3: 15 x 18432 6.88 / 8.75, 36 x 18432 8.15 / 9.12, 30 x 24576 9.02 /
//     9.55, 24 x 32768 10.8 / 11.7, 28 x 32768 13.0 / 11.7, 12 x 65536 17.2 / 19.4,
//     14 x 65536 21.0 / 19.4, 6 x 131072 29.8 / 36.2
//   256 and more, 4: 4 x 262144 69.5 / 69.7, 1 x 1048576 263 / 271, 2 x 1048576 539 / 271
inline bool rms_per_block(int64_t n_tok, int64_t nhb, int64_t cus) {
    const int64_t per_cu = nhb < 15 ? 1 : nhb < 18 ? 2 : nhb < 256 ? 3 : 4;
    return n_tok <= per_cu * cus && n_tok * nhb <= per_cu * cus;
}

// Rows (16 rt) and waves over K (ks) of a workgroup of the streamed kernel for 9
// to 16 tokens.  8 ways over K keep more loads in flight than 4, but their ring
// fills a CU where two 4-way ones fit, so they pay in one round of CUs only, on
// 16 rows or else on 32.  Measured on MI355X (256 CUs, us, 9 / 12 / 16 tokens, 16
// rows and 4 ways -> this): 16 rows, 1024x5120 5.9 6.0 6.2 -> 5.5 5.5 5.6, 4096x17408
// 15.8 16.0 16.4 -> 12.2 12.4 12.8; 32 rows, 5120x6144 8.9 8.9 9.0 -> 8.0 8.0 8.4,
// 5120x17408 18.6 18.6 18.8 -> 16.5 16.6 17.2, 8192x8192 11.2 11.4 11.6 -> 10.7 10.6
// 10.9.  On 40 to 47 blocks the 32-row gain is small (6144x5120 2 %) and gone at
// either end (4097x5120 7.5 -> 7.6..7.8, 8192x5120 8.4 -> 8.5), so the range stops
// short of both there.  Below 40 blocks 8 partial sums are further from 64 bits than
// 4, from 40 on no further (4 / 8 ways, 1e-8: 2048 columns 5.7 / 6.4, 3072 6.2 /
// 6.6, 4096 6.75 / 6.88, 5120 7.20 / 7.13, 6144 7.65 / 7.35, 17408 11.4 / 9.5).
struct SmallShape {
    int rt, ks;
};
inline SmallShape small_shape(int64_t n_out, int nb, int64_t cus) {
    if (nb < 40) return {1, 4};
    if (n_out <= 16 * cus) return {1, 8};
    if (nb < 48 ? 2 * n_out > 33 * cus && n_out <= 28 * cus : n_out <= 32 * cus) return {2, 8};
    return {1, 4};
}

// Tile shapes of the small-tile GEMM (gemm_mid.hip): 16 mi rows x 16 ni tokens
// (sum: the stored sums are read, batches of up to 16 tokens only), and the time
// of one step of 8 blocks on one CU (MI355X, us, the slope over K of one round of
// workgroups).  A CU holds one workgroup of the wider tiles, whose registers or
// LDS leave no room for a second.  Of the 16-token tiles it holds two (116 and 95
// VGPRs, 72 and 52 KB of LDS): us2 is a step of both, so a second one costs about
// 0.6 of a round.  Measured (us, 5120 columns, 256 / 257 / 512 / 513 workgroups): 80 x 32
// 18.7 32.0 35.9 48.8, 80 x 16 13.7 18.1 20.9 28.2, 48 x 16 10.2 13.3 14.6 19.3.
struct MidShape {
    int mi, ni;
    float us, us2;
    bool sum;
};
constexpr int MID_SHAPES = 9, MID_SUM = 6;
constexpr MidShape mid_shapes[MID_SHAPES] = {
    {5, 3, 3.6f, 0.0f, false},  {3, 2, 1.8f, 0.0f, false},  {5, 2, 2.5f, 0.0f, false},
    {4, 2, 2.05f, 0.0f, false}, {4, 3, 2.8f, 0.0f, false},  {2, 2, 1.45f, 0.0f, false},
    {5, 1, 1.9f, 3.0f, true},   {5, 1, 1.8f, 2.85f, false}, {3, 1, 1.2f, 1.98f, false}};

// The fastest shape for n_tok tokens of rows of nb blocks, and its estimated time:
// rounds of workgroups, 4 us to start and reduce, and a clock that many full
// rounds lower (17408x5120 with 400 tokens: 8 rounds of 80 x 48 in 171 us, 33
// tokens: one in 22).  32-bit arithmetic, this runs on every call: the caller has
// seen that there are under 2^22 tiles of 32 x 16.
inline int mid_pick(int64_t n_out, int64_t n_tok, int nb, int cus, float * us) {
    int pick = -1;
    const uint32_t c = (uint32_t)cus;
    for (int k = 0; k < MID_SHAPES; ++k) {
        const MidShape & s = mid_shapes[k];
        if (s.sum) continue;
        const uint32_t bm = 16 * s.mi, bn = 16 * s.ni;
        const uint32_t wgs = (((uint32_t)n_out + bm - 1) / bm) * (((uint32_t)n_tok + bn - 1) / bn);
        const uint32_t rounds = (wgs + c - 1) / c;
        const float r = (float)rounds;
        const float step = s.us2 == 0.0f ? r * s.us : (float)(rounds / 2) * s.us2 + (float)(rounds % 2) * s.us;
        const float t = 4.0f + (1.0f + 0.02f * (r < 8.0f ? r : 8.0f)) * (float)(nb / 8) * step;
        if (pick < 0 || t < *us) *us = t, pick = k;
    }
    return pick;
}

}  // namespace pq2

#endif
