// launch_rules.h -- rules that choose a kernel or a shape from sizes alone:
// plain host C++, so that they are tested without a GPU.
#ifndef PQ2_LAUNCH_RULES_H
#define PQ2_LAUNCH_RULES_H

#include <stdint.h>

#include <initializer_list>

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

// ---- more than 16 tokens ---------------------------------------------------
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// What the wide kernel (gemm_wide.hip) needs of the sizes: whole pairs of blocks,
// and buffer ranges that are ints
inline bool wide_fits(int64_t n_out, int64_t n_tok, int nb) {
    return nb >= 2 && nb % 2 == 0 && (uint64_t)n_out * 34 * (uint64_t)nb < (1ull << 31) &&
           (uint64_t)n_tok * 36 * 4 * (uint64_t)nb < (1ull << 31);
}

// Rows [0, rows) of the product that the wide kernel takes, and its tile
// height (*mi = 8: 256 rows, 5: 160 rows): the whole 256-row tiles whose
// 256 x 256 tiles fill whole rounds of the device's CUs (the caller runs the
// remaining rows on the 128-row kernel), or, short of one round, every row on
// 256- or 160-row tiles where one round of them holds at least 3/4 of a full
// round's outputs; 0 where the kernel's requirements do not hold or its tiles
// would fill too little of a round.
inline int64_t wide_rows(int64_t n_out, int64_t n_tok, int nb, int cus, int * mi) {
    *mi = 8;
    if (!wide_fits(n_out, n_tok, nb)) return 0;
    const int64_t T = ceil_div(n_tok, 256);
    if (4 * n_tok < 3 * T * 256) return 0;                                        // token tiles mostly empty
    // 256-row tiles over the rows whose tiles fill whole rounds
    const int64_t R = n_out / 256, rounds = R * T / cus;
    if (rounds >= 1) return (rounds * cus / T < R ? rounds * cus / T : R) * 256;
    // Less than one round: a round of wide tiles takes about the same time
    // however many CUs it fills, so one pays where at least 3/4 of a full
    // round's outputs are real (measured on MI355X, one process, us, LDS kernel
    // -> wide: 17408x5120 M = 768 225 -> 181 (256 rows), M = 512 165 -> 138
    // (160 rows), 6144x5120 M = 2048 191 -> 183 (256 rows); at 5/8 and below
    // the LDS kernel stays faster: 17408x5120 M = 384 116 against 137,
    // 5120x6144 M = 1024 126 against 160)
    const int64_t outputs = n_out * n_tok;
    if (ceil_div(n_out, 256) * T <= cus && 4 * outputs >= 3 * (int64_t)cus * 256 * 256) return n_out;
    if (ceil_div(n_out, 160) * T <= cus && 4 * outputs >= 3 * (int64_t)cus * 160 * 256) {
        *mi = 5;
        return n_out;
    }
    return 0;
}

// Time (us) of tokens [0, cols) on the large tiles, rows as wide_rows gives
// them: rounds of workgroups times what a round takes a block of K (MI355X: 4.5
// us on 256-row tiles, 3.45 on 160-row ones, 1.42 on 128 x 128, 1.05 on 128 x 64;
// a product that fills three rounds of 128 x 128 or more exactly takes 1.55 to 1.6
// each, so that three do not pass for faster than one of 256-row tiles: 12288x5120
// with 1024 tokens 184 us against 177, 8192x2048 with 1536 82 against 78)
inline float large_us(int64_t n_out, int64_t cols, int nb, int cus, int64_t rows, int mi) {
    float us = 0.0f;
    if (rows > 0) us = (mi == 8 ? 4.5f : 3.45f) * (float)ceil_div(ceil_div(rows, 32 * mi) * ceil_div(cols, 256), cus);
    if (rows < n_out) {
        // gemm_prefill_f16's choice
        const int64_t R = ceil_div(n_out - rows, 128), T = ceil_div(cols, 128);
        const int64_t full = R * T / cus, rest = R * T - full * cus;
        if (2 * R * T <= cus) us += 1.05f;
        else if (full >= 1 && rest > 0 && 2 * rest <= cus && full * cus % T == 0 &&
                 (R - full * cus / T) * ceil_div(cols, 64) <= cus)
            us += 1.42f * (float)full + 1.05f;
        else us += (rows == 0 && rest == 0 && full >= 3 ? 1.55f : 1.42f) * (float)ceil_div(R * T, cus);
    }
    return us * (float)nb;
}

// The tiles of a prefill: tokens [0, cols) on the large ones, the first rows of
// them on the wide kernel (tile height mi), tokens [cols, n_tok) on the small
// ones (gemm_mid.hip; cols = 0: all of them).  wide, small: the pointers let
// these kernels run (and, for the small one, the sizes).  rows and mi come as
// wide_rows gives them for every token; another plan has to be 5 % faster by its
// estimate.  Small tiles take over the whole product where large ones would leave
// most CUs idle, or the tokens past the whole large tiles where these would start
// another round, and rows whose wide tiles are short of a round take 128-row
// tiles where those have fewer empty tokens.  Measured (us, large tiles as
// wide_rows has them -> this plan): 17408x5120 with 20 tokens 57 -> 17, 33 54 ->
// 22, 100 57 -> 48, 140 101 -> 63, 400 159 -> 126; 5120x17408 with 100 132 -> 45, 800
// 361 -> 213; 10240x5120 with 386 102 -> 69, 777 139 -> 129 (768 + 9 tokens), 1166 229 ->
// 180; unchanged 17408x5120 with 1500, 10240x5120 with 1900.  Not a matter of the
// workspace, with which wide tiles are up to 5 % faster: the bytes have to be the
// same with and without one (8704x5120 with 960 tokens and a workspace pays 3 %).
inline void prefill_plan(bool wide, bool small, int64_t n_out, int64_t n_tok, int nb, int cus, int64_t * cols,
                         int64_t * rows, int * mi) {
    float best = 0.95f * large_us(n_out, n_tok, nb, cus, *rows, *mi);
    float us = 0.0f;
    if (small) mid_pick(n_out, n_tok, nb, cus, &us);
    if (small && us < best) best = us, *cols = 0, *rows = 0;
    // wide_rows looks at the tokens that it is given only
    if ((uint64_t)n_tok * 36 * 4 * (uint64_t)nb >= (1ull << 31)) return;
    for (int64_t c : {n_tok, n_tok / 128 * 128, n_tok / 256 * 256}) {
        if (c == 0 || (c < n_tok && !small)) continue;
        us = 0.0f;
        if (c < n_tok) mid_pick(n_out, n_tok - c, nb, cus, &us);
        int m = 8;
        const int64_t r = wide ? wide_rows(n_out, c, nb, cus, &m) : 0;
        const float with = us + large_us(n_out, c, nb, cus, r, m), plain = us + large_us(n_out, c, nb, cus, 0, 8);
        if (r > 0 && (c == n_tok || c % 256 == 0) && with < best) best = with, *cols = c, *rows = r, *mi = m;
        if (plain < best) best = plain, *cols = c, *rows = 0;
    }
}

}  // namespace pq2

#endif
