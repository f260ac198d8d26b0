// gemm_mid.hip -- PQ2_0 x Q8_1 GEMM for a few dozen to a few hundred tokens.
//
// Contract as gemm_wide.hip: Y[r*n_tok + t] = sum_b f16(dw[r,b]) * sum_p
// f16(da[4b+p, t]) * S(r, b, p, t), S the integer dot of chunk p of block b
// (reference tests/test_p40.cpp:449-470), X chunk-major.
//
// Shape.  At these sizes the 128-row tiles of gemm_f16_kernel leave most CUs
// idle, so the workgroup tile is small (16 MI rows x 16 NI tokens) and the 8
// waves of a workgroup split K instead: step s of the loop is 8 PQ2_0 blocks
// (272 bytes of every row, 16-byte aligned), one block per wave, and every
// wave runs the whole tile over its blocks; the 8 partial tiles meet in LDS at
// the end, added in wave order.
//   * W: a step's rows arrive by 16-byte LDS-DMA (17 lanes a row), double
//     buffered; a row's pitch of 68 dwords puts 16 rows' reads on distinct
//     banks.
//   * X: a wave needs 4 runs of 16 NI Q8_1 blocks; it loads them as contiguous
//     16-byte pieces one step ahead (per-token loads at a 36-byte stride cost
//     the L1 an access a lane) and passes them through its own LDS region.
// Arithmetic: v_mfma_f32_16x16x32_f16 gives the exact chunk dot S (below); U =
// sum_p da_p * S_p in fp32, then acc += dw * U: 5 FMAs per 16 x 16 tile and
// chunk, the scales stay in fp32 whatever their size.
//
// What bounds it is the VALU, so the operands are made in few instructions: a
// code becomes the f16 1024 + code (or 1024 + 4 code, against q / 4) with one
// mask, and what that adds to the dot, (1024 + 1) q per code too much, is
// taken off by the accumulator's start: one MFMA per 16 tokens and chunk with
// a constant A (-1025, -1028) gives it for every row tile.  All of these are
// integers below 2^24, so S is exact.  80 x 16 tiles, which run batches of up to
// 16 tokens, start from -1024 and the block's stored sum s instead, as every
// kernel of those batches does.
#include <hip/hip_runtime.h>

#include "pq2_device.h"
#include "host_state.h"
#include "launch_rules.h"
#include "../../include/bonsai_p40.h"

#include <stdint.h>

using namespace pq2;

namespace {

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int M_STEP = 8 * PQ2_BYTES;                            // bytes of a row per step

__device__ __forceinline__ v8h as_v8h(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(v8h, (v4u){a, b, c, d});
}

// The lane's 8 codes of a chunk (bit pairs 0 and 1 of every byte of v) as f16
// bit patterns: 0x6400 | code is 1024 + code, and a code two bits up is
// 1024 + 4 code, which saves the shift (its q is divided by 4 instead).
__device__ __forceinline__ v8h codes_f16(uint32_t v, uint32_t e, uint32_t m0, uint32_t m1) {
    const uint32_t u = v >> 8;
    return as_v8h((v & m0) | e, (u & m0) | e, (v & m1) | e, (u & m1) | e);
}

// The 8 q that go with them (bytes of the position words of bit pairs 0 and 1)
// as f16 q and q / 4: the half 0x6400 + (q + 128) is 1152 + q
__device__ __forceinline__ v8h q_f16(uint32_t q0, uint32_t q1) {
    const uint32_t x0 = q0 ^ 0x80808080u, x1 = q1 ^ 0x80808080u, e = 0x64646464u;
    const v2h m = {(_Float16)-1152.0f, (_Float16)-1152.0f}, m4 = {(_Float16)-288.0f, (_Float16)-288.0f};
    const v2h r4 = {(_Float16)0.25f, (_Float16)0.25f};
    const v2h a = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(x0, e, 0x00060004u)) + m;
    const v2h b = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(x0, e, 0x00070005u)) + m;
    const v2h c = __builtin_elementwise_fma(__builtin_bit_cast(v2h, __builtin_amdgcn_perm(x1, e, 0x00060004u)), r4, m4);
    const v2h d = __builtin_elementwise_fma(__builtin_bit_cast(v2h, __builtin_amdgcn_perm(x1, e, 0x00070005u)), r4, m4);
    return as_v8h(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, c),
                  __builtin_bit_cast(uint32_t, d));
}

// 16 bytes a lane from a buffer to LDS (a function of its own: the host pass
// does not know the size 16 and drops a kernel template that names it)
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint8_t * to, uint32_t off, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)to, 16, off, soff, 0, 0);
}

template <int MI, int NI, bool SUM>
__global__ void __launch_bounds__(512)
gemm_mid_kernel(const uint8_t * __restrict__ W, const uint8_t * __restrict__ X, float * __restrict__ Y, int n_out,
                int n_tok, int nb, int tok_first, int tok_tiles) {
    constexpr int BM = 16 * MI, BN = 16 * NI;
    constexpr int WP = BM * 17, WL = (WP + 511) / 512;           // 16-byte pieces of a W step; DMAs per wave
    constexpr int SW = (WP + 63) / 64 * 1024;
    constexpr int RUN = BN * Q81_BYTES / 16;                     // pieces of a run
    constexpr int XP = 4 * RUN, XL = (XP + 63) / 64;             // pieces of a wave's X step; loads
    constexpr int SX = XL * 1024;
    constexpr int MAIN = 2 * SW + 8 * SX + 8 * BM * 4, RED = 8 * BM * BN * 4;
    __shared__ __attribute__((aligned(16))) uint8_t lds[MAIN > RED ? MAIN : RED];
    uint8_t * const sW = lds;                                    // [2][SW]
    uint8_t * const sX = lds + 2 * SW;                    // [8][SX]
    float * const sD = reinterpret_cast<float *>(lds + 2 * SW + 8 * SX);   // [8][BM]

    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // each XCD (workgroups go to them in turn) gets a contiguous run of tiles,
    // token tiles of one row tile next to each other: they share W in its L2
    const int total = gridDim.x, xcd = blockIdx.x & 7;
    const int tile = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
    const int row0 = tile / tok_tiles * BM, tok0 = tok_first + tile % tok_tiles * BN;

    const uint32_t rs = (uint32_t)PQ2_BYTES * nb;
    uint32_t w_off[WL];
#pragma unroll
    for (int k = 0; k < WL; ++k) {
        const int p = tid + 512 * k, row = min(p / 17, min(BM, n_out - row0) - 1);
        w_off[k] = row * rs + 16u * (uint32_t)(p % 17);
    }
    auto load_w = [&](int s) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rw =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(W) + (size_t)row0 * rs, 0, -1, 0x00020000);
#pragma unroll
        for (int k = 0; k < WL; ++k)
            if (512 * (k + 1) <= WP || 512 * k + 64 * wave < WP) dma16(rw, sW + (s & 1) * SW + 8192 * k + 1024 * wave, w_off[k], M_STEP * s);
    };
    uint32_t x_off[XL];
    const uint32_t run_bytes = (uint32_t)n_tok * Q81_BYTES;
#pragma unroll
    for (int k = 0; k < XL; ++k) {
        const int i = min(64 * k + lane, XP - 1);
        x_off[k] = (uint32_t)(i / RUN) * run_bytes + 16u * (uint32_t)(i % RUN);
    }
    const size_t x_all = (size_t)nb * 4 * run_bytes;
    v4u xr[XL];
    auto load_x = [&](int s) __attribute__((always_inline)) {
        // pieces past the last token run into the next chunk's blocks (their
        // columns are not stored), past X's end they read as zeros
        const size_t at = (size_t)(8 * s + wave) * 4 * run_bytes + (size_t)tok0 * Q81_BYTES;
        const size_t left = x_all - at;
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(X) + at, 0, (int)(left > 0xffffffffu ? 0xffffffffu : (uint32_t)left), 0x00020000);
#pragma unroll
        for (int k = 0; k < XL; ++k) xr[k] = __builtin_amdgcn_raw_buffer_load_b128(rx, x_off[k], 0, 0);
    };
    auto put_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < XL; ++k) *reinterpret_cast<v4u *>(sX + wave * SX + 1024 * k + 16 * lane) = xr[k];
    };

    v4f acc[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};

    auto compute = [&](int s) __attribute__((always_inline)) {
        const uint8_t * w = sW + (s & 1) * SW + PQ2_BYTES * wave;          // the wave's block of row 0
        // the block's scales, a row a lane (here to fp32 in LDS, below by groups
        // of 4 rows)
        float * const d = sD + wave * BM;
        uint32_t dr[(BM + 63) / 64];
#pragma unroll
        for (int r = 0; r < BM; r += 64)
            dr[r / 64] = *reinterpret_cast<const uint16_t *>(w + min(r + lane, BM - 1) * M_STEP);
        // codes: dword g / 2 of a chunk starts 2 bytes past a dword in even blocks
        const uint32_t sh = wave & 1 ? 0u : 2u;
        const uint8_t * wc = w + 2 - sh + l16 * M_STEP + 4 * (g >> 1);
        const uint32_t shift = 8 * sh + 4 * (g & 1);             // and bit pair 2 (g & 1) to the bottom
        // opaque, so that mask and exponent share one v_and_or (a VGPR and an SGPR)
        uint32_t ex = 0x64006400u, m0 = 0x00030003u, m1 = 0x000C000Cu;
        asm("" : "+v"(ex));
        asm("" : "+s"(m0), "+s"(m1));
        // f16 -1025 and -1028; with the stored sum taken off instead, -1024 for both
        const v8h fix = SUM ? as_v8h(0xE400E400u, 0xE400E400u, 0xE400E400u, 0xE400E400u)
                            : as_v8h(0xE401E401u, 0xE401E401u, 0xE404E404u, 0xE404E404u);
        v4f U[MI][NI];
        // software pipeline over i = (chunk, row tile): while tile i's MFMAs are
        // issued, products LAG MFMAs old are folded and tile i + 1's words read
        constexpr int LAG = 2, N = 4 * MI * NI;    // MFMA n = i * NI + ni, its product in S[n % (LAG + 1)]
        uint32_t wr[2][2], xw[NI][3];
        v8h Bf[NI];
        v4f E[NI];
        float da[2][NI];
        v4f S[LAG + 1];
        uint32_t wb[MI];                                         // LDS addresses of the row tiles, kept in registers
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
            wb[mi] = (uint32_t)(uintptr_t)(lds_void *)(wc + 16 * mi * M_STEP);
            asm("" : "+v"(wb[mi]));
        }
        auto read_w = [&](int i) __attribute__((always_inline)) {
            const auto * p = reinterpret_cast<const __attribute__((address_space(3))) uint32_t *>((uintptr_t)(wb[i % MI] + 8 * (i / MI)));
            wr[i & 1][0] = p[0];
            wr[i & 1][1] = p[1];
        };
        auto read_x = [&](int c) __attribute__((always_inline)) {
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                const uint32_t * x = reinterpret_cast<const uint32_t *>(sX + wave * SX + (c * BN + 16 * ni + l16) * Q81_BYTES);
                xw[ni][0] = x[0];
                xw[ni][1] = x[1 + 2 * g];
                xw[ni][2] = x[2 + 2 * g];
            }
        };
        auto fold = [&](int n) __attribute__((always_inline)) {
            const int ni = n % NI, mi = n / NI % MI, c = n / (NI * MI);
            const v4f & p = S[n % (LAG + 1)];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                U[mi][ni][k] = c == 0 ? da[0][ni] * p[k] : fmaf(da[c & 1][ni], p[k], U[mi][ni][k]);
            asm volatile("" : "+v"(U[mi][ni]));
        };
        read_x(0);
        read_w(0);
#pragma unroll
        for (int i = 0; i < 4 * MI; ++i) {
            const int mi = i % MI, c = i / MI;
            if (mi == 0) {
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
                    Bf[ni] = q_f16(xw[ni][1], xw[ni][2]);
                    da[c & 1][ni] = f16_bits_to_f32(xw[ni][0] & 0xffffu);
                    asm("" : "+v"(da[c & 1][ni]));              // fp32 from here on, not an f16 source of each FMA
                    const float ns = SUM ? (float)-((int)xw[ni][0] >> 16) : 0.0f;
                    E[ni] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fix, Bf[ni], (v4f){ns, ns, ns, ns}, 0, 0, 0);
                }
            }
            if (i == MI) {
#pragma unroll
                for (int r = 0; r < BM; r += 64)
                    if (r + lane < BM) d[r + lane] = f16_bits_to_f32(dr[r / 64]);
            }
            if (i + 1 < 4 * MI) read_w(i + 1);
            if (mi == (MI > 1 ? 1 : 0) && c < 3) read_x(c + 1);
            const v8h A = codes_f16(__builtin_amdgcn_alignbit(wr[i & 1][1], wr[i & 1][0], shift), ex, m0, m1);
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                const int n = i * NI + ni;
                S[n % (LAG + 1)] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, Bf[ni], E[ni], 0, 0, 0);
                if (n >= LAG) fold(n - LAG);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int n = N - LAG; n < N; ++n) fold(n);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
            const v4f dw = *reinterpret_cast<const v4f *>(d + 16 * mi + 4 * g);
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[mi][ni][i] = fmaf(dw[i], U[mi][ni][i], acc[mi][ni][i]);
        }
    };
    // every load of this wave landed, its X in LDS, then the barrier
    auto step_end = [&]() __attribute__((always_inline)) {
        put_x();
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    const int steps = nb / 8;
    load_w(0);
    load_x(0);
    step_end();
#pragma clang loop unroll(disable)
    for (int s = 0; s < steps; ++s) {
        if (s + 1 < steps) {
            load_w(s + 1);
            load_x(s + 1);
        }
        compute(s);
        step_end();
    }

    // the 8 partial tiles, [row][token] each
    float * const red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[wave * BM * BN + (16 * mi + 4 * g + i) * BN + 16 * ni + l16] = acc[mi][ni][i];
    __syncthreads();
#pragma unroll 2
    for (int o = tid; o < BM * BN; o += 512) {
        float y = red[o];
#pragma unroll
        for (int w = 1; w < 8; ++w) y += red[w * BM * BN + o];
        const int row = row0 + o / BN, tok = tok0 + o % BN;
        if (row < n_out && tok < n_tok) Y[(size_t)row * n_tok + tok] = y;
    }
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

template <int MI, int NI, bool SUM = false>
int launch_mid(const uint8_t * w, const uint8_t * x, float * Y, int64_t n_out, int64_t first, int64_t n_tok, int nb,
               hipStream_t st) {
    const int64_t R = cdiv(n_out, 16 * MI), T = cdiv(n_tok - first, 16 * NI);
    hipLaunchKernelGGL((gemm_mid_kernel<MI, NI, SUM>), dim3((unsigned)(R * T)), dim3(512), 0, st, w, x, Y, (int)n_out,
                       (int)n_tok, nb, (int)first, (int)T);
    return (int)hipGetLastError();
}

// Whole steps of 8 blocks, 16-byte DMA of W's rows, 32-bit offsets (80 rows of
// W, a block's 4 chunks of X), a grid of under 2^32 threads
bool mid_takes(const void * W, int64_t n_out, int64_t n_tok, int nb) {
    return nb % 8 == 0 && ((uintptr_t)W & 15u) == 0 && nb <= (1 << 20) && n_tok <= (1 << 24) &&
           cdiv(n_out, 32) * cdiv(n_tok, 16) <= (1 << 22);
}

int run_mid(const void * W, const void * Xq, float * Y, int64_t n_out, int64_t first, int64_t n_tok, int nb, int pick,
            hipStream_t st) {
    const uint8_t * w = (const uint8_t *)W, * x = (const uint8_t *)Xq;
    switch (pick) {
        case 0: return launch_mid<5, 3>(w, x, Y, n_out, first, n_tok, nb, st);
        case 1: return launch_mid<3, 2>(w, x, Y, n_out, first, n_tok, nb, st);
        case 2: return launch_mid<5, 2>(w, x, Y, n_out, first, n_tok, nb, st);
        case 3: return launch_mid<4, 2>(w, x, Y, n_out, first, n_tok, nb, st);
        case 4: return launch_mid<4, 3>(w, x, Y, n_out, first, n_tok, nb, st);
        case 5: return launch_mid<2, 2>(w, x, Y, n_out, first, n_tok, nb, st);
        case MID_SUM: return launch_mid<5, 1, true>(w, x, Y, n_out, first, n_tok, nb, st);
        case 7: return launch_mid<5, 1>(w, x, Y, n_out, first, n_tok, nb, st);
        default: return launch_mid<3, 1>(w, x, Y, n_out, first, n_tok, nb, st);
    }
}

}  // namespace

namespace pq2 {

// Y = W . X of up to 16 tokens where the kernel's requirements hold and it is
// the faster one; -1: nothing launched.  BONSAI_GEMM_MID: 0 never, 1..9 that tile
// shape, whatever the tokens (tests).
int gemm_mid(const void * W, const void * Xq, float * Y, int64_t n_out, int64_t n_tok, int nb, int cus, hipStream_t st) {
    const int forced = pq2host::knob(pq2host::K_GEMM_MID, -1);
    int pick = MID_SUM;
    if (forced > 0) {
        pick = (forced < MID_SHAPES ? forced : MID_SHAPES) - 1;
    } else if (forced == 0 || n_tok > 16 || nb < 40 || n_out <= 64 * (int64_t)cus ||
               cdiv(n_out, 80 * (int64_t)cus) * 64 * cus > n_out) {
        // 9 to 16 tokens on tall matrices.  The streamed kernel (gemm_small_kernel)
        // costs by the rows, about one unit for each 64 of a CU; the tiles here by
        // whole multiples of 80 rows a CU, each about that unit too (two workgroups
        // share a CU, the second adds what a further round would).  So the tiles are
        // taken where their multiples, rounded up, are no more than those units as a
        // fraction, past the first.  Measured on MI355X (256 CUs, us, streamed /
        // tiles, 9, 12, 16 tokens): 17408x5120 13.6 13.8 14.5 / 13.2 13.2 13.3, 20481
        // rows 14.9 14.8 15.8 / 18.1 18.1 18.0, 28000 19.5 19.9 21.4 / 19.8 19.8 20.1, 32768
        // 22.0 22.4 24.0 / 20.6 20.2 20.3, 40961 25.2 25.9 27.7 / 27.7 28.3 28.2, 49152
        // 28.4 28.4 30.4 / 28.8 28.8 29.1, 57344 34.6 35.7 38.7 / 30.3 30.3 30.1; 17408x8192
        // 21.2 21.8 23.8 / 19.8 19.8 19.8, 24576x8192 23.5 23.9 25.4 / 27.7 27.6 27.9.
        // Below 40 blocks 8 partial sums are further from 64 bits than that kernel's
        // 4 (3072 columns 6.6e-8 against 6.2e-8; at 5120 7.1e-8 against 7.2e-8).
        // More tokens: gemm_dispatch's plan.
        return -1;
    }
    if (!mid_takes(W, n_out, n_tok, nb)) return -1;
    return run_mid(W, Xq, Y, n_out, 0, n_tok, nb, pick, st);
}

// Whether the kernel's requirements hold for more than 16 tokens (and
// BONSAI_GEMM_MID does not decide)
bool gemm_mid_takes(const void * W, int64_t n_out, int64_t n_tok, int nb) {
    return pq2host::knob(pq2host::K_GEMM_MID, -1) < 0 && mid_takes(W, n_out, n_tok, nb);
}

// Tokens [first, n_tok) of the product (gemm_mid_takes it)
int gemm_mid_tail(const void * W, const void * Xq, float * Y, int64_t n_out, int64_t first, int64_t n_tok, int nb,
                  int cus, hipStream_t st) {
    float us = 0.0f;
    return run_mid(W, Xq, Y, n_out, first, n_tok, nb, mid_pick(n_out, n_tok - first, nb, cus, &us), st);
}

}  // namespace pq2
