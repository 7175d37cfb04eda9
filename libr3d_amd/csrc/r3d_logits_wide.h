/* r3d_logits_wide.h -- logits_gemm_e4m3 for 9 and more activation rows: up to 64 of them
 * against one pass over the head (the 4-row walk of r3d_logits.hip takes 8 a pass).
 *
 * A workgroup of 8 waves owns blocks of 128 TW head rows (a wave TW tiles of 16), each over
 * the whole of K in 256-wide windows, as one stream of windows across its blocks.  The codes
 * arrive in whole 128-byte lines straight into registers, one window ahead (two loads per
 * 16 rows x 128 bytes, rows 0-7 and 8-15, eight lanes a line, put in operand order through 2 KB
 * of the wave's LDS, r3d_lines_turn; a load of a row a lane with the shuffle in registers takes
 * 242 us where this takes 228): lane 16 kb + p then holds head row p's 16-byte chunks kb and
 * 4 + kb of a line -- one 128-wide scale block -- which widen exactly to the operands of four
 * v_mfma_f32_16x16x32_bf16.  All 16 columns of the MFMA are activation rows, against the 4 of
 * 16 products that the 4-row walk uses.  A window's activation rows (16 NTG of them, zero past
 * M and past K) sit in LDS, double-buffered, XOR-swizzled by row so that eight lanes reading
 * one chunk of eight rows hit distinct banks; they are fetched two windows ahead, so that the
 * fetch never waits behind the codes.  The block sum is scaled once, tot = fma(scale, block,
 * tot), as in the 4-row walk; each wave keeps its rows' scales of two windows in an LDS table.
 *
 * Bound: the head's bytes from HBM.  262144 x 5376 (1.43 GB), bf16 scale per row x 128, us:
 *
 *   M                                     16    32    64
 *   8-row passes                         475   949  1899
 *   a row a lane, TW = 1                 260   290   371
 *   a row a lane, TW = 2                 243   259   321
 *   this walk (eight lanes a line), TW 2 228   243   316
 *
 * TW = 1 restages the activation rows twice as often per head row but balances twice as
 * finely over the workgroups (151936 x 4096, M = 16: 132 against 146 us with a row a lane, 122
 * now; 32000 x 4096: 31 against 42); logits_wide_tiles picks.  Measured without gain: three windows of codes in
 * flight (TW = 1: 262 us), four waves a workgroup (293), sixteen (spills). */
#ifndef R3D_LOGITS_WIDE_H
#define R3D_LOGITS_WIDE_H

#include "r3d_gemv_lines.h"
#include "r3d_logits_device.h"

namespace r3d {

template <int NTG, int TW, int SDT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
void logits_wide_kernel(
    const uint16_t* __restrict__ X, int64_t x_pitch, const uint8_t* __restrict__ codes,
    const uint8_t* __restrict__ scale, int64_t s_pitch, int64_t s_bytes, int br,
    float* __restrict__ Y, int64_t y_pitch, int N, int K, int M, int nwin, LogitsGuard guard) {
    constexpr int ESZ = SDT == 2 ? 4 : 2;
    constexpr int RB = 128 * TW;                      /* head rows a block */
    static_assert(TW <= 2, "one scale load covers a window's tiles");
    extern __shared__ __align__(16) uint8_t lg_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63, p = l & 15, kb = l >> 4;
    const int mb = blockIdx.y * 64;
    const int live = M - mb < 16 * NTG ? M - mb : 16 * NTG;
    const int blocks = (N + RB - 1) / RB;

    if (!lg_header_ok(guard)) {                       /* the head changed under the plan */
        for (int b = blockIdx.x; b < blocks; b += gridDim.x)
            for (int i = threadIdx.x; i < RB * live; i += 512) {
                const int n = b * RB + i % RB;
                if (n < N) Y[(int64_t)(mb + i / RB) * y_pitch + n] = __builtin_nanf("");
            }
        return;
    }
    const int nw = (K + 255) / 256;
    float* tab = reinterpret_cast<float*>(lg_lds + 2 * 8192 * NTG) + wave * 128;
    const __amdgpu_buffer_rsrc_t rs = r3d_rsrc(scale, s_bytes);
    const __amdgpu_buffer_rsrc_t rx =
        r3d_rsrc(X + (int64_t)mb * x_pitch, ((live - 1) * x_pitch + K) * 2);
    /* staging: thread t brings columns 8 (t % 32) .. + 8 of row t / 32 of each group */
    const int sr = threadIdx.x >> 5, sk = threadIdx.x & 31;
    const int sdst = 512 * sr + 16 * (sk ^ (sr & 7));
    /* B operands: chunk kb of a line, halves 0 and 1, of row p; chunk 4 + kb is eight 16-byte
     * units on (the swizzle moves the low three bits only) */
    const int x0 = 512 * p + 16 * ((2 * kb) ^ (p & 7)), x1 = x0 ^ 16;
    /* codes: a load's row and chunk of this lane, and their turn into operands */
    const int lr = l >> 3, lc8 = l & 7;
    uint8_t* const turn = lg_lds + 2 * 8192 * NTG + 8 * 2 * 256 + kLinesTurn * wave;
    const int twr = 128 * lr + 16 * (lc8 ^ lr), trd = 128 * p + 16 * (kb ^ (p & 7));

    const int nb = (blocks - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    auto row0 = [&](int bi) -> int64_t {              /* past the last block: rows past N */
        return bi < nb ? ((int64_t)blockIdx.x + (int64_t)bi * gridDim.x) * RB + wave * (16 * TW)
                       : (int64_t)N;
    };
    /* cursors over the workgroup's stream of windows (nw a block): x and scales two ahead,
     * codes one */
    struct Cur { int bi, w; };
    auto step = [&](Cur& c) __attribute__((always_inline)) {
        if (++c.w == nw) { c.w = 0; ++c.bi; }
    };
    r3d_i32x4 xr[2][NTG];
    auto load_x = [&](Cur& c, int buf) __attribute__((always_inline)) {
        const int k = 256 * c.w + 8 * sk;
#pragma unroll
        for (int g = 0; g < NTG; ++g) {
            const int m = 16 * g + sr;
            const uint32_t o = m < live && k < K ? (uint32_t)((m * x_pitch + k) * 2) : kLgOob;
            xr[buf][g] = __builtin_bit_cast(
                r3d_i32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)o, 0, 0));
        }
    };
    auto put_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < NTG; ++g)
            *reinterpret_cast<r3d_i32x4*>(lg_lds + 8192 * (buf * NTG + g) + sdst) = xr[buf][g];
    };
    /* lane 16 kb + p brings the scale of tile kb / 2, row p, the window's block kb % 2 */
    float sv[2];
    auto load_s = [&](Cur& c, int buf) __attribute__((always_inline)) {
        const int blk = 2 * c.w + (kb & 1);
        const int64_t row = row0(c.bi) + 16 * (kb >> 1) + p;
        sv[buf] = lg_scale<SDT>(rs, kb < 2 * TW && row < N && blk < nwin
                                        ? (uint32_t)(((row / br) * s_pitch + blk) * ESZ)
                                        : kLgOob);
    };
    r3d_i32x4 cw[2][TW][4];                           /* [window % 2][tile][line, rows half] */
    auto load_c = [&](Cur& c, int buf) __attribute__((always_inline)) {
        const int64_t n0 = row0(c.bi);
        const int64_t rows = N - n0 < 16 * TW ? (N - n0 > 0 ? N - n0 : 0) : 16 * TW;
        const __amdgpu_buffer_rsrc_t rc = r3d_rsrc(codes + (rows ? n0 : 0) * K, rows * K);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ka = 256 * c.w + 128 * j + 16 * lc8;
#pragma unroll
            for (int t = 0; t < TW; ++t) {
                cw[buf][t][2 * j] = r3d_buf_ld16_stream(
                    rc, ka < K ? (uint32_t)((16 * t + lr) * K + ka) : kLgOob);
                cw[buf][t][2 * j + 1] = r3d_buf_ld16_stream(
                    rc, ka < K ? (uint32_t)((16 * t + 8 + lr) * K + ka) : kLgOob);
            }
        }
    };
    /* even and odd blocks of K apart: with one sum of all 42 the error against 64 bits at
     * K = 5376 was 1.21e-7, over the 4-row walk's 0.95e-7; with two it is 0.93e-7 */
    r3d_f32x4 tot[2][TW][NTG];
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int g = 0; g < NTG; ++g) tot[0][t][g] = tot[1][t][g] = r3d_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto consume = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            r3d_i32x4 v[TW][2];
#pragma unroll
            for (int t = 0; t < TW; ++t)
                r3d_lines_turn(turn, twr, trd, cw[buf][t][2 * j], cw[buf][t][2 * j + 1], v[t][0], v[t][1]);
            r3d_f32x4 blk[TW][NTG];
#pragma unroll
            for (int t = 0; t < TW; ++t)
#pragma unroll
                for (int g = 0; g < NTG; ++g) blk[t][g] = r3d_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int c = 0; c < 4; ++c) {             /* 8 columns a lane: chunk c / 2, half c % 2 */
                lg_bf16x8 wv[TW];
#pragma unroll
                for (int t = 0; t < TW; ++t)
                    wv[t] = lg_codes8(v[t][c >> 1][2 * (c & 1)], v[t][c >> 1][2 * (c & 1) + 1]);
                const uint8_t* xb = lg_lds + 8192 * NTG * buf + 256 * j + 128 * (c >> 1) +
                                    ((c & 1) ? x1 : x0);
#pragma unroll
                for (int g = 0; g < NTG; ++g) {
                    const lg_bf16x8 bv = *reinterpret_cast<const lg_bf16x8*>(xb + 8192 * g);
#pragma unroll
                    for (int t = 0; t < TW; ++t)
                        blk[t][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[t], bv, blk[t][g], 0, 0, 0);
                }
            }
#pragma unroll
            for (int t = 0; t < TW; ++t) {
                const r3d_f32x4 sc = *reinterpret_cast<const r3d_f32x4*>(
                    tab + 64 * buf + 32 * t + 16 * j + 4 * kb);
#pragma unroll
                for (int g = 0; g < NTG; ++g)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        tot[j][t][g][i] = fmaf(sc[i], blk[t][g][i], tot[j][t][g][i]);
            }
            if (j == 0) __builtin_amdgcn_sched_barrier(0);
        }
    };
    const bool v4 = ((uintptr_t)Y & 15) == 0 && (y_pitch & 3) == 0;
    auto store = [&](int bi) __attribute__((always_inline)) {
        const int64_t n0 = row0(bi);
        /* every accumulator complete in every lane before the lane-divergent stores */
        r3d_f32x4 o[TW][NTG];
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int g = 0; g < NTG; ++g) {
                o[t][g] = tot[0][t][g] + tot[1][t][g];
                tot[0][t][g] = tot[1][t][g] = r3d_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                asm volatile("" : "+v"(o[t][g]));
            }
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int g = 0; g < NTG; ++g) {
                const int m = 16 * g + p;
                const int64_t n = n0 + 16 * t + 4 * kb;
                if (m < live && n < N) {
                    float* yp = Y + (int64_t)(mb + m) * y_pitch + n;
                    if (v4 && n + 4 <= N) {
                        *reinterpret_cast<r3d_f32x4*>(yp) = o[t][g];
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (n + i < N) yp[i] = o[t][g][i];
                    }
                }
            }
    };

    Cur at{0, 0}, lx{0, 0}, ls{0, 0}, lc{0, 0};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        load_x(lx, i);
        load_s(ls, i);
        step(lx);
        step(ls);
    }
    load_c(lc, 0);
    step(lc);
    __builtin_amdgcn_sched_barrier(0);
    put_x(0);
    tab[l] = sv[0];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int total = nb * nw;
    for (int t = 0; t < total; t += 2) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            if (t + b >= total) break;
            load_x(lx, b);                            /* window t + b + 2, into the registers of t + b */
            load_s(ls, b);
            load_c(lc, b ^ 1);
            step(lx);
            step(ls);
            step(lc);
            __builtin_amdgcn_sched_barrier(0);
            consume(b);
            __builtin_amdgcn_sched_barrier(0);
            put_x(b ^ 1);                             /* window t + b + 1 */
            tab[64 * (b ^ 1) + l] = sv[b ^ 1];
            /* the other buffers were last read before the barrier that ended the window before */
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            const int bi = at.bi;
            step(at);
            if (at.w == 0) store(bi);
        }
    }
}

}  // namespace r3d

#endif /* R3D_LOGITS_WIDE_H */
