/* r3d_prefill_f8.h -- the fp8a8 prefill's wide tile: 256 weight rows x 32 WMW tokens on eight
 * waves (4 along N x 2 along M, two a SIMD), a wave 4 weight fragments x WMW token fragments.
 *
 * Y[m, n] = sum_g (D_g[m, n] * sa[m, g]) * sb[n, g], D_g the e4m3 x e4m3 product of a 128-wide
 * K group: one v_mfma_scale_f32_16x16x128_f8f6f4 per 16 x 16 sub-tile and group, its result
 * flushed into the f32 accumulator three MFMAs later (src/r3d_gemm_fp8a8.hip:9-15).
 *
 * Why this tile.  An MFMA takes 32 cycles of its SIMD and a lone wave hides few of the flush's
 * VALU cycles behind its own MFMAs (47.6 cycles an MFMA with four multiply-adds beside it, 53
 * with eight; two waves: 39 and 50, measured in a bare loop), so the tile wants two waves a
 * SIMD -- and then the LDS is next: a wave reads 2 KB a fragment and step, so 4 x 4 fragments a
 * wave (128 x 256) read 1024 cycles and take 384 to fill against 1248 of matrix work, 4 x 8
 * (256 x 256) 1536 + 512 against 2496.  256 x 128 is for launches too small for that tile.
 *
 * A stage (a K group's 64 KB) leaves room for a ring of two only.  The weights of a stage are
 * in registers when its step begins (fragment ni of step s + 1 is read right after step s's
 * last MFMA on it), so two barriers a step free the ring in halves, and every load has one and
 * a half steps to land:
 *   mid  (group WMW/2 - 2)  the stage's weights, row scales and first-half activations are
 *                           read: stage s + 2's go out in their place; its second half is here;
 *   end  (group WMW - 2)    the rest is read: stage s + 2's token scales and second half go
 *                           out; stage s + 1's weights, scales and first half are here.
 * With one barrier and everything issued at it: 132 -> 100 us instead of 91 at M = 512,
 * N = 5376, K = 21504 on 256 x 128 (three chunks).  No branch may stand in the walk: a choice of
 * scale load by wave split its live ranges (230 registers spilled).
 *
 * Measured (us; before: 128 x 256 on four waves and 128 x 128, r3d_prefill.h):
 *   2048 x 21504 x 5376   128 x 128 blocks 283 -> 251, one scale a row 343 -> 258
 *                         (1.83 PFLOP/s), scales that vary along a row 353 -> 340
 *   512 x 5376 x 21504    (K split six ways, r3d_plan.cpp; with the planes' sum, 11 of it)
 *                         133 -> 89, 168 -> 94, 169 -> 120
 * At full load the clock gives way before anything else: the same walk with no loads and no
 * LDS reads at all (a variant, not kept) takes 1.83 us a step on 256 CUs and 1.15 on 42. */
#ifndef R3D_PREFILL_F8_H
#define R3D_PREFILL_F8_H

#include "r3d_device.h"
#include "r3d_prefill_layout.h"

namespace r3d {

/* How a tile's weight scales enter the flush: one bf16 a 128 x 128 block, folded into the
 * token's scale (acc += D * (sa * sb), one rounding off libref's order); one a row and group
 * (libref's order); or one a row for the whole walk (a per-channel checkpoint on the per-row
 * grid), applied once at its end: sum(D * sa) * sb, one multiply-add an element where the
 * per-row flush takes two and the unpacking of sb. */
enum { F8_BLOCK, F8_ROW, F8_CHAN };

struct F8Args {
    const uint8_t* A;
    const float* AS;
    const uint8_t* B;
    const uint16_t* BS;
    uint16_t* Y;
    int M, N;
    int64_t a_pitch, as_pitch, b_pitch, bs_pitch, y_pitch;
    float* part;                     /* this unit's f32 plane, or null: the whole walk into Y */
};

/* One tile at (n0, m0) over the groups [s0, s0 + steps).  F8_CHAN: false, and nothing written,
 * where some row's scale is not one finite value over them or a result is not finite. */
template <int WMW, int SC>
__device__ __forceinline__ bool prefill_f8_tile(const F8Args& P, uint8_t* smem, int64_t n0,
                                                int64_t m0, int s0, int steps) {
    using L = PrefillF8Layout<WMW>;
    constexpr int WNF = 4, RR = 4, LAG = 3, RB = SC == F8_BLOCK ? 128 : 1;
    constexpr bool gen = SC == F8_ROW;
    const uint8_t* const A = P.A;
    const float* const AS = P.AS;
    const uint8_t* const B = P.B;
    const uint16_t* const BS = P.BS;
    const int M = P.M, N = P.N;
    const int64_t a_pitch = P.a_pitch, as_pitch = P.as_pitch, b_pitch = P.b_pitch,
                  bs_pitch = P.bs_pitch, y_pitch = P.y_pitch;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, q = lane >> 4;
    const int wn = wave & 3, wm = wave >> 2;

    const int64_t k0 = 128 * (int64_t)s0;
    const __amdgpu_buffer_rsrc_t rB = r3d_rsrc(B + n0 * b_pitch + k0, (N - n0) * b_pitch - k0);
    const __amdgpu_buffer_rsrc_t rA = r3d_rsrc(A + m0 * a_pitch + k0, (M - m0) * a_pitch - k0);
    /* scales, 64 rows a wave: the weight rows' bf16 (of scale row n / RB) and the tokens' f32.
     * Waves w and w + 4 fetch the same ones: a choice by wave would be a branch, and branches
     * in the walk split every live range of it (230 registers spilled) */
    const int64_t sr0 = n0 / RB, srn = (N - 1) / RB + 1;
    const __amdgpu_buffer_rsrc_t rW = r3d_rsrc(BS + sr0 * bs_pitch + s0, (srn - sr0) * bs_pitch * 2 - 2 * s0);
    const __amdgpu_buffer_rsrc_t rT = r3d_rsrc(AS + m0 * as_pitch + s0, (M - m0) * as_pitch * 4 - 4 * s0);
    /* a 1 KB plane load: 16 rows x 64 bytes, four lanes a row, chunk swizzled by row / 2 % 4
     * (r3d_prefill.h) */
    const int lr = lane >> 2, lc = (lane & 3) ^ ((lr >> 1) & 3);
    uint32_t woff[L::WLD], aoff[L::ALD], wsoff, tsoff;
#pragma unroll
    for (int i = 0; i < L::WLD; ++i) {
        const int j = wave + 8 * i;
        int64_t n = n0 + 16 * (j >> 1) + lr;
        if (n > N - 1) n = N - 1;
        woff[i] = (uint32_t)((n - n0) * b_pitch + 64 * (j & 1) + 16 * lc);
    }
#pragma unroll
    for (int i = 0; i < L::ALD; ++i) {
        const int j = wave + 8 * i;
        const int f = j >> 1;                          /* fragment mi = f / 2 of half wm = f % 2 */
        int64_t m = m0 + 16 * ((f & 1) * WMW + (f >> 1)) + lr;
        if (m > M - 1) m = M - 1;
        aoff[i] = (uint32_t)((m - m0) * a_pitch + 64 * (j & 1) + 16 * lc);
    }
    {
        const int r0 = 64 * (wave & 3) + lane;
        int64_t n = n0 + r0, m = m0 + (r0 < L::BM ? r0 : L::BM - 1);
        if (n > N - 1) n = N - 1;
        if (m > M - 1) m = M - 1;
        wsoff = (uint32_t)((n / RB - sr0) * bs_pitch * 2);
        tsoff = (uint32_t)((m - m0) * as_pitch * 4);
    }
    /* the loads of a stage in their order: k = 0 the weight rows' scales, 1 .. WLD the weights,
     * then the activations' first half (MID loads so far), the tokens' scales, the second half */
    constexpr int WS = SC == F8_CHAN ? 0 : 1;          /* F8_CHAN reads its scales at the end */
    constexpr int LOADS = WS + L::WLD + L::ALD + 1, MID = WS + L::WLD + L::ALD / 2;
    auto load = [&](int k, int s, uint8_t* st) __attribute__((always_inline)) {
        const int sc = s < steps ? s : steps - 1;
        const int w = k - WS, i = w - L::WLD - (k < MID ? 0 : 1);
        if (k < WS)
            r3d_buf_lds<2>(rW, st + L::S + 256 * (wave & 3), wsoff, 2 * sc);
        else if (w < L::WLD)
            r3d_buf_lds<16>(rB, st + L::W + 1024 * (wave + 8 * w), woff[w], 128 * sc);
        else if (k == MID)
            r3d_buf_lds<4>(rT, st + L::AS + 256 * (wave & 3), tsoff, 4 * sc);
        else
            r3d_buf_lds<16>(rA, st + L::A + 1024 * (wave + 8 * i), aoff[i], 128 * sc);
    };
    auto issue = [&](int from, int to, int s, uint8_t* st) __attribute__((always_inline)) {
#pragma unroll
        for (int k = from; k < to; ++k) load(k, s, st);
    };

    r3d_f32x4 acc[WNF][WMW];
#pragma unroll
    for (int a = 0; a < WNF; ++a)
#pragma unroll
        for (int b = 0; b < WMW; ++b) acc[a][b] = r3d_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    r3d_i32x8 wF[WNF], ar[2];
    float af[2], sprev = 0.0f, sbv = 1.0f;
    r3d_f32x4 d[RR];
#pragma unroll
    for (int r = 0; r < RR; ++r) d[r] = r3d_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t sbP[WNF][2];                              /* general walk: the lane's row scales */
#pragma unroll
    for (int a = 0; a < WNF; ++a) sbP[a][0] = sbP[a][1] = 0u;
    const int rd = 16 * (4 * li + (q ^ ((li >> 1) & 3)));
    auto read_w = [&](const uint8_t* st, int ni) __attribute__((always_inline)) {
        const uint8_t* p = st + L::W + 2048 * (wn * WNF + ni) + rd;
        const r3d_i32x4 lo = *reinterpret_cast<const r3d_i32x4*>(p);
        const r3d_i32x4 hi = *reinterpret_cast<const r3d_i32x4*>(p + 1024);
        wF[ni] = r3d_i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto read_a = [&](const uint8_t* st, int mi) __attribute__((always_inline)) {
        const uint8_t* p = st + L::A + 2048 * (2 * mi + wm) + rd;
        const r3d_i32x4 lo = *reinterpret_cast<const r3d_i32x4*>(p);
        const r3d_i32x4 hi = *reinterpret_cast<const r3d_i32x4*>(p + 1024);
        ar[mi & 1] = r3d_i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        af[mi & 1] = *reinterpret_cast<const float*>(st + L::AS + 4 * (16 * (wm * WMW + mi) + li));
    };
    auto read_sb = [&](const uint8_t* st, int ni) __attribute__((always_inline)) {
        const r3d_i32x4 v = *reinterpret_cast<const r3d_i32x4*>(st + L::S + 4 * (16 * (wn * WNF + ni) + 4 * q));
        sbP[ni][0] = __builtin_amdgcn_perm((uint32_t)v[1], (uint32_t)v[0], 0x05040100u);
        sbP[ni][1] = __builtin_amdgcn_perm((uint32_t)v[3], (uint32_t)v[2], 0x05040100u);
    };
    /* the scale slot of one of the wave's 64 weight rows (a row a lane), bf16 bits */
    auto row_slot = [&](const uint8_t* st, int r) -> uint32_t {
        return *reinterpret_cast<const uint16_t*>(st + L::S + 4 * (64 * wn + r));
    };
    float sbn = 0.0f;                                  /* RB 128: the next step's block scale */

    auto flush = [&](int tt, int mi, float scur) __attribute__((always_inline)) {
        const int t2 = tt < 0 ? tt + WMW * WNF : tt;
        const int nf = t2 % WNF, mf = t2 / WNF;
        const float sv = tt >= 0 && mf == mi ? scur : sprev;
        const r3d_f32x4 v = d[t2 % RR];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (gen) {
                const uint32_t pw = sbP[nf][i >> 1];
                const float sb = __uint_as_float((i & 1) ? (pw & 0xFFFF0000u) : (pw << 16));
                acc[nf][mf][i] = acc[nf][mf][i] + (v[i] * sv) * sb;
            } else {
                acc[nf][mf][i] = __builtin_fmaf(v[i], sv, acc[nf][mf][i]);
            }
        }
    };
    auto step = [&](int s, uint8_t* cur, uint8_t* nxt) __attribute__((always_inline)) {
#pragma unroll
        for (int mi = 0; mi < WMW; ++mi) {
            const float scur = RB == 128 ? af[mi & 1] * sbv : af[mi & 1];
#pragma unroll
            for (int ni = 0; ni < WNF; ++ni) {
                const int tt = mi * WNF + ni;
                d[tt % RR] = r3d_mfma_fp8_fp8(wF[ni], ar[mi & 1]);
                if (mi == WMW - 1) read_w(nxt, ni);
                flush(tt - LAG, mi, scur);
                if (gen && tt < LAG) read_sb(cur, WNF - LAG + tt);   /* after its last use */
                if (gen && tt == WMW * WNF - 1) read_sb(nxt, 0);
            }
            sprev = scur;
            if (mi == WMW / 2 - 2) {
                /* mid: this stage's weights (in registers since the last step) and first-half
                 * activations are read, its second half has landed */
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LOADS) : "memory");
                issue(0, MID / 2, s + 2, cur);
                read_a(cur, mi + 2);
            } else if (mi + 2 == WMW) {
                /* end: the stage is read, the next one's scales, weights and first half are here */
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LOADS - 1) : "memory");
                issue(MID, LOADS, s + 2, cur);
                read_a(nxt, 0);
                if (RB == 128) sbn = __uint_as_float(row_slot(nxt, 0) << 16);
            } else if (mi + 2 < WMW) {
                if (mi == WMW / 2 - 1) issue(MID / 2, MID, s + 2, cur);
                read_a(cur, mi + 2);
            } else {
                read_a(nxt, 1);
                if (RB == 128) sbv = sbn;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    uint8_t* const r0 = smem;
    uint8_t* const r1 = smem + L::STAGE;
    /* F8_CHAN: is every row's scale one finite value over the unit's groups?  Two lanes a row,
     * each every other dword, 16 loads at once and ahead of the stages' so that their wait is not
     * the stages' (one at a time cost 15 us a tile).  A row may start or end inside a dword; its
     * other half, at the plane's ends two bytes outside the operand, is read with it (an aligned
     * dword lies in one page) and looked at by neither lane */
    uint32_t* const flag = reinterpret_cast<uint32_t*>(smem + L::LDS);
    constexpr int CB = 16;
    uint32_t cv[CB], c0 = 0;
    int odd = 0, nd = 0;
    const uint32_t* cd = nullptr;
    auto chan_load = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int i = i0 + 2 * j + (lane & 1);
            cv[j] = cd[i < nd ? i : nd - 1];
        }
    };
    if (SC == F8_CHAN) {
        int64_t n = n0 + 32 * wave + (lane >> 1);
        if (n > N - 1) n = N - 1;
        const uint16_t* row = BS + n * bs_pitch + s0;
        odd = (int)((uintptr_t)row >> 1) & 1;
        cd = reinterpret_cast<const uint32_t*>(row - odd);
        nd = (steps + odd + 1) >> 1;
        c0 = cd[0] >> (16 * odd) & 0xFFFFu;
        chan_load(0);
        __builtin_amdgcn_sched_barrier(0);
    }
    issue(0, LOADS, 0, r0);
    issue(0, MID, 1, r1);
    if (SC == F8_CHAN) {
        __builtin_amdgcn_sched_barrier(0);
        bool one = (c0 & 0x7F80u) != 0x7F80u;
        for (int i0 = 0;;) {
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                const int i = i0 + 2 * j + (lane & 1), e = 2 * (i < nd ? i : nd - 1);
                if (e >= odd && (cv[j] & 0xFFFFu) != c0) one = false;
                if (e + 1 < steps + odd && (cv[j] >> 16) != c0) one = false;
            }
            if ((i0 += 2 * CB) >= nd) break;
            chan_load(i0);
        }
        const uint32_t all = __all(one);
        if (lane == 0) flag[wave] = all;
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LOADS - 1) : "memory");
    if (SC == F8_CHAN) {
        uint32_t f = 1;
#pragma unroll
        for (int i = 0; i < 8; ++i) f &= flag[i];
        if (__builtin_amdgcn_readfirstlane(f) == 0) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            return false;
        }
    }
    issue(MID, LOADS, 1, r1);
#pragma unroll
    for (int ni = 0; ni < WNF; ++ni) read_w(r0, ni);
    read_a(r0, 0);
    read_a(r0, 1);
    if (RB == 128) sbv = __uint_as_float(row_slot(r0, 0) << 16);
    /* F8_ROW: the others stay zero until the first flushes, of empty results, are past */
    if (gen) read_sb(r0, 0);
    int s = 0;
    for (; s + 2 <= steps; s += 2) {
        step(s, r0, r1);
        step(s + 1, r1, r0);
    }
    if (s < steps) step(s, r0, r1);
#pragma unroll
    for (int tt = WMW * WNF - LAG; tt < WMW * WNF; ++tt) flush(tt, WMW - 1, sprev);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   /* drain the tail reloads */
#pragma unroll
    for (int ni = 0; ni < WNF; ++ni)
#pragma unroll
        for (int mi = 0; mi < WMW; ++mi) asm volatile("" : "+v"(acc[ni][mi]));
    if (SC == F8_CHAN) {
        /* sum(D * sa) leaves the f32 range before sum((D * sa) * sb) does where sb < 1, and a sum
         * that left it stays Inf or NaN: a tile with such a result takes the per-group walk.  The
         * largest magnitude, NaN above all, in half an instruction an element
         * (300 x 2050 x 8192 split 30.1 -> 30.6 us, 512 x 5376 x 21504 94.0 -> 94.8). */
        float big = 0.0f;
#pragma unroll
        for (int ni = 0; ni < WNF; ++ni)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t n = n0 + 16 * (wn * WNF + ni) + 4 * q + i;
                const float sb = __uint_as_float((uint32_t)BS[(n < N ? n : N - 1) * bs_pitch + s0] << 16);
#pragma unroll
                for (int mi = 0; mi < WMW; ++mi) acc[ni][mi][i] *= sb;
#pragma unroll
                for (int mi = 0; mi < WMW; mi += 2)
                    big = __builtin_elementwise_maximum(
                        __builtin_elementwise_maximum(fabsf(acc[ni][mi][i]), fabsf(acc[ni][mi + 1][i])), big);
            }
        const uint32_t fin = __all(big < __builtin_inff());
        if (lane == 0) flag[wave] = fin;
        __syncthreads();
        uint32_t f = 1;
#pragma unroll
        for (int i = 0; i < 8; ++i) f &= flag[i];
        if (__builtin_amdgcn_readfirstlane(f) == 0) return false;
    }

    uint16_t* const Y = P.Y;
    if (P.part) {
        float* const pp = P.part;
#pragma unroll
        for (int ni = 0; ni < WNF; ++ni)
#pragma unroll
            for (int mi = 0; mi < WMW; ++mi) {
                const int64_t m = m0 + 16 * (wm * WMW + mi) + li;
                const int64_t n = n0 + 16 * (wn * WNF + ni) + 4 * q;
                if (m >= M || n >= N) continue;
                const r3d_f32x4 v = acc[ni][mi];
                float* o = pp + m * N + n;
                if (n + 4 <= N) {
                    *reinterpret_cast<r3d_f32x4_u4*>(o) = v;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < N) o[i] = v[i];
                }
            }
        return true;
    }
    constexpr int YP = L::YP, CPR = L::BN / 8;
    __syncthreads();                                   /* every wave is done with the ring */
#pragma unroll
    for (int ni = 0; ni < WNF; ++ni)
#pragma unroll
        for (int mi = 0; mi < WMW; ++mi) {
            const int ml = 16 * (wm * WMW + mi) + li, nl = 16 * (wn * WNF + ni) + 4 * q;
            const r3d_f32x4 v = acc[ni][mi];
            *reinterpret_cast<uint2*>(smem + ml * YP + 2 * nl) =
                make_uint2(r3d_pack_bf16x2(v[0], v[1]), r3d_pack_bf16x2(v[2], v[3]));
        }
    __syncthreads();
    for (int e = threadIdx.x; e < L::BM * CPR; e += 512) {
        const int r = e / CPR, c = e - (e / CPR) * CPR;
        const int64_t m = m0 + r, n = n0 + 8 * c;
        if (m >= M || n >= N) continue;
        const r3d_i32x4 v = *reinterpret_cast<const r3d_i32x4*>(smem + r * YP + 16 * c);
        uint16_t* yp = Y + m * y_pitch + n;
        if (n + 8 <= N) {
            *reinterpret_cast<r3d_i32x4_u2*>(yp) = v;
        } else {
            const uint16_t* h = reinterpret_cast<const uint16_t*>(&v);
            for (int i = 0; i < 8; ++i)
                if (n + i < N) yp[i] = h[i];
        }
    }
    return true;
}

template <int WMW, int RB>
__global__ __launch_bounds__(512) void prefill_f8_kernel(F8Args P, int ksteps, int grid_m,
                                                         int tiles, int kc, int cst) {
    using L = PrefillF8Layout<WMW>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    /* units and tiles as in r3d_prefill.h: chunk u / tiles of tile u % tiles, a contiguous run
     * of units an XCD, tiles in groups of GN weight tiles, token tile major */
    const int bid = blockIdx.x;
    const int units = tiles * kc;
    const int per = units >> 3, rem = units & 7, x = bid & 7;
    const int u = x * per + (x < rem ? x : rem) + (bid >> 3);
    const int kci = u / tiles, t = u - kci * tiles;
    const int s0 = kci * cst;
    const int steps = ksteps - s0 < cst ? ksteps - s0 : cst;
    int tm, tn;
    {
        constexpr int GN = 8;
        const int grid_n = tiles / grid_m;
        const int grp = t / (GN * grid_m), in = t - grp * GN * grid_m, gn0 = grp * GN;
        const int gw = grid_n - gn0 < GN ? grid_n - gn0 : GN;
        tm = in / gw;
        tn = gn0 + (in - tm * gw);
    }
    const int64_t n0 = (int64_t)tn * L::BN, m0 = (int64_t)tm * L::BM;
    if (P.part) P.part += (int64_t)kci * P.M * P.N;
    if (RB == 128) {
        prefill_f8_tile<WMW, F8_BLOCK>(P, smem, n0, m0, s0, steps);
    } else if (!prefill_f8_tile<WMW, F8_CHAN>(P, smem, n0, m0, s0, steps)) {
        __syncthreads();
        prefill_f8_tile<WMW, F8_ROW>(P, smem, n0, m0, s0, steps);
    }
}

}  // namespace r3d

#endif /* R3D_PREFILL_F8_H */
