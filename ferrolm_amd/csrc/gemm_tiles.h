// The tiled GEMM of batched verify steps and prompt chunks (MM activations:
// two bf16 pieces per value, internal.h): v_mfma_f32_16x16x32_bf16 on operand
// tiles in the layouts the producers and the upload wrote them in, so nothing
// is rearranged on the way.
//
// A workgroup of NWN x NWK waves owns 16 RT rows x 64 NWN columns. Its activation
// blocks (1 KB each: one row tile, k-block and piece, in the lanes' order) are
// copied straight to LDS (global_load_lds_dwordx4) one stage ahead; a stage is a
// pair of k-blocks for each of the NWK shares of K. A wave owns 64 columns of one
// share: it alone loads and converts its weights, in registers, so every weight is
// converted once per workgroup and serves RT row tiles, and the activations are read
// from LDS by NWN waves. The K shares' sums meet in LDS, each share finishing some of
// the row tiles, and the epilogues run on a wave's own 16 x 64 tiles, without barriers.
//
// Bound: the issue of a SIMD's matrix and vector instructions, and on tiles of few rows what a stage
// costs whatever its rows. The group scale is applied to every k-block's product (four FMAs for every
// two MFMAs) and a weight's conversion takes about 1.7 operations; measured alone, an MFMA of 16 x 16 x
// 32 and two FMAs take 20 cycles with two waves per SIMD, 16 without the FMAs. So a step's MFMAs, FMAs,
// conversions and copies are interleaved by hand and two waves share each SIMD. A row tile of a stage is
// then 0.21 us of MFMA issue, 0.27 with the FMAs; the four-share tiles take 0.35 us for each row tile and
// 0.27 (bf16), 0.46 (int8) or 0.58 us (int4) besides (launch_mm's costs): a stage opens with a wait for
// every load in flight and a barrier, and with two to five row tiles little is left to cover them.
// Whole products of int4 weights, the packing of their inputs included, k_gemm -> here: 1024 rows, 16384
// x 2048 217 -> 153 us, 6144 x 2048 95 -> 77, 2048 x 8192 134 -> 96, 28672 x 4096 677 -> 458; of 28672 x
// 4096, 80 rows 60 -> 52, 160 rows 115 -> 92 us. Three stages in LDS with one workgroup per CU were no
// faster for single tiles and slower for full ones (16384 x 2048 158 us for the product alone, 137 with two).
#pragma once
#include "devutil.h"

#include <hip/hip_ext.h>


namespace fg {

// bytes b, b+1 of w (two's-complement int8) as two bf16, exactly
__device__ __forceinline__ uint32_t codes_bf16(uint32_t w, int b) {
    const float f0 = (float)(int8_t)(w >> (8 * b)), f1 = (float)(int8_t)(w >> (8 * b + 8));
    return __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
}

// 1 KB per wave from global memory (base uniform, off the lane's byte) to LDS byte `lds` + 16 lane.
// The compiler does not see the write: the kernel waits (vmcnt) and meets at a barrier itself. M0
// holds the LDS address.
__device__ __forceinline__ void copy_to_lds(uint32_t lds, const uint8_t* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
                 : "m0", "memory");
}

// The epilogues (internal.h) on one wave's 16 x 64 tile d (D layout), row tile rt, columns from
// col0, through its own LDS rows lw; rs: 1/rms of the tile's rows. Lane l finishes row l / 4,
// columns 16 (l % 4) .. + 15 (SILU: channels 8 (l % 4) .. + 7). No barrier: only this wave's data.
template <int EPI>
__device__ __forceinline__ void wave_epilogue(const GemvArgs& a, const f32x4 (&d)[4], int rt, int col0, float* lw,
                                              const float* rs, int lane) {
    constexpr int YS = 68;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) lw[(4 * (lane >> 4) + r) * YS + t * 16 + (lane & 15)] = d[t][r];
    const int rr = lane >> 2, q4 = lane & 3, row = rt * 16 + rr, tile = col0 / 64;
    const bool live = row < a.m;
    const float* y = lw + rr * YS;
    if (EPI == EPI_SILU) {
        const int c = q4 * 8, b = c / a.il, j = c % a.il;
        const float* g = y + b * 2 * a.il + j;
        const float r = rs[rr];
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float gt = g[e] * r, up = g[a.il + e] * r;
            v[e] = live ? gt / (1.0f + dev_exp(-gt)) * up : 0.0f;
        }
        if (a.cap && live)
#pragma unroll
            for (int e = 0; e < 8; e++) a.cap[(size_t)row * a.ldcap + tile * 32 + c + e] = v[e];
        if (live && a.pa) {
            const int prt = (a.pa_passes + 3) >> 2;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                u16x8 o;
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = (uint16_t)bf16_piece(v[e], h);
                ((u16x8*)a.pa)[(((size_t)tile * prt + rt) * 2 + h) * 64 + q4 * 16 + rr] = o;
            }
        }
    } else {
        const int col = col0 + q4 * 16;
        const bool in = live && col < a.N;
        float v[16];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const f32x4 f = *(const f32x4*)(y + q4 * 16 + 4 * e);
#pragma unroll
            for (int i = 0; i < 4; i++) v[4 * e + i] = f[i];
        }
        if (EPI == EPI_STORE || EPI == EPI_QKV) {
            if (in) {
                const float r = EPI == EPI_QKV ? rs[rr] : 1.0f;
                float* o = a.out + (size_t)row * a.ldo + col;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    if (EPI == EPI_QKV) v[e] *= r;
                    if (a.bias) v[e] += a.bias[col + e];
                }
                if (EPI == EPI_STORE && ((size_t)a.out & 15)) {  // a caller's buffer may be aligned to a float only
#pragma unroll
                    for (int e = 0; e < 16; e++) o[e] = v[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        *(float4*)(o + 4 * e) = make_float4(v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]);
                }
            }
        } else if (EPI == EPI_ARGMAX) {
            const float r = rs[rr];
            float bv = -INFINITY;
            int bi = 0;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                v[e] *= r;
                const float c = v[e] != v[e] ? -INFINITY : v[e];
                if (e == 0 || c > bv) {
                    bv = c;
                    bi = e;
                }
            }
            if (in && a.logits) {
                float* o = a.logits + (size_t)row * a.N + col;
#pragma unroll
                for (int e = 0; e < 4; e++) *(float4*)(o + 4 * e) = make_float4(v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]);
            }
            // (max, first index) of the 32-column tile: its other half sits in lane ^ 1
            bi += (q4 & 1) * 16;
            const float ov = lane_xor1(bv);
            const int oi = __float_as_int(lane_xor1(__int_as_float(bi)));
            if (q4 & 1 ? ov >= bv : ov > bv) {
                bv = ov;
                bi = oi;
            }
            if (in && !(q4 & 1))
                a.best[(size_t)(col >> 5) * a.m + row] = make_float2(bv, __int_as_float((col & ~31) + bi));
        } else {  // EPI_RESID
            float ssq = 0.0f;
            float* x = a.x + (size_t)row * a.ldx + col;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float4 xo = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (in) xo = *(const float4*)(x + 4 * e);
                v[4 * e] = in ? xo.x + v[4 * e] : 0.0f;
                v[4 * e + 1] = in ? xo.y + v[4 * e + 1] : 0.0f;
                v[4 * e + 2] = in ? xo.z + v[4 * e + 2] : 0.0f;
                v[4 * e + 3] = in ? xo.w + v[4 * e + 3] : 0.0f;
            }
#pragma unroll
            for (int e = 0; e < 16; e++) ssq = fmaf(v[e], v[e], ssq);
            if (in)
#pragma unroll
                for (int e = 0; e < 4; e++) *(float4*)(x + 4 * e) = make_float4(v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]);
            ssq = group_reduce<4, false>(ssq);
            if (q4 == 0 && live) a.ss_out[(size_t)tile * a.ss_m + row] = ssq;
            if (live && a.pa) {
                const int prt = (a.pa_passes + 3) >> 2;
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const int q8 = q4 * 2 + s, kb = col0 / 32 + q8 / 4;
                    if (col + 8 * s >= a.N) continue;
                    float w[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) w[e] = a.g_next ? a.g_next[col + 8 * s + e] * v[8 * s + e] : v[8 * s + e];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        u16x8 o;
#pragma unroll
                        for (int e = 0; e < 8; e++) o[e] = (uint16_t)bf16_piece(w[e], h);
                        ((u16x8*)a.pa)[(((size_t)kb * prt + rt) * 2 + h) * 64 + (q8 & 3) * 16 + rr] = o;
                    }
                }
            }
        }
    }
    // the consumer's zero padding past the last k-block, by the wave of the last columns
    if ((EPI == EPI_SILU || EPI == EPI_RESID) && a.pa && live && col0 + 64 >= a.N) {
        const int prt = (a.pa_passes + 3) >> 2, covered = EPI == EPI_RESID ? (a.N + 31) / 32 : (a.N + 63) / 64;
        const u16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int kb = covered; kb < a.pa_kb; kb++)
#pragma unroll
            for (int h = 0; h < 2; h++) ((u16x8*)a.pa)[(((size_t)kb * prt + rt) * 2 + h) * 64 + q4 * 16 + rr] = z;
    }
}

// Holds a value's place in the program order (no instruction)
template <class T>
__device__ __forceinline__ void pin(T& v) {
    asm volatile("" : "+v"(v));
}

template <int KIND, int EPI, int RT, int NWN, int NWK>
__global__ __launch_bounds__(64 * NWN * NWK, 2) void k_mm(const GemvArgs a) {
    constexpr bool Q = KIND != BF16;
    constexpr bool NEED_R = EPI == EPI_QKV || EPI == EPI_SILU || EPI == EPI_ARGMAX;
    constexpr int NW = NWN * NWK, NTHR = 64 * NW, BN = 64 * NWN;
    constexpr int STAGE = NWK * RT * 4 * 1024;   // bytes of a stage's activations
    constexpr int NA = NWK * RT * 4 / NW;        // 1 KB blocks of a stage that each wave copies
    static_assert(NA * NW == NWK * RT * 4, "the blocks of a stage divide among the waves");
    constexpr int YS = 68, EPW = 16 * YS * 4;    // a wave's epilogue rows
    constexpr int XCH = NWN * RT * (NWK - 1) * 4 * 1024;  // the K shares' exchange
    constexpr int FIN = (XCH > NW * EPW ? XCH : NW * EPW);
    constexpr int LDS = (2 * STAGE > FIN + RT * 64 ? 2 * STAGE : FIN + RT * 64);
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
    __shared__ __align__(1024) uint8_t smem[LDS];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % NWN, kw = wave / NWN;
    const int RTt = (a.p_total + 3) >> 2, groups = (RTt + RT - 1) / RT, cg = (a.N + BN - 1) / BN;
    // Workgroup i runs on XCD i % 8: an XCD takes whole column groups, its row groups one after the
    // other, so a column group's weights are read from memory once and then from that XCD's L2. Where
    // the column groups are not a multiple of eight it takes an eighth of the tiles in that order (bf16
    // 3584 x 3584, 272 rows: 41.2 -> 28.8 us; taking them so everywhere made int8 49152 x 576 3% slower).
    int cgi, gi;
    if (cg % 8 == 0) {
        const int y = blockIdx.x / 8;
        cgi = (int)(blockIdx.x % 8) + 8 * (y / groups);
        gi = y % groups;
    } else {
        const int tiles = cg * groups, xcd = blockIdx.x % 8;
        const int at = xcd * (tiles / 8) + min(xcd, tiles % 8) + (int)(blockIdx.x / 8);
        cgi = at / groups;
        gi = at % groups;
    }
    const int rt0 = gi * RT, col0 = cgi * BN + wn * 64, ntl = a.N >> 4, KB = a.KB, KC = KB >> 2;
    // n-tiles past the end re-read the last one (their results are discarded)
    int tl[4];
#pragma unroll
    for (int t = 0; t < 4; t++) tl[t] = min((col0 >> 4) + t, ntl - 1);
    // the k-block pairs, in stages of NWK; in a last stage that is not full the shares past the end
    // have nothing to add (their loads and copies take the last pair again)
    const int NP = KB >> 1, ns = (NP + NWK - 1) / NWK;

    // block q of the wave's share of stage s, into buffer s & 1
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)smem;
    auto copy_block = [&](int s, int q) {
        const int b = wave * NA + q, kbl = b / (2 * RT), rem = b % (2 * RT);
        const int kb = min(2 * s * NWK + kbl, 2 * NP - 2 + (kbl & 1)), i = min(rt0 + (rem >> 1), RTt - 1);
        copy_to_lds(lds0 + (s & 1) * STAGE + b * 1024, a.XA + (((size_t)kb * RTt + i) * 2 + (rem & 1)) * 1024, lane * 16);
    };
    // The wave's weights of a pair of k-blocks as stored (BF16: the operands), and their scales
    struct Raw {
        u32x4 w[KIND == BF16 ? 8 : 4];
    };
    struct Scales {
        f32x2 v[4];
    };
    auto load_weights = [&](int s, Raw& r) {
        const int pr = min(s * NWK + kw, NP - 1), c = pr >> 1, half = pr & 1;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const size_t tile = tl[t];
            if (KIND == INT4) {
                const u32x2 v = *((const u32x2*)a.W + ((tile * KC + c) * 64 + lane) * 2 + half);
                r.w[t][0] = v[0];
                r.w[t][1] = v[1];
            } else if (KIND == INT8) {
                r.w[t] = *((const u32x4*)a.W + (tile * (KB >> 1) + pr) * 64 + lane);
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++)
                    r.w[2 * t + j] = *((const u32x4*)a.W + (tile * KB + 2 * pr + j) * 64 + lane);
            }
        }
    };
    auto load_scales = [&](int s, Scales& sc) {
        const int pr = min(s * NWK + kw, NP - 1), c = pr >> 1, half = pr & 1;
        if (Q)
#pragma unroll
            for (int t = 0; t < 4; t++)
                sc.v[t] = *((const f32x2*)a.S + (((size_t)tl[t] * KC + c) * 16 + (lane & 15)) * 2 + half);
    };
    // the operands of k-block j, [n-tile][word of two inputs]; word w (of 16) converted
    u32x4 B[2][4];
    auto convert = [&](const Raw& r, int j, int w) {
        const int t = w >> 2, q = w & 3;
        if (KIND == INT4) {
            const uint32_t c = r.w[t][j];
            B[j][t][q] = codes_bf16(q < 2 ? (c << 4) & 0xF0F0F0F0u : c & 0xF0F0F0F0u, 2 * (q & 1));
        } else if (KIND == INT8) {
            B[j][t][q] = codes_bf16(r.w[t][2 * j + (q >> 1)], 2 * (q & 1));
        }
    };

    f32x4 acc[RT][4];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[i][t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    const f32x4 fzero = {0.0f, 0.0f, 0.0f, 0.0f};

    // One stage: two k-blocks of RT row tiles, 16 RT MFMAs, as 4 RT half-steps of four (two n-tiles,
    // hi then lo). The order is written out: beside each MFMA, which holds the matrix pipe for 16
    // cycles, go two FMAs of the half-step before (its products scaled and added), the conversion of
    // the next k-block's weights, and the next step's activations from LDS. cur: this stage's weights
    // (k-block 1 is converted during k-block 0, then the stage after next is loaded there); next: the
    // next stage's (k-block 0 is converted during k-block 1).
    auto stage = [&](int s, Raw& cur, Raw& next, const Scales& sc, Scales& scn) {
        // stage s has landed, here and in every wave, and every wave is done with the other buffer
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        // (a product with a zero scale would not be zero where it has overflowed)
        if (NWK > 1 && s * NWK + kw >= NP) return;
        if (KIND == BF16) load_weights(s + 1, next);
        load_scales(s + 1, scn);
        const bf16x8* st = (const bf16x8*)(smem + (s & 1) * STAGE + kw * (4 * RT * 1024)) + lane;
        bf16x8 ah = st[0], al = st[64];
        f32x4 dp[2] = {fzero, fzero};
        constexpr int WP = (16 + 2 * RT - 1) / (2 * RT);  // words converted per half-step
#pragma unroll
        for (int n = 0; n < 2 * RT; n++) {
            const int i = n % RT, j = n / RT;
            if (KIND != BF16 && n == RT) load_weights(s + 2, cur);
            // the next stage's copies, spread over the first k-block's steps
            constexpr int PER = (NA + RT - 1) / RT;
            if (s + 1 < ns)
#pragma unroll
                for (int q = n * PER; q < n * PER + PER && q < NA; q++) copy_block(s + 1, q);
            bf16x8 nh = ah, nl = al;
            if (n + 1 < 2 * RT) {
                nh = st[(n + 1) * 128];
                nl = st[(n + 1) * 128 + 64];
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int t0 = 2 * h, t1 = t0 + 1;
                bf16x8 b0, b1;
                if (Q) {
                    b0 = as_bf16x8(B[j][t0]);
                    b1 = as_bf16x8(B[j][t1]);
                } else {
                    b0 = as_bf16x8(cur.w[2 * t0 + j]);
                    b1 = as_bf16x8(cur.w[2 * t1 + j]);
                }
                // the products of the half-step before: row tile pi, n-tiles pt and pt + 1, k-block pj
                const int m = 2 * n + h - 1, pn = m >> 1, pi = pn % RT, pj = pn / RT, pt = 2 * (m & 1);
                f32x4 d0, d1;
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    if (Q) {
                        if (g == 0) d0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, b0, fzero, 0, 0, 0);
                        if (g == 1) d1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, b1, fzero, 0, 0, 0);
                        if (g == 2) d0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, b0, d0, 0, 0, 0);
                        if (g == 3) d1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, b1, d1, 0, 0, 0);
                        if (g & 1)
                            pin(d1);
                        else
                            pin(d0);
                        if (m >= 0) {
                            const int tt = g >> 1;
#pragma unroll
                            for (int r = 2 * (g & 1); r < 2 * (g & 1) + 2; r++)
                                acc[pi][pt + tt][r] = fmaf(dp[tt][r], sc.v[pt + tt][pj], acc[pi][pt + tt][r]);
                            pin(acc[pi][pt + tt]);
                        }
                        const int w = (i * 2 + h) * WP + g;
                        if (g < WP && w < 16) {
                            convert(j == 0 ? cur : next, 1 - j, w);
                            pin(B[1 - j][w >> 2]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    } else {
                        const int t = g & 1 ? t1 : t0;
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g < 2 ? ah : al, g & 1 ? b1 : b0, acc[i][t], 0, 0, 0);
                    }
                }
                if (Q) {
                    dp[0] = d0;
                    dp[1] = d1;
                } else {
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            ah = nh;
            al = nl;
        }
        if (Q)
#pragma unroll
            for (int tt = 0; tt < 2; tt++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[RT - 1][2 + tt][r] = fmaf(dp[tt][r], sc.v[2 + tt][1], acc[RT - 1][2 + tt][r]);
    };

    Raw ra, rb;
    Scales sa, sb;
#pragma unroll
    for (int q = 0; q < NA; q++) copy_block(0, q);
    load_weights(0, ra);
    load_scales(0, sa);
    if (KIND != BF16) {
        load_weights(1, rb);
#pragma unroll
        for (int w = 0; w < 16; w++) convert(ra, 0, w);
    }
    int s = 0;
    for (; s + 1 < ns; s += 2) {
        stage(s, ra, rb, sa, sb);
        stage(s + 1, rb, ra, sb, sa);
    }
    if (s < ns) stage(s, ra, rb, sa, sb);
    __syncthreads();  // every wave is done with the stages: the LDS is free

    float* rs = (float*)(smem + FIN);
    if (NEED_R) {
        // 1/rms of the rows from the producers' sums of squares: four lanes per row
        for (int e = tid; e < RT * 64; e += NTHR) {
            const int row = min(rt0 * 16 + (e >> 2), a.m - 1), src = a.rows_src ? a.rows_src[row] : row;
            float v = 0.0f;
#pragma unroll 8
            for (int t = e & 3; t < a.ss_tiles; t += 4) v += a.ss_in[(size_t)t * a.ss_m + src];
            v = group_reduce<4, false>(v);
            if (!(e & 3)) rs[e >> 2] = 1.0f / sqrtf(v / (float)a.hidden + a.eps);
        }
    }
    if constexpr (NWK > 1) {
        // each K share hands its sums of row tile i to share i % NWK (in the lanes' own layout), which
        // adds them in the shares' order
        f32x4* xs = (f32x4*)smem + (size_t)wn * RT * (NWK - 1) * 256 + lane;
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int to = i % NWK;
            if (kw != to)
#pragma unroll
                for (int t = 0; t < 4; t++) xs[((i * (NWK - 1) + (kw < to ? kw : kw - 1)) * 4 + t) * 64] = acc[i][t];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RT; i++)
            if (kw == i % NWK)
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int k = 0; k < NWK; k++) {
                        const f32x4 x = k == i % NWK ? acc[i][t]
                                                     : xs[((i * (NWK - 1) + (k < i % NWK ? k : k - 1)) * 4 + t) * 64];
                        v = k == 0 ? x : v + x;
                    }
                    acc[i][t] = v;
                }
    }
    __syncthreads();  // rs; the exchange is read
    float* lw = (float*)(smem + wave * EPW);
#pragma unroll
    for (int i = 0; i < RT; i++) {
        if (NWK > 1 && kw != i % NWK) continue;
        if ((rt0 + i) * 16 >= a.m || col0 >= a.N) continue;
        wave_epilogue<EPI>(a, acc[i], rt0 + i, col0, lw, rs + i * 16, lane);
    }
}

// The tile shapes (RT, NWN, NWK), in launch_mm's order.
template <int KIND, int EPI>
static void run_mm_epi(hipStream_t st, int cfg, const GemvArgs& a, hipEvent_t e0, hipEvent_t e1) {
    auto run = [&](auto kern, int rt, int nwn, int nwk) {
        const int groups = ((a.p_total + 3) / 4 + rt - 1) / rt, cg = (a.N + 64 * nwn - 1) / (64 * nwn);
        if (e0 || e1)
            hipExtLaunchKernelGGL(kern, dim3(cg * groups), dim3(64 * nwn * nwk), 0, st, e0, e1, 0, a);
        else
            hipLaunchKernelGGL(kern, dim3(cg * groups), dim3(64 * nwn * nwk), 0, st, a);
    };
    switch (cfg) {
        case 0: run(k_mm<KIND, EPI, 8, 4, 1>, 8, 4, 1); break;
        case 1: run(k_mm<KIND, EPI, 5, 4, 1>, 5, 4, 1); break;
        case 2: run(k_mm<KIND, EPI, 8, 4, 2>, 8, 4, 2); break;
        case 3: run(k_mm<KIND, EPI, 5, 2, 2>, 5, 2, 2); break;
        case 4: run(k_mm<KIND, EPI, 4, 2, 2>, 4, 2, 2); break;
        case 5: run(k_mm<KIND, EPI, 5, 2, 4>, 5, 2, 4); break;
        case 6: run(k_mm<KIND, EPI, 4, 2, 4>, 4, 2, 4); break;
        case 7: run(k_mm<KIND, EPI, 3, 2, 4>, 3, 2, 4); break;
        case 8: run(k_mm<KIND, EPI, 2, 2, 4>, 2, 2, 4); break;
    }
}

template <int KIND>
void run_mm(hipStream_t st, int epi, int cfg, const GemvArgs& a, hipEvent_t e0, hipEvent_t e1) {
    switch (epi) {
        case EPI_STORE: run_mm_epi<KIND, EPI_STORE>(st, cfg, a, e0, e1); break;
        case EPI_QKV: run_mm_epi<KIND, EPI_QKV>(st, cfg, a, e0, e1); break;
        case EPI_RESID: run_mm_epi<KIND, EPI_RESID>(st, cfg, a, e0, e1); break;
        case EPI_SILU: run_mm_epi<KIND, EPI_SILU>(st, cfg, a, e0, e1); break;
        case EPI_ARGMAX: run_mm_epi<KIND, EPI_ARGMAX>(st, cfg, a, e0, e1); break;
    }
}

}  // namespace fg
