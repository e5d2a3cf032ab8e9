// split_gemm.h - the kernels of the products over split rows (split.h), shared
// by the forward's products (split.hip) and the training step's
// (split_train.hip).
#pragma once
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "split.h"

namespace {

constexpr int SP_BK = 16;  // k per stage and per matrix instruction

__device__ __forceinline__ int xcd_order(int pid, int nt) {
    const int per = nt / 8, rem = nt % 8;
    const int xcd = pid % 8, idx = pid / 8;
    return (xcd < rem) ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

// Tile of work id p: groups of 8 row tiles, so that neighbours share X and W
// rows in the XCD's L2 (4 and 16 measured 1-3 % slower).
__device__ __forceinline__ void group_coords(int p, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int GM = 8;
    const int group = p / (GM * tiles_n);
    const int first_m = group * GM;
    const int gsize = min(tiles_m - first_m, GM);
    const int in_group = p % (GM * tiles_n);
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

template <int EPI>
__device__ __forceinline__ float epi_value(float v, float b, float old) {
    if (EPI == EPI_STORE) return v;
    if (EPI == EPI_BIAS || EPI == EPI_QKV) return v + b;
    if (EPI == EPI_BIAS_GELU) return gelu_tanh(v + b);
    return (old + v) + b;
}

// A workgroup of WR x WC wavefronts owns a tile of 64 WR rows x 32 CB WC
// columns, each wavefront 2 x CB blocks of 32 x 32. Both operands go from
// global memory straight into LDS (lds_dma16) through a ring of S stages of 16
// k, 64 bytes a row: granule 2 q + p of a row is plane p (hi, lo) of its k
// octet q, stored at slot (2 q + p) ^ (row / 4 % 4), so that the 16 rows a
// quarter wavefront reads at one granule fall in 16 different granules of a
// 256-byte bank line. A step waits for stage kt + 1, passes one barrier
// (every wavefront has stage kt in registers by then, so its slot is free for
// stage kt + S), and then multiplies stage kt while it reads stage kt + 1 and
// issues the loads of stage kt + S, one such instruction between two matrix
// instructions: issued together ahead of them they left the matrix cores idle
// for as long as the LDS queue took (QKV at M=16384, 181 -> 171 us; proj 224
// -> 208). Wave priority as in gemm.hip.
//
// The bound is the matrix cores at the clock the chip holds under them: a
// register-only loop of these instructions on random data reaches 1300-1560
// TFLOP/s (2500 nominal), and the 256 x 192 tiles at K = 3072 run 1200 of
// raw products (399 of fp32 work, against 134 on the fp32 cores).
//
// VEC: the operands swapped, so that a lane holds four consecutive columns of
// a row and moves them as 16 bytes (N, ldy and the pointers multiples of
// four); without it 32 lanes cover 32 columns of a row, which takes any
// alignment (the lm_head's odd row length). The GELU and QKV epilogues write
// split rows, the next product's or the attention's operands. KS > 1 (EPI_STORE):
// K split over workgroups, partials to a.part + ks M N.
//
// KM >= 0 (the training backward): each operand carries one scale, that of
// split_scale of *a.xmax and *a.wmax, or (xstep, wstep 1) one for each row and
// column of Y, and a K-major operand (KM & 1: X, KM & 2:
// W; rows of ldx / ldw values, one per k) is used as it is stored: a stage
// holds 16 of its rows, TM / 4 (TN / 4) granules each, and the reads turn 4 x 16
// corners of it (read_turned) into the lanes' eight k. Granules are XORed with
// bit 0 of k at bit 0 and bit 1 of k at bit 3, so that the four rows x 32
// columns a read touches fill a 256-byte bank line. Columns past the end re-read the
// last octet of a row (their results are not stored).
template <int EPI, int KM, int WR, int WC, int CB, int S, int OCC, bool VEC>
__global__ void __launch_bounds__(64 * WR * WC, OCC * WR * WC / 4)
    k_gemm_split(SplitGemmArgs a, int tiles_m, int tiles_n, int KR, int KS) {
    constexpr int NW = WR * WC, TM = 64 * WR, TN = 32 * CB * WC;
    constexpr int ROWS = (TM + TN + 16 * NW - 1) / (16 * NW) * 16 * NW;  // padded: whole loads
    constexpr int NI = ROWS / (16 * NW);  // load instructions per wavefront and stage
    constexpr int STAGE = ROWS * 64;      // bytes
    constexpr bool OUT_SPLIT = EPI == EPI_BIAS_GELU || EPI == EPI_QKV;
    static_assert(S >= 2 && OCC * S * STAGE <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) char sm[S * STAGE];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int tiles = tiles_m * tiles_n;
    int p = xcd_order(blockIdx.x, tiles * KS);
    const int ks = p / tiles;
    p -= ks * tiles;
    int tm, tn;
    group_coords(p, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * TM, n0 = tn * TN, K = a.K, kb = ks * KR;
    const int nk = (min(KR, K - kb)) / SP_BK;

    // load instruction i of this wavefront covers stage rows 16 (NW i + wave)
    // .. +15 (X rows, then W rows, then padding): lane -> row lane / 4, slot
    // lane % 4; rows past M or N re-read the last one (their results are not
    // stored)
    constexpr bool XT = KM >= 0 && (KM & 1), WT = KM >= 0 && (KM & 2);
    const char* src[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int row = 16 * (NW * i + wave) + (lane >> 2);
        if (XT && row < TM) {
            const int q = (NW * i + wave) * 64 + lane, k = q / (TM / 4);
            const int g = (q % (TM / 4)) ^ ((k & 1) | ((k & 2) << 2));
            src[i] = (const char*)a.X + ((long)(kb + k) * a.ldx + 8l * min(m0 / 8 + (g >> 1), (int)(a.ldx / 8) - 1)) * 4 +
                     16 * (g & 1);
        } else if (WT && row >= TM) {
            // (padding granules wrap to the first rows)
            const int q = (NW * i + wave) * 64 + lane - 4 * TM, k = (q / (TN / 4)) & 15;
            const int g = (q % (TN / 4)) ^ ((k & 1) | ((k & 2) << 2));
            src[i] = (const char*)a.W + ((long)(kb + k) * a.ldw + 8l * min(n0 / 8 + (g >> 1), (int)(a.ldw / 8) - 1)) * 4 +
                     16 * (g & 1);
        } else {
            const int g = (lane & 3) ^ ((row >> 2) & 3);
            src[i] = (row < TM ? (const char*)a.X + (long)min(m0 + row, a.M - 1) * K * 4
                               : (const char*)a.W + (long)min(n0 + row - TM, a.N - 1) * K * 4) +
                     (long)kb * 4 + 16 * g;
        }
    }
    const long xstep = XT ? 64 * a.ldx : 64, wstep = WT ? 64 * a.ldw : 64;
    auto issue1 = [&](int kt, int slot, int i) {
        lds_dma16(src[i] + (long)kt * (16 * (NW * i + wave) < TM ? xstep : wstep),
                  (const float*)(sm + slot * STAGE + (NW * i + wave) * 1024));
    };
    const int wm = (wave / WC) * 64, wn = (wave % WC) * 32 * CB;
    const int lr = lane & 31, lh = lane >> 5;
    // byte offsets of this lane's hi granules in a stage (lo: bit 4 flipped)
    const int sw = 16 * ((2 * lh) ^ ((lr >> 2) & 3));
    const int ah = (wm + lr) * 64 + sw, bh = (TM + wn + lr) * 64 + sw;
    const int al = ah ^ 16, bl = bh ^ 16;
    // and of the turned reads, per block of 32 columns
    int at[2], bt[CB];
    if constexpr (KM > 0) {
        const int k = 8 * lh + ((lane >> 2) & 3), x = (k & 1) | ((k & 2) << 2);
        const int g = 4 * ((lane >> 4) & 1) + (lane & 2);
#pragma unroll
        for (int i = 0; i < 2; i++)
            at[i] = k * TM * 4 + 16 * ((wm / 4 + 8 * i + g) ^ x) + 8 * (lane & 1);
#pragma unroll
        for (int j = 0; j < CB; j++)
            bt[j] = TM * 64 + k * TN * 4 + 16 * ((wn / 4 + 8 * j + g) ^ x) + 8 * (lane & 1);
    }

    f32x16 acc[2][CB];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < CB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    struct Ops {
        f16x8 ah[2], al[2], bh[CB], bl[CB];
    };
    constexpr int NR = 2 * CB + 4, NM = 6 * CB;  // reads and products of a step
    constexpr int NQ = (NR + NI + NM - 1) / NM;  // reads and loads per product
    // read q of a stage, in the order the products use them
    auto read1 = [&](int slot, Ops& o, int q) {
        const char* base = sm + slot * STAGE;
        auto rx = [&](int i, bool l) {
            if constexpr (XT) return read_turned(base + (l ? at[i] ^ 16 : at[i]), TM * 16);
            else return *(const f16x8*)(base + (l ? al : ah) + i * 2048);
        };
        auto rw = [&](int j, bool l) {
            if constexpr (WT) return read_turned(base + (l ? bt[j] ^ 16 : bt[j]), TN * 16);
            else return *(const f16x8*)(base + (l ? bl : bh) + j * 2048);
        };
        if (q < CB) o.bh[q] = rw(q, false);
        else if (q < CB + 2) o.al[q - CB] = rx(q - CB, true);
        else if (q < CB + 4) o.ah[q - CB - 2] = rx(q - CB - 2, false);
        else o.bl[q - CB - 4] = rw(q - CB - 4, true);
    };
    // product q: lo hi, hi hi, hi lo over the blocks
    auto mul1 = [&](const Ops& o, int q) {
        const int pr = q / (2 * CB), j = (q % (2 * CB)) / 2, i = q & 1;
        const f16x8 x = pr == 0 ? o.al[i] : o.ah[i], w = pr == 2 ? o.bl[j] : o.bh[j];
        acc[i][j] = VEC ? __builtin_amdgcn_mfma_f32_32x32x16_f16(w, x, acc[i][j], 0, 0, 0)
                        : __builtin_amdgcn_mfma_f32_32x32x16_f16(x, w, acc[i][j], 0, 0, 0);
    };

#pragma unroll
    for (int st = 0; st < S; st++)
        if (st < nk)
#pragma unroll
            for (int i = 0; i < NI; i++) issue1(st, st, i);
    if (nk >= S) wait_vmcnt<NI * (S - 1)>();
    else wait_vmcnt<0>();
    asm volatile("s_barrier" ::: "memory");
    Ops o0, o1;
#pragma unroll
    for (int q = 0; q < NR; q++) read1(0, o0, q);
    int slot = 0;  // kt % S
    // FULL: stage kt + S exists
    auto step = [&](int kt, const Ops& cur, Ops& nxt, auto full) {
        const int next = slot + 1 == S ? 0 : slot + 1;
        if constexpr (decltype(full)::value) {
            // stage kt + 1 has landed once at most stages kt + 2 .. kt + S - 1
            // are in flight
            wait_vmcnt<NI * (S - 2)>();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int q = 0; q < NM; q++) {
#pragma unroll
                for (int u = NQ * q; u < NQ * q + NQ; u++) {
                    if (u < NR) read1(next, nxt, u);
                    else if (u - NR < NI) issue1(kt + S, slot, u - NR);
                }
                mul1(cur, q);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
        } else {
            if (kt + 1 < nk) {
                if (kt + S - 1 < nk) wait_vmcnt<NI * (S - 2)>();
                else wait_vmcnt<0>();
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                if (kt + S < nk)
#pragma unroll
                    for (int i = 0; i < NI; i++) issue1(kt + S, slot, i);
#pragma unroll
                for (int q = 0; q < NR; q++) read1(next, nxt, q);
            }
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int q = 0; q < NM; q++) mul1(cur, q);
            __builtin_amdgcn_s_setprio(0);
        }
        slot = next;
    };
    int kt = 0;
    for (; kt + 1 + S < nk; kt += 2) {
        step(kt, o0, o1, std::true_type{});
        step(kt + 1, o1, o0, std::true_type{});
    }
    for (; kt + 1 < nk; kt += 2) {
        step(kt, o0, o1, std::false_type{});
        step(kt + 1, o1, o0, std::false_type{});
    }
    if (kt < nk) step(kt, o0, o1, std::false_type{});

    if constexpr (VEC) {
        unsigned top = 0;
        // acc[i][j][4 g + e]: row m0 + wm + 32 i + lane % 32, column n0 + wn
        // + 32 j + 8 g + 4 (lane / 32) + e. The scales, bias and residual of
        // block column j + 1 are loaded before block column j is stored: a
        // load after a store would wait for that store too (the vector-memory
        // counter counts both).
        const bool part = EPI == EPI_STORE && KS > 1;
        float *yrow[2], *srow[2];
        const float sign = KM == 2 && (lr & 1) ? -1.f : 1.f;  // (odd rows are stored negated)
        int ex[2] = {0, 0};                                   // exponents that undo the scales
        int ew[2][4][4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = min(m0 + wm + 32 * i + lr, a.M - 1);
            srow[i] = EPI == EPI_QKV ? a.Ys + (long)row * a.N : nullptr;
            const long orow = a.seg ? (long)(row / a.seg) * a.seg_stride + row % a.seg : row;
            yrow[i] = part ? a.part + ((long)ks * a.M + row) * a.N : a.Y + orow * a.ldy;
            if (KM >= 0) ex[i] = -split_exp(a.xmax[row * a.xstep]);
        }
        const float os0 = OUT_SPLIT ? a.out_scale[0] : 1.f;
        const float os1 = EPI == EPI_QKV ? a.out_scale[1] : 1.f;
        const float os2 = EPI == EPI_QKV ? a.out_scale[2] : 1.f;
        const int third = a.N / 3;
        constexpr bool BIAS = EPI != EPI_STORE && KM < 0;  // (the backward's is zero)
        constexpr bool AHEAD = EPI != EPI_RESID || OCC < 3;  // (three per CU: registers)
        f32x4 s[2][4], b[2][4], old[2][2][4];
        auto load = [&](int j, int t) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int c = min(n0 + wn + 32 * j + 4 * lh + 8 * g, a.N - 4);
                if constexpr (KM < 0) {
                    s[t][g] = *(const f32x4*)(a.winv + c);
                } else {
                    u32x4 u;
                    if (a.wstep) u = *(const u32x4*)(a.wmax + c);
                    else u = u32x4{*a.wmax, *a.wmax, *a.wmax, *a.wmax};
#pragma unroll
                    for (int e = 0; e < 4; e++) ew[t][g][e] = -split_exp(u[e]);
                }
                if (BIAS) b[t][g] = *(const f32x4*)(a.bias + c);
                if (EPI == EPI_RESID)
#pragma unroll
                    for (int i = 0; i < 2; i++) old[t][i][g] = *(const f32x4*)(yrow[i] + c);
            }
        };
        if (AHEAD) load(0, 0);
#pragma unroll
        for (int j = 0; j < CB; j++) {
            const int t = AHEAD ? j & 1 : 0;
            if (!AHEAD) load(j, 0);
            else if (j + 1 < CB) load(j + 1, t ^ 1);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const bool rok = m0 + wm + 32 * i + lr < a.M;
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int c = n0 + wn + 32 * j + 4 * lh + 8 * g;
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float y = KM >= 0 ? __builtin_amdgcn_ldexpf(acc[i][j][4 * g + e] * sign,
                                                                          ex[i] + ew[t][g][e])
                                                : acc[i][j][4 * g + e] * s[t][g][e];
                        v[e] = epi_value<EPI>(y, BIAS ? b[t][g][e] : 0.f,
                                              EPI == EPI_RESID ? old[t][i][g][e] : 0.f);
                    }
                    if constexpr (OUT_SPLIT) {
                        // lanes l and l + 32 hold columns 0-3 and 4-7 of an
                        // octet: the lower lane stores its hi granule, the
                        // upper its lo granule
                        const float os = EPI == EPI_QKV && c >= third
                                             ? (c >= 2 * third ? os2 : os1)
                                             : os0;
                        unsigned h0, h1, l0, l1;
                        split_pair(v[0] * os, v[1] * os, h0, l0);
                        split_pair(v[2] * os, v[3] * os, h1, l1);
                        swap32(h0, l0);
                        swap32(h1, l1);
                        if (rok && c < a.N) {
                            *(u32x4*)((EPI == EPI_QKV ? srow[i] : yrow[i]) + c) = u32x4{h0, h1, l0, l1};
                            if (EPI == EPI_QKV && a.Y) *(f32x4*)(yrow[i] + c) = v;
                        }
                    } else if (rok && c < a.N) {
                        *(f32x4*)(yrow[i] + c) = v;
                        if (KM >= 0) top = max(top, abs_bits(v));
                    }
                }
            }
        }
        if (KM >= 0 && a.amax && !part) block_atomic_max<NW>(a.amax, top);
    } else {
        // acc[i][j][r]: row m0 + wm + 32 i + 8 (r / 4) + 4 (lane / 32) + r %
        // 4, column n0 + wn + 32 j + lane % 32 (stored only: the lm_head)
        static_assert(VEC || (EPI == EPI_STORE && KM < 0), "plain stores");
        float s[CB];
#pragma unroll
        for (int j = 0; j < CB; j++) s[j] = a.winv[min(n0 + wn + 32 * j + lr, a.N - 1)];
        const bool inside = m0 + TM <= a.M && n0 + TN <= a.N;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = m0 + wm + 32 * i + 8 * (r >> 2) + 4 * lh + (r & 3);
                float* yr = a.Y + (long)row * a.ldy + n0 + wn + lr;
#pragma unroll
                for (int j = 0; j < CB; j++)
                    if (inside || (row < a.M && n0 + wn + 32 * j + lr < a.N))
                        yr[32 * j] = acc[i][j][r] * s[j];
            }
    }
}

// Y = epi(sum of the KS partials in order), eight columns per thread.
template <int EPI>
__global__ void __launch_bounds__(256) k_split_reduce(SplitGemmArgs a, int KS) {
    const int n8 = a.N >> 3;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    const long i = min(id, (long)a.M * n8 - 1);  // (past the end: the last again)
    const int row = (int)(i / n8), c = (int)(i - (long)row * n8) * 8;
    const long MN = (long)a.M * a.N;
    const float* p = a.part + (long)row * a.N + c;
    const long orow = a.seg ? (long)(row / a.seg) * a.seg_stride + row % a.seg : row;
    float* y = a.Y + orow * a.ldy + c;
    f32x4 b[2] = {}, old[2] = {}, v[2] = {};
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if (EPI != EPI_STORE) b[h] = *(const f32x4*)(a.bias + c + 4 * h);
        if (EPI == EPI_RESID) old[h] = *(const f32x4*)(y + 4 * h);
    }
    for (int q0 = 0; q0 < KS; q0 += 4) {
        f32x4 t[4][2];
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                t[j][h] = *(const f32x4*)(p + min(q0 + j, KS - 1) * MN + 4 * h);
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (q0 + j < KS)
#pragma unroll
                for (int h = 0; h < 2; h++) v[h] += t[j][h];
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) v[h][e] = epi_value<EPI>(v[h][e], b[h][e], old[h][e]);
    if (a.amax) block_atomic_max<4>(a.amax, max(abs_bits(v[0]), abs_bits(v[1])));
    if (id != i) return;
    if (EPI == EPI_BIAS_GELU || EPI == EPI_QKV) {
        const float os = a.out_scale[EPI == EPI_QKV ? c / (a.N / 3) : 0];
        u32x4 hi, lo;
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                unsigned hp, lp;
                split_pair(v[h][2 * e] * os, v[h][2 * e + 1] * os, hp, lp);
                hi[2 * h + e] = hp;
                lo[2 * h + e] = lp;
            }
        float* ys = EPI == EPI_QKV ? a.Ys + (long)row * a.N + c : y;
        *(u32x4*)ys = hi;
        *(u32x4*)(ys + 4) = lo;
    }
    if (EPI != EPI_BIAS_GELU && (EPI != EPI_QKV || a.Y)) {
        *(f32x4*)y = v[0];
        *(f32x4*)(y + 4) = v[1];
    }
}

}  // namespace
