// split.hip - fp32 products Y[M,N] = epi(X[M,K] . W[N,K]^T) on the fp16
// matrix cores of gfx950.
//
// Each fp32 operand value is held as hi + lo, two fp16 values (split.h): hi is
// the value rounded to 11 bits, lo the remainder rounded to 11 bits, exact for
// three values in four and off by one unit of fp32's last place otherwise. A
// product is hi hi + hi lo + lo hi, three v_mfma_f32_32x32x16_f16 summed in
// fp32 (the missing lo lo is below 2^-22 of the product). The fp32 matrix
// instructions add their products to the accumulator two k at a time, and
// that chain's rounding is what their error is made of; sixteen k at a time
// it is a quarter as long, so the split products are the nearer of the two to
// float64 (M=300 N=500 K=768, unit inputs: 2.7e-7 against 4.4e-7 relative in
// the 2-norm for an fp32 chain). The fp16 units run at 16 times the fp32 rate,
// so three instructions per product are about five times the fp32 peak.
//
// Range: fp16 reaches 65504, and its smallest step is 2^-24. Operands are
// scaled by powers of two (exact) so that no value can exceed 2^15: a weight
// row by its own largest value, an input by a bound that follows from the
// weights alone. LayerNorm outputs are at most sqrt(C) max|g| + max|b|; a
// product of one, y = w . (g x^ + b) + c with |x^| <= sqrt(C), is at most
// sqrt(C) |w g| + |w . b + c|, which bounds v, so the attention's output (an
// average of v rows), and fc, so GELU's. The scales are powers of two, so
// results do not depend on them until values fall 2^-16 below their bound and
// lo starts losing bits: an absolute error of 2^-39 of the bound. k_split_w
// compares that with each output's typical size and flags matrices where it
// could exceed 2^-24 of it (gains or rows many thousands of times apart, or
// values that are not finite), k_split_scores heads whose scores lose accuracy
// or could be too large for their probabilities, k_split_scales bounds further than
// 2^40 from 1; a model with a flag keeps the fp32 kernels.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "kernels.h"
#include "split.h"
#include "split_gemm.h"

namespace {

// ---------------------------------------------------------------- scales

__device__ __forceinline__ float block_max(float v, float* red) {
    v = wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// max that keeps a NaN (fmaxf drops it)
__device__ __forceinline__ float max_nan(float m, float v) { return m != m || v <= m ? m : v; }

// Bounds of the LayerNorm outputs; the other slots are cleared for
// k_split_bound.
__global__ void __launch_bounds__(256) k_split_ln_bound(const LayerW* layers, const float* lnf_w,
                                                        const float* lnf_b, int L, int C,
                                                        float* bound, int* bad) {
    __shared__ float red[4];
    const int i = blockIdx.x, l = i >> 1;
    const float* g = i == 2 * L ? lnf_w : i & 1 ? layers[l].ln2_w : layers[l].ln1_w;
    const float* b = i == 2 * L ? lnf_b : i & 1 ? layers[l].ln2_b : layers[l].ln1_b;
    float mg = 0.f, mb = 0.f;
    bool fin = true;
    for (int c = threadIdx.x; c < C; c += 256) {
        mg = fmaxf(mg, fabsf(g[c]));
        mb = fmaxf(mb, fabsf(b[c]));
        fin = fin && fabsf(g[c]) < 1e30f && fabsf(b[c]) < 1e30f;
    }
    mg = block_max(mg, red);
    mb = block_max(mb, red);
    if (!fin) atomicOr(bad, 1);
    if (threadIdx.x == 0) {
        float* slot = bound + SPLIT_SLOTS * l;
        slot[i & 1 ? SLOT_LN2 : SLOT_LN1] = sqrtf((float)C) * mg + mb;
        if (i < 2 * L && !(i & 1)) slot[SLOT_Q] = slot[SLOT_Q + 1] = slot[SLOT_V] = slot[SLOT_HID] = 0.f;
    }
}

__global__ void k_split_clear(int* bad) { *bad = 0; }

// Of each row n of W [N, K] applied to a LayerNorm output (gains g, biases
// b): typ[n], the output's size for inputs of unit variance, and the
// largest possible |output| over each `part` rows (a multiple of 16) into bound[n /
// part]. Four rows per wavefront and one atomic per workgroup: one per row
// followed each other on the same word (2304 x 768: 34 us a launch).
__global__ void __launch_bounds__(256) k_split_bound(const float* __restrict__ W,
                                                     const float* __restrict__ g,
                                                     const float* __restrict__ b,
                                                     const float* __restrict__ bias, int N, int K,
                                                     int part, float* __restrict__ typ, float* bound,
                                                     int* bad) {
    const int n0 = blockIdx.x * 16 + (threadIdx.x >> 6) * 4, lane = threadIdx.x & 63;
    unsigned top = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int n = n0 + r;
        if (n >= N) break;
        float s2 = 0.f, sb = 0.f;
        for (int k = 4 * lane; k < K; k += 256) {
            const f32x4 w = *(const f32x4*)(W + (long)n * K + k);
            const f32x4 gg = *(const f32x4*)(g + k), bb = *(const f32x4*)(b + k);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                s2 += (w[e] * gg[e]) * (w[e] * gg[e]);
                sb += w[e] * bb[e];
            }
        }
        s2 = wave_sum(s2);
        sb = wave_sum(sb) + bias[n];
        const float y = sqrtf((float)K) * sqrtf(s2) + fabsf(sb);
        if (lane == 0) {
            typ[n] = sqrtf(s2 + sb * sb);
            if (!(y < 1e30f)) atomicOr(bad, 1);
        }
        if (y < 1e30f) top = max(top, __builtin_bit_cast(unsigned, y));  // non-negative: ordered as bits
    }
    block_atomic_max<4>((unsigned*)bound + blockIdx.x * 16 / part, top);
}

// Per layer and head: whether scores keep their accuracy. q and k values too
// small for a full lo are off by 2^-39 of their bounds, which must move a score
// (in units of log2 e) by no more than its fp32 roundings would: 2^-24 of its
// typical size, or of a quarter. And whether a score can be so large that its rounding
// takes a probability out of fp16's range: k_attn_split's exponents reach 15 and
// half a unit of the maximum's last place (0.25 at 2^22, 1 at 2^24) and must stay
// below 16. |q| <= sqrt(C) |w g| + |w b + c| <= sqrt(C + 1) of its typical size.
__global__ void __launch_bounds__(64) k_split_scores(const float* __restrict__ typ,
                                                     const float* __restrict__ bound, int C, int H,
                                                     int* bad) {
    const int l = blockIdx.x / H, hs = C / H, h = blockIdx.x % H, lane = threadIdx.x;
    const float* t = typ + (long)l * 7 * C + h * hs;
    float tq = 0.f, tk = 0.f, top = 0.f;
    for (int d = lane; d < hs; d += 64) {
        tq = fmaxf(tq, t[d]);
        tk = fmaxf(tk, t[C + d]);
        top += t[d] * t[C + d];
    }
    tq = wave_max(tq);
    tk = wave_max(tk);
    top = wave_sum(top) * (C + 1.f) * (1.4426950408889634f / sqrtf((float)hs));
    const float bq = bound[SPLIT_SLOTS * l + SLOT_Q], bk = bound[SPLIT_SLOTS * l + SLOT_Q + 1];
    const float err = 0x1p-39f * (bq * tk + bk * tq);  // sqrt(hs) terms, over sqrt(hs)
    if (lane == 0 && !(err <= 0x1p-24f * fmaxf(0.25f, tq * tk) && top <= 0x1p22f)) atomicOr(bad, 1);
}

// scale = the power of two that takes the bound into [2^14, 2^15), 1 where the
// values are all zero. Bounds within 2^40 of 1 keep the products of two scales (a weight
// row's is within 2^65 of 1), and what undoes them, normal floats.
__global__ void k_split_scales(const float* bound, float* scale, int n, int* bad) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    const float b = bound[i];
    const bool fits = b >= 0x1p-40f && b <= 0x1p40f;
    scale[i] = fits ? ldexpf(1.f, 14 - ilogbf(b)) : 1.f;
    if (!fits && b != 0.f) atomicOr(bad, 1);
}

// Split rows of W [N, K], each scaled so that its largest value lies in [2^14,
// 2^15), and winv[n] = 1 / (row scale x input scale), which undoes both. typ:
// the typical sizes of the K inputs, as |g| and |b| (typ_b set) or their own.
// One wavefront per row.
__global__ void __launch_bounds__(256) k_split_w(const float* __restrict__ W,
                                                 unsigned* __restrict__ Ws,
                                                 float* __restrict__ winv, int N, int K,
                                                 const float* __restrict__ typ,
                                                 const float* __restrict__ typ_b,
                                                 const float* __restrict__ bound,
                                                 const float* __restrict__ xscale, int* bad) {
    const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (n >= N) return;
    const float* w = W + (long)n * K;
    float mx = 0.f, s2 = 0.f, st = 0.f;
    for (int k = 4 * lane; k < K; k += 256) {
        const f32x4 v = *(const f32x4*)(w + k), t = *(const f32x4*)(typ + k);
        f32x4 tb = {0.f, 0.f, 0.f, 0.f};
        if (typ_b) tb = *(const f32x4*)(typ_b + k);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            mx = max_nan(mx, fabsf(v[e]));
            s2 += v[e] * v[e];
            st += (v[e] * v[e]) * (t[e] * t[e] + tb[e] * tb[e]);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max_nan(mx, __shfl_xor(mx, o, 64));
    s2 = wave_sum(s2);
    st = wave_sum(st);
    // absolute error of inputs and weights too small for a full lo (2^-39 of
    // the bound, and of the row's largest weight) against the output's
    // typical size
    const float x = *bound;
    const float err = 0x1p-39f * (x * sqrtf(s2) + mx * sqrtf((float)K) * x);
    const bool fits = (mx == 0.f || mx > 1e-15f) && mx < 1e15f && s2 < 1e30f && err <= 0x1p-24f * sqrtf(st);
    const float sc = mx > 0.f && fits ? ldexpf(1.f, 14 - ilogbf(mx)) : 1.f;
    if (lane == 0) {
        winv[n] = 1.f / (sc * *xscale);
        if (!fits) atomicOr(bad, 1);
    }
    unsigned* o = Ws + (long)n * K;
    for (int k = 8 * lane; k < K; k += 512) {
        u32x4 hi, lo;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const f32x4 v = *(const f32x4*)(w + k + 4 * h);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                unsigned hp, lp;
                split_pair(v[2 * e] * sc, v[2 * e + 1] * sc, hp, lp);
                hi[2 * h + e] = hp;
                lo[2 * h + e] = lp;
            }
        }
        *(u32x4*)(o + k) = hi;
        *(u32x4*)(o + k + 4) = lo;
    }
}

// ---------------------------------------------------------------- dispatch

// Tile shapes, by estimated time. A step of 16 k costs a workgroup sharing its
// CU with w - 1 others step[w - 1] us (measured on launches that leave the chip
// part-idle; 0.71 us for 256 x 256 is 2290 TFLOP/s of raw products, 92 % of
// nominal), but a full chip is held by its power, the larger tiles with fewer
// LDS bytes per product the least: all steps running at a time together take
// no less than their raw products at rate TFLOP/s. start covers a workgroup's
// first loads and its epilogue. Measured against it (us, best
// shape first): 2048 x 2304 x 768 128x192 28.8, 128x128 32.8, 256x192 40.2;
// 2048 x 768 x 768 64x128 15.7, 128x128 17.7, 128x192 21.7; 4096 x 1600 x 1600
// 128x128 69.5, 256x192 73.7, 128x192 87.5; 16384 x 3072 x 768 256x256 209,
// 256x192 220, 128x192 223. Splitting K pays where the tiles leave CUs idle
// over a long K (2048 x 768 x 3072: 64x128 53.7, four splits of 128x192 39.3);
// its partials cost about 0.25 us per MB written and summed.
struct Shape {
    int TM, TN, occ;
    double step[4], start, rate;
};
constexpr Shape SHAPES[] = {{256, 256, 1, {0.71}, 11.0, 1310},
                            {256, 192, 1, {0.565}, 8.0, 1250},
                            {128, 192, 2, {0.42, 0.80}, 6.0, 1140},
                            {128, 128, 3, {0.378, 0.60, 0.95}, 4.0, 970},
                            {64, 128, 4, {0.256, 0.49, 0.65, 0.80}, 3.5, 900}};

struct Plan {
    int shape, KS, KR;
};

bool vec_ok(const SplitGemmArgs& a) {
    return a.N % 4 == 0 && a.ldy % 4 == 0 && (size_t)a.Y % 16 == 0 && (size_t)a.bias % 16 == 0 &&
           (size_t)a.winv % 16 == 0;
}

double round_us(const Shape& s, long wgs, int steps) {
    const int w = (int)((wgs + 255) / 256);
    // (a part-filled round draws its power at a higher clock and gets less for
    // it: 192 of 256 workgroups of 256 x 256 ran at 1227, all of them at 1310)
    const double rate = s.rate * (0.75 + 0.25 * wgs / (256.0 * s.occ));
    const double raw = (double)wgs * s.TM * s.TN * SP_BK * 6 / (rate * 1e6);  // us a step
    return s.start + steps * std::max(s.step[w - 1], raw);
}

// Splits that keep the error no larger than the fp32 kernels' where those split
// K over idle CUs, into sums of c k each. Measured (relative 2-norm, unit
// inputs): an fp32 sum of c k 0.73e-7 + 0.155e-7 sqrt(c) (in quadrature), a
// split one 0.90e-7 + 0.107e-7 sqrt(c), so sums of up to 2.1 c - 25 are as good
// (K = 256, M = 384: 1.93e-7 whole, 1.50e-7 in fp32, whose 4 splits sum 64 k);
// 1.5 c - 20 leaves a margin.
int min_splits(const SplitGemmArgs& a) {
    GemmArgs g{};
    g.M = a.M; g.N = a.N; g.K = a.K;
    g.part = a.part; g.part_cap = a.part_cap;
    const int ks = launch_gemm_splits(g);
    return ks <= 1 ? 1 : (int)std::ceil(a.K / (1.5 * a.K / ks - 20.0));
}

Plan plan(const SplitGemmArgs& a) {
    const int nk = a.K / SP_BK;
    const bool can = a.part && vec_ok(a) && a.N % 8 == 0;
    const int min_ks = can ? min_splits(a) : 1;
    const int max_ks = can ? std::max(min_ks, std::min(8, nk / 8)) : 1;
    Plan best{3, 1, a.K};
    double best_us = 1e30;
    for (int i = 0; i < (int)(sizeof(SHAPES) / sizeof(SHAPES[0])); i++) {
        const Shape& s = SHAPES[i];
        const long tiles = (long)((a.M + s.TM - 1) / s.TM) * ((a.N + s.TN - 1) / s.TN);
        for (int want = min_ks; want <= max_ks; want++) {
            const int per = (nk + want - 1) / want, ks = (nk + per - 1) / per;
            if (ks > 1 && (long)ks * a.M * a.N > a.part_cap) continue;
            const long wgs = tiles * ks, slots = 256L * s.occ;
            double us = (wgs / slots) * round_us(s, slots, per);
            if (wgs % slots) us += round_us(s, wgs % slots, per);
            if (ks > 1) us += 2.0 + 1e-6 * ks * a.M * a.N;
            if (us < best_us) {
                best_us = us;
                best = Plan{i, ks, per * SP_BK};
            }
        }
    }
    return best;
}

template <int EPI, bool VEC>
hipError_t run_shape(const SplitGemmArgs& a, const Plan& p, hipStream_t s) {
    const Shape& sh = SHAPES[p.shape];
    const int tm = (a.M + sh.TM - 1) / sh.TM, tn = (a.N + sh.TN - 1) / sh.TN;
    const unsigned grid = (unsigned)(tm * tn * p.KS);
    switch (p.shape) {
        case 0: k_gemm_split<EPI, -1, 4, 2, 4, 4, 1, VEC><<<grid, 512, 0, s>>>(a, tm, tn, p.KR, p.KS); break;
        case 1: k_gemm_split<EPI, -1, 4, 2, 3, 4, 1, VEC><<<grid, 512, 0, s>>>(a, tm, tn, p.KR, p.KS); break;
        case 2: k_gemm_split<EPI, -1, 2, 2, 3, 3, 2, VEC><<<grid, 256, 0, s>>>(a, tm, tn, p.KR, p.KS); break;
        case 3: k_gemm_split<EPI, -1, 2, 2, 2, 3, 3, VEC><<<grid, 256, 0, s>>>(a, tm, tn, p.KR, p.KS); break;
        default: k_gemm_split<EPI, -1, 1, 2, 2, 3, 4, VEC><<<grid, 128, 0, s>>>(a, tm, tn, p.KR, p.KS); break;
    }
    return hipGetLastError();
}

template <int EPI>
hipError_t reduce(const SplitGemmArgs& a, int KS, hipStream_t s) {
    const long n = (long)a.M * (a.N / 8);
    k_split_reduce<EPI><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(a, KS);
    return hipGetLastError();
}

}  // namespace

int launch_split_gemm_splits(const SplitGemmArgs& a) {
    return a.M > 0 && a.N > 0 && a.K > 0 ? plan(a).KS : 1;
}

int launch_split_gemm_plan(const SplitGemmArgs& a) {
    const Plan p = plan(a);
    return p.KS + 256 * p.shape;
}

hipError_t launch_split_gemm(const SplitGemmArgs& a, hipStream_t s) {
    if (a.M <= 0 || a.N <= 0) return hipSuccess;
    if (a.K <= 0 || a.K % SP_BK || !a.winv) return hipErrorInvalidValue;
    const bool vec = vec_ok(a);
    if (a.epi != EPI_STORE && (!vec || !a.bias)) return hipErrorInvalidValue;
    const bool split_out = a.epi == EPI_BIAS_GELU || a.epi == EPI_QKV;
    if (split_out != (a.out_scale != nullptr)) return hipErrorInvalidValue;
    if (split_out && a.N % (a.epi == EPI_QKV ? 24 : 8)) return hipErrorInvalidValue;
    if (a.epi == EPI_QKV && (!a.Ys || (size_t)a.Ys % 16)) return hipErrorInvalidValue;
    if (!vec && a.seg) return hipErrorInvalidValue;
    const Plan p = plan(a);
    // the LayerNorm is formed by the split sum; without splits the caller
    // launches it
    if (a.ln_out && (p.KS == 1 || a.epi != EPI_RESID || a.seg)) return hipErrorInvalidValue;
    if (p.KS > 1) {
        const hipError_t e = run_shape<EPI_STORE, true>(a, p, s);
        if (e != hipSuccess) return e;
        if (a.ln_out) {
            GemmArgs g{};
            g.M = a.M; g.N = a.N; g.K = a.K;
            g.bias = a.bias; g.Y = a.Y; g.ldy = a.ldy;
            g.part = a.part; g.part_cap = a.part_cap;
            g.ln_w = a.ln_w; g.ln_b = a.ln_b; g.ln_out = a.ln_out; g.ln_scale = a.ln_scale;
            g.epi = EPI_RESID;
            return launch_sum_heads(g, p.KS, s);
        }
        switch (a.epi) {
            case EPI_STORE: return reduce<EPI_STORE>(a, p.KS, s);
            case EPI_BIAS: return reduce<EPI_BIAS>(a, p.KS, s);
            case EPI_BIAS_GELU: return reduce<EPI_BIAS_GELU>(a, p.KS, s);
            case EPI_RESID: return reduce<EPI_RESID>(a, p.KS, s);
            case EPI_QKV: return reduce<EPI_QKV>(a, p.KS, s);
        }
        return hipErrorInvalidValue;
    }
    switch (a.epi) {
        case EPI_STORE:
            return vec ? run_shape<EPI_STORE, true>(a, p, s) : run_shape<EPI_STORE, false>(a, p, s);
        case EPI_BIAS: return run_shape<EPI_BIAS, true>(a, p, s);
        case EPI_BIAS_GELU: return run_shape<EPI_BIAS_GELU, true>(a, p, s);
        case EPI_RESID: return run_shape<EPI_RESID, true>(a, p, s);
        case EPI_QKV: return run_shape<EPI_QKV, true>(a, p, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_split_scales(const LayerW* d_layers, const LayerW* layers, const float* lnf_w,
                               const float* lnf_b, int L, int C, int H, float* bound,
                               float* scale, float* typ, int* bad, hipStream_t s) {
    k_split_clear<<<1, 1, 0, s>>>(bad);
    k_split_ln_bound<<<2 * L + 1, 256, 0, s>>>(d_layers, lnf_w, lnf_b, L, C, bound, bad);
    for (int l = 0; l < L; l++) {
        const LayerW& w = layers[l];
        float* t = typ + (long)l * 7 * C;
        float* slot = bound + SPLIT_SLOTS * l;
        // the QKV product's three thirds; fc
        k_split_bound<<<(3 * C + 15) / 16, 256, 0, s>>>(w.attn_w, w.ln1_w, w.ln1_b, w.attn_b, 3 * C, C,
                                                      C, t, slot + SLOT_Q, bad);
        k_split_bound<<<(4 * C + 15) / 16, 256, 0, s>>>(w.fc_w, w.ln2_w, w.ln2_b, w.fc_b, 4 * C, C, 4 * C, t + 3 * C,
                                        slot + SLOT_HID, bad);
    }
    k_split_scores<<<L * H, 64, 0, s>>>(typ, bound, C, H, bad);
    k_split_scales<<<(split_slots(L) + 63) / 64, 64, 0, s>>>(bound, scale, split_slots(L), bad);
    return hipGetLastError();
}

hipError_t launch_split_w(const float* W, const SplitWeights& o, int N, int K, const float* typ,
                          const float* typ_b, const float* bound, const float* scale, int* bad,
                          hipStream_t s) {
    if (N <= 0 || K <= 0 || K % SP_BK) return hipErrorInvalidValue;
    k_split_w<<<(N + 3) / 4, 256, 0, s>>>(W, (unsigned*)o.W, o.winv, N, K, typ, typ_b, bound, scale,
                                          bad);
    return hipGetLastError();
}
