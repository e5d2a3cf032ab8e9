// split_train.hip - the training backward's products on the fp16 matrix cores
// (split_gemm.h), and the passes that bring its tensors into split rows.
//
// Weights, activations and gradients change with every step, so each tensor
// carries one power-of-two scale taken from its own largest magnitude, found on
// the device in the same step: by the kernel that writes the tensor, from a bound
// that its producer implies (LayerNorm, GELU's gradient), or by a pass
// over it. One scale per tensor, not per row, is what lets one split copy serve both
// products it is in, with K along its rows in one and across them in the other. A
// value loses bits of lo once it is 2^-16 below its tensor's largest (2^-39 of that
// largest at most), so a product's error stays within 2^-24 of its operands' norms.
//
// The fp16 matrix instructions round their sums down (4096 x 768 x 3072, unit
// inputs: mean error -4.5e-8 of the result's size, against -3e-10 of the fp32
// ones). That is small beside the error itself (3.6e-7, fp32 5.0e-7), but the same
// for every row of a dX, and the sums over all rows that follow (LayerNorm's and
// attention's gradients) pile it up: LayerNorm gains' gradients were off by 2.1e-6 for
// 0.9e-6 in fp32. So the odd rows of activations and gradients are stored
// negated. A dX is negated back where it is written, which turns every second
// row's rounding up; in a dW both factors of a row's product carry the sign.
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "split.h"
#include "split_gemm.h"

namespace {

__device__ __forceinline__ float bits_to_float(unsigned u) { return __builtin_bit_cast(float, u); }

// Raises *t.amax to the largest magnitude of a tensor. Few large workgroups: their
// atomics to one word follow each other (768 of them took 15 us for 12.6 MB).
__global__ void __launch_bounds__(1024) k_tensor_max(SplitTensor t) {
    const long n4 = t.n >> 2, step = (long)gridDim.x * 1024;
    unsigned m = 0;
    const f32x4* p = (const f32x4*)t.src;
    long i = (long)blockIdx.x * 1024 + threadIdx.x;
    for (; i + 3 * step < n4; i += 4 * step) {
        const f32x4 a = p[i], b = p[i + step], c = p[i + 2 * step], d = p[i + 3 * step];
        m = max(max(m, max(abs_bits(a), abs_bits(b))), max(abs_bits(c), abs_bits(d)));
    }
    for (; i < n4; i += step) m = max(m, abs_bits(p[i]));
    block_atomic_max<16>(t.amax, m);
}

__device__ __forceinline__ void tensor_split(const SplitTensor& t) {
    const float sc = split_scale(*t.amax);
    const long n8 = t.n >> 3;
    const f32x4* p = (const f32x4*)t.src;
    u32x4* o = (u32x4*)t.dst;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n8; i += (long)gridDim.x * 256) {
        u32x4 hi, lo;
        const bool odd = t.alt && ((unsigned)i / (unsigned)(t.alt >> 3) & 1);
        split_octet(p[2 * i], p[2 * i + 1], odd ? -sc : sc, hi, lo);
        o[2 * i] = hi;
        o[2 * i + 1] = lo;
    }
}

// Weight matrices: the largest magnitude and each column's, over rows blockIdx.x,
// blockIdx.x + gridDim.x, ...
__global__ void __launch_bounds__(256) k_weights_max(const SplitTensor* d) {
    const SplitTensor t = d[blockIdx.y];
    const int rows = (int)(t.n / t.K), q4 = t.K >> 2, step = gridDim.x;
    unsigned top = 0;
    for (int q = threadIdx.x; q < q4; q += 256) {
        const f32x4* p = (const f32x4*)t.src + q;
        unsigned m[4] = {0, 0, 0, 0};
        auto take = [&](const f32x4& v) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                m[e] = max(m[e], __builtin_bit_cast(unsigned, (float)v[e]) & 0x7fffffffu);
        };
        int r = blockIdx.x;
        for (; r + 7 * step < rows; r += 8 * step) {
            f32x4 v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = p[(long)(r + i * step) * q4];
#pragma unroll
            for (int i = 0; i < 8; i++) take(v[i]);
        }
        for (; r < rows; r += step) take(p[(long)r * q4]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (m[e]) atomicMax(t.colmax + 4 * q + e, m[e]);
            top = max(top, m[e]);
        }
    }
    wave_atomic_max(t.amax, top);
}

// The split, and whether one scale keeps the accuracy of a product that sums over
// the rows: a column's values are off by at most 2^-39 of the matrix's largest, so
// columns (other than zero ones) whose largest is within 2^-12 of it keep 2^-27 of
// their own. Values that are not finite, or of no ordinary size, do not fit either.
__global__ void __launch_bounds__(256) k_weights_split(const SplitTensor* d, int* bad) {
    const SplitTensor t = d[blockIdx.y];
    const unsigned top = *t.amax;
    const float least = bits_to_float(top) * 0x1p-12f;
    bool fits = bits_to_float(top) < 1e15f && (top == 0 || bits_to_float(top) > 1e-15f);
    if (blockIdx.x == 0)
        for (int c = threadIdx.x; c < t.K; c += 256)
            fits = fits && (t.colmax[c] == 0 || bits_to_float(t.colmax[c]) >= least);
    if (!fits) atomicOr(bad, 1);
    tensor_split(t);
}
__global__ void __launch_bounds__(256) k_tensor_split(SplitTensor t) { tensor_split(t); }

__global__ void __launch_bounds__(256) k_split_slots(unsigned* slots, long n) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) slots[i] = 0u;
}

// |LayerNorm(x)| <= sqrt(C) max|g| + max|b|
__global__ void __launch_bounds__(256) k_split_ln(const LayerW* layers, const float* lnf_w,
                                                  const float* lnf_b, int L, int C,
                                                  unsigned* amax) {
    __shared__ unsigned red[2];
    const int i = blockIdx.x, l = i >> 1;
    const float* g = i == 2 * L ? lnf_w : i & 1 ? layers[l].ln2_w : layers[l].ln1_w;
    const float* b = i == 2 * L ? lnf_b : i & 1 ? layers[l].ln2_b : layers[l].ln1_b;
    if (threadIdx.x < 2) red[threadIdx.x] = 0;
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += 256) {
        atomicMax(red, __builtin_bit_cast(unsigned, fabsf(g[c])));
        atomicMax(red + 1, __builtin_bit_cast(unsigned, fabsf(b[c])));
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const float top = sqrtf((float)C) * bits_to_float(red[0]) + bits_to_float(red[1]);
        amax[i] = __builtin_bit_cast(unsigned, fabsf(top));
    }
}

__global__ void __launch_bounds__(256) k_split_gelu_bwd(f32x4* __restrict__ d,
                                                        const f32x4* __restrict__ x,
                                                        u32x4* __restrict__ ds, long n8, int cols,
                                                        const unsigned* __restrict__ amax) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    f32x4 v[2] = {d[2 * i], d[2 * i + 1]};
    const f32x4 u[2] = {x[2 * i], x[2 * i + 1]};
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[h][e] *= gelu_grad(u[h][e]);
        d[2 * i + h] = v[h];
    }
    u32x4 hi, lo;
    const float sc = split_scale(*amax);
    split_octet(v[0], v[1], (unsigned)i / (unsigned)(cols >> 3) & 1 ? -sc : sc, hi, lo);
    ds[2 * i] = hi;
    ds[2 * i + 1] = lo;
}

unsigned grid_of(long n, int per) { return (unsigned)std::min((n + per - 1) / per, 2048l); }

template <int EPI, int KM, int WR, int WC, int CB, int S, int OCC>
void run(const SplitGemmArgs& a, int KS, hipStream_t s) {
    const int tm = (a.M + 64 * WR - 1) / (64 * WR), tn = (a.N + 32 * CB * WC - 1) / (32 * CB * WC);
    const int per = (a.K / SP_BK + KS - 1) / KS;
    k_gemm_split<EPI, KM, WR, WC, CB, S, OCC, true>
        <<<(unsigned)(tm * tn * KS), 64 * WR * WC, 0, s>>>(a, tm, tn, per * SP_BK, KS);
}

// (the tile shapes and the splits of K of launch_split_gemm)
template <int EPI, int KM>
hipError_t run_shape(const SplitGemmArgs& a, int plan, hipStream_t s) {
    const int KS = plan & 255;
    switch (plan >> 8) {
        case 0: run<EPI, KM, 4, 2, 4, 4, 1>(a, KS, s); break;
        case 1: run<EPI, KM, 4, 2, 3, 4, 1>(a, KS, s); break;
        case 2: run<EPI, KM, 2, 2, 3, 3, 2>(a, KS, s); break;
        case 3: run<EPI, KM, 2, 2, 2, 3, 3>(a, KS, s); break;
        default: run<EPI, KM, 1, 2, 2, 3, 4>(a, KS, s); break;
    }
    return hipGetLastError();
}

template <int EPI, int KM>
hipError_t run_epi(const SplitGemmArgs& a, int plan, hipStream_t s) {
    const int KS = plan & 255;
    if (KS == 1) return run_shape<EPI, KM>(a, plan, s);
    const hipError_t e = run_shape<EPI_STORE, KM>(a, plan, s);
    if (e != hipSuccess) return e;
    const long n = (long)a.M * (a.N / 8);
    k_split_reduce<EPI><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(a, KS);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_split_train(const SplitGemmArgs& a, hipStream_t s) {
    if (a.M <= 0 || a.N <= 0) return hipSuccess;
    if (a.K <= 0 || a.K % SP_BK || !a.xmax || !a.wmax || a.seg || a.ln_out || a.out_scale)
        return hipErrorInvalidValue;
    if (a.N % 8 || a.ldy % 4 || (size_t)a.Y % 16 || (size_t)a.bias % 16) return hipErrorInvalidValue;
    if ((a.km & 1) && (a.ldx % 8 || a.ldx < a.M)) return hipErrorInvalidValue;
    if (a.ldw % 8 || a.ldw < a.N) return hipErrorInvalidValue;
    const int plan = launch_split_gemm_plan(a);
    if (a.km == 2 && a.epi == EPI_STORE) return run_epi<EPI_STORE, 2>(a, plan, s);
    if (a.km == 3 && a.epi == EPI_RESID && a.bias && !a.amax) return run_epi<EPI_RESID, 3>(a, plan, s);
    return hipErrorInvalidValue;
}

hipError_t launch_split_weights(const SplitTensor* d, int count, unsigned* colmax, long ncol, int* bad,
                                hipStream_t s) {
    if (count <= 0) return hipSuccess;
    const hipError_t e = launch_split_slots(colmax, ncol, s);
    if (e != hipSuccess) return e;
    k_weights_max<<<dim3(32, count), 256, 0, s>>>(d);
    k_weights_split<<<dim3(256, count), 256, 0, s>>>(d, bad);
    return hipGetLastError();
}

hipError_t launch_split_tensor(const SplitTensor& t, bool measure, hipStream_t s) {
    if (t.n <= 0) return hipSuccess;
    if ((t.n & 7) || (t.alt & 7) || t.n >> 35) return hipErrorInvalidValue;
    if (measure) k_tensor_max<<<(unsigned)std::min((t.n + 4095) / 4096, 256l), 1024, 0, s>>>(t);
    k_tensor_split<<<grid_of(t.n, 256 * 8), 256, 0, s>>>(t);
    return hipGetLastError();
}

hipError_t launch_split_slots(unsigned* slots, long n, hipStream_t s) {
    k_split_slots<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(slots, n);
    return hipGetLastError();
}

hipError_t launch_split_ln(const LayerW* layers, const float* lnf_w, const float* lnf_b, int L, int C,
                           unsigned* amax, hipStream_t s) {
    k_split_ln<<<2 * L + 1, 256, 0, s>>>(layers, lnf_w, lnf_b, L, C, amax);
    return hipGetLastError();
}

hipError_t launch_split_gelu_bwd(float* d, const float* x, float* ds, long n, int cols,
                                 const unsigned* amax, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (cols <= 0 || (cols & 7) || n % cols || n >> 35) return hipErrorInvalidValue;
    k_split_gelu_bwd<<<(unsigned)((n / 8 + 255) / 256), 256, 0, s>>>((f32x4*)d, (const f32x4*)x,
                                                                     (u32x4*)ds, n / 8, cols, amax);
    return hipGetLastError();
}
