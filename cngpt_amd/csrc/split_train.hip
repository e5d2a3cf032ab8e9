// split_train.hip - the training backward's products on the fp16 matrix cores
// (split_gemm.h), and the passes that bring its tensors into split rows.
//
// Weights, activations and gradients change with every step, so their scales (powers
// of two from the largest magnitudes) are found on the device in the same step. Small
// rows and columns have to keep their accuracy, since the update divides each
// gradient by its own size, so a scale is shared only over what a product sums:
//   dW[o][i] = sum over rows n of dY[n][o] X[n][i]: one scale for each column of dY
//   and of X, each a factor of a whole row or column of dW. (One scale per tensor lost
//   columns far below the tensor's largest: a LayerNorm gain 2^-28 of the others
//   left 1.3e-2 of error in its columns of dW, a hidden unit that never opens all of its
//   column; fp32 1e-6.)
//   dX[n][i] = sum over outputs o of dY[n][o] W[o][i]: one scale for each row of dY
//   (a second copy of it), and one for W, whose rows and columns must not be too far
//   apart (k_weights_split); others keep the fp32 products.
// A value loses bits of lo once it is 2^-16 below the largest that shares its scale
// (2^-40 of that at most), so a product's error stays within 2^-24 of its operands'
// norms.
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

__global__ void __launch_bounds__(256) k_tensor_split(SplitTensor t) {
    const float sc = split_scale(*t.amax);
    const long n8 = t.n >> 3;
    const f32x4* p = (const f32x4*)t.src;
    u32x4* o = (u32x4*)t.dst;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n8; i += (long)gridDim.x * 256) {
        u32x4 hi, lo;
        const bool odd = t.alt && ((unsigned)i / (unsigned)(t.alt >> 3) & 1);
        const float f = odd ? -sc : sc;
        split_octet(p[2 * i] * f, p[2 * i + 1] * f, hi, lo);
        o[2 * i] = hi;
        o[2 * i + 1] = lo;
    }
}

// Raises colmax[c] to the largest magnitude of column c. A workgroup takes 256
// columns of CM_ROWS rows, a wavefront every fourth row, eight loads in flight. The
// atomics are contiguous and few: over the 48 tensors of a GPT-2 small step at 4096 rows
// (7/4 x 768 columns on average) 6.8, 6.4 and 7.0 us a launch with 32, 64 and 128 rows;
// from the lanes that hold four columns each 13.7 with 32 rows, 9.7 with 64.
constexpr int CM_ROWS = 64;
__global__ void __launch_bounds__(256) k_cols_max(const float* __restrict__ x, int rows, int cols,
                                                  unsigned* __restrict__ colmax) {
    __shared__ unsigned red[4][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = blockIdx.x * 256 + 4 * lane, r0 = blockIdx.y * CM_ROWS;
    const int r1 = min(rows, r0 + CM_ROWS);
    u32x4 m = {0, 0, 0, 0};
    if (c < cols) {
        for (int r = r0 + wave; r < r1; r += 32) {
            f32x4 v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = *(const f32x4*)(x + (long)min(r + 4 * i, r1 - 1) * cols + c);
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    m[e] = max(m[e], __builtin_bit_cast(unsigned, (float)v[i][e]) & 0x7fffffffu);
        }
    }
    *(u32x4*)(red[wave] + 4 * lane) = m;
    __syncthreads();
    const int t = threadIdx.x;
    const unsigned top = max(max(red[0][t], red[1][t]), max(red[2][t], red[3][t]));
    if (top) atomicMax(colmax + blockIdx.x * 256 + t, top);  // (zero past the last column)
}

// The copies of activations and gradients x [rows][cols] (a.cols, a multiple of 8), odd
// rows negated: by_col with a scale per column, rows .. rows_p-1 of it zero, and, if
// wanted, by_row with a scale per row, whose largest magnitudes go to rowmax. One
// wavefront per row. Bound by memory (4096 rows
// of 768 to 3072 columns, half of them both copies: 13.4 us on average, 4.8 TB/s).
__global__ void __launch_bounds__(256) k_split_rows(SplitRows a) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= a.rows_p) return;
    u32x4* col = (u32x4*)(a.by_col + (long)r * a.cols);
    if (r >= a.rows) {
        for (int q = lane; q < a.cols >> 2; q += 64) col[q] = u32x4{0, 0, 0, 0};
        return;
    }
    const f32x4* x = (const f32x4*)(a.src + (long)r * a.cols);
    const float sign = r & 1 ? -1.f : 1.f;
    float rs = sign;
    if (a.by_row) {
        unsigned m = 0;
        for (int q = lane; q < a.cols >> 2; q += 64) m = max(m, abs_bits(x[q]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
        if (lane == 0) a.rowmax[r] = m;
        rs *= split_scale(m);
    }
    u32x4* row = (u32x4*)(a.by_row + (long)r * a.cols);
    for (int q = 2 * lane; q < a.cols >> 2; q += 128) {
        const f32x4 v0 = x[q], v1 = x[q + 1];
        const u32x4 m0 = ((const u32x4*)a.colmax)[q], m1 = ((const u32x4*)a.colmax)[q + 1];
        f32x4 c0, c1;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            c0[e] = v0[e] * (sign * split_scale(m0[e]));
            c1[e] = v1[e] * (sign * split_scale(m1[e]));
        }
        u32x4 hi, lo;
        split_octet(c0, c1, hi, lo);
        col[q] = hi;
        col[q + 1] = lo;
        if (a.by_row) {
            split_octet(v0 * rs, v1 * rs, hi, lo);
            row[q] = hi;
            row[q + 1] = lo;
        }
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
// the rows, one wavefront per row. A column's values are off by at most 2^-40 of the
// matrix's largest, so columns (other than zero ones) whose largest is within 2^-12 of
// it keep 2^-28 of their own. The other operand's scale follows its largest value,
// whose share of a sum is of the size of its row of this matrix: rows whose largest is
// within 2^-10 keep the values of a sum far below it at 2^-30 of that share. Values that
// are not finite, or of no ordinary size, do not fit either.
__global__ void __launch_bounds__(256) k_weights_split(const SplitTensor* d, int* bad) {
    const SplitTensor t = d[blockIdx.y];
    const int rows = (int)(t.n / t.K), lane = threadIdx.x & 63;
    const unsigned top = *t.amax;
    const float sc = split_scale(top);
    bool fits = bits_to_float(top) < 1e15f && (top == 0 || bits_to_float(top) > 1e-15f);
    if (blockIdx.x == 0)
        for (int c = threadIdx.x; c < t.K; c += 256)
            fits = fits && (t.colmax[c] == 0 || bits_to_float(t.colmax[c]) >= bits_to_float(top) * 0x1p-12f);
    for (int r = blockIdx.x * 4 + (threadIdx.x >> 6); r < rows; r += gridDim.x * 4) {
        const f32x4* x = (const f32x4*)(t.src + (long)r * t.K);
        u32x4* o = (u32x4*)(t.dst + (long)r * t.K);
        unsigned m = 0;
        for (int q = 2 * lane; q < t.K >> 2; q += 128) {
            const f32x4 v0 = x[q], v1 = x[q + 1];
            m = max(m, max(abs_bits(v0), abs_bits(v1)));
            u32x4 hi, lo;
            split_octet(v0 * sc, v1 * sc, hi, lo);
            o[q] = hi;
            o[q + 1] = lo;
        }
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, s, 64));
        fits = fits && bits_to_float(m) >= bits_to_float(top) * 0x1p-10f;
    }
    if (!fits) atomicOr(bad, 1);
}

__global__ void __launch_bounds__(256) k_clear_max(unsigned* slots, long n) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) slots[i] = 0u;
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
    if ((a.xstep | a.wstep) & ~1 || (a.wstep && (size_t)a.wmax % 16)) return hipErrorInvalidValue;
    if ((a.km & 1) && (a.ldx % 8 || a.ldx < a.M)) return hipErrorInvalidValue;
    if (a.ldw % 8 || a.ldw < a.N) return hipErrorInvalidValue;
    const int plan = launch_split_gemm_plan(a);
    if (a.km == 2 && a.epi == EPI_STORE) return run_epi<EPI_STORE, 2>(a, plan, s);
    if (a.km == 3 && a.epi == EPI_RESID && a.bias && !a.amax) return run_epi<EPI_RESID, 3>(a, plan, s);
    return hipErrorInvalidValue;
}

hipError_t launch_split_weights(const SplitTensor* d, int count, int* bad, hipStream_t s) {
    if (count <= 0) return hipSuccess;
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

hipError_t launch_cols_max(const float* x, int rows, int cols, unsigned* colmax, hipStream_t s) {
    if (rows <= 0 || cols <= 0) return hipSuccess;
    if ((cols & 3) || (size_t)x % 16) return hipErrorInvalidValue;
    k_cols_max<<<dim3((cols + 255) / 256, (rows + CM_ROWS - 1) / CM_ROWS), 256, 0, s>>>(x, rows, cols,
                                                                                       colmax);
    return hipGetLastError();
}

hipError_t launch_split_rows(const SplitRows& a, hipStream_t s) {
    if (a.rows <= 0) return hipSuccess;
    if ((a.cols & 7) || a.rows_p < a.rows || !a.by_col || !a.by_row != !a.rowmax || (size_t)a.src % 16 ||
        (size_t)a.by_col % 16 || (size_t)a.by_row % 16 || (size_t)a.colmax % 16)
        return hipErrorInvalidValue;
    k_split_rows<<<(unsigned)((a.rows_p + 3) / 4), 256, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_clear_max(unsigned* slots, long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    k_clear_max<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(slots, n);
    return hipGetLastError();
}
