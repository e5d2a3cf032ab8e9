// split.cpp - test-only C entry points into the split-operand products
// (split.hip): operands split on the device as the forward splits them, the
// product through launch_split_gemm, split outputs joined again on the host.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "../../cngpt_amd/csrc/common.h"
#include "../../cngpt_amd/csrc/ctx_view.h"
#include "../../cngpt_amd/csrc/kernels.h"

namespace {

struct Dev {
    std::vector<void*> ptrs;
    bool ok = true;
    ~Dev() {
        for (void* p : ptrs) (void)hipFree(p);
    }
    template <class T>
    T* put(const T* host, size_t n) {
        void* p = nullptr;
        if (hipMalloc(&p, n * sizeof(T) + 16) != hipSuccess) return ok = false, nullptr;
        ptrs.push_back(p);
        const hipError_t e = host ? hipMemcpy(p, host, n * sizeof(T), hipMemcpyHostToDevice)
                                  : hipMemset(p, 0, n * sizeof(T));
        if (e != hipSuccess) ok = false;
        return (T*)p;
    }
};

float join(const _Float16* row, int c, float scale) {
    const _Float16* g = row + c / 8 * 16 + c % 8;
    return ((float)g[0] + (float)g[8]) / scale;
}

}  // namespace

extern "C" {

// K splits (low byte) and tile shape (second byte) that a plain product takes.
int kat_split_plan(int M, int N, int K) {
    SplitGemmArgs a{};
    a.M = M; a.N = N; a.K = K; a.ldy = N;
    a.part = (float*)16; a.part_cap = 1 << 24;
    return launch_split_gemm_plan(a);
}

// Y = epi(X . W^T), rows of Y ldy floats apart at the row mapping of seg /
// seg_stride (Y holds y_rows rows). xbound: the largest |X| the scales allow
// for. With lnout, also LayerNorm(Y rows) (gains lnw, biases lnb): formed in
// the split-K sum, or by the LayerNorm launch. Returns the verdict on W (0:
// accurate), -1 on failure.
int kat_split_gemm(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K,
                   int ldy, int seg, int seg_stride, int y_rows, int epi, float xbound,
                   const float* lnw, const float* lnb, float* lnout) {
    Dev d;
    std::vector<float> ones(K > N ? K : N, 1.f);
    float* dw = d.put(W, (size_t)N * K);
    float* db = d.put(bias, N);
    float* dy = d.put(Y, (size_t)y_rows * ldy);
    float* dxs = d.put<float>(nullptr, (size_t)M * K);
    float* dws = d.put<float>(nullptr, (size_t)N * K);
    float* winv = d.put<float>(nullptr, N);
    float* typ = d.put(ones.data(), K);
    const float scale = ldexpf(1.f, 14 - ilogbf(xbound));
    const float oscale = 64.f, qkv_scale[3] = {64.f, 256.f, 32.f};
    float* bound = d.put(&xbound, 1);
    float* xs = d.put(&scale, 1);
    float* os = d.put(&oscale, 1);
    int* bad = d.put<int>(nullptr, 2);
    float* part = d.put<float>(nullptr, 1 << 24);
    float* dlw = lnout ? d.put(lnw, N) : nullptr;
    float* dlb = lnout ? d.put(lnb, N) : nullptr;
    float* dln = lnout ? d.put<float>(nullptr, (size_t)M * N) : nullptr;
    if (!d.ok) return -1;
    SplitWeights o{dws, winv};
    if (launch_split_w(dw, o, N, K, typ, nullptr, bound, xs, bad, nullptr) != hipSuccess) return -1;
    std::vector<_Float16> split((size_t)M * K * 2);
    for (int r = 0; r < M; r++)
        for (int k = 0; k < K; k++) {
            const float v = X[(size_t)r * K + k] * scale;
            _Float16* g = &split[((size_t)r * K + k / 8 * 8) * 2 + k % 8];
            g[0] = (_Float16)v;
            g[8] = (_Float16)(v - (float)g[0]);
        }
    if (hipMemcpy(dxs, split.data(), split.size() * 2, hipMemcpyHostToDevice) != hipSuccess) return -1;
    SplitGemmArgs a{};
    a.X = dxs; a.W = dws; a.winv = winv; a.bias = db; a.Y = dy;
    a.M = M; a.N = N; a.K = K;
    a.ldy = ldy;
    a.seg = seg; a.seg_stride = seg_stride;
    a.epi = epi;
    a.out_scale = epi == EPI_BIAS_GELU ? os : epi == EPI_QKV ? d.put(qkv_scale, 3) : nullptr;
    if (epi == EPI_QKV) a.Ys = dln;
    if (!d.ok) return -1;
    a.part = part; a.part_cap = 1 << 24;
    const bool ln = lnout && epi != EPI_QKV;
    const bool in_sum = ln && launch_split_gemm_splits(a) > 1;
    if (in_sum) {
        a.ln_w = dlw; a.ln_b = dlb; a.ln_out = dln; a.ln_scale = os;
    }
    if (launch_split_gemm(a, nullptr) != hipSuccess) return -1;
    if (ln && !in_sum &&
        launch_layernorm(dy, ldy, dlw, dlb, dln, N, M, N, nullptr, nullptr, nullptr, os) != hipSuccess)
        return -1;
    int verdict = 0;
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(&verdict, bad, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(Y, dy, (size_t)y_rows * ldy * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    std::vector<_Float16> row(2 * (size_t)N);
    auto join_rows = [&](float* rows, int n, long stride) {
        for (int r = 0; r < n; r++) {
            float* p = rows + r * stride;
            memcpy(row.data(), p, (size_t)N * sizeof(float));
            for (int c = 0; c < N; c++)
                p[c] = join(row.data(), c, epi == EPI_QKV ? qkv_scale[c / (N / 3)] : oscale);
        }
    };
    if (epi == EPI_BIAS_GELU) join_rows(Y, M, ldy);
    if (lnout) {
        if (hipMemcpy(lnout, dln, (size_t)M * N * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
            return -1;
        join_rows(lnout, M, N);
    }
    return verdict;
}

// The training backward's products (launch_split_train) in Y [M][N], and the fp32
// product of the same operands in Y32: km 2, Y = X [M][K] . W [K][ldw]; km 3, Y
// += X [K][ldx]^T . W [K][ldw]. Returns the largest |Y| that the launch reports as
// bits (km 2), 0 otherwise; -1 on failure.
long kat_split_train(const float* X, const float* W, float* Y, float* Y32, int M, int N, int K, int ldx,
                     int ldw, int km) {
    Dev d;
    const long nx = km == 3 ? (long)K * ldx : (long)M * K, nw = (long)K * ldw;
    std::vector<float> zero(N, 0.f);
    float *dx = d.put(X, nx), *dw = d.put(W, nw), *dy = d.put(Y, (size_t)M * N), *dy2 = d.put(Y32, (size_t)M * N);
    float *dxs = d.put<float>(nullptr, nx), *dws = d.put<float>(nullptr, nw), *db = d.put(zero.data(), N);
    float* part = d.put<float>(nullptr, 1 << 24);
    unsigned* slot = d.put<unsigned>(nullptr, 3);
    if (!d.ok) return -1;
    SplitTensor tx{}, tw{};
    tx.src = dx; tx.dst = dxs; tx.n = nx; tx.amax = slot; tx.alt = km == 3 ? ldx : K;
    tw.src = dw; tw.dst = dws; tw.n = nw; tw.amax = slot + 1; tw.alt = km == 3 ? ldw : 0;
    if (launch_split_tensor(tx, true, nullptr) != hipSuccess || launch_split_tensor(tw, true, nullptr) != hipSuccess)
        return -1;
    SplitGemmArgs a{};
    a.X = dxs; a.W = dws; a.Y = dy; a.bias = db;
    a.M = M; a.N = N; a.K = K;
    a.ldy = N; a.ldx = ldx; a.ldw = ldw; a.km = km;
    a.epi = km == 3 ? EPI_RESID : EPI_STORE;
    a.xmax = slot; a.wmax = slot + 1;
    if (km == 2) a.amax = slot + 2;
    a.part = part; a.part_cap = 1 << 24;
    if (launch_split_train(a, nullptr) != hipSuccess) return -1;
    if (K % 32 == 0 && M > SKINNY_MAX_M) {
        GemmArgs g{};
        g.X = dx; g.W = dw; g.Y = dy2; g.bias = db;
        g.M = M; g.N = N; g.K = K;
        g.ldy = N; g.ldx = ldx; g.ldw = ldw; g.km = km;
        g.epi = a.epi;
        g.part = part; g.part_cap = 1 << 24;
        if (launch_gemm(g, nullptr) != hipSuccess) return -1;
    }
    unsigned top = 0;
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(Y, dy, (size_t)M * N * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(Y32, dy2, (size_t)M * N * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(&top, slot + 2, sizeof(top), hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    return top;
}

// The same products with the scales of the training step: km 2, a scale per row of X
// [M][K] and one for W [K][ldw]; km 3, one per column of X [K][ldx] and of W. X holds
// K - pad rows (M - pad with km 2), which launch_split_rows pads with zero rows.
int kat_split_train_rows(const float* X, const float* W, float* Y, int M, int N, int K, int ldx, int ldw,
                         int km, int pad) {
    Dev d;
    const int xrows = km == 3 ? K : M, xcols = km == 3 ? ldx : K;
    std::vector<float> zero(N, 0.f);
    float *dx = d.put(X, (size_t)(xrows - pad) * xcols), *dw = d.put(W, (size_t)K * ldw);
    float *dy = d.put(Y, (size_t)M * N), *db = d.put(zero.data(), N);
    std::vector<unsigned> ff((size_t)xrows * xcols, 0xffffffffu);  // (padding must be written)
    float* xcol = (float*)d.put(ff.data(), ff.size());
    float *xrow = d.put<float>(nullptr, (size_t)xrows * xcols), *wcol = d.put<float>(nullptr, (size_t)K * ldw);
    float* part = d.put<float>(nullptr, 1 << 24);
    unsigned *xmax = d.put<unsigned>(nullptr, xcols), *wmax = d.put<unsigned>(nullptr, ldw);
    unsigned* rmax = d.put<unsigned>(nullptr, xrows);
    if (!d.ok) return -1;
    if (launch_cols_max(dx, xrows - pad, xcols, xmax, nullptr) != hipSuccess ||
        launch_split_rows({dx, xrows - pad, xrows, xcols, xmax, xcol, km == 2 ? xrow : nullptr,
                           km == 2 ? rmax : nullptr}, nullptr) != hipSuccess)
        return -1;
    SplitGemmArgs a{};
    a.Y = dy; a.bias = db;
    a.M = M; a.N = N; a.K = K;
    a.ldy = N; a.ldx = ldx; a.ldw = ldw; a.km = km;
    a.X = km == 3 ? xcol : xrow; a.W = wcol;
    a.xmax = km == 3 ? xmax : rmax; a.wmax = wmax;
    a.xstep = 1; a.wstep = km == 3;
    a.epi = km == 3 ? EPI_RESID : EPI_STORE;
    a.part = part; a.part_cap = 1 << 24;
    if (km == 3) {
        if (launch_cols_max(dw, K - pad, ldw, wmax, nullptr) != hipSuccess ||
            launch_split_rows({dw, K - pad, K, ldw, wmax, wcol, nullptr, nullptr}, nullptr) != hipSuccess)
            return -1;
    } else {
        SplitTensor t{};
        t.src = dw; t.dst = wcol; t.n = (long)K * ldw; t.amax = wmax;
        if (launch_split_tensor(t, true, nullptr) != hipSuccess) return -1;
    }
    if (launch_split_train(a, nullptr) != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(Y, dy, (size_t)M * N * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    return 0;
}

// Causal attention over qkv [B, T, 3C] through the split kernel: out [B, T, C].
// smax: the largest magnitude of q, k and v the scales allow for.
int kat_attention_split(const float* qkv, float* out, int B, int T, int C, int H, const float* smax) {
    const size_t rows = (size_t)B * T;
    float scale[3];
    for (int i = 0; i < 3; i++) scale[i] = ldexpf(1.f, 14 - ilogbf(smax[i]));
    std::vector<_Float16> split(rows * 3 * C * 2);
    for (size_t r = 0; r < rows; r++)
        for (int c = 0; c < 3 * C; c++) {
            const float v = qkv[r * 3 * C + c] * scale[c / C];
            _Float16* g = &split[(r * 3 * C + c / 8 * 8) * 2 + c % 8];
            g[0] = (_Float16)v;
            g[8] = (_Float16)(v - (float)g[0]);
        }
    Dev d;
    _Float16* dq = d.put(split.data(), split.size());
    float* ds = d.put(scale, 3);
    float* dout = d.put<float>(nullptr, rows * C);
    if (!d.ok) return -1;
    if (launch_attention_split((const float*)dq, dout, B, T, C, H, ds, nullptr) != hipSuccess ||
        hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(out, dout, rows * C * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    std::vector<_Float16> row(2 * (size_t)C);
    for (size_t r = 0; r < rows; r++) {
        memcpy(row.data(), out + r * C, (size_t)C * sizeof(float));
        for (int c = 0; c < C; c++) out[r * C + c] = join(row.data(), c, scale[2]);
    }
    return 0;
}

// cngpt_hip_forward_noalloc captured on the handle's stream (device pointers as there):
// the graph, null on failure.
hipGraphExec_t kat_capture_noalloc(cngpt_hip_ctx* h, const int* tokens, int B, int T, int mode, float* logits) {
    CtxView v;
    if (ctx_view(h, &v) || hipStreamBeginCapture(v.stream, hipStreamCaptureModeThreadLocal) != hipSuccess)
        return nullptr;
    const int rc = cngpt_hip_forward_noalloc(h, tokens, B, T, mode, logits, nullptr);
    hipGraph_t g = nullptr;
    hipGraphExec_t ex = nullptr;
    if (hipStreamEndCapture(v.stream, &g) != hipSuccess || rc) return nullptr;
    if (hipGraphInstantiate(&ex, g, nullptr, nullptr, 0) != hipSuccess) ex = nullptr;
    (void)hipGraphDestroy(g);
    return ex;
}

int kat_replay(cngpt_hip_ctx* h, hipGraphExec_t ex) {
    CtxView v;
    return ctx_view(h, &v) || hipGraphLaunch(ex, v.stream) != hipSuccess ||
                   hipStreamSynchronize(v.stream) != hipSuccess
               ? -1
               : 0;
}

void kat_drop(hipGraphExec_t ex) { (void)hipGraphExecDestroy(ex); }

}  // extern "C"
