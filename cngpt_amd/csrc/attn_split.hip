// attn_split.hip - causal self-attention on the fp16 matrix cores, every
// operand a pair of fp16 values (split.h). The computation of k_attn_causal
// (attention.hip: online softmax in base 2 over tiles of keys, S^T = K Q^T
// so that a lane owns one query, probabilities fed to O^T += V^T P^T from the
// accumulators) with each product as hi hi + hi lo + lo hi.
#include "common.h"
#include "kernels.h"
#include "split.h"

namespace {

// hi and lo operands of 8 values
struct Pair8 {
    f16x8 h, l;
};
__device__ __forceinline__ Pair8 split8(const float (&v)[8]) {
    u32x4 h, l;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        unsigned hp, lp;
        split_pair(v[2 * e], v[2 * e + 1], hp, lp);
        h[e] = hp;
        l[e] = lp;
    }
    return Pair8{__builtin_bit_cast(f16x8, h), __builtin_bit_cast(f16x8, l)};
}

__device__ __forceinline__ f32x16 mfma(const f16x8& a, const f16x8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// One workgroup = 4 wavefronts = 128 queries of one (sequence, head). The qkv
// rows are split rows (the QKV product writes them), so a tile of KT keys goes
// from global memory straight into LDS (lds_dma16, double-buffered): K and V
// rows of HS / 4 granules (granule 2 o + p: octet o of d, plane p). K granules
// are XOR-swizzled by key, so that the rows a read touches at one granule fall
// in different banks. V is read turned (read_turned: a lane gets four keys at
// its d), the keys 16 t + 4 lh + {0..3, 8..11} of step t, which are those the
// lane's half lh holds of S^T in accumulator registers 8 (t % 2) .. +7; its
// granules are swizzled by key % 4, over bits that the 32 d of a read leave
// free. Splitting fp32 rows while staging them instead took 147 of the 440
// vector instructions a wavefront issues per tile, and those are the bound
// (GPT-2 small B=16 T=1024: 113 us against 98 per layer; 285 in fp32).
//
// scales: q, k and v carry scales[0], [1] and [2] (powers of two); the output
// is split rows times scales[2]. A probability carries a factor 2^12, which
// cancels against the sum, so that lo keeps its bits down to 2^-26 of the
// row's largest. The running max is moved only when some score of the
// wavefront passes it by more than 3 (probabilities up to 2^15 then, and half a
// unit of the maximum's last place in the exponent more: k_split_scores holds
// scores below 2^22), which leaves the output unscaled on most tiles.
template <int HS, int KT, int OCC>
__global__ void __launch_bounds__(256, OCC)
    k_attn_split(const float* __restrict__ qkv, float* __restrict__ out, int B, int T, int C, int H,
                 int nqb, const float* __restrict__ scales) {
    constexpr int ST = HS / 16;         // 16-d steps of a score
    constexpr int NKB = KT / 32;        // 32-key blocks of a tile
    constexpr int NDB = HS / 32;        // 32-row blocks of O^T
    constexpr int GK = HS / 4;          // granules of a row
    constexpr int RB = HS * 4;          // bytes of a row
    constexpr int KB = KT * RB;         // bytes of a K (or V) tile
    constexpr int NI = KT * GK / 256;   // load instructions per wavefront for each
    __shared__ __attribute__((aligned(1024))) char sm[2][2 * KB];
    auto swk = [](int key) { return GK >= 16 ? key & 15 : (key / (16 / GK)) & (GK - 1); };
    auto swv = [](int key) {
        const int k0 = key & 1, k1 = (key >> 1) & 1;
        return GK >= 16 ? k0 | (k1 << 3) : k1;
    };

    const int BH = B * H;
    const int qb = nqb - 1 - (int)(blockIdx.x / BH);  // longest query blocks first
    const int bh = blockIdx.x % BH;
    const int b = bh / H, h = bh % H;
    const long C3 = 3L * C;
    const char* base = (const char*)(qkv + (long)b * T * C3 + h * HS);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int lr = lane & 31, lh = lane >> 5;
    const int q0 = qb * 128 + wave * 32, qi = q0 + lr;
    const int ntiles = min(qb * 128 + 127, T - 1) / KT + 1;
    // scores in units of log2
    const float cs = 1.4426950408889634f / (sqrtf((float)HS) * scales[0] * scales[1]);

    // load instruction i of this wavefront covers granules (4 i + wave) 64 ..
    // +63 of a tile; keys past T re-read the last one (masked below)
    auto issue = [&](int kt, int buf) {
        char* ks = sm[buf];
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int g = (4 * i + wave) * 64 + lane, key = g / GK, slot = g % GK;
            const char* row = base + (long)min(kt * KT + key, T - 1) * C3 * 4;
            lds_dma16(row + 4 * C + 16 * (slot ^ swk(key)), (float*)(ks + (4 * i + wave) * 1024));
            lds_dma16(row + 8 * C + 16 * (slot ^ swv(key)), (float*)(ks + KB + (4 * i + wave) * 1024));
        }
    };

    issue(0, 0);
    Pair8 q[ST];
    const char* qp = base + (long)min(qi, T - 1) * C3 * 4 + 32 * lh;
#pragma unroll
    for (int s = 0; s < ST; s++) {
        q[s].h = *(const f16x8*)(qp + 64 * s);
        q[s].l = *(const f16x8*)(qp + 64 * s + 16);
    }
    // this lane's hi granules: of K row lr, and of the turned reads (lo: bit 4
    // flipped; d block j: bits 7 and up flipped by j)
    const int ko = lr * RB + 16 * ((2 * lh) ^ swk(lr));
    const int vkey = 4 * lh + ((lane >> 2) & 3);
    const int vo = vkey * RB + 16 * ((4 * ((lane >> 4) & 1) + (lane & 2)) ^ swv(vkey)) + 8 * (lane & 1);

    f32x16 o[NDB];
#pragma unroll
    for (int j = 0; j < NDB; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[j][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    wait_vmcnt<0>();
    __syncthreads();
    for (int kt = 0; kt < ntiles; kt++) {
        const int cur = kt & 1;
        if (kt + 1 < ntiles) issue(kt + 1, cur ^ 1);
        // Wave-uniform: skip tiles entirely above this wavefront's queries.
        if (q0 < T && kt * KT <= q0 + 31) {
            const char* ks = sm[cur];
            const char* vs = ks + KB;
            f32x16 s[NKB];
#pragma unroll
            for (int kb = 0; kb < NKB; kb++)
#pragma unroll
                for (int r = 0; r < 16; r++) s[kb][r] = 0.f;
#pragma unroll
            for (int t = 0; t < ST; t++) {
                Pair8 k[NKB];
#pragma unroll
                for (int kb = 0; kb < NKB; kb++) {
                    // granule 2 (2 t + lh): 64 t bytes on, under the swizzle
                    const char* p = ks + kb * 32 * RB + (ko ^ (64 * t));
                    k[kb].h = *(const f16x8*)p;
                    k[kb].l = *(const f16x8*)(ks + kb * 32 * RB + (ko ^ (64 * t) ^ 16));
                }
#pragma unroll
                for (int kb = 0; kb < NKB; kb++) s[kb] = mfma(k[kb].l, q[t].h, s[kb]);
#pragma unroll
                for (int kb = 0; kb < NKB; kb++) s[kb] = mfma(k[kb].h, q[t].l, s[kb]);
#pragma unroll
                for (int kb = 0; kb < NKB; kb++) s[kb] = mfma(k[kb].h, q[t].h, s[kb]);
            }
            // s[kb][r]: key kt*64 + 32 kb + 8 (r/4) + 4 lh + r%4, query qi
            if (kt * KT + KT - 1 > q0) {
#pragma unroll
                for (int kb = 0; kb < NKB; kb++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int key = kt * KT + kb * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                        s[kb][r] = (key > qi) ? -INFINITY : s[kb][r];
                    }
            }
            float mt = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < NKB; kb++)
#pragma unroll
                for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[kb][r]);
            mt = fmaxf(mt, __shfl_xor(mt, 32, 64)) * cs;
            if (__any(mt > m_run + 3.f)) {
                const float m_new = fmaxf(m_run, mt);
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int j = 0; j < NDB; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[j][r] *= alpha;
            }
            const float off = 12.f - m_run;
            float ps = 0.f;
            Pair8 p[2 * NKB];
#pragma unroll
            for (int t = 0; t < 2 * NKB; t++) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    v[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t >> 1][8 * (t & 1) + e], cs, off));
                    ps += v[e];
                }
                p[t] = split8(v);
            }
            l_run += ps;
#pragma unroll
            for (int t = 0; t < 2 * NKB; t++) {
                Pair8 v[NDB];
#pragma unroll
                for (int j = 0; j < NDB; j++) {
                    const char* p0 = vs + t * 16 * RB + (vo ^ (128 * j));
                    v[j].h = read_turned(p0, 8 * RB);
                    v[j].l = read_turned(vs + t * 16 * RB + (vo ^ (128 * j) ^ 16), 8 * RB);
                }
#pragma unroll
                for (int j = 0; j < NDB; j++) o[j] = mfma(v[j].l, p[t].h, o[j]);
#pragma unroll
                for (int j = 0; j < NDB; j++) o[j] = mfma(v[j].h, p[t].l, o[j]);
#pragma unroll
                for (int j = 0; j < NDB; j++) o[j] = mfma(v[j].h, p[t].h, o[j]);
            }
        }
        wait_vmcnt<0>();
        __syncthreads();
    }

    // o[j][r]: d = 32 j + 8 (r / 4) + 4 lh + r % 4 of query qi, times v's
    // scale, which is the output's; each half of the lanes holds the sum over
    // its own keys (both lanes of a query take the same branch)
    l_run += __shfl_xor(l_run, 32, 64);
    if (qi < T) {
        const float inv = 1.0f / l_run;
        float* op = out + ((long)b * T + qi) * C + h * HS;
#pragma unroll
        for (int j = 0; j < NDB; j++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                unsigned h0, h1, l0, l1;
                split_pair(o[j][4 * g] * inv, o[j][4 * g + 1] * inv, h0, l0);
                split_pair(o[j][4 * g + 2] * inv, o[j][4 * g + 3] * inv, h1, l1);
                swap32(h0, l0);
                swap32(h1, l1);
                *(u32x4*)(op + 32 * j + 8 * g + 4 * lh) = u32x4{h0, h1, l0, l1};
            }
    }
}

}  // namespace

bool attention_split_takes(int HS) { return HS == 32 || HS == 64 || HS == 128; }

hipError_t launch_attention_split(const float* qkv, float* out, int B, int T, int C, int H,
                                  const float* scales, hipStream_t s) {
    if (B <= 0 || T <= 0) return hipSuccess;
    const int nqb = (T + 127) / 128;
    const unsigned grid = (unsigned)nqb * B * H;
    switch (C / H) {
        case 32:
            k_attn_split<32, 64, 4><<<grid, 256, 0, s>>>(qkv, out, B, T, C, H, nqb, scales);
            break;
        case 64:
            k_attn_split<64, 64, 2><<<grid, 256, 0, s>>>(qkv, out, B, T, C, H, nqb, scales);
            break;
        case 128:
            k_attn_split<128, 32, 2><<<grid, 256, 0, s>>>(qkv, out, B, T, C, H, nqb, scales);
            break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
