// split.h - fp32 values as pairs of fp16 values (hi + lo), the operand form of
// the products on the fp16 matrix cores (split.hip).
//
// A split row of K values (K a multiple of 16) has the bytes of K floats: each
// group of 8 values is 16 bytes of hi halves, then 16 bytes of lo halves, so a
// lane's operand of a 16-k matrix instruction is one 16-byte granule.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// hi and lo halves of two values (round to nearest, so that lo is at most
// half a unit of hi's last place): |v - hi - lo| <= 2^-23 |v| while |v| <=
// 2^15 and lo is a normal fp16, at most 2^-25 below that. The values are pinned
// to their fp32 roundings first: a product that the compiler forms again,
// rounded straight to fp16, for one of its two uses can round to the other side
// of a tie, and hi would be off by a whole unit.
__device__ __forceinline__ void split_pair(float x, float y, unsigned& hi, unsigned& lo) {
    asm("" : "+v"(x), "+v"(y));
    const f16x2 hp = {(_Float16)x, (_Float16)y};
    hi = __builtin_bit_cast(unsigned, hp);
    float dx, dy;  // v - hi: exact
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(dx) : "v"(hi), "v"(x));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(dy) : "v"(hi), "v"(y));
    const f16x2 l = {(_Float16)dx, (_Float16)dy};
    lo = __builtin_bit_cast(unsigned, l);
}

// lanes 32-63 of a <-> lanes 0-31 of b
__device__ __forceinline__ void swap32(unsigned& a, unsigned& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// Four consecutive values (columns c .. c + 3 of a split row, c = 4 x the
// lane's place in the row, neighbouring lanes holding neighbouring quads):
// an even lane gets the pair's hi granule, an odd lane its lo granule, each
// stored at the byte offset 4 c of the row. Both lanes of a pair are active.
__device__ __forceinline__ u32x4 split_quad(const f32x4& v, int lane) {
    unsigned h0, h1, l0, l1;
    split_pair(v[0], v[1], h0, l0);
    split_pair(v[2], v[3], h1, l1);
    const bool odd = lane & 1;
    const unsigned s0 = odd ? h0 : l0, s1 = odd ? h1 : l1;
    const unsigned r0 = __builtin_amdgcn_mov_dpp(s0, 0xB1, 0xF, 0xF, false);
    const unsigned r1 = __builtin_amdgcn_mov_dpp(s1, 0xB1, 0xF, 0xF, false);
    return odd ? u32x4{r0, r1, l0, l1} : u32x4{h0, h1, r0, r1};
}

typedef __fp16 h16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) h16x4 lds_h16x4;

// Rows r and r + 4 of a 4-row x 16-lane corner turn: each lane reads 8 bytes
// of its row (ds_read_b64_tr_b16: within 16 lanes, lane s reads row s / 4, four
// halves from 4 (s % 4); lane i receives half i of the four rows).
__device__ __forceinline__ f16x8 read_turned(const char* p, int second) {
    const h16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h16x4*)p);
    const h16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h16x4*)(p + second));
    f16x8 r;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        r[e] = (_Float16)a[e];
        r[4 + e] = (_Float16)b[e];
    }
    return r;
}

// The scale of values whose largest magnitude has the bits amax, 2 to the
// power of this: it takes that into [2^14, 2^15) (held where the scale is a normal
// float); 0 for zero, infinity and NaN.
__device__ __forceinline__ int split_exp(unsigned amax) {
    return amax - 1u < 0x7f7fffffu ? min(141 - (int)(amax >> 23), 127) : 0;
}
__device__ __forceinline__ float split_scale(unsigned amax) {
    return __builtin_bit_cast(float, (unsigned)(split_exp(amax) + 127) << 23);
}

// Largest magnitude of four values, as bits (ordered as the values are, NaN
// above infinity), and the wavefront's into *dst (no order: a maximum).
__device__ __forceinline__ unsigned abs_bits(const f32x4& v) {
    unsigned m = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) m = max(m, __builtin_bit_cast(unsigned, (float)v[e]) & 0x7fffffffu);
    return m;
}
__device__ __forceinline__ void wave_atomic_max(unsigned* dst, unsigned v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (unsigned)__shfl_xor((int)v, o, 64));
    if ((threadIdx.x & 63) == 0 && v) atomicMax(dst, v);
}
// The same of a workgroup of NW wavefronts.
template <int NW>
__device__ __forceinline__ void block_atomic_max(unsigned* dst, unsigned v) {
    __shared__ unsigned red[NW];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (unsigned)__shfl_xor((int)v, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < NW; w++) v = max(v, red[w]);
        if (v) atomicMax(dst, v);
    }
}

// Eight values as the two granules of an octet.
__device__ __forceinline__ void split_octet(const f32x4& a, const f32x4& b, u32x4& hi, u32x4& lo) {
#pragma unroll
    for (int e = 0; e < 2; e++) {
        unsigned h, l;
        split_pair(a[2 * e], a[2 * e + 1], h, l);
        hi[e] = h;
        lo[e] = l;
        split_pair(b[2 * e], b[2 * e + 1], h, l);
        hi[2 + e] = h;
        lo[2 + e] = l;
    }
}
