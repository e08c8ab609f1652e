// split.h -- fp32 products on the fp16 matrix cores at fp32 accuracy.
//
// A float x times a power of two s that brings it into fp16's normal range is
// x s = h + l + e, h = fp16(x s), l = fp16(x s - h) (both rounded to nearest),
// |l| <= 2^-11 |x s|, |e| <= max(2^-24 |x s|, 2^-25).  A product is then
//   (x s)(y t) = h h' + (h l' + l h') + O(2^-22 |x s y t|),
// three fp16 MFMAs with fp32 accumulation; the terms cost two VALU operations
// a value, three with the scale.  One fp16 32x32x16 MFMA takes 33 cycles and 16
// contraction indices, one fp32 32x32x2 MFMA 65 and 2; on random data the
// matrix clocks reach 1.62 PFLOP/s (fp16) and 154 TFLOP/s (fp32), so the ceiling
// of fp32 products rises from 154 to 540 TFLOP/s.  fp32 MFMAs also keep the
// vector ALUs from issuing; these do not (8 MFMAs with 64 v_fma interleaved,
// cycles: 820 against 520 + 268 apart; 340 against 264 + 268).
//
// Error against 64-bit sums on tiles of normal deviates, relative 2-norm,
// fp32 MFMA -> this: K = 32 1.02e-7 -> 0.94e-7, K = 64 1.44e-7 -> 1.12e-7,
// K = 256 2.9e-7 -> 1.9e-7, K = 2048 8.1e-7 -> 5.0e-7: the terms' own error
// (about 9e-8) is less than what an accumulator rounded 8 times as often adds.
// (Three bf16 terms, six MFMAs, hold every bit of x over its whole range, but
// reached 83 us where this takes 57: B8 H12 S1024 D64 causal forward.)
//
// The scale decides where this holds: |x s| < 65504, or the result is inf or
// NaN; and the largest |x s| of what is summed should be 2^-1 or more, so that
// 2^-25 is below its rounding.  Each kernel says how it picks its scales and
// what it does with data outside them.
#pragma once

#include "common.h"

namespace hipgpt {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));

// An MFMA operand (eight contraction indices per lane): t[0] = h, t[1] = l.
struct Half8 {
    halfx8 t[2];
};

// (x, y) as packed terms.  (The empty asm keeps the compiler from
// converting each half again to get at it, and 1.0 opaque keeps x - h a single
// mixed-precision FMA.)
__device__ __forceinline__ void half_pair(float x, float y, unsigned& h, unsigned& l) {
    h = __builtin_bit_cast(unsigned, halfx2{(_Float16)x, (_Float16)y});
    asm("" : "+v"(h));
    const halfx2 hh = __builtin_bit_cast(halfx2, h);
    float one = 1.f;
    asm("" : "+s"(one));
    l = __builtin_bit_cast(unsigned, halfx2{(_Float16)__builtin_fmaf(x, one, -(float)hh[0]),
                                            (_Float16)__builtin_fmaf(y, one, -(float)hh[1])});
}
// The terms of eight values in registers, times s if SCALED.
template <bool SCALED>
__device__ __forceinline__ Half8 half8(const float (&x)[8], float s) {
    u32x4 w[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned h, l;
        half_pair(SCALED ? x[2 * i] * s : x[2 * i], SCALED ? x[2 * i + 1] * s : x[2 * i + 1], h, l);
        w[0][i] = h;
        w[1][i] = l;
    }
    Half8 r;
#pragma unroll
    for (int p = 0; p < 2; ++p) r.t[p] = __builtin_bit_cast(halfx8, w[p]);
    return r;
}

__device__ __forceinline__ floatx16 mfma_f16(const halfx8& a, const halfx8& b, const floatx16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// acc += a b without h h'; and all of it, small terms first.  Where one sum
// takes several steps from zero, all the small terms go first: an addition
// rounds at the size the sum then has.
__device__ __forceinline__ floatx16 mfma_half_small(const Half8& a, const Half8& b, floatx16 acc) {
    acc = mfma_f16(a.t[1], b.t[0], acc);
    return mfma_f16(a.t[0], b.t[1], acc);
}
__device__ __forceinline__ floatx16 mfma_half(const Half8& a, const Half8& b, floatx16 acc) {
    return mfma_f16(a.t[0], b.t[0], mfma_half_small(a, b, acc));
}

// Power of two that brings a magnitude to [2^7, 2^8), and its inverse
// (magnitudes below 2^-87 as if at 2^-87).
__device__ __forceinline__ unsigned scale_exp(float m) {
    const unsigned e = __float_as_uint(m) >> 23;
    return e < 40u ? 40u : e > 254u ? 254u : e;
}
__device__ __forceinline__ float scale_of(unsigned e) { return __uint_as_float((261u - e) << 23); }
__device__ __forceinline__ float unscale_of(unsigned e) { return __uint_as_float((e - 7u) << 23); }

__device__ __forceinline__ float max4(const floatx4& v) {
    return fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
}

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

// Operand that contracts over the rows of a row-major LDS tile of 16-bit
// values: column `lane & 15` of the 16 columns the lane's group of 16 points
// at, four rows from its first one and four from eight rows on (rows8: 16-bit
// elements from a row to the eighth after it).  Within the group lane r passes
// the address of row r / 4, columns 4 (r % 4) ..; see fa_bf16.hip.
__device__ __forceinline__ halfx8 read_rows_tr(const unsigned short* p, int rows8) {
    const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)p));
    const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + rows8)));
    return __builtin_bit_cast(halfx8, uint4{lo.x, lo.y, hi.x, hi.y});
}

// 16 values in accumulator register order as the operand that contracts over
// them, times s if SCALED.
struct HalfP {
    Half8 s[2];
};
template <bool SCALED>
__device__ __forceinline__ HalfP half_p(const floatx16& p, float s) {
    HalfP h;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = p[8 * i + j];
        h.s[i] = half8<SCALED>(x, s);
    }
    return h;
}

}  // namespace hipgpt
