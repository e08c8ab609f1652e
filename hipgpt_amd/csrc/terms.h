// terms.h -- fp32 products on the bf16 matrix cores, every operand bit kept.
//
// A float has 24 significand bits and bf16 8 at fp32's exponent range, so
//   x = a + b + c,  a = bf16(x), b = bf16(x - a), c = x - a - b
// (rounded to nearest: |b| <= 2^-8 |x|, |c| <= 2^-17 |x|, both differences and c
// exact).  A product is
//   x y = a a' + (a b' + b a') + (a c' + b b' + c a') + e,  |e| <= 2^-24 |x y|,
// six bf16 MFMAs with fp32 accumulation.  Neither the split nor its error knows
// any other value: no scale is shared, and a product by a power of two is exact.
//
// Operands carry 2^24 (kTermScale), so that the terms of every normal float are
// normal bf16 values and sums of products down to fp32's smallest are held; it
// is taken out of the result as 2^-48.  What that carries past fp32's largest (an
// operand of 2^103, a sum of 2^80), and infinities and NaN, whose terms are
// inf - inf, end in a result that is not finite.  Every kernel tests for that
// before it stores and then forms the tile again on fp32 MFMA.
//
// Six 32x32x16 MFMAs take 6 x 33 cycles for 16 contraction indices, the eight
// fp32 32x32x2 ones they stand for 8 x 65; and fp32 MFMAs keep the vector ALUs
// from issuing, these do not (8 MFMAs with 64 v_fma interleaved, cycles: 820
// against 520 + 268 apart; 340 against 264 + 268).
#pragma once

#include "common.h"

namespace hipgpt {

constexpr float kTermScale = 16777216.f;                   // 2^24
constexpr float kTermUnscale = 1.f / 16777216.f;           // of one operand
constexpr float kTermUnscale2 = kTermUnscale * kTermUnscale;  // of a product

// An MFMA operand (eight contraction indices per lane): t[0] = a, t[1] = b, t[2] = c.
struct Term8 {
    bf16x8 t[3];
};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// The packed terms of (x, y).
__device__ __forceinline__ void term_pair(float x, float y, unsigned (&w)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        w[i] = __builtin_bit_cast(unsigned, bf16x2{(__bf16)x, (__bf16)y});
        if (i < 2) {
            x -= __uint_as_float(w[i] << 16);
            y -= __uint_as_float(w[i] & 0xffff0000u);
        }
    }
}
// The terms of eight values in registers.
__device__ __forceinline__ Term8 term8(const float (&x)[8]) {
    u32x4 w[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned p[3];
        term_pair(x[2 * i], x[2 * i + 1], p);
#pragma unroll
        for (int t = 0; t < 3; ++t) w[t][i] = p[t];
    }
    Term8 r;
#pragma unroll
    for (int t = 0; t < 3; ++t) r.t[t] = __builtin_bit_cast(bf16x8, w[t]);
    return r;
}
// The terms of four values times kTermScale to three planes of 16-bit values, `plane` elements apart.
__device__ __forceinline__ void store_terms(unsigned short* dst, int plane, const floatx4& v) {
    unsigned lo[3], hi[3];
    term_pair(v[0] * kTermScale, v[1] * kTermScale, lo);
    term_pair(v[2] * kTermScale, v[3] * kTermScale, hi);
#pragma unroll
    for (int t = 0; t < 3; ++t) *reinterpret_cast<uint2*>(dst + t * plane) = uint2{lo[t], hi[t]};
}

__device__ __forceinline__ floatx16 mfma_bf16(const bf16x8& a, const bf16x8& b, const floatx16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// acc += a b without a[0] b[0]; and all of it.  Smallest terms first: an
// addition rounds at the size the sum then has.  (Where one sum takes several
// steps from zero, all their small terms go first.)
__device__ __forceinline__ floatx16 mfma_terms_small(const Term8& a, const Term8& b, floatx16 acc) {
    acc = mfma_bf16(a.t[2], b.t[0], acc);
    acc = mfma_bf16(a.t[0], b.t[2], acc);
    acc = mfma_bf16(a.t[1], b.t[1], acc);
    acc = mfma_bf16(a.t[1], b.t[0], acc);
    return mfma_bf16(a.t[0], b.t[1], acc);
}
__device__ __forceinline__ floatx16 mfma_terms(const Term8& a, const Term8& b, floatx16 acc) {
    return mfma_bf16(a.t[0], b.t[0], mfma_terms_small(a, b, acc));
}

// Bits of the larger magnitude; an infinity or NaN is 0x7f800000 or more.
__device__ __forceinline__ unsigned top_bits(unsigned top, float x) {
    return max(top, __float_as_uint(x) & 0x7fffffffu);
}
constexpr unsigned kInfBits = 0x7f800000u;

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

// Operand that contracts over the rows of a row-major LDS tile of 16-bit
// values: column `lane & 15` of the 16 columns the lane's group of 16 points
// at, four rows from its first one and four from eight rows on (rows8: 16-bit
// elements from a row to the eighth after it).  Within the group lane r passes
// the address of row r / 4, columns 4 (r % 4) ..; see fa_bf16.hip.
__device__ __forceinline__ bf16x8 read_rows_tr(const unsigned short* p, int rows8) {
    const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)p));
    const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + rows8)));
    return __builtin_bit_cast(bf16x8, uint4{lo.x, lo.y, hi.x, hi.y});
}

// 16 values in accumulator register order as the operand that contracts over
// them.
struct TermP {
    Term8 s[2];
};
__device__ __forceinline__ TermP term_p(const floatx16& p) {
    TermP h;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = p[8 * i + j];
        h.s[i] = term8(x);
    }
    return h;
}

}  // namespace hipgpt
