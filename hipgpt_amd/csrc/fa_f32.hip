// fa_f32.hip -- fp32 attention forward on gfx950 MFMA.
//
// Replaces flash_attention_kernel<32|64> and multihead_attention_kernel_fallback
// (HipGPT src/hip_kernels.cpp:263-325, :329-402) for head dims up to 128
// (D = 16, 48, 96, ... run zero-padded to the next of 32/64/128).  The kernel
// body is fa_kernel.h; this file supplies the operand traits -- F32HalfTraits
// below, and F32Traits, the fp32 MFMA ones it falls back to:
//   * S^T = K Q^T on v_mfma_f32_32x32x2_f32.  Q is held in registers,
//     pre-scaled by scale*log2(e) (so scores are already in the log2
//     domain).  Lane (c, h) takes the contraction indices d = h*DP/2 + s:
//     its K operand is 4 consecutive floats of K row c per ds_read_b128.
//   * O^T = V^T P^T: for accumulator register r the lane needs
//     V[acc_key(r, h)][d]; V is stored transposed in LDS so the four
//     consecutive keys of each register group are one ds_read_b128.
//   * K pitch DP+4 floats and V^T pitch 36 floats keep the 16-lane phases
//     of ds_read_b128 on distinct banks.
//
// MFMA 32x32x2 f32 operand layout (lane l, c = l & 31, h = l >> 5):
//   A[m][k]: lane holds A[c][h]          B[k][n]: lane holds B[h][c]
//   D[m][n]: register r holds D[8*(r/4) + 4*h + (r%4)][c]
#include "common.h"
#include "fa_kernel.h"
#include "kernels.h"

namespace hipgpt {

namespace {

using fa::BK;

template <int DP_, bool VPRE_ = (DP_ <= 32), int SRES_ = (DP_ == 32 ? 4 : 0)>
struct F32Traits {
    static constexpr int DP = DP_;
    using elem = float;
    using gelem = float;
    using chunk = floatx4;
    static constexpr int KSTR = DP + 4;
    static constexpr int VTP = BK + 4;
    static constexpr int KTILE = BK * KSTR;
    static constexpr int VTILE = DP * VTP;

    struct QReg {
        float v[DP / 2];
    };

    template <bool VEC>
    __device__ __forceinline__ static void load_q(QReg& q, const float* qrow, int hf, bool valid, int D,
                                                  float qscale) {
        const float* p = qrow + hf * (DP / 2);
        if (!valid) {
#pragma unroll
            for (int s = 0; s < DP / 2; ++s) q.v[s] = 0.f;
        } else if (VEC) {
#pragma unroll
            for (int s = 0; s < DP / 2; s += 4) {
                const floatx4 t = *reinterpret_cast<const floatx4*>(p + s);
#pragma unroll
                for (int j = 0; j < 4; ++j) q.v[s + j] = t[j] * qscale;
            }
        } else {
#pragma unroll
            for (int s = 0; s < DP / 2; ++s) q.v[s] = (hf * (DP / 2) + s < D) ? p[s] * qscale : 0.f;
        }
    }

    __device__ __forceinline__ static chunk from_u32x4(u32x4 v) { return __builtin_bit_cast(chunk, v); }

    // Q already carries scale*log2(e).
    __device__ __forceinline__ static float score_scale(const QReg&, float) { return 1.0f; }

    template <bool VEC>
    __device__ __forceinline__ static chunk load_chunk(const float* base, int64_t rowoff, int cc, int D, bool ok) {
        if (VEC) return ok ? *reinterpret_cast<const floatx4*>(base + rowoff + cc * 4) : floatx4{0.f, 0.f, 0.f, 0.f};
        chunk r;
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = (ok && cc * 4 + j < D) ? base[rowoff + cc * 4 + j] : 0.f;
        return r;
    }
    __device__ __forceinline__ static void store_k_chunk(float* Kt, int r, int cc, const chunk& v) {
        *reinterpret_cast<floatx4*>(Kt + r * KSTR + cc * 4) = v;
    }
    __device__ __forceinline__ static void store_vt_chunk(float* Vt, int r, int cc, const chunk& v) {
#pragma unroll
        for (int j = 0; j < 4; ++j) Vt[(cc * 4 + j) * VTP + r] = v[j];
    }

    // K operands are read in groups of up to 8 x 16 bytes ahead of the MFMA
    // chain (the whole tile for DP <= 64), so the LDS latency is paid once
    // per group rather than per read.
    static constexpr int KG = DP / 8 < 8 ? DP / 8 : 8;
    __device__ __forceinline__ static floatx16 qk(const float* Kt, const QReg& q, int c, int hf) {
        const float* kr = Kt + c * KSTR + hf * (DP / 2);
        floatx16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int j0 = 0; j0 < DP / 8; j0 += KG) {
            floatx4 kv[KG];
#pragma unroll
            for (int j = 0; j < KG; ++j) kv[j] = *reinterpret_cast<const floatx4*>(kr + 4 * (j0 + j));
#pragma unroll
            for (int j = 0; j < KG; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[j][u], q.v[4 * (j0 + j) + u], s, 0, 0, 0);
        }
        return s;
    }

    // V^T operands of a tile: lane (c, hf) of block db needs
    // V[acc_key(t, hf)][db*32 + c], t = 0..15 -- four ds_read_b128 per block.
    // VPRE: read before the softmax (VReg holds them) -- the streaming kernel
    // at DP = 32; otherwise each block is read just
    // before use.  That brings the streaming kernel at DP = 64 to 128 VGPRs:
    // with WAVES_PER_EU = 4 two 8-wave workgroups share a CU (c3: 132 -> 128
    // us; prefetching V under the same cap spills).
    static constexpr bool VPRE = VPRE_;
    static constexpr int WAVES_PER_EU = (DP == 64 && !VPRE) ? 4 : 1;
    // With probs, rows of up to SRES stages keep their score tiles in
    // registers between the two sweeps (DP = 32: 4 stages, Sk <= 256 at two
    // key splits).
    static constexpr int PROBS_RES_STAGES = SRES_;
    struct VReg {
        floatx4 v[VPRE ? DP / 32 : 1][4];
        const float* vt;
    };
    __device__ __forceinline__ static void load_block(floatx4 (&dst)[4], const float* Vt, int db, int c, int hf) {
        const float* p = Vt + (db * 32 + c) * VTP + 4 * hf;
#pragma unroll
        for (int g = 0; g < 4; ++g) dst[g] = *reinterpret_cast<const floatx4*>(p + 8 * g);
    }
    __device__ __forceinline__ static void load_v(VReg& vr, const float* Vt, int c, int hf) {
        vr.vt = Vt;
        if (VPRE)
#pragma unroll
            for (int db = 0; db < DP / 32; ++db) load_block(vr.v[VPRE ? db : 0], Vt, db, c, hf);
    }
    using PReg = floatx16;
    template <bool SCALED = false>
    __device__ __forceinline__ static const floatx16& to_p(const floatx16& p) { return p; }
    __device__ __forceinline__ static void pv(const VReg& vr, const floatx16& p, floatx16* o, int c, int hf) {
#pragma unroll
        for (int db = 0; db < DP / 32; ++db) {
            floatx4 blk[4];
            if (VPRE) {
#pragma unroll
                for (int g = 0; g < 4; ++g) blk[g] = vr.v[VPRE ? db : 0][g];
            } else {
                load_block(blk, vr.vt, db, c, hf);
            }
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(blk[g][u], p[4 * g + u], o[db], 0, 0, 0);
        }
    }
};

// The products on operands split into two fp16 terms (split.h), the traits
// every problem runs unless its data need F32Traits (`exact`).  Tiles are two
// row-major planes; operand layouts as in fa_bf16.hip (v_mfma_f32_32x32x16).
//   Q: each row is scaled by the power of two that brings its largest
//     magnitude to [2^7, 2^8), taken out of the scores by score_scale.
//   K: times 2^6.  Whatever K's own scale, its terms are off by at most
//     max(2^-24 |k|, 2^-31), so a score (log2 units) by a few 2^-31 |q|: the
//     rows where that is not far below the rounding of the exponential have
//     an entry of 16 or more (big()) and take the exact traits.
//   V: times 2^8; exact traits if every |v| is below 2^-9.
//   P: below 2^15 (kHalfPShift, kHalfPScale).
// What overflows fp16 (|k| >= 1023, |v| >= 255) or is not finite ends in O as
// inf or NaN and takes the exact traits.
// B8 H12 S1024 D64 causal 124 -> 57 us, B4 H16 S2048 D128 causal 577 -> 219,
// B32 H8 S256 D32 causal 15.6 -> 11.2, with probs unmasked 30.0 -> 22.9; error
// against 64 bits 2.8e-7 -> 2.5e-7, 4.5e-7 -> 3.1e-7, 1.8e-7 -> 1.7e-7,
// 4.2e-7 -> 3.6e-7.
template <int DP_, int SRES_ = 0>
struct F32HalfTraits {
    static constexpr int DP = DP_;
    using elem = unsigned short;
    using gelem = float;
    using exact = F32Traits<DP>;
    using chunk = floatx4;
    static constexpr int KSTR = DP + 8;
    static constexpr int VRP = DP + 16;
    static constexpr int KPL = BK * KSTR;  // one term's plane
    static constexpr int VPL = BK * VRP;
    static constexpr int KTILE = 2 * KPL;
    static constexpr int VTILE = 2 * VPL;
    static constexpr int WAVES_PER_EU = DP == 64 ? 3 : 2;
    static constexpr int PROBS_RES_STAGES = SRES_;

    struct QReg {
        Half8 v[DP / 16];
        float unscale;
        unsigned top;  // bits of the row's largest |q|
        __device__ __forceinline__ bool big() const { return top >= 0x41800000u; }  // 16
    };

    template <bool VEC>
    __device__ __forceinline__ static void load_q(QReg& q, const float* qrow, int hf, bool valid, int D, float qscale) {
        const float* p = qrow + hf * (DP / 2);
        float x[DP / 2];
        float mx = 0.f;
#pragma unroll
        for (int u = 0; u < DP / 2; u += 4) {
            floatx4 t = {0.f, 0.f, 0.f, 0.f};
            if (VEC) {
                if (valid) t = *reinterpret_cast<const floatx4*>(p + u);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (valid && hf * (DP / 2) + u + i < D) t[i] = p[u + i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[u + i] = t[i] * qscale;
                mx = fmaxf(mx, fabsf(x[u + i]));
            }
        }
        mx = fa::halves_max(mx);
        q.top = __float_as_uint(mx);
        // the row's largest magnitude to [2^7, 2^8); rows below 2^-64 as if at 2^-64
        const unsigned e = max(q.top >> 23, 63u);
        const float scale = __uint_as_float((261u - e) << 23);
        q.unscale = __uint_as_float((e - 7u) << 23) * (1.f / fa::kHalfKScale);
#pragma unroll
        for (int j = 0; j < DP / 16; ++j) {
            float y[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] = x[8 * j + u] * scale;
            q.v[j] = half8<false>(y, 1.f);
        }
    }

    __device__ __forceinline__ static chunk from_u32x4(u32x4 v) { return __builtin_bit_cast(chunk, v); }
    __device__ __forceinline__ static float score_scale(const QReg& q, float) { return q.unscale; }
    template <bool VEC>
    __device__ __forceinline__ static chunk load_chunk(const float* base, int64_t rowoff, int cc, int D, bool ok) {
        return F32Traits<DP>::template load_chunk<VEC>(base, rowoff, cc, D, ok);
    }
    template <int PLANE>
    __device__ __forceinline__ static void store_chunk(unsigned short* dst, const chunk& v, float s) {
        uint2 w[2];
        half_pair(v[0] * s, v[1] * s, w[0].x, w[1].x);
        half_pair(v[2] * s, v[3] * s, w[0].y, w[1].y);
#pragma unroll
        for (int t = 0; t < 2; ++t) *reinterpret_cast<uint2*>(dst + t * PLANE) = w[t];
    }
    __device__ __forceinline__ static void store_k_chunk(unsigned short* Kt, int r, int cc, const chunk& v) {
        store_chunk<KPL>(Kt + r * KSTR + cc * 4, v, fa::kHalfKScale);
    }
    __device__ __forceinline__ static void store_vt_chunk(unsigned short* Vt, int r, int cc, const chunk& v) {
        store_chunk<VPL>(Vt + r * VRP + cc * 4, v, fa::kHalfVScale);
    }

    __device__ __forceinline__ static floatx16 qk(const unsigned short* Kt, const QReg& q, int c, int hf) {
        const unsigned short* kr = Kt + c * KSTR + hf * (DP / 2);
        floatx16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
        Half8 k[DP / 16];
#pragma unroll
        for (int j = 0; j < DP / 16; ++j) {
#pragma unroll
            for (int t = 0; t < 2; ++t) k[j].t[t] = *reinterpret_cast<const halfx8*>(kr + t * KPL + 8 * j);
            s = mfma_half_small(k[j], q.v[j], s);
        }
#pragma unroll
        for (int j = 0; j < DP / 16; ++j) s = mfma_f16(k[j].t[0], q.v[j].t[0], s);
        return s;
    }

    struct VReg {
        const unsigned short* vt;
    };
    __device__ __forceinline__ static void load_v(VReg& vr, const unsigned short* Vt, int, int) { vr.vt = Vt; }
    // V terms of step s, block db: V[16s + 4hf + 0..3][db*32 + c] and the four
    // rows eight further on, transposed by ds_read_b64_tr_b16.
    __device__ __forceinline__ static Half8 v_terms(const unsigned short* Vt, int db, int s, int c, int hf) {
        const int r = c & 15;
        const unsigned short* p = Vt + (16 * s + 4 * hf + (r >> 2)) * VRP + db * 32 + (c & 16) + 4 * (r & 3);
        Half8 v;
#pragma unroll
        for (int t = 0; t < 2; ++t) v.t[t] = read_rows_tr(p + t * VPL, 8 * VRP);
        return v;
    }
    using PReg = HalfP;
    template <bool SCALED = false>
    __device__ __forceinline__ static PReg to_p(const floatx16& p) {
        return half_p<SCALED>(p, fa::kHalfPScale);
    }
    __device__ __forceinline__ static void pv(const VReg& vr, const PReg& pb, floatx16* o, int c, int hf) {
#pragma unroll
        for (int db = 0; db < DP / 32; ++db)
#pragma unroll
            for (int s = 0; s < 2; ++s) o[db] = mfma_half(v_terms(vr.vt, db, s, c, hf), pb.s[s], o[db]);
    }
};

// Workgroup shapes, NQS query sub-blocks of 32 rows x NKS key splits, by how
// far 128-query blocks (n128 of them over all (batch, head) pairs) fill the
// device's 256 CUs.  Few: the keys of a row are split over up to four waves
// and the workgroups are small, so that more CUs have work and a row's serial
// chain is shorter.  Many: no key split (no merge, no wave idle in the
// diagonal stages), two or three workgroups per CU.  SRES: probs rows of up
// to SRES stages keep their scores in registers between the two sweeps.
// us, shapes at n128 (head dim, entry, keys):
//   D=32 causal, 256 keys: 2x2 9.2, 4x1 10.6 at 256; 14.8, 11.7 at 512; 1024
//     keys: 1x4 13.6, 2x4 15.1, 2x2 17.8 at 64; 18.0, 15.2, 17.9 at 128; 2x2
//     18.3, 4x1 24.7 at 256; 46.2, 41.1 at 1024.
//   D=32 probs, 256 keys: 1x4 7.6, 2x2 9.7 at 64; 2x2 22.9, 4x1 29.1 at 512;
//     1024 keys: 2x4 26.5, 2x2 31.2 at 128.
//   D=64 causal, 256 keys: 1x4 10.0, 2x4 11.2, 4x2 11.7 at 64; 4x1 17.0, 4x2
//     22.4 at 512; 1024 keys: 2x4 23.6, 2x2 27.3, 4x2 28.8 at 128; 4x2 37.7,
//     4x1 39.9 at 384; 4x1 58.4, 4x2 68.3 at 768.
//   D=64 probs, 256 keys: 2x2 33.9, 4x2 39.9, 4x1 45.0 at 512; 1024 keys: 2x4
//     40.6, 4x2 49.5 at 128; 4x2 78, 4x1 90 at 256; level from 384 on.
//   D=128 causal, 1024 keys: 2x2 51, 4x1 64, 8x1 74 at 128; 4x1 78, 8x1 81 at
//     512; 8x1 136, 4x1 143 at 1024.  Probs, 256 keys: 2x2 22.5, 4x1 34 at
//     128; 4x1 36, 2x2 39 at 256.
template <int DP, int NQS, int NKS, int SRES = 0, bool VEC = true>
hipError_t launch_shape(const AttnArgs& a, bool causal, bool probs, hipStream_t s) {
    return fa::launch_fa_flags<F32HalfTraits<DP, SRES>, NQS, NKS, VEC>(a, causal, probs, s);
}

// Head dims below the padded one and unaligned rows (guarded loads): two
// shapes each, for grids that do and do not fill the device.
hipError_t launch_guarded(const AttnArgs& a, bool causal, bool probs, int64_t n128, hipStream_t s) {
    switch (fa_f32_padded_dim(a.D)) {
        case 32: return launch_shape<32, 2, 2, 4, false>(a, causal, probs, s);
        case 64:
            return n128 <= 128 ? launch_shape<64, 2, 4, 0, false>(a, causal, probs, s)
                               : launch_shape<64, 4, 2, 0, false>(a, causal, probs, s);
        case 128:
            return n128 <= 128 ? launch_shape<128, 2, 2, 0, false>(a, causal, probs, s)
                               : launch_shape<128, 8, 1, 0, false>(a, causal, probs, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

int fa_f32_padded_dim(int D) {
    if (D <= 32) return 32;
    if (D <= 64) return 64;
    if (D <= 128) return 128;
    return 0;
}

hipError_t launch_fa_f32(const AttnArgs& a, bool causal, bool vec, hipStream_t s) {
    const bool probs = a.probs != nullptr;
    const int64_t n128 = (int64_t)a.B * a.H * ((a.Sq + 127) / 128);
    const int Sk = a.Sk;
    if (!vec) return launch_guarded(a, causal, probs, n128, s);
    switch (fa_f32_padded_dim(a.D)) {
        case 32:
            if (n128 <= 64 && Sk > 128) return launch_shape<32, 1, 4, 2>(a, causal, probs, s);
            if (n128 <= 128 && Sk > 256) return launch_shape<32, 2, 4, 2>(a, causal, probs, s);
            if (n128 < 512 || probs) return launch_shape<32, 2, 2, 4>(a, causal, probs, s);
            return launch_shape<32, 4, 1>(a, causal, probs, s);
        case 64:
            if (n128 <= 64 && Sk <= 256 && Sk > 128) return launch_shape<64, 1, 4, 2>(a, causal, probs, s);
            if (n128 <= 128) return launch_shape<64, 2, 4>(a, causal, probs, s);
            if (probs && Sk <= 256) return launch_shape<64, 2, 2, 4>(a, causal, probs, s);
            if (n128 <= 256 || (causal && n128 <= 512 && Sk > 512))
                return launch_shape<64, 4, 2>(a, causal, probs, s);
            return launch_shape<64, 4, 1>(a, causal, probs, s);
        case 128:
            if (n128 <= 128) return launch_shape<128, 2, 2>(a, causal, probs, s);
            if (n128 <= 512 || probs) return launch_shape<128, 4, 1>(a, causal, probs, s);
            return launch_shape<128, 8, 1>(a, causal, probs, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace hipgpt
