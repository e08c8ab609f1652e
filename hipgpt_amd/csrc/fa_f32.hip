// fa_f32.hip -- fp32 attention forward on gfx950 MFMA.
//
// Replaces flash_attention_kernel<32|64> and multihead_attention_kernel_fallback
// (HipGPT src/hip_kernels.cpp:263-325, :329-402) for head dims up to 128
// (D = 16, 48, 96, ... run zero-padded to the next of 32/64/128).  The kernel
// body is fa_kernel.h; this file supplies the operand traits -- F32TermTraits
// below, and F32Traits, the fp32 MFMA ones it falls back to and small grids run:
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

template <int DP_, int NBUF_>
struct F32Traits {
    static constexpr int DP = DP_;
    static constexpr int NBUF = NBUF_;
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
    __device__ __forceinline__ static float score_scale(float) { return 1.0f; }

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
    struct VReg {
        const float* vt;
    };
    __device__ __forceinline__ static void load_v(VReg& vr, const float* Vt, int, int) { vr.vt = Vt; }
    using PReg = floatx16;
    __device__ __forceinline__ static const floatx16& to_p(const floatx16& p) { return p; }
    __device__ __forceinline__ static void pv(const VReg& vr, const floatx16& p, floatx16* o, int c, int hf) {
#pragma unroll
        for (int db = 0; db < DP / 32; ++db) {
            const float* const v = vr.vt + (db * 32 + c) * VTP + 4 * hf;
            floatx4 blk[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) blk[g] = *reinterpret_cast<const floatx4*>(v + 8 * g);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(blk[g][u], p[4 * g + u], o[db], 0, 0, 0);
        }
    }
};

// The products on operands split into three bf16 terms (terms.h), the traits
// every problem runs; a workgroup with a result that is not finite runs again
// with F32Traits (`exact`).  Tiles are three row-major planes; operand layouts
// as in fa_bf16.hip (v_mfma_f32_32x32x16).  Q, K, V and P carry 2^24 each, taken
// out of the scores by score_scale and out of O in the epilogue.
// Against fp32 MFMA, us: B8 H12 S1024 D64 causal 124 -> 86, B4 H16 S2048 D128 causal
// 579 -> 351, B32 H8 S256 D32 causal 15.8 -> 14.1, with probs unmasked 30.2 -> 27.9,
// 333 queries x 1357 keys B3 H12 D64 93 -> 42.  Bound by the matrix cores (six
// MFMAs per product: 0.9-1.2 PFLOP/s at the two longest) and the vector ALUs
// beside them (the softmax and the split of P, K and V).
template <int DP_, int NBUF_ = 1, int SRES_ = 0, int WPE_ = (DP_ <= 64 ? 3 : 2)>
struct F32TermTraits {
    static constexpr int DP = DP_;
    static constexpr int NBUF = NBUF_;
    using elem = unsigned short;
    using gelem = float;
    using exact = F32Traits<DP, NBUF_>;
    using chunk = floatx4;
    static constexpr int KSTR = DP + 8;
    static constexpr int VRP = DP + 16;
    static constexpr int KPL = BK * KSTR;  // one term's plane
    static constexpr int VPL = BK * VRP;
    static constexpr int KTILE = 3 * KPL;
    static constexpr int VTILE = 3 * VPL;
    static constexpr int WAVES_PER_EU = WPE_;
    static constexpr int PROBS_RES_STAGES = SRES_;

    struct QReg {
        Term8 v[DP / 16];
    };

    template <bool VEC>
    __device__ __forceinline__ static void load_q(QReg& q, const float* qrow, int hf, bool valid, int D, float qscale) {
        const float* p = qrow + hf * (DP / 2);
        const float scale = qscale * kTermScale;
#pragma unroll
        for (int j = 0; j < DP / 16; ++j) {
            float x[8];
#pragma unroll
            for (int u = 0; u < 8; u += 4) {
                floatx4 t = {0.f, 0.f, 0.f, 0.f};
                if (VEC) {
                    if (valid) t = *reinterpret_cast<const floatx4*>(p + 8 * j + u);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (valid && hf * (DP / 2) + 8 * j + u + i < D) t[i] = p[8 * j + u + i];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) x[u + i] = t[i] * scale;
            }
            q.v[j] = term8(x);
        }
    }

    __device__ __forceinline__ static chunk from_u32x4(u32x4 v) { return __builtin_bit_cast(chunk, v); }
    __device__ __forceinline__ static float score_scale(float) { return kTermUnscale2; }
    template <bool VEC>
    __device__ __forceinline__ static chunk load_chunk(const float* base, int64_t rowoff, int cc, int D, bool ok) {
        return exact::template load_chunk<VEC>(base, rowoff, cc, D, ok);
    }
    __device__ __forceinline__ static void store_k_chunk(unsigned short* Kt, int r, int cc, const chunk& v) {
        store_terms(Kt + r * KSTR + cc * 4, KPL, v);
    }
    __device__ __forceinline__ static void store_vt_chunk(unsigned short* Vt, int r, int cc, const chunk& v) {
        store_terms(Vt + r * VRP + cc * 4, VPL, v);
    }

    __device__ __forceinline__ static floatx16 qk(const unsigned short* Kt, const QReg& q, int c, int hf) {
        const unsigned short* kr = Kt + c * KSTR + hf * (DP / 2);
        floatx16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int j = 0; j < DP / 16; ++j) {
            Term8 k;
#pragma unroll
            for (int t = 0; t < 3; ++t) k.t[t] = *reinterpret_cast<const bf16x8*>(kr + t * KPL + 8 * j);
            s = mfma_terms_small(k, q.v[j], s);
        }
        asm volatile("" ::: "memory");  // the first terms are read again: held, they spill
#pragma unroll
        for (int j = 0; j < DP / 16; ++j) s = mfma_bf16(*reinterpret_cast<const bf16x8*>(kr + 8 * j), q.v[j].t[0], s);
        return s;
    }

    struct VReg {
        const unsigned short* vt;
    };
    __device__ __forceinline__ static void load_v(VReg& vr, const unsigned short* Vt, int, int) { vr.vt = Vt; }
    // V terms of step s, block db: V[16s + 4hf + 0..3][db*32 + c] and the four
    // rows eight further on, transposed by ds_read_b64_tr_b16.
    __device__ __forceinline__ static Term8 v_terms(const unsigned short* Vt, int db, int s, int c, int hf) {
        const int r = c & 15;
        const unsigned short* p = Vt + (16 * s + 4 * hf + (r >> 2)) * VRP + db * 32 + (c & 16) + 4 * (r & 3);
        Term8 v;
#pragma unroll
        for (int t = 0; t < 3; ++t) v.t[t] = read_rows_tr(p + t * VPL, 8 * VRP);
        return v;
    }
    using PReg = TermP;
    __device__ __forceinline__ static PReg to_p(const floatx16& p) {
        floatx16 x;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = p[r] * kTermScale;
        return term_p(x);
    }
    __device__ __forceinline__ static void pv(const VReg& vr, const PReg& pb, floatx16* o, int c, int hf) {
#pragma unroll
        for (int db = 0; db < DP / 32; ++db)
#pragma unroll
            for (int s = 0; s < 2; ++s) o[db] = mfma_terms(v_terms(vr.vt, db, s, c, hf), pb.s[s], o[db]);
    }
};

// Workgroup shapes, NQS query sub-blocks of 32 rows x NKS key splits, by how
// far 128-query blocks (n128 of them over all (batch, head) pairs) fill the
// device's 256 CUs.  Few: the keys of a row are split over up to four waves
// and the workgroups are small, so that more CUs have work and a row's serial
// chain is shorter.  Many: no key split (no merge, no wave idle in the
// diagonal stages), two or three workgroups per CU.  One stage buffer (NBUF)
// unless a second costs no workgroup.  SRES: probs rows of up to SRES stages
// keep their scores in registers between the two sweeps.
// us, shapes (x NBUF) at n128; c: causal, f: unmasked, p: unmasked with probs:
//   D=32, 256 keys: 128 c 1x4 9.0, 2x2x2 9.5, 2x4 9.6, f 10.6, 9.2, 9.4; 256 c
//     2x2x2 10.3, 4x2 11.4, f 12.1, 11.6; 1024 c 4x1x2 22.8, 4x2 25.0, 2x2x2 30.8.
//     1024 keys: 64 c 1x4 18.1, 2x4 19.4, 2x2x2 22.5; 128 p 2x4 37.8, 1x4 45.7; 256 c 2x2x2 24.3, 2x4
//     25.2, 4x2 29.0, f 34.9, 37.5, 30.8, p 69.5, 59.6, 65.6; 1024 c 4x2 60.4,
//     4x1x2 62.9, 2x2x2 71.8.
//   D=64, 256 keys: 128 2x2 14.0, 2x4 14.1, 4x2 16.9; 256 c 2x2 14.7, 4x2 17.5, f
//     19.9, 18.8, p 25.6, 28.9; 512 c 4x1x2 26.4, 4x1 27.8, with probs 43.8, 49.7; 1024 c
//     4x1 42.0, 8x1 54.4, 2x2 51.7.  1024 keys: 128 2x4 32.5, 2x2 38.0, 4x2 45.8; 256 c 2x2 41.4, 2x4 42.6, 4x2 46.9, f 60.2,
//     65.1, 52.4, p 98.6, 107.9, 92.6; 512 c 4x2 60.5, 4x1 69.3, f 104, 98.8; 768 c
//     4x1 85.6, 4x1x2 89.3, 4x2 92.6, p 246, 264, 275.
//   D=128, 256 keys: 128 2x2 26.4, 4x1x2 33.5; 256 2x2 38.1, 4x1x2 34.1; 512 4x1
//     43.2, 8x1x2 43.6.  1024 keys: 256 c 2x2 86.4, 4x1x2 109, f 147, 109, p 219,
//     170; 512 c 4x1 128, 8x1x2 132, f 185, 171, p 293, 297; 768 c 176, 185; 1024 c
//     224, 199; 2048 keys: 1024 c 393, 351.
template <int DP, int NQS, int NKS, int NBUF, int SRES = 0, int WPE = (DP <= 64 ? 3 : 2), bool VEC = true>
hipError_t launch_shape(const AttnArgs& a, bool causal, bool probs, hipStream_t s) {
    return fa::launch_fa_flags<F32TermTraits<DP, NBUF, SRES, WPE>, NQS, NKS, VEC>(a, causal, probs, s);
}

// Short calls on fp32 MFMA itself, rows of at most 32 NKS SRES keys (with probs
// their scores stay in registers): in small grids each call is one short chain of
// load, scores, softmax and product per wave, which the terms' conversion
// lengthens, and at D = 32 with probs the stores bound the larger ones.  us, terms
// against this, blocks of 128 rows: D=32, 256 keys, unmasked probs 16 8.5, 7.6; 128
// 12.3, 11.7; 512 34.0, 31.5; 1024 66.1, 60.9; causal probs 512 31.1, 26.9; 1024 60.2,
// 51.4 (without probs 22.8, 30.8); 128 keys, causal probs 1024 46.4, 38.5.  D=64, 64
// blocks 12.5, 12.3; 128 19.8, 22.1.
template <int DP, int NQS, int NKS, int SRES>
hipError_t launch_f32(const AttnArgs& a, bool causal, bool probs, hipStream_t s) {
    using T = F32Traits<DP, 2>;
    if (probs)
        return causal ? fa::launch_fa<T, NQS, NKS, true, true, true, SRES>(a, s)
                      : fa::launch_fa<T, NQS, NKS, false, true, true, SRES>(a, s);
    return causal ? fa::launch_fa<T, NQS, NKS, true, false, true>(a, s)
                  : fa::launch_fa<T, NQS, NKS, false, false, true>(a, s);
}

// Head dims below the padded one and unaligned rows (guarded loads): two
// shapes each, for grids that do and do not fill the device.
hipError_t launch_guarded(const AttnArgs& a, bool causal, bool probs, int64_t n128, hipStream_t s) {
    switch (fa_f32_padded_dim(a.D)) {
        case 32: return launch_shape<32, 2, 2, 2, 4, 1, false>(a, causal, probs, s);
        case 64:
            return n128 <= 128 ? launch_shape<64, 2, 4, 1, 0, 1, false>(a, causal, probs, s)
                               : launch_shape<64, 4, 2, 1, 0, 1, false>(a, causal, probs, s);
        case 128:
            return n128 <= 128 ? launch_shape<128, 2, 2, 1, 0, 1, false>(a, causal, probs, s)
                               : launch_shape<128, 8, 1, 1, 0, 1, false>(a, causal, probs, s);
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
    const bool small = n128 <= 64 && Sk > 128 && Sk <= 256;
    switch (fa_f32_padded_dim(a.D)) {
        case 32:
            if (probs && Sk <= 256)
                return n128 <= 128 && Sk > 128 ? launch_f32<32, 1, 4, 2>(a, causal, probs, s)
                                               : launch_f32<32, 2, 2, 4>(a, causal, probs, s);
            if (small) return launch_f32<32, 1, 4, 2>(a, causal, probs, s);
            if (n128 <= 64 || (n128 <= 128 && Sk <= 256 && causal))
                return launch_shape<32, 1, 4, 1>(a, causal, probs, s);
            if (n128 <= 128 && Sk > 256) return launch_shape<32, 2, 4, 1, 2>(a, causal, probs, s);
            if (n128 <= 128 || (n128 <= 256 && causal && !probs)) return launch_shape<32, 2, 2, 2>(a, causal, probs, s);
            if (n128 >= 512 && Sk <= 256) return launch_shape<32, 4, 1, 2>(a, causal, probs, s);
            return launch_shape<32, 4, 2, 1>(a, causal, probs, s);
        case 64:
            if (small) return launch_f32<64, 1, 4, 2>(a, causal, probs, s);
            if (n128 <= 128 && Sk > 256) return launch_shape<64, 2, 4, 1>(a, causal, probs, s);
            if (n128 <= 128 || (n128 <= 256 && (causal || (probs && Sk <= 256))))
                return launch_shape<64, 2, 2, 1, 4>(a, causal, probs, s);
            if (n128 <= 256 || (causal && n128 <= 512 && Sk > 512))
                return launch_shape<64, 4, 2, 1>(a, causal, probs, s);
            if (Sk <= 256) return launch_shape<64, 4, 1, 2>(a, causal, probs, s);
            return launch_shape<64, 4, 1, 1>(a, causal, probs, s);
        case 128:
            if (n128 <= 128 || (n128 <= 256 && causal && Sk > 512)) return launch_shape<128, 2, 2, 1>(a, causal, probs, s);
            if (n128 <= 256) return launch_shape<128, 4, 1, 2>(a, causal, probs, s);
            if (n128 < 1024) return launch_shape<128, 4, 1, 1>(a, causal, probs, s);
            return launch_shape<128, 8, 1, 2>(a, causal, probs, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace hipgpt
