// bwd_terms.h -- the attention backward (HipGPT src/hip_kernels.cpp:1159-1272)
// on operands split into three bf16 terms (terms.h): head dims up to 128.
//
// The math and the two kernels of bwd_tiled.h and bwd_wide.h -- one keeps 32
// queries per wave and walks the keys (dQ, and with stored probs the row dots
// Dq), one keeps 32 keys and walks the queries (dK, dV) -- with the head dim
// split over DH waves above 64 as there.  What differs is the operands: a
// staged tile is three row-major planes of terms, which serve both the
// products over the head dim (rows read with ds_read_b128) and those over the
// tile's rows (ds_read_b64_tr_b16), so no transposed copies are staged and a
// product takes 6 x 16 indices per MFMA instead of 2.
//
// Every operand carries 2^24 (kTermScale): the staged rows and the rows a wave
// keeps as they are split, dS = P (dP - Dq) through the factors of dP and Dq, P
// by a multiplication.  A workgroup with a result that is not finite stores
// nothing and runs again on the fp32 MFMA kernels.
//
// One LDS stage: the next tiles wait in registers, and where registers allow two
// workgroups share a CU, one multiplying while another converts.  Against the
// fp32 MFMA kernels, us: from lse, B8 H12 S1024 D64 causal 447 -> 297; stored causal
// probs, B8 H12 S1024 D64 410 -> 300, B2 H8 S999 D128 493 -> 253.  Bound by the
// matrix cores (six MFMAs per product, 0.8-0.9 PFLOP/s in the larger calls) and
// the conversions, of every staged tile by each workgroup that stages it and
// of P and dS.
#pragma once

#include <type_traits>

#include "bwd_tiled.h"
#include "bwd_wide.h"
#include "common.h"
#include "fa_common.h"
#include "kernels.h"
#include "rowtiles.h"
#include "terms.h"

namespace hipgpt {
namespace bwd {

template <int DP, int DH>
struct TermTiles {
    static constexpr int HP = DP + 8;    // row pitch, 16-bit elements
    static constexpr int PL = BK * HP;   // one term's plane
    static constexpr int TILE = 3 * PL;
    static constexpr int CPR = DP / 4;   // 16-byte chunks of a row
    static constexpr int CPT = BK * CPR;
    static constexpr int DW = DP / DH;   // head dims per wave
    static constexpr int NDBW = DW / 32;
    static constexpr int NJ = DW / 16;   // MFMA steps over the wave's dims

    // acc[m = row c of the tile][n = c] += sum over the wave's dims of tile[c][d] b[d]
    __device__ __forceinline__ static void dchain(floatx16& acc, const unsigned short* tile, const Term8 (&b)[NJ],
                                                  int c, int hf, int dh) {
        const unsigned short* rr = tile + c * HP + dh * DW + hf * (DW / 2);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            Term8 a;
#pragma unroll
            for (int t = 0; t < 3; ++t) a.t[t] = *reinterpret_cast<const bf16x8*>(rr + t * PL + 8 * j);
            acc = mfma_terms_small(a, b[j], acc);
        }
        asm volatile("" ::: "memory");  // the first terms are read again: held, they spill
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc = mfma_bf16(*reinterpret_cast<const bf16x8*>(rr + 8 * j), b[j].t[0], acc);
    }
    // acc[n][db][m = d][n = c] += sum_k tile[k][d] x[n][k][c] over the 32 tile rows
    template <int N>
    __device__ __forceinline__ static void rchain(floatx16 (*acc)[NDBW], const unsigned short* tile, const TermP* x,
                                                  int c, int hf, int dh) {
        const int r = c & 15;
#pragma unroll
        for (int db = 0; db < NDBW; ++db)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const unsigned short* p =
                    tile + (16 * s + 4 * hf + (r >> 2)) * HP + dh * DW + db * 32 + (c & 16) + 4 * (r & 3);
                Term8 a;
#pragma unroll
                for (int t = 0; t < 3; ++t) a.t[t] = read_rows_tr(p + t * PL, 8 * HP);
#pragma unroll
                for (int n = 0; n < N; ++n) acc[n][db] = mfma_terms(a, x[n].s[s], acc[n][db]);
            }
    }
    // The terms of the lane's dims of row `row`, times mul.
    __device__ __forceinline__ static void load_row(Term8 (&v)[NJ], const float* x, int row, int S, int D, int64_t ts,
                                                    int dh, int hf, float mul) {
        float t[DW / 2];
        RowTiles<DP, DH>::load_lane_row(t, x, row, S, D, ts, dh, hf);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            float y[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] = t[8 * j + u] * mul;
            v[j] = term8(y);
        }
    }
};

// Two tiles of 32 rows per stage, chunks i < PER / 2 of a thread from tile 0.
template <int DP, int NT>
struct TermStage {
    static constexpr int CPR = DP / 4, CPT = BK * CPR, HP = DP + 8, PL = BK * HP;
    static constexpr int PER = 2 * CPT / NT;
    static_assert(CPT % NT == 0, "a thread's chunks split evenly over the two tiles");
    floatx4 v[PER];

    __device__ __forceinline__ static int row(int i, int tid) { return (tid + i * NT) % CPT / CPR; }
    __device__ __forceinline__ void load(const RowLoader& l0, const RowLoader& l1, int row0, int D, int tid) {
        const int cc = tid % CPR;  // NT is a multiple of CPR
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const floatx4 t = (i < PER / 2 ? l0 : l1).load(row0 + row(i, tid), cc);
            v[i] = cc * 4 < D ? t : floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    __device__ __forceinline__ void store(unsigned short* dst, int tid) const {
        const int cc = tid % CPR;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            store_terms(dst + (i < PER / 2 ? 0 : 3 * PL) + row(i, tid) * HP + cc * 4, PL, v[i]);
    }
};

template <int N, int NDB>
__device__ __forceinline__ bool not_finite(const floatx16 (&acc)[N][NDB]) {
    unsigned top = 0;
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) top = top_bits(top, acc[n][db][r]);
    return top >= kInfBits;
}

// ----------------------------------------------------------------- dQ, Dq
// Workgroup: NB query sub-blocks x DH dim slices.  run() is false, for all waves
// alike and with nothing stored, when the results need the fp32 kernel (flag: an
// int of LDS, zero, ordered by run's barriers).
template <int DP, int NB, int DH, bool CAUSAL, bool RECOMP>
struct TermQ {
    using T = TermTiles<DP, DH>;
    using X = RowTiles<DP, DH>;  // partial-tile exchange
    static constexpr int NW = NB * DH, NT = NW * 64;
    static constexpr int NACC = RECOMP ? 1 : 2;
    static constexpr int STAGE = 2 * T::TILE;  // V, K
    static constexpr int XCH = DH > 1 ? NW * 16 * 64 * (RECOMP ? 2 : 1) : 0;  // floats
    static constexpr int LDS_BYTES = STAGE * 2 + XCH * 4;

    __device__ __forceinline__ static bool run(const BwdArgs& a, unsigned char* lds_raw, int* simd_slots, int* flag,
                                               int nqb, int bh, int rank) {
        unsigned short* const lds = reinterpret_cast<unsigned short*>(lds_raw);
        floatx4* const xch = reinterpret_cast<floatx4*>(lds_raw + STAGE * 2);
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int c = lane & 31, hf = lane >> 5;
        const int role = DH > 1 ? wave : role_of(fa::simd_rank<NW>(simd_slots, wave, lane), rank, nqb, NW, CAUSAL);
        const int sb = role / DH, dh = role % DH;
        const int qb = CAUSAL ? nqb - 1 - rank : rank;
        const int b = bh / a.H, h = bh % a.H;
        const int S = a.S, D = a.D;
        const int q0 = qb * NB * BK, qw0 = q0 + sb * BK, qi = qw0 + c;
        const int64_t base = (int64_t)b * a.bs + (int64_t)h * a.hs;
        const int kend = CAUSAL ? min(S, q0 + NB * BK) : S;
        const int nstages = (kend + BK - 1) / BK;
        const int wtiles = qw0 < S ? (CAUSAL ? (min(S, qw0 + BK) + BK - 1) / BK : nstages) : 0;

        RowLoader vl, kl;
        vl.init(a.v + base, a.ts, S, D);
        kl.init(a.k + base, a.ts, S, D);
        TermStage<DP, NT> stg;
        stg.load(vl, kl, 0, D, tid);

        Term8 go[T::NJ];  // dO[qi], B operand of dP^T = V dO^T
        T::load_row(go, a.go + base, qi, S, D, a.ts, dh, hf, kTermScale);
        Term8 q2[RECOMP ? T::NJ : 1];  // Q[qi] in log2 units, B operand of S'^T = K Q^T
        float lse2 = 0.f, dqv = 0.f;
        if constexpr (RECOMP) {
            T::load_row(q2, a.q + base, qi, S, D, a.ts, dh, hf, a.scale * kLog2e * kTermScale);
            float dsum = 0.f;
            if (qi < S) {
                const float* gp = a.go + base + (int64_t)qi * a.ts;
                const float* op = a.o + base + (int64_t)qi * a.ts;
                for (int d0 = hf * 4; d0 < D; d0 += 8) {
                    const floatx4 g4 = *reinterpret_cast<const floatx4*>(gp + d0);
                    const floatx4 o4 = *reinterpret_cast<const floatx4*>(op + d0);
#pragma unroll
                    for (int j = 0; j < 4; ++j) dsum = fmaf(g4[j], o4[j], dsum);
                }
                lse2 = a.lse[(int64_t)bh * S + qi] * kLog2e;
            }
            dqv = halves_sum(dsum);
        }

        // dP accumulators count 2^-48, scores likewise; dS carries 2^24
        const float dqt = dqv * kTermScale;

        floatx16 acc[NACC][T::NDBW];
#pragma unroll
        for (int n = 0; n < NACC; ++n)
#pragma unroll
            for (int db = 0; db < T::NDBW; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][db][r] = 0.f;
        float ld = 0.f;
        const float* prow = RECOMP ? nullptr : a.probs + ((int64_t)bh * S + qi) * S;
        // P of key tile t in accumulator order; rows of a length that is no
        // multiple of 4 are read in unaligned 16-byte pieces
        auto load_p = [&](floatx4 (&pv)[4], int t) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int k0 = t * BK + 8 * g + 4 * hf;
                if (qi < S && k0 + 3 < S) {
                    __builtin_memcpy(&pv[g], prow + k0, 16);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) pv[g][j] = (qi < S && k0 + j < S) ? prow[k0 + j] : 0.f;
                }
            }
        };
        floatx4 pnext[4];
        if (!RECOMP && wtiles > 0) load_p(pnext, 0);

        stg.store(lds, tid);
        __syncthreads();
        for (int st = 0; st < nstages; ++st) {
            if (st + 1 < nstages) stg.load(vl, kl, (st + 1) * BK, D, tid);
            const bool act = st < wtiles;  // wave-uniform
            floatx16 dp, sc;  // register r <-> key acc_key(r, h)
            if (DH > 1 || act) {
#pragma unroll
                for (int r = 0; r < 16; ++r) dp[r] = sc[r] = 0.f;
            }
            if (act) {
                T::dchain(dp, lds, go, c, hf, dh);
                if constexpr (RECOMP) T::dchain(sc, lds + T::TILE, q2, c, hf, dh);
            }
            if constexpr (DH > 1) {
                if (act) {
                    X::publish(dp, xch, wave, lane);
                    if constexpr (RECOMP) X::publish(sc, xch + NW * 256, wave, lane);
                }
                __syncthreads();
                if (act) {
                    dp = X::total(dp, xch, sb, dh, lane);
                    if constexpr (RECOMP) sc = X::total(sc, xch + NW * 256, sb, dh, lane);
                }
            }
            if (act) {
                if constexpr (RECOMP) {
                    const int kb0 = st * BK;
                    floatx16 x;
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        x[r] = fast_exp2(fmaf(sc[r], kTermUnscale2, -lse2)) * fmaf(dp[r], kTermUnscale, -dqt);
                    if (kb0 + BK > S || (CAUSAL && kb0 + BK - 1 > qw0)) {
                        asm volatile("");  // a branch, not 16 selects in every tile
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int key = kb0 + acc_key(r, hf);
                            if (!(key < S && (!CAUSAL || key <= qi))) x[r] = 0.f;
                        }
                    }
                    const TermP xs = term_p(x);
                    T::template rchain<1>(acc, lds + T::TILE, &xs, c, hf, dh);  // (dS K)^T += K^T dS^T
                } else {
                    floatx16 p, x;
#pragma unroll
                    for (int g = 0; g < 4; ++g)
#pragma unroll
                        for (int j = 0; j < 4; ++j) p[4 * g + j] = pnext[g][j];
                    if (st + 1 < wtiles) load_p(pnext, st + 1);
                    float s = 0.f;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        x[r] = p[r] * (dp[r] * kTermUnscale);
                        s += x[r];
                        p[r] *= kTermScale;
                    }
                    ld += s;
                    const TermP xs[2] = {term_p(x), term_p(p)};
                    T::template rchain<2>(acc, lds + T::TILE, xs, c, hf, dh);  // A^T, Bm^T
                }
            }
            __syncthreads();
            if (st + 1 < nstages) {
                stg.store(lds, tid);
                __syncthreads();
            }
        }

        const float dq = RECOMP ? dqv : halves_sum(ld) * kTermUnscale;
        if (qi < S && (not_finite(acc) || top_bits(0, dq) >= kInfBits)) *flag = 1;
        __syncthreads();
        if (*flag) return false;
        if (qi < S) {
            if (a.dvec && dh == 0 && hf == 0) a.dvec[(int64_t)bh * S + qi] = dq;
            float* out = a.dq + base + (int64_t)qi * a.ts;
            const float us = kTermUnscale2 * a.scale;
#pragma unroll
            for (int db = 0; db < T::NDBW; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int d0 = dh * T::DW + db * 32 + 8 * g + 4 * hf;
                    if (d0 < D) {
                        floatx4 v;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float x = RECOMP ? acc[0][db][4 * g + j]
                                                   : fmaf(-dq, acc[NACC - 1][db][4 * g + j], acc[0][db][4 * g + j]);
                            v[j] = x * us;
                        }
                        *reinterpret_cast<floatx4*>(out + d0) = v;
                    }
                }
        }
        return true;
    }
};

// ----------------------------------------------------------------- dK, dV
// SELF_DQ (recompute mode without a workspace): the row dots are formed from
// the staged rows of dO and O.
template <int DP, int NB, int DH, bool CAUSAL, bool RECOMP, bool SELF_DQ>
struct TermKV {
    using T = TermTiles<DP, DH>;
    using X = RowTiles<DP, DH>;
    static constexpr int NW = NB * DH, NT = NW * 64;
    static constexpr int TILES = 2 * T::TILE;               // dO, Q
    static constexpr int STAGE = TILES + 2 * 2 * BK;        // + Dq, lse' (floats)
    static constexpr int XCH = DH > 1 ? NW * 16 * 64 * (RECOMP ? 2 : 1) : 0;
    static constexpr int LDS_BYTES = STAGE * 2 + XCH * 4;
    static_assert(!SELF_DQ || (RECOMP && DH == 1), "row dots need whole rows in one wave's lanes");

    __device__ __forceinline__ static bool run(const BwdArgs& a, unsigned char* lds_raw, int* simd_slots, int* flag,
                                               int nkb, int bh, int rank) {
        unsigned short* const lds = reinterpret_cast<unsigned short*>(lds_raw);
        floatx4* const xch = reinterpret_cast<floatx4*>(lds_raw + STAGE * 2);
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int c = lane & 31, hf = lane >> 5;
        const int kb = rank;  // causal: key block 0 sees the most query tiles and launches first
        const int role = DH > 1 ? wave : role_of(fa::simd_rank<NW>(simd_slots, wave, lane), rank, nkb, NW, CAUSAL);
        const int sb = role / DH, dh = role % DH;
        const int b = bh / a.H, h = bh % a.H;
        const int S = a.S, D = a.D;
        const int k0 = kb * NB * BK, kw0 = k0 + sb * BK, kj = kw0 + c;
        const int64_t base = (int64_t)b * a.bs + (int64_t)h * a.hs;
        const int nq = (S + BK - 1) / BK;
        const int it0 = CAUSAL ? k0 / BK : 0;
        const int wit0 = CAUSAL ? kw0 / BK : 0;
        const int nstages = nq - it0;

        RowLoader gl, ql, ol;
        gl.init(a.go + base, a.ts, S, D);
        ql.init(a.q + base, a.ts, S, D);
        if (SELF_DQ) ol.init(a.o + base, a.ts, S, D);
        TermStage<DP, NT> stg;
        constexpr int NG = TermStage<DP, NT>::PER / 2;
        floatx4 ostg[SELF_DQ ? NG : 1];
        float dqs = 0.f, lses = 0.f;
        auto load = [&](int st) {
            const int row0 = (it0 + st) * BK;
            stg.load(gl, ql, row0, D, tid);
            if constexpr (SELF_DQ) {
#pragma unroll
                for (int i = 0; i < NG; ++i) ostg[i] = ol.load(row0 + stg.row(i, tid), tid % T::CPR);
            }
            if (tid < BK) {
                if (!SELF_DQ) dqs = row0 + tid < S ? a.dvec[(int64_t)bh * S + row0 + tid] : 0.f;
                // +inf past the last row: P = 0
                if (RECOMP) lses = row0 + tid < S ? a.lse[(int64_t)bh * S + row0 + tid] * kLog2e : kInf;
            }
        };
        load(0);

        Term8 vr[T::NJ];  // V[kj], B operand of dP = dO V^T
        T::load_row(vr, a.v + base, kj, S, D, a.ts, dh, hf, kTermScale);
        Term8 kr[RECOMP ? T::NJ : 1];  // K[kj] in log2 units, B operand of S' = Q K^T
        if constexpr (RECOMP) T::load_row(kr, a.k + base, kj, S, D, a.ts, dh, hf, a.scale * kLog2e * kTermScale);

        // dP accumulators count 2^-48, scores likewise; Dq and dS carry 2^24
        auto store = [&] {
            stg.store(lds, tid);
            float* const f = reinterpret_cast<float*>(lds + TILES);
            if constexpr (SELF_DQ) {
                // the chunk dots summed over the row's CPR lanes (rows past S: 0)
#pragma unroll
                for (int i = 0; i < NG; ++i) {
                    float d = stg.v[i][0] * ostg[i][0];
#pragma unroll
                    for (int j = 1; j < 4; ++j) d = fmaf(stg.v[i][j], ostg[i][j], d);
#pragma unroll
                    for (int m = 1; m < T::CPR; m <<= 1) d += __shfl_xor(d, m);
                    if (tid % T::CPR == 0) f[stg.row(i, tid)] = d * kTermScale;
                }
            }
            if (tid < BK) {
                if (!SELF_DQ) f[tid] = dqs * kTermScale;
                if (RECOMP) f[BK + tid] = lses;
            }
        };

        floatx16 acc[2][T::NDBW];  // dV^T, dK^T
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int db = 0; db < T::NDBW; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][db][r] = 0.f;
        const float* pcol = RECOMP ? nullptr : a.probs + (int64_t)bh * S * S + kj;
        auto load_p = [&](floatx16& pv, int it) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int qr = it * BK + acc_key(r, hf);
                pv[r] = (qr < S && kj < S) ? pcol[(int64_t)qr * S] : 0.f;
            }
        };
        floatx16 pnext;
        if (!RECOMP && wit0 < nq) load_p(pnext, wit0);

        store();
        __syncthreads();
        for (int st = 0; st < nstages; ++st) {
            if (st + 1 < nstages) load(st + 1);
            const int it = it0 + st;
            const bool act = it >= wit0;  // wave-uniform
            const float* f = reinterpret_cast<const float*>(lds + TILES);
            floatx16 dp, sc;  // register r <-> query acc_key(r, h)
            auto zero = [](floatx16& t) {
#pragma unroll
                for (int r = 0; r < 16; ++r) t[r] = 0.f;
            };
            if constexpr (DH > 1) {
                zero(dp);
                zero(sc);
                if (act) {
                    T::dchain(dp, lds, vr, c, hf, dh);
                    X::publish(dp, xch, wave, lane);
                    if constexpr (RECOMP) {
                        T::dchain(sc, lds + T::TILE, kr, c, hf, dh);
                        X::publish(sc, xch + NW * 256, wave, lane);
                    }
                }
                __syncthreads();
                if (act) {
                    dp = X::total(dp, xch, sb, dh, lane);
                    if constexpr (RECOMP) sc = X::total(sc, xch + NW * 256, sb, dh, lane);
                }
            }
            if (act) {
                floatx16 p, x;
                if constexpr (RECOMP) {
                    if constexpr (DH == 1) {
                        zero(sc);
                        T::dchain(sc, lds + T::TILE, kr, c, hf, dh);
                    }
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const floatx4 l4 = *reinterpret_cast<const floatx4*>(f + BK + 8 * g + 4 * hf);
#pragma unroll
                        for (int j = 0; j < 4; ++j) p[4 * g + j] = fast_exp2(fmaf(sc[4 * g + j], kTermUnscale2, -l4[j]));
                    }
                    if (CAUSAL && it * BK < kw0 + BK - 1) {  // some query of the tile precedes some key of the wave
                        asm volatile("");
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            if (!(it * BK + acc_key(r, hf) >= kj)) p[r] = 0.f;
                    }
                } else {
                    p = pnext;
                    if (it + 1 < nq) load_p(pnext, it + 1);
                }
                {
#pragma unroll
                    for (int r = 0; r < 16; ++r) x[r] = p[r] * kTermScale;
                    const TermP ps = term_p(x);
                    T::template rchain<1>(&acc[0], lds, &ps, c, hf, dh);  // dV^T += dO^T P
                }
                if constexpr (DH == 1) {
                    zero(dp);
                    T::dchain(dp, lds, vr, c, hf, dh);
                }
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const floatx4 dq = *reinterpret_cast<const floatx4*>(f + 8 * g + 4 * hf);
#pragma unroll
                    for (int j = 0; j < 4; ++j) x[4 * g + j] = p[4 * g + j] * fmaf(dp[4 * g + j], kTermUnscale, -dq[j]);
                }
                const TermP xs = term_p(x);
                T::template rchain<1>(&acc[1], lds + T::TILE, &xs, c, hf, dh);  // dK^T += Q^T dS
            }
            __syncthreads();
            if (st + 1 < nstages) {
                store();
                __syncthreads();
            }
        }

        // (a key past the last row: its lane's P is exp2(-lse), perhaps infinite, and never stored)
        if (kj < S && not_finite(acc)) *flag = 1;
        __syncthreads();
        if (*flag) return false;
        if (kj < S) {
            float* dvp = a.dv + base + (int64_t)kj * a.ts;
            float* dkp = a.dk + base + (int64_t)kj * a.ts;
            const float us = kTermUnscale2 * a.scale;
#pragma unroll
            for (int db = 0; db < T::NDBW; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int d0 = dh * T::DW + db * 32 + 8 * g + 4 * hf;
                    if (d0 < D) {
                        floatx4 v, k;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            v[j] = acc[0][db][4 * g + j] * kTermUnscale2;
                            k[j] = acc[1][db][4 * g + j] * us;
                        }
                        *reinterpret_cast<floatx4*>(dvp + d0) = v;
                        *reinterpret_cast<floatx4*>(dkp + d0) = k;
                    }
                }
        }
        return true;
    }
};

// The fp32 MFMA kernels behind them: head dims of exactly 32 or 64 (TIGHT) the
// tiled ones, which need no workspace in recompute mode, else the wide ones.
template <int DP, int NB, int DH, bool CAUSAL, bool RECOMP, bool TIGHT>
struct TermPair {
    using Q = TermQ<DP, NB, DH, CAUSAL, RECOMP>;
    using KV = TermKV<DP, NB, DH, CAUSAL, RECOMP, RECOMP && TIGHT>;
    using XQ = std::conditional_t<TIGHT, BwdQ<TIGHT ? DP : 32, NB, CAUSAL, RECOMP>, WideQ<DP, NB, DH, CAUSAL, RECOMP>>;
    using XKV =
        std::conditional_t<TIGHT, BwdKV<TIGHT ? DP : 32, NB, CAUSAL, RECOMP>, WideKV<DP, NB, DH, CAUSAL, RECOMP>>;
    static constexpr int QB = Q::LDS_BYTES > 4 * XQ::LDS_FLOATS ? Q::LDS_BYTES : 4 * XQ::LDS_FLOATS;
    static constexpr int KB = KV::LDS_BYTES > 4 * XKV::LDS_FLOATS ? KV::LDS_BYTES : 4 * XKV::LDS_FLOATS;
    static constexpr int NT = NB * DH * 64;

    // redo: an int of LDS, zero, ordered by run's barriers
    __device__ __forceinline__ static void q(const BwdArgs& a, unsigned char* lds, int* simd, int* redo, int nb, int bh,
                                             int rank) {
        if (Q::run(a, lds, simd, redo, nb, bh, rank)) return;
        if constexpr (TIGHT)
            XQ::run(a, reinterpret_cast<float*>(lds), simd, nb, bh, rank);
        else
            XQ::run(a, reinterpret_cast<float*>(lds), nb, bh, rank);
    }
    __device__ __forceinline__ static void kv(const BwdArgs& a, unsigned char* lds, int* simd, int* redo, int nb,
                                              int bh, int rank) {
        if (KV::run(a, lds, simd, redo, nb, bh, rank)) return;
        if constexpr (TIGHT)
            XKV::run(a, reinterpret_cast<float*>(lds), simd, nb, bh, rank);
        else
            XKV::run(a, reinterpret_cast<float*>(lds), bh, rank);
    }
};

// WHICH: 0 queries, 1 keys, 2 both kinds in one grid, dealt in chunks of B*H
// workgroups in turn (recompute mode: neither needs the other's results).
template <int WHICH, int DP, int NB, int DH, bool CAUSAL, bool RECOMP, bool TIGHT>
__global__ __launch_bounds__(NB* DH * 64) __attribute__((amdgpu_waves_per_eu(DH == 1 ? 2 : 1)))
void bwd_terms_kernel(BwdArgs a, int nb) {
    using P = TermPair<DP, NB, DH, CAUSAL, RECOMP, TIGHT>;
    constexpr int LB = WHICH == 0 ? P::QB : WHICH == 1 ? P::KB : P::QB > P::KB ? P::QB : P::KB;
    __shared__ __attribute__((aligned(16))) unsigned char lds[LB];
    __shared__ int simd[NB * DH];
    __shared__ int redo;
    if (threadIdx.x == 0) redo = 0;
    const int BH = a.B * a.H;
    const int chunk = blockIdx.x / BH, bh = blockIdx.x % BH;
    if (WHICH == 0)
        P::q(a, lds, simd, &redo, nb, bh, chunk);
    else if (WHICH == 1)
        P::kv(a, lds, simd, &redo, nb, bh, chunk);
    else if (chunk & 1)
        P::kv(a, lds, simd, &redo, nb, bh, chunk >> 1);
    else
        P::q(a, lds, simd, &redo, nb, bh, chunk >> 1);
}

template <int DP, int NB, int DH, bool TIGHT, bool CAUSAL, bool RECOMP>
hipError_t launch_terms_mode(const BwdArgs& a, hipStream_t s) {
    const int BH = a.B * a.H;
    const int nb = (a.S + NB * BK - 1) / (NB * BK);
    const int64_t g = (int64_t)nb * BH;
    if (g <= 0 || 2 * g > 0x7fffffff) return hipErrorInvalidConfiguration;
    const dim3 block(NB * DH * 64);
    if constexpr (RECOMP && TIGHT) {
        hipLaunchKernelGGL((bwd_terms_kernel<2, DP, NB, DH, CAUSAL, RECOMP, TIGHT>), dim3((unsigned)(2 * g)), block, 0,
                           s, a, nb);
    } else {
        hipLaunchKernelGGL((bwd_terms_kernel<0, DP, NB, DH, CAUSAL, RECOMP, TIGHT>), dim3((unsigned)g), block, 0, s, a,
                           nb);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((bwd_terms_kernel<1, DP, NB, DH, CAUSAL, RECOMP, TIGHT>), dim3((unsigned)g), block, 0, s, a,
                           nb);
    }
    return hipGetLastError();
}

template <int DP, int NB, int DH, bool TIGHT>
hipError_t launch_terms(const BwdArgs& a, hipStream_t s) {
    if (!a.probs)
        return a.causal ? launch_terms_mode<DP, NB, DH, TIGHT, true, true>(a, s)
                        : launch_terms_mode<DP, NB, DH, TIGHT, false, true>(a, s);
    return a.causal ? launch_terms_mode<DP, NB, DH, TIGHT, true, false>(a, s)
                    : launch_terms_mode<DP, NB, DH, TIGHT, false, false>(a, s);
}

}  // namespace bwd
}  // namespace hipgpt
