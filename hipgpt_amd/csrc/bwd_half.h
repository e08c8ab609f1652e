// bwd_half.h -- the attention backward (HipGPT src/hip_kernels.cpp:1159-1272)
// on operands split into two fp16 terms (split.h): head dims up to 128.
//
// The math and the two kernels of bwd_tiled.h and bwd_wide.h -- one keeps 32
// queries per wave and walks the keys (dQ, and with stored probs the row dots
// Dq), one keeps 32 keys and walks the queries (dK, dV) -- with the head dim
// split over DH waves above 64 as there.  What differs is the operands: a
// staged tile is two row-major planes of fp16 terms, which serve both the
// products over the head dim (rows read with ds_read_b128) and those over the
// tile's rows (ds_read_b64_tr_b16), so no transposed copies are staged and a
// product takes 3 x 16 indices per MFMA instead of 2.
//
// Scales, all powers of two.  The rows a wave keeps carry one each (largest
// magnitude to [2^7, 2^8)); the staged tensors one each per workgroup, from
// its first stage, so a value up to 255 times the first stage's largest fits
// and every value is held to 2^-32 of that.  P carries 2^14.  dS = P (dP - Dq)
// is formed in units in which a product of the two largest magnitudes
// (dO and V) is 2^9 .. 2^11: sums over the head dim stay below fp16's 2^16 and
// typical P of 2^-10 still leave dS near 1, 2^-24 of it above fp16's last bit.
// A workgroup whose first stage is all zeros, or whose results are not finite,
// runs again on the fp32 MFMA kernels.
//
// us before -> after, causal: forward and backward from lse, B8 H12 S1024 D64
// 571 -> 240 (of it the forward 124 -> 56); stored probs, B2 H8 S999 D128 499 ->
// 190; error against 64 bits 7.3e-7 -> 5.0e-7 and 6.3e-7 -> 4.0e-7.
#pragma once

#include <type_traits>

#include "bwd_tiled.h"
#include "bwd_wide.h"
#include "common.h"
#include "fa_common.h"
#include "kernels.h"
#include "rowtiles.h"
#include "split.h"

namespace hipgpt {
namespace bwd {

constexpr float kBwdPScale = 16384.f;  // P before its split
constexpr int kDsExp = 9;              // dS units: see above

template <int DP, int DH>
struct HalfTiles {
    static constexpr int HP = DP + 8;    // row pitch, 16-bit elements
    static constexpr int PL = BK * HP;   // one term's plane
    static constexpr int TILE = 2 * PL;
    static constexpr int CPR = DP / 4;   // 16-byte chunks of a row
    static constexpr int CPT = BK * CPR;
    static constexpr int DW = DP / DH;   // head dims per wave
    static constexpr int NDBW = DW / 32;
    static constexpr int NJ = DW / 16;   // MFMA steps over the wave's dims

    // acc[m = row c of the tile][n = c] += sum over the wave's dims of tile[c][d] b[d]
    __device__ __forceinline__ static void dchain(floatx16& acc, const unsigned short* tile, const Half8 (&b)[NJ],
                                                  int c, int hf, int dh) {
        const unsigned short* rr = tile + c * HP + dh * DW + hf * (DW / 2);
        Half8 a[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
#pragma unroll
            for (int t = 0; t < 2; ++t) a[j].t[t] = *reinterpret_cast<const halfx8*>(rr + t * PL + 8 * j);
            acc = mfma_half_small(a[j], b[j], acc);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc = mfma_f16(a[j].t[0], b[j].t[0], acc);
    }
    // acc[n][db][m = d][n = c] += sum_k tile[k][d] x[n][k][c] over the 32 tile rows
    template <int N>
    __device__ __forceinline__ static void rchain(floatx16 (*acc)[NDBW], const unsigned short* tile, const HalfP* x,
                                                  int c, int hf, int dh) {
        const int r = c & 15;
#pragma unroll
        for (int db = 0; db < NDBW; ++db)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const unsigned short* p =
                    tile + (16 * s + 4 * hf + (r >> 2)) * HP + dh * DW + db * 32 + (c & 16) + 4 * (r & 3);
                Half8 a;
#pragma unroll
                for (int t = 0; t < 2; ++t) a.t[t] = read_rows_tr(p + t * PL, 8 * HP);
#pragma unroll
                for (int n = 0; n < N; ++n) acc[n][db] = mfma_half(a, x[n].s[s], acc[n][db]);
            }
    }
    // The lane's dims of row `row` times mul, scaled by the power of two of
    // their largest magnitude over the wave's dims (its exponent is returned).
    __device__ __forceinline__ static unsigned load_row(Half8 (&v)[NJ], const float* x, int row, int S, int D,
                                                        int64_t ts, int dh, int hf, float mul) {
        float t[DW / 2];
        RowTiles<DP, DH>::load_lane_row(t, x, row, S, D, ts, dh, hf);
        float m = 0.f;
#pragma unroll
        for (int s = 0; s < DW / 2; ++s) {
            t[s] *= mul;
            m = fmaxf(m, fabsf(t[s]));
        }
        const unsigned e = scale_exp(fa::halves_max(m));
        const float sc = scale_of(e);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            float y[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] = t[8 * j + u] * sc;
            v[j] = half8<false>(y, 1.f);
        }
        return e;
    }
};

// Two tiles of 32 rows per stage, chunks i < PER / 2 of a thread from tile 0.
template <int DP, int NT>
struct HalfStage {
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
    __device__ __forceinline__ float top(int tile) const {
        float m = 0.f;
#pragma unroll
        for (int i = tile * PER / 2; i < (tile + 1) * PER / 2; ++i)
            m = fmaxf(fmaxf(m, fmaxf(fabsf(v[i][0]), fabsf(v[i][1]))), fmaxf(fabsf(v[i][2]), fabsf(v[i][3])));
        return m;
    }
    __device__ __forceinline__ void store(unsigned short* dst, float s0, float s1, int tid) const {
        const int cc = tid % CPR;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const float s = i < PER / 2 ? s0 : s1;
            uint2 t[2];
            half_pair(v[i][0] * s, v[i][1] * s, t[0].x, t[1].x);
            half_pair(v[i][2] * s, v[i][3] * s, t[0].y, t[1].y);
            unsigned short* p = dst + (i < PER / 2 ? 0 : 2 * PL) + row(i, tid) * HP + cc * 4;
            *reinterpret_cast<uint2*>(p) = t[0];
            *reinterpret_cast<uint2*>(p + PL) = t[1];
        }
    }
};

// Maxima over the workgroup of N values per thread (two barriers).
template <int NW, int N>
__device__ __forceinline__ void wg_max(float (&m)[N], float* slots, int wave, int lane) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
        m[n] = wave_max(m[n]);
        if (lane == 0) slots[wave * N + n] = m[n];
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int w = 0; w < NW; ++w) m[n] = fmaxf(m[n], slots[w * N + n]);
    __syncthreads();
}

template <int N, int NDB>
__device__ __forceinline__ bool not_finite(const floatx16 (&acc)[N][NDB]) {
    unsigned top = 0;
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) top = max(top, __float_as_uint(acc[n][db][r]) & 0x7fffffffu);
    return top >= 0x7f800000u;
}

// 2^n (n >= -126)
__device__ __forceinline__ float pow2(int n) { return __uint_as_float((unsigned)(127 + n) << 23); }

// ----------------------------------------------------------------- dQ, Dq
// Workgroup: NB query sub-blocks x DH dim slices.  run() is true when a wave's
// results need the fp32 kernel.
template <int DP, int NB, int DH, bool CAUSAL, bool RECOMP>
struct HalfQ {
    using T = HalfTiles<DP, DH>;
    using X = RowTiles<DP, DH>;  // partial-tile exchange
    static constexpr int NW = NB * DH, NT = NW * 64;
    static constexpr int NACC = RECOMP ? 1 : 2;
    static constexpr int STAGE = 2 * T::TILE;  // V, K
    static constexpr int XCH = DH > 1 ? NW * 16 * 64 * (RECOMP ? 2 : 1) : 0;  // floats
    static constexpr int LDS_BYTES = 2 * STAGE * 2 + XCH * 4 + NW * 2 * 4;

    __device__ __forceinline__ static bool run(const BwdArgs& a, unsigned char* lds_raw, int* simd_slots, int nqb,
                                               int bh, int rank) {
        unsigned short* const lds = reinterpret_cast<unsigned short*>(lds_raw);
        floatx4* const xch = reinterpret_cast<floatx4*>(lds_raw + 2 * STAGE * 2);
        float* const slots = reinterpret_cast<float*>(lds_raw + 2 * STAGE * 2 + XCH * 4);
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
        HalfStage<DP, NT> stg;
        stg.load(vl, kl, 0, D, tid);

        Half8 go[T::NJ];  // dO[qi], B operand of dP^T = V dO^T
        const unsigned ego = T::load_row(go, a.go + base, qi, S, D, a.ts, dh, hf, 1.f);
        Half8 q2[RECOMP ? T::NJ : 1];  // Q[qi] in log2 units, B operand of S'^T = K Q^T
        unsigned eq = 0;
        float lse2 = 0.f, dqv = 0.f;
        if constexpr (RECOMP) {
            eq = T::load_row(q2, a.q + base, qi, S, D, a.ts, dh, hf, a.scale * kLog2e);
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

        float mx[2] = {stg.top(0), stg.top(1)};
        wg_max<NW, 2>(mx, slots, wave, lane);
        const unsigned ev = __builtin_amdgcn_readfirstlane(scale_exp(mx[0]));
        const unsigned ek = __builtin_amdgcn_readfirstlane(scale_exp(mx[1]));
        const float sv = scale_of(ev), sk = scale_of(ek);
        bool redo = mx[0] == 0.f || mx[1] == 0.f;

        // dP accumulators are 2^(134 - ego) 2^(134 - ev) dP.  dS is formed
        // times t = 2^(kDsExp + 127 - er) 2^(127 - ev), er the exponent of the
        // row (its largest over the DH slices), so a slice's accumulator
        // counts 2^(kDsExp - 14 + ego - er).
        unsigned er = ego;
        if constexpr (DH > 1) {
            // slices of one sub-block: each lane's row exponents through LDS
            float* const ex = reinterpret_cast<float*>(xch);
            ex[wave * 64 + lane] = __uint_as_float(ego);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < DH; ++j) er = max(er, __float_as_uint(ex[(sb * DH + j) * 64 + lane]));
            __syncthreads();
        }
        const float fdp = pow2(max(kDsExp - 14 + (int)ego - (int)er, -126));
        const float t0 = pow2(max(-126, min(127, kDsExp + 127 - (int)er))), t1 = pow2(max(-126, min(127, 127 - (int)ev)));
        const float it0 = pow2(max(-126, min(127, (int)er - 127 - kDsExp))), it1 = pow2(max(-126, min(127, (int)ev - 127)));
        const float dqt = dqv * t0 * t1;
        const float us = RECOMP ? unscale_of(eq) * unscale_of(ek) : 0.f;

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

        stg.store(lds, sv, sk, tid);
        __syncthreads();
        for (int st = 0; st < nstages; ++st) {
            const unsigned short* cur = lds + (st & 1) * STAGE;
            if (st + 1 < nstages) stg.load(vl, kl, (st + 1) * BK, D, tid);
            const bool act = st < wtiles;  // wave-uniform
            floatx16 dp, sc;  // register r <-> key acc_key(r, h)
            if (DH > 1 || act) {
#pragma unroll
                for (int r = 0; r < 16; ++r) dp[r] = sc[r] = 0.f;
            }
            if (act) {
                T::dchain(dp, cur, go, c, hf, dh);
                if constexpr (RECOMP) T::dchain(sc, cur + T::TILE, q2, c, hf, dh);
            }
            if constexpr (DH > 1) {
                if (act) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) dp[r] *= fdp;
                    X::publish(dp, xch, wave, lane);
                    if constexpr (RECOMP) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) sc[r] *= us;
                        X::publish(sc, xch + NW * 256, wave, lane);
                    }
                }
                __syncthreads();
                if (act) {
                    dp = X::total(dp, xch, sb, dh, lane);
                    if constexpr (RECOMP) sc = X::total(sc, xch + NW * 256, sb, dh, lane);
                }
            }
            const float fd = DH > 1 ? 1.f : fdp, fs = DH > 1 ? 1.f : us;
            if (act) {
                if constexpr (RECOMP) {
                    const int kb0 = st * BK;
                    floatx16 x;
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        x[r] = fast_exp2(fmaf(sc[r], fs, -lse2)) * fmaf(dp[r], fd, -dqt);
                    if (kb0 + BK > S || (CAUSAL && kb0 + BK - 1 > qw0)) {
                        asm volatile("");  // a branch, not 16 selects in every tile
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int key = kb0 + acc_key(r, hf);
                            if (!(key < S && (!CAUSAL || key <= qi))) x[r] = 0.f;
                        }
                    }
                    const HalfP xs = half_p<false>(x, 1.f);
                    T::template rchain<1>(acc, cur + T::TILE, &xs, c, hf, dh);  // (dS K)^T += K^T dS^T
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
                        x[r] = p[r] * (dp[r] * fd);
                        s += x[r];
                    }
                    ld += s;
                    const HalfP xs[2] = {half_p<false>(x, 1.f), half_p<true>(p, kBwdPScale)};
                    T::template rchain<2>(acc, cur + T::TILE, xs, c, hf, dh);  // A^T, Bm^T
                }
            }
            if (st + 1 < nstages) stg.store(lds + ((st + 1) & 1) * STAGE, sv, sk, tid);
            __syncthreads();
        }

        const float dq = RECOMP ? dqt : halves_sum(ld);  // times t
        redo |= not_finite(acc) || (__float_as_uint(dq) & 0x7fffffffu) >= 0x7f800000u;
        if (qi < S) {
            if (a.dvec && dh == 0 && hf == 0) a.dvec[(int64_t)bh * S + qi] = RECOMP ? dqv : dq * it0 * it1;
            float* out = a.dq + base + (int64_t)qi * a.ts;
            const float uk = unscale_of(ek) * a.scale, dqp = dq * (1.f / kBwdPScale);
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
                                                   : fmaf(-dqp, acc[NACC - 1][db][4 * g + j], acc[0][db][4 * g + j]);
                            v[j] = x * uk * it0 * it1;
                        }
                        *reinterpret_cast<floatx4*>(out + d0) = v;
                    }
                }
        }
        return redo;
    }
};

// ----------------------------------------------------------------- dK, dV
// SELF_DQ (recompute mode without a workspace): the row dots are formed from
// the staged rows of dO and O.
template <int DP, int NB, int DH, bool CAUSAL, bool RECOMP, bool SELF_DQ>
struct HalfKV {
    using T = HalfTiles<DP, DH>;
    using X = RowTiles<DP, DH>;
    static constexpr int NW = NB * DH, NT = NW * 64;
    static constexpr int TILES = 2 * T::TILE;               // dO, Q
    static constexpr int STAGE = TILES + 2 * 2 * BK;        // + Dq, lse' (floats)
    static constexpr int XCH = DH > 1 ? NW * 16 * 64 * (RECOMP ? 2 : 1) : 0;
    static constexpr int LDS_BYTES = 2 * STAGE * 2 + XCH * 4 + NW * 3 * 4;
    static_assert(!SELF_DQ || (RECOMP && DH == 1), "row dots need whole rows in one wave's lanes");

    __device__ __forceinline__ static bool run(const BwdArgs& a, unsigned char* lds_raw, int* simd_slots, int nkb,
                                               int bh, int rank) {
        unsigned short* const lds = reinterpret_cast<unsigned short*>(lds_raw);
        floatx4* const xch = reinterpret_cast<floatx4*>(lds_raw + 2 * STAGE * 2);
        float* const slots = reinterpret_cast<float*>(lds_raw + 2 * STAGE * 2 + XCH * 4);
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
        HalfStage<DP, NT> stg;
        constexpr int NG = HalfStage<DP, NT>::PER / 2;
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
        load(k0 / BK - it0);  // the scales' rows: the same with and without a causal mask, so that both round alike

        Half8 vr[T::NJ];  // V[kj], B operand of dP = dO V^T
        const unsigned evj = T::load_row(vr, a.v + base, kj, S, D, a.ts, dh, hf, 1.f);
        Half8 kr[RECOMP ? T::NJ : 1];  // K[kj] in log2 units, B operand of S' = Q K^T
        unsigned ekj = 0;
        if constexpr (RECOMP) ekj = T::load_row(kr, a.k + base, kj, S, D, a.ts, dh, hf, a.scale * kLog2e);

        float mx[3] = {stg.top(0), stg.top(1), evj > 40u ? __uint_as_float(evj << 23) : 0.f};
        if (!CAUSAL && k0 > 0) load(0);
        wg_max<NW, 3>(mx, slots, wave, lane);
        const unsigned eg = __builtin_amdgcn_readfirstlane(scale_exp(mx[0]));
        const unsigned eq = __builtin_amdgcn_readfirstlane(scale_exp(mx[1]));
        const unsigned ev = __builtin_amdgcn_readfirstlane(scale_exp(mx[2]));
        const float sg = scale_of(eg), sq = scale_of(eq);
        bool redo = mx[0] == 0.f || mx[1] == 0.f || mx[2] == 0.f;

        // dP accumulators are 2^(134 - evj) 2^(134 - eg) dP; dS is formed times
        // t = 2^(kDsExp + 127 - eg) 2^(127 - ev), ev the exponent of the
        // workgroup's largest |v|
        const float fdp = pow2(max(kDsExp - 14 + (int)evj - (int)ev, -126));
        const float t0 = pow2(max(-126, min(127, kDsExp + 127 - (int)eg))), t1 = pow2(max(-126, min(127, 127 - (int)ev)));
        const float i0 = pow2(max(-126, min(127, (int)eg - 127 - kDsExp))), i1 = pow2(max(-126, min(127, (int)ev - 127)));
        const float us = RECOMP ? unscale_of(ekj) * unscale_of(eq) : 0.f;

        auto store = [&](unsigned short* dst) {
            stg.store(dst, sg, sq, tid);
            float* const f = reinterpret_cast<float*>(dst + TILES);
            if constexpr (SELF_DQ) {
                // the chunk dots summed over the row's CPR lanes (rows past S: 0)
#pragma unroll
                for (int i = 0; i < NG; ++i) {
                    float d = stg.v[i][0] * ostg[i][0];
#pragma unroll
                    for (int j = 1; j < 4; ++j) d = fmaf(stg.v[i][j], ostg[i][j], d);
#pragma unroll
                    for (int m = 1; m < T::CPR; m <<= 1) d += __shfl_xor(d, m);
                    if (tid % T::CPR == 0) f[stg.row(i, tid)] = d * t0 * t1;
                }
            }
            if (tid < BK) {
                if (!SELF_DQ) f[tid] = dqs * t0 * t1;
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

        store(lds);
        __syncthreads();
        for (int st = 0; st < nstages; ++st) {
            const unsigned short* cur = lds + (st & 1) * STAGE;
            if (st + 1 < nstages) load(st + 1);
            const int it = it0 + st;
            const bool act = it >= wit0;  // wave-uniform
            floatx16 dp, sc;  // register r <-> query acc_key(r, h)
            if (DH > 1 || act) {
#pragma unroll
                for (int r = 0; r < 16; ++r) dp[r] = sc[r] = 0.f;
            }
            if (act) {
                T::dchain(dp, cur, vr, c, hf, dh);
                if constexpr (RECOMP) T::dchain(sc, cur + T::TILE, kr, c, hf, dh);
            }
            if constexpr (DH > 1) {
                if (act) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) dp[r] *= fdp;
                    X::publish(dp, xch, wave, lane);
                    if constexpr (RECOMP) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) sc[r] *= us;
                        X::publish(sc, xch + NW * 256, wave, lane);
                    }
                }
                __syncthreads();
                if (act) {
                    dp = X::total(dp, xch, sb, dh, lane);
                    if constexpr (RECOMP) sc = X::total(sc, xch + NW * 256, sb, dh, lane);
                }
            }
            const float fd = DH > 1 ? 1.f : fdp, fs = DH > 1 ? 1.f : us;
            if (act) {
                const float* f = reinterpret_cast<const float*>(cur + TILES);
                floatx16 p, x;
                if constexpr (RECOMP) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const floatx4 l4 = *reinterpret_cast<const floatx4*>(f + BK + 8 * g + 4 * hf);
#pragma unroll
                        for (int j = 0; j < 4; ++j) p[4 * g + j] = fast_exp2(fmaf(sc[4 * g + j], fs, -l4[j]));
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
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const floatx4 dq = *reinterpret_cast<const floatx4*>(f + 8 * g + 4 * hf);
#pragma unroll
                    for (int j = 0; j < 4; ++j) x[4 * g + j] = p[4 * g + j] * fmaf(dp[4 * g + j], fd, -dq[j]);
                }
                const HalfP ps = half_p<true>(p, kBwdPScale), xs = half_p<false>(x, 1.f);
                T::template rchain<1>(&acc[0], cur, &ps, c, hf, dh);            // dV^T += dO^T P
                T::template rchain<1>(&acc[1], cur + T::TILE, &xs, c, hf, dh);  // dK^T += Q^T dS
            }
            if (st + 1 < nstages) store(lds + ((st + 1) & 1) * STAGE);
            __syncthreads();
        }

        redo |= not_finite(acc);
        if (kj < S) {
            float* dvp = a.dv + base + (int64_t)kj * a.ts;
            float* dkp = a.dk + base + (int64_t)kj * a.ts;
            const float ug = unscale_of(eg) * (1.f / kBwdPScale), uq = unscale_of(eq) * a.scale;
#pragma unroll
            for (int db = 0; db < T::NDBW; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int d0 = dh * T::DW + db * 32 + 8 * g + 4 * hf;
                    if (d0 < D) {
                        floatx4 v, k;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            v[j] = acc[0][db][4 * g + j] * ug;
                            k[j] = acc[1][db][4 * g + j] * uq * i0 * i1;
                        }
                        *reinterpret_cast<floatx4*>(dvp + d0) = v;
                        *reinterpret_cast<floatx4*>(dkp + d0) = k;
                    }
                }
        }
        return redo;
    }
};

// The fp32 MFMA kernels behind them: head dims of exactly 32 or 64 (TIGHT) the
// tiled ones, which need no workspace in recompute mode, else the wide ones.
template <int DP, int NB, int DH, bool CAUSAL, bool RECOMP, bool TIGHT>
struct HalfPair {
    using Q = HalfQ<DP, NB, DH, CAUSAL, RECOMP>;
    using KV = HalfKV<DP, NB, DH, CAUSAL, RECOMP, RECOMP && TIGHT>;
    using XQ = std::conditional_t<TIGHT, BwdQ<TIGHT ? DP : 32, NB, 1, CAUSAL, RECOMP>, WideQ<DP, NB, DH, 2, CAUSAL, RECOMP>>;
    using XKV =
        std::conditional_t<TIGHT, BwdKV<TIGHT ? DP : 32, NB, 1, CAUSAL, RECOMP>, WideKV<DP, NB, DH, 2, CAUSAL, RECOMP>>;
    static constexpr int QB = Q::LDS_BYTES > 4 * XQ::LDS_FLOATS ? Q::LDS_BYTES : 4 * XQ::LDS_FLOATS;
    static constexpr int KB = KV::LDS_BYTES > 4 * XKV::LDS_FLOATS ? KV::LDS_BYTES : 4 * XKV::LDS_FLOATS;
    static constexpr int NT = NB * DH * 64;

    // redo: an int of LDS, zero, ordered by run's barriers
    __device__ __forceinline__ static void q(const BwdArgs& a, unsigned char* lds, int* simd, int* redo, int nb, int bh,
                                             int rank) {
        if (Q::run(a, lds, simd, nb, bh, rank)) *redo = 1;
        __syncthreads();
        if (!*redo) return;
        if constexpr (TIGHT)
            XQ::run(a, reinterpret_cast<float*>(lds), simd, nb, bh, rank);
        else
            XQ::run(a, reinterpret_cast<float*>(lds), nb, bh, rank);
    }
    __device__ __forceinline__ static void kv(const BwdArgs& a, unsigned char* lds, int* simd, int* redo, int nb,
                                              int bh, int rank) {
        if (KV::run(a, lds, simd, nb, bh, rank)) *redo = 1;
        __syncthreads();
        if (!*redo) return;
        if constexpr (TIGHT)
            XKV::run(a, reinterpret_cast<float*>(lds), simd, nb, bh, rank);
        else
            XKV::run(a, reinterpret_cast<float*>(lds), bh, rank);
    }
};

// WHICH: 0 queries, 1 keys, 2 both kinds in one grid, dealt in chunks of B*H
// workgroups in turn (recompute mode: neither needs the other's results).
template <int WHICH, int DP, int NB, int DH, bool CAUSAL, bool RECOMP, bool TIGHT>
__global__ __launch_bounds__(NB* DH * 64) void bwd_half_kernel(BwdArgs a, int nb) {
    using P = HalfPair<DP, NB, DH, CAUSAL, RECOMP, TIGHT>;
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
hipError_t launch_half_mode(const BwdArgs& a, hipStream_t s) {
    const int BH = a.B * a.H;
    const int nb = (a.S + NB * BK - 1) / (NB * BK);
    const int64_t g = (int64_t)nb * BH;
    if (g <= 0 || 2 * g > 0x7fffffff) return hipErrorInvalidConfiguration;
    const dim3 block(NB * DH * 64);
    if constexpr (RECOMP && TIGHT) {
        hipLaunchKernelGGL((bwd_half_kernel<2, DP, NB, DH, CAUSAL, RECOMP, TIGHT>), dim3((unsigned)(2 * g)), block, 0,
                           s, a, nb);
    } else {
        hipLaunchKernelGGL((bwd_half_kernel<0, DP, NB, DH, CAUSAL, RECOMP, TIGHT>), dim3((unsigned)g), block, 0, s, a,
                           nb);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((bwd_half_kernel<1, DP, NB, DH, CAUSAL, RECOMP, TIGHT>), dim3((unsigned)g), block, 0, s, a,
                           nb);
    }
    return hipGetLastError();
}

template <int DP, int NB, int DH, bool TIGHT>
hipError_t launch_half(const BwdArgs& a, hipStream_t s) {
    if (!a.probs)
        return a.causal ? launch_half_mode<DP, NB, DH, TIGHT, true, true>(a, s)
                        : launch_half_mode<DP, NB, DH, TIGHT, false, true>(a, s);
    return a.causal ? launch_half_mode<DP, NB, DH, TIGHT, true, false>(a, s)
                    : launch_half_mode<DP, NB, DH, TIGHT, false, false>(a, s);
}

}  // namespace bwd
}  // namespace hipgpt
