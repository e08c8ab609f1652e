// bwd_tiled.h -- LDS-tiled MFMA kernels of the attention backward on the
// forward's probabilities (HipGPT src/hip_kernels.cpp:1159-1272), for head
// dims 32 and 64 with 16-byte aligned rows.  The workgroups of bwd_terms.h run
// them where a result on bf16 terms is not finite.
//
// Math per (b, h), scale c = 1/sqrt(D):
//   dP = dO V^T,  Dq_i = sum_j P_ij dP_ij,  dS = P o (dP - Dq),
//   dQ = c dS K,  dK = c dS^T Q,  dV = P^T dO.
// Two kernels, every gradient element written once (no atomics, no memset):
//   * BwdQ (query-stationary): a wave owns 32 queries.  One pass over the keys
//     accumulates
//       A = (P o dP) K,  Bm = P K,  Dq = rowsum(P o dP),
//     and dQ = c (A - Dq Bm), so P and V are read once.  Dq goes to the
//     workspace for the second kernel.
//   * BwdKV (key-stationary): a wave owns 32 keys (V in registers); dP = dO V^T
//     lands with one key per lane and the queries in the accumulator's register
//     order, which is the B-operand layout of dV^T += dO^T P and dK^T += Q^T dS,
//     so P and dS never leave registers.
// Operand tiles go global -> registers -> LDS, double buffered, one barrier
// per tile, with the next tile's loads in flight during the MFMAs.  LDS tiles are row-major (pitch DP+4:
// conflict-free ds_read_b128 along the head dim) or transposed (pitch 36:
// ds_read_b128 along the 32 rows).  P is read straight from global memory in
// the layout each kernel needs: rows of 16 bytes (query-stationary) or
// 128-byte row segments per half-wave (key-stationary).
// Causal (probs zero above the diagonal) skips key tiles past a query
// tile's diagonal (query-stationary) and query tiles before a key tile's
// diagonal (key-stationary).
// Recompute mode (RECOMP; FlashAttention-2's backward): no probs buffer.  The
// forward's O and row log-sum-exp give Dq_i = dO_i . O_i up front (each kernel
// forms it from the dO rows it loads; the query-stationary one then forms
// dQ = c dS K directly) and P is rebuilt per tile as exp2(S' - lse'),
// S' = (c log2 e) q.k from the operand tiles already in LDS plus a row-major K
// (resp. Q) tile, with the causal mask applied on the diagonal tiles.  Neither
// kernel then reads the other's output.
#pragma once

#include <type_traits>

#include "common.h"
#include "fa_common.h"
#include "kernels.h"

namespace hipgpt {
namespace bwd {

using fa::acc_key;
using fa::BK;
using fa::halves_sum;

constexpr int TP = BK + 4;  // pitch of a transposed tile (rows are head dims)

template <int DP>
struct Tiles {
    static constexpr int RP = DP + 4;           // pitch of a row-major tile
    static constexpr int ROW = BK * RP;         // floats of a row-major tile
    static constexpr int TR = DP * TP;          // floats of a transposed tile
    static constexpr int CPR = DP / 4;          // 16-byte chunks per row
    static constexpr int CPT = BK * CPR;        // chunks per tile

    __device__ __forceinline__ static void store_row(float* t, int r, int cc, const floatx4& v) {
        *reinterpret_cast<floatx4*>(t + r * RP + cc * 4) = v;
    }
    __device__ __forceinline__ static void store_tr(float* t, int r, int cc, const floatx4& v) {
#pragma unroll
        for (int j = 0; j < 4; ++j) t[(cc * 4 + j) * TP + r] = v[j];
    }
    // Chain over the head dim: D[m = row c of `rt`][n = c] += sum_d rt[c][d] b[d],
    // lane (c, h) taking d = h*DP/2 + s (b holds the lane's DP/2 values).
    __device__ __forceinline__ static void dchain(floatx16& acc, const float* rt, const float* b, int c, int hf) {
        const float* rr = rt + c * RP + hf * (DP / 2);
#pragma unroll
        for (int j = 0; j < DP / 8; ++j) {
            const floatx4 kv = *reinterpret_cast<const floatx4*>(rr + 4 * j);
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[u], b[4 * j + u], acc, 0, 0, 0);
        }
    }
    // Chain over the 32 tile rows: acc[n][db][m = d][n = c] += sum_k tt[d][k] x[n][k][c]
    // for N right-hand operands sharing the A tile, x in accumulator register
    // order (register t <-> row acc_key(t, h)).
    template <int N>
    __device__ __forceinline__ static void rchain(floatx16 (*acc)[DP / 32], const float* tt, const floatx16* x, int c,
                                                  int hf) {
#pragma unroll
        for (int db = 0; db < DP / 32; ++db) {
            const float* p = tt + (db * 32 + c) * TP + 4 * hf;
            floatx4 blk[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) blk[g] = *reinterpret_cast<const floatx4*>(p + 8 * g);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int n = 0; n < N; ++n)
                        acc[n][db] = __builtin_amdgcn_mfma_f32_32x32x2f32(blk[g][u], x[n][4 * g + u], acc[n][db], 0, 0, 0);
        }
    }
};

// Wave role from its SIMD rank sr and the workgroup's launch rank.  The
// launch ranks of one (b, h) are dealt to the same CUs in turn, so a CU holds
// one workgroup of each rank.  Rotating the roles by the rank spreads causal
// work when there are as many ranks as roles; with two ranks (the c1 / c2
// shapes: 4 roles of 5..8 and 1..4 tiles, resp. 8..5 and 4..1) the second rank
// takes the roles in reverse SIMD order, so every SIMD carries 9 tiles instead
// of 7..11.
__device__ __forceinline__ int role_of(int sr, int rank, int nranks, int nw, bool causal) {
    if (causal && nranks == 2) return rank ? nw - 1 - sr : sr;
    return (sr + rank) % nw;
}

// ----------------------------------------------------------------- dQ, Dq
template <int DP, int NQS, bool CAUSAL, bool RECOMP>
struct BwdQ {
    using T = Tiles<DP>;
    static constexpr int NW = NQS;
    static constexpr int NT = NW * 64;
    static constexpr int NDB = DP / 32;
    static constexpr int NACC = RECOMP ? 1 : 2;  // accumulators: A (, Bm)
    // stage: a key tile, V row-major + K transposed (+ K row-major, the A operand
    // of S^T = K Q^T, when P is recomputed)
    static constexpr int STAGE = T::ROW + T::TR + (RECOMP ? T::ROW : 0);
    static constexpr int PER = (2 * T::CPT + NT - 1) / NT;  // chunks per thread per stage
    static constexpr int LDS_FLOATS = 2 * STAGE;

    // Workgroup `rank` of the nqb query blocks of problem bh.
    __device__ __forceinline__ static void run(const BwdArgs& a, float* lds, int* simd_slots, int nqb, int bh, int rank) {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));  // as a second pass: nothing of the first stays live for it
        const int lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int c = lane & 31, hf = lane >> 5;
        const int qb = CAUSAL ? nqb - 1 - rank : rank;
        const int qs = role_of(fa::simd_rank<NW>(simd_slots, wave, lane), rank, nqb, NW, CAUSAL);
        const int b = bh / a.H, h = bh % a.H;
        const int S = a.S;
        const int q0 = qb * NQS * BK, qw0 = q0 + qs * BK, qi = qw0 + c;
        const int64_t base = (int64_t)b * a.bs + (int64_t)h * a.hs;
        const int kend = CAUSAL ? min(S, q0 + NQS * BK) : S;
        const int ntiles = (kend + BK - 1) / BK;
        const int wtiles = qw0 < S ? (CAUSAL ? (min(S, qw0 + BK) + BK - 1) / BK : ntiles) : 0;

        // dO (B operand of dP^T = V dO^T): lane (c, h) holds dO[qi][h*DP/2 + s]
        float go[DP / 2];
        {
            const float* g = a.go + base + (int64_t)qi * a.ts + hf * (DP / 2);
#pragma unroll
            for (int s = 0; s < DP / 2; s += 4) {
                const floatx4 t = qi < S ? *reinterpret_cast<const floatx4*>(g + s) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; ++j) go[s + j] = t[j];
            }
        }
        // Recompute mode: Q (B operand of S^T = K Q^T) pre-scaled to log2
        // units, the row's log-sum-exp in the same units, and the row dot
        // Dq_i = dO_i . O_i.
        float q2[RECOMP ? DP / 2 : 1];
        float lse2 = 0.f, dqv = 0.f;
        if constexpr (RECOMP) {
            const float qsc = a.scale * kLog2e;
            const float* qp = a.q + base + (int64_t)qi * a.ts + hf * (DP / 2);
            const float* op = a.o + base + (int64_t)qi * a.ts + hf * (DP / 2);
            float dsum = 0.f;
#pragma unroll
            for (int s = 0; s < DP / 2; s += 4) {
                const floatx4 qv = qi < S ? *reinterpret_cast<const floatx4*>(qp + s) : floatx4{0.f, 0.f, 0.f, 0.f};
                const floatx4 ov = qi < S ? *reinterpret_cast<const floatx4*>(op + s) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    q2[s + j] = qv[j] * qsc;
                    dsum = fmaf(go[s + j], ov[j], dsum);
                }
            }
            dqv = halves_sum(dsum);
            if (qi < S) lse2 = a.lse[(int64_t)bh * S + qi] * kLog2e;
        }
        RowLoader kl, vl;
        kl.init(a.k + base, a.ts, S, a.D);
        vl.init(a.v + base, a.ts, S, a.D);
        floatx4 stg[PER];
        static_assert((T::CPT) % 64 == 0, "a wave's chunks are all K or all V");
        auto load = [&](int st) {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int f = tid + i * NT;
                if ((2 * T::CPT) % NT != 0 && f >= 2 * T::CPT) break;
                const int isk = f >= T::CPT;
                const int g = isk ? f - T::CPT : f;
                const int row = st * BK + g / T::CPR;
                // K or V is wave-uniform (CPT is a multiple of 64): a scalar
                // branch instead of a per-lane select of two buffer resources
                if (__builtin_amdgcn_readfirstlane(isk))
                    stg[i] = kl.load(row, g % T::CPR);
                else
                    stg[i] = vl.load(row, g % T::CPR);
            }
        };
        auto store = [&](float* dst) {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int f = tid + i * NT;
                if ((2 * T::CPT) % NT != 0 && f >= 2 * T::CPT) break;
                const int isk = f >= T::CPT;
                const int g = isk ? f - T::CPT : f;
                const int r = g / T::CPR, cc = g % T::CPR;
                if (isk) {
                    T::store_tr(dst + T::ROW, r, cc, stg[i]);
                    if (RECOMP) T::store_row(dst + T::ROW + T::TR, r, cc, stg[i]);
                } else {
                    T::store_row(dst, r, cc, stg[i]);
                }
            }
        };

        floatx16 acc[NACC][NDB];  // [0] = A^T (recompute: dS K, unscaled), [1] = Bm^T, both [d][query]
#pragma unroll
        for (int n = 0; n < NACC; ++n)
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][db][r] = 0.f;
        float ld = 0.f;
        const float* prow = RECOMP ? nullptr : a.probs + ((int64_t)bh * S + qi) * S;
        const bool pvec = (S & 3) == 0;

        // P of key tile t in accumulator order: piece g holds keys
        // t*32 + 8g + 4h .. +3 (register 4g + j <-> key t*32 + acc_key(4g + j, h)).
        auto load_p = [&](floatx4 (&pv)[4], int t) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int k0 = t * BK + 8 * g + 4 * hf;
                if (pvec && qi < S && k0 + 3 < S) {
                    pv[g] = *reinterpret_cast<const floatx4*>(prow + k0);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) pv[g][j] = (qi < S && k0 + j < S) ? prow[k0 + j] : 0.f;
                }
            }
        };
        // The next tile's P is requested while this tile's MFMAs run.
        floatx4 pnext[4];
        if (!RECOMP && wtiles > 0) load_p(pnext, 0);

        auto compute = [&](int t, const float* tile) {
            if (t >= wtiles) return;
            floatx16 x[2];
            if constexpr (RECOMP) {
                floatx16 sc;
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = 0.f;
                T::dchain(sc, tile + T::ROW + T::TR, q2, c, hf);  // S'^T, register r <-> key acc_key(r, h)
                const int kb0 = t * BK;
                const bool edge = kb0 + BK > S || (CAUSAL && kb0 + BK - 1 > qw0);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = kb0 + acc_key(r, hf);
                    const float p = fast_exp2(sc[r] - lse2);
                    x[1][r] = (!edge || (key < S && (!CAUSAL || key <= qi))) ? p : 0.f;
                }
            } else {
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int j = 0; j < 4; ++j) x[1][4 * g + j] = pnext[g][j];
                if (t + 1 < wtiles) load_p(pnext, t + 1);
            }
            floatx16 dp;
#pragma unroll
            for (int r = 0; r < 16; ++r) dp[r] = 0.f;
            T::dchain(dp, tile, go, c, hf);  // dP^T, register r <-> key acc_key(r, h)
            if constexpr (RECOMP) {
#pragma unroll
                for (int r = 0; r < 16; ++r) x[0][r] = x[1][r] * (dp[r] - dqv);
                T::template rchain<1>(acc, tile + T::ROW, x, c, hf);  // (dS K)^T += K^T dS^T
            } else {
                float s = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    x[0][r] = x[1][r] * dp[r];
                    s += x[0][r];
                }
                ld += s;
                T::template rchain<2>(acc, tile + T::ROW, x, c, hf);  // A^T += K^T (P o dP)^T, Bm^T += K^T P^T
            }
        };

        if (ntiles > 0) {
            load(0);
            store(lds);
        }
        __syncthreads();
        for (int st = 0; st < ntiles; ++st) {
            if (st + 1 < ntiles) load(st + 1);
            compute(st, lds + (st & 1) * STAGE);
            if (st + 1 < ntiles) store(lds + ((st + 1) & 1) * STAGE);
            __syncthreads();
        }

        if (qi < S) {
            const float dq = RECOMP ? dqv : halves_sum(ld);
            if (!RECOMP && hf == 0) a.dvec[(int64_t)bh * S + qi] = dq;
            float* out = a.dq + base + (int64_t)qi * a.ts;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    floatx4 v;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        v[j] = RECOMP ? a.scale * acc[0][db][4 * g + j]
                                      : a.scale * fmaf(-dq, acc[NACC - 1][db][4 * g + j], acc[0][db][4 * g + j]);
                    *reinterpret_cast<floatx4*>(out + db * 32 + 8 * g + 4 * hf) = v;
                }
        }
    }
};

// ----------------------------------------------------------------- dK, dV
template <int DP, int NKB, bool CAUSAL, bool RECOMP>
struct BwdKV {
    using T = Tiles<DP>;
    static constexpr int NW = NKB;
    static constexpr int NT = NW * 64;
    static constexpr int NDB = DP / 32;
    // stage: a query tile, dO row-major + dO transposed + Q transposed + Dq (+ lse' + Q row-major, the A operand of S' = Q K^T, when P is
    // recomputed)
    static constexpr int DQ_OFF = T::ROW + 2 * T::TR;
    static constexpr int LSE_OFF = DQ_OFF + BK;
    static constexpr int QROW_OFF = LSE_OFF + BK;
    static constexpr int STAGE = DQ_OFF + BK + (RECOMP ? BK + T::ROW : 0);
    static constexpr int PER = (2 * T::CPT + NT - 1) / NT;
    static constexpr int LDS_FLOATS = 2 * STAGE;
    // Recompute mode forms Dq from the staged dO chunks: chunks i < NG of a
    // thread are dO, and a row's CPR chunks sit in consecutive lanes.
    static constexpr int NG = T::CPT / NT;
    static_assert(!RECOMP || (T::CPT) % NT == 0, "dO chunks must fill whole passes");

    // Workgroup `rank` (the key block) of the nkb key blocks of problem bh.
    __device__ __forceinline__ static void run(const BwdArgs& a, float* lds, int* simd_slots, int nkb, int bh, int rank) {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));  // as a second pass: nothing of the first stays live for it
        const int lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int c = lane & 31, hf = lane >> 5;
        const int kb = rank;  // key block; causal: block 0 sees the most query tiles and launches first
        const int ksub = role_of(fa::simd_rank<NW>(simd_slots, wave, lane), rank, nkb, NW, CAUSAL);
        const int b = bh / a.H, h = bh % a.H;
        const int S = a.S;
        const int k0 = kb * NKB * BK, kw0 = k0 + ksub * BK, kj = kw0 + c;
        const int64_t base = (int64_t)b * a.bs + (int64_t)h * a.hs;
        const int nq = (S + BK - 1) / BK;
        // query tiles [it0, nq): causal starts at the workgroup's first key tile
        const int it0 = CAUSAL ? k0 / BK : 0;
        const int wit0 = CAUSAL ? kw0 / BK : 0;  // this wave's first useful query tile
        const int nstages = nq - it0;

        // V (B operand of dP = dO V^T): lane (c, h) holds V[kj][h*DP/2 + s]
        float vr[DP / 2];
        {
            const float* vp = a.v + base + (int64_t)kj * a.ts + hf * (DP / 2);
#pragma unroll
            for (int s = 0; s < DP / 2; s += 4) {
                const floatx4 t = kj < S ? *reinterpret_cast<const floatx4*>(vp + s) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; ++j) vr[s + j] = t[j];
            }
        }
        // Recompute mode: K (B operand of S' = Q K^T) pre-scaled to log2 units
        float kr2[RECOMP ? DP / 2 : 1];
        if constexpr (RECOMP) {
            const float qsc = a.scale * kLog2e;
            const float* kp = a.k + base + (int64_t)kj * a.ts + hf * (DP / 2);
#pragma unroll
            for (int s = 0; s < DP / 2; s += 4) {
                const floatx4 t = kj < S ? *reinterpret_cast<const floatx4*>(kp + s) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; ++j) kr2[s + j] = t[j] * qsc;
            }
        }
        RowLoader gl, ql, ol;
        gl.init(a.go + base, a.ts, S, a.D);
        ql.init(a.q + base, a.ts, S, a.D);
        if (RECOMP) ol.init(a.o + base, a.ts, S, a.D);
        floatx4 stg[PER];
        floatx4 ostg[RECOMP ? NG : 1];  // O chunks matching the dO chunks (recompute mode)
        float dqs = 0.f;   // Dq value this thread stages (stored-probs mode)
        float lses = 0.f;  // lse' value this thread stages (+inf past the last row: P = 0)
        static_assert((T::CPT) % 64 == 0, "a wave's chunks are all Q or all dO");
        auto load = [&](int st) {
            const int qt0 = it0 + st;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int f = tid + i * NT;
                if ((2 * T::CPT) % NT != 0 && f >= 2 * T::CPT) break;
                const int isq = f >= T::CPT;
                const int g = isq ? f - T::CPT : f;
                const int row = qt0 * BK + g / T::CPR;
                if (__builtin_amdgcn_readfirstlane(isq))  // wave-uniform, as above
                    stg[i] = ql.load(row, g % T::CPR);
                else
                    stg[i] = gl.load(row, g % T::CPR);
                if constexpr (RECOMP) {
                    if (i < NG) ostg[i] = ol.load(row, g % T::CPR);
                }
            }
            if (tid < BK) {
                const int qrow = qt0 * BK + tid;
                if (RECOMP)
                    lses = qrow < S ? a.lse[(int64_t)bh * S + qrow] * kLog2e : kInf;
                else
                    dqs = qrow < S ? a.dvec[(int64_t)bh * S + qrow] : 0.f;
            }
        };
        auto store = [&](float* dst) {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int f = tid + i * NT;
                if ((2 * T::CPT) % NT != 0 && f >= 2 * T::CPT) break;
                const int isq = f >= T::CPT;
                const int g = isq ? f - T::CPT : f;
                const int r = g / T::CPR, cc = g % T::CPR;
                if (isq) {
                    T::store_tr(dst + T::ROW + T::TR, r, cc, stg[i]);
                    if (RECOMP) T::store_row(dst + QROW_OFF, r, cc, stg[i]);
                } else {
                    T::store_row(dst, r, cc, stg[i]);
                    T::store_tr(dst + T::ROW, r, cc, stg[i]);
                }
                if constexpr (RECOMP) {
                    // Dq of row r: the chunk dots summed over the row's CPR lanes
                    // (rows past S load as zero: Dq = 0)
                    if (i < NG) {
                        float d = stg[i][0] * ostg[i][0];
#pragma unroll
                        for (int j = 1; j < 4; ++j) d = fmaf(stg[i][j], ostg[i][j], d);
#pragma unroll
                        for (int m = 1; m < T::CPR; m <<= 1) d += __shfl_xor(d, m);
                        if (cc == 0) dst[DQ_OFF + r] = d;
                    }
                }
            }
            if (tid < BK) {
                if (RECOMP)
                    dst[LSE_OFF + tid] = lses;
                else
                    dst[DQ_OFF + tid] = dqs;
            }
        };

        floatx16 acc[2][NDB];  // [0] = dV^T, [1] = dK^T (unscaled), both [d][key]
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][db][r] = 0.f;
        const float* pcol = RECOMP ? nullptr : a.probs + (int64_t)bh * S * S + kj;

        // P column of query tile it, register r <-> query it*32 + acc_key(r, h)
        auto load_p = [&](floatx16& pv, int it) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int qr = it * BK + acc_key(r, hf);
                pv[r] = (qr < S && kj < S) ? pcol[(int64_t)qr * S] : 0.f;
            }
        };
        // The next tile's P is requested while this one's MFMAs run.
        floatx16 pnext;
        if (!RECOMP && wit0 < nq) load_p(pnext, wit0);

        auto compute = [&](int st, const float* tile) {
            const int it = it0 + st;
            if (it < wit0) return;
            floatx16 x[2];  // [0] = P, [1] = dS, register r <-> query it*32 + acc_key(r, h)
            if constexpr (RECOMP) {
                floatx16 sc;
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = 0.f;
                T::dchain(sc, tile + QROW_OFF, kr2, c, hf);  // S', register r <-> query acc_key(r, h)
                const float* lt = tile + LSE_OFF;
                // causal: some query of this tile precedes some key of the wave
                const bool edge = CAUSAL && it * BK < kw0 + BK - 1;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const floatx4 l4 = *reinterpret_cast<const floatx4*>(lt + 8 * g + 4 * hf);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float p = fast_exp2(sc[4 * g + j] - l4[j]);
                        x[0][4 * g + j] = (!edge || it * BK + acc_key(4 * g + j, hf) >= kj) ? p : 0.f;
                    }
                }
            } else {
                x[0] = pnext;
                if (it + 1 < nq) load_p(pnext, it + 1);
            }
            floatx16 dp;
#pragma unroll
            for (int r = 0; r < 16; ++r) dp[r] = 0.f;
            T::dchain(dp, tile, vr, c, hf);  // dP, register r <-> query acc_key(r, h)
            const float* dqt = tile + DQ_OFF;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const floatx4 dq = *reinterpret_cast<const floatx4*>(dqt + 8 * g + 4 * hf);
#pragma unroll
                for (int j = 0; j < 4; ++j) x[1][4 * g + j] = x[0][4 * g + j] * (dp[4 * g + j] - dq[j]);
            }
            // dV^T += dO^T P, dK^T += Q^T dS: two A tiles, one per product
            T::template rchain<1>(&acc[0], tile + T::ROW, &x[0], c, hf);
            T::template rchain<1>(&acc[1], tile + T::ROW + T::TR, &x[1], c, hf);
        };

        if (nstages > 0) {
            load(0);
            store(lds);
        }
        __syncthreads();
        for (int st = 0; st < nstages; ++st) {
            if (st + 1 < nstages) load(st + 1);
            compute(st, lds + (st & 1) * STAGE);
            if (st + 1 < nstages) store(lds + ((st + 1) & 1) * STAGE);
            __syncthreads();
        }

        if (kj < S) {
            float* dvp = a.dv + base + (int64_t)kj * a.ts;
            float* dkp = a.dk + base + (int64_t)kj * a.ts;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int d0 = db * 32 + 8 * g + 4 * hf;
                    *reinterpret_cast<floatx4*>(dvp + d0) =
                        floatx4{acc[0][db][4 * g], acc[0][db][4 * g + 1], acc[0][db][4 * g + 2], acc[0][db][4 * g + 3]};
                    *reinterpret_cast<floatx4*>(dkp + d0) =
                        floatx4{a.scale * acc[1][db][4 * g], a.scale * acc[1][db][4 * g + 1],
                                a.scale * acc[1][db][4 * g + 2], a.scale * acc[1][db][4 * g + 3]};
                }
        }
    }
};

}  // namespace bwd
}  // namespace hipgpt
