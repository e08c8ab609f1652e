// gemm.hip -- fp32 GEMM + bias on gfx950 MFMA: the projections either side
// of the attention (QKV projection and output projection).
//
// Replaces matmul_add_bias_tiled_kernel / launch_matmul_add_bias and
// matmul_tiled_kernel / launch_matmul (HipGPT src/hip_kernels.cpp:113-154,
// :70-109), called from TransformerLayer::self_attention_forward
// (src/transformer_layer.cpp:217, :220):
//     C[m][n] = sum_k A[m][k] W[k][n] (+ bias[n])
// with A [M][K] (row stride lda), W [K][N] (row stride ldw).  Output column
// n goes to C + (n / seg_w) * seg_stride + m * ldc + n % seg_w, which is the
// plain row-major [M][N] buffer for seg_w = N and, for the QKV projection
// (N = 3E, seg_w = E, seg_stride = M*E), the planar [Q|K|V] buffer the
// attention launcher reads.  Output fp32 or bf16 (RNE).
//
// Tiling: a workgroup owns a BM x BN tile of C and walks K in steps of 32.
// Each wave computes a WM x WN sub-tile as C^T = W^T A^T, so an accumulator
// register group holds four consecutive output columns of one row (16-byte
// stores, 16-byte bias loads).  Operand staging: global -> registers -> LDS; the
// next tile's global loads are in flight during the MFMAs.
//
// gemm_terms_tile runs every problem with 16-byte rows on operands split into
// three bf16 terms (terms.h; v_mfma_f32_32x32x16_bf16, six per product).  Against
// the fp32 tile, us, and error against 64 bits: M 8192 N 2304 K 768 227 -> 173,
// 3.5e-7 -> 1.2e-7; M 8192 N 768 K 256 30.0 -> 28.2, 2.0e-7 -> 6.9e-8; M 1024 N
// 768 K 256 13.2 -> 10.8.  Bound by the matrix cores and, in turn with them, the
// conversion of the next k-tile: six MFMAs per product at 173 us are 1.0
// PFLOP/s of the 1.62 that bf16 MFMAs alone reach on random data.
//
// gemm_f32_tile (v_mfma_f32_32x32x2_f32) takes tiles with a result that is not
// finite on the terms, and operands without 16-byte rows:
//   A tile [BM][GBK] (pitch GBK+4 floats): lane (c, h) reads row c,
//     k = (GBK/2)h + s as ds_read_b128 (four k-steps per read).
//   W tile [GBK][BN] (pitch BN+4, second half of the k rows shifted by 32
//     floats so the two lane halves read different banks): lane (c, h) reads
//     W[(GBK/2)h + s][c] as one dword per k-step.
// MFMA 32x32x2 f32 operand layout (lane l, c = l & 31, h = l >> 5): A-operand
// value = row c of the MFMA's M dim, B-operand value = column c of its N dim,
// both at contraction index h of the step; here contraction index
// k = (GBK/2)h + s at step s, the same bijection for both operands.
#include "common.h"
#include "kernels.h"
#include "terms.h"

namespace hipgpt {

namespace {

template <int BM, int BN, int WM, int WN, int GBK_ = 32>
struct Cfg {
    static constexpr int GBK = GBK_;         // k per tile
    static constexpr int APITCH = GBK + 4;   // A tile row pitch, floats
    static constexpr int ACPR = GBK / 4;     // 16-byte chunks per A tile row
    static constexpr int WAVES_M = BM / WM;
    static constexpr int WAVES_N = BN / WN;
    static constexpr int NW = WAVES_M * WAVES_N;
    static constexpr int NT = NW * 64;
    static constexpr int MB = WM / 32;  // m blocks per wave (MFMA N dim)
    static constexpr int NB = WN / 32;  // n blocks per wave (MFMA M dim)
    static constexpr int WPITCH = BN + 4;
    static constexpr int A_ELEMS = BM * APITCH;
    static constexpr int W_ELEMS = GBK * WPITCH + 32;
    static constexpr int STAGE = A_ELEMS + W_ELEMS;
    static constexpr int A_CHUNKS = BM * GBK / 4;
    static constexpr int W_CHUNKS = GBK * BN / 4;
    static constexpr int A_PER = A_CHUNKS / NT;
    static constexpr int W_PER = W_CHUNKS / NT;
    static_assert(A_CHUNKS % NT == 0 && W_CHUNKS % NT == 0, "tile loads must split evenly over the workgroup");
    static_assert(WM % 32 == 0 && WN % 32 == 0 && BM % WM == 0 && BN % WN == 0, "bad tile shape");
    // W row r of the tile lives at r * WPITCH + (r >= GBK/2 ? 32 : 0).
    __device__ __forceinline__ static int wrow(int r) { return r * WPITCH + (r >= GBK / 2 ? 32 : 0); }
};

__device__ __forceinline__ floatx4 zero4() { return floatx4{0.f, 0.f, 0.f, 0.f}; }

// Tile results of one wave (+ bias) to C: rows mw.., columns nw...
template <class C, bool VEC, bool BF16OUT>
__device__ __forceinline__ void store_tile(const GemmArgs& g, const floatx16 (&acc)[C::NB][C::MB], float* lds, int mw,
                                           int nw, int wave, int lane) {
    const int c = lane & 31, h = lane >> 5;
    // ---- epilogue, whole-row path: each 32 x 32 block (+ bias) goes through
    // a per-wave scratch in the (now idle) stage buffers and leaves as whole
    // 128-byte row segments, non-temporally, when the block is inside C, fp32,
    // and its 32 columns stay in one segment ----
    constexpr bool ROWS_T = VEC && !BF16OUT && C::NW * 32 * 36 <= 2 * C::STAGE;
    if constexpr (ROWS_T) {
        float* const X = lds + wave * 32 * 36;
        const int rr = lane >> 3, cc = 4 * (lane & 7);
#pragma unroll
        for (int i = 0; i < C::NB; ++i) {
            const int nb = nw + 32 * i;  // first column of the block
#pragma unroll
            for (int j = 0; j < C::MB; ++j) {
                const int mb = mw + 32 * j;  // first row of the block
                const bool whole = mb + 32 <= g.M && nb + 32 <= g.N && nb / g.seg_w == (nb + 31) / g.seg_w;
                if (!whole) continue;  // left to the general path below
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int n = nb + 8 * q + 4 * h;
                    const floatx4 bv = g.bias ? *reinterpret_cast<const floatx4*>(g.bias + n) : zero4();
                    floatx4 v;
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        v[u] = acc[i][j][4 * q + u] + bv[u];

                    *reinterpret_cast<floatx4*>(X + c * 36 + 8 * q + 4 * h) = v;
                }
                asm volatile("" ::: "memory");  // other lanes' writes (the wave's LDS accesses are in order)
                float* const cb = static_cast<float*>(g.C) + (int64_t)(nb / g.seg_w) * g.seg_stride + nb % g.seg_w;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int row = 8 * k + rr;
                    const floatx4 v = *reinterpret_cast<const floatx4*>(X + row * 36 + cc);
                    __builtin_nontemporal_store(v, reinterpret_cast<floatx4*>(cb + (int64_t)(mb + row) * g.ldc + cc));
                }
                asm volatile("" ::: "memory");  // the next block's writes come after these reads
            }
        }
    }

    // ---- epilogue: + bias, store (register group q -> columns 8q + 4h .. +3) ----
#pragma unroll
    for (int i = 0; i < C::NB; ++i) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = nw + 32 * i + 8 * q + 4 * h;
            floatx4 bv = zero4();
            if (g.bias) {
                if (VEC) {
                    if (n < g.N) bv = *reinterpret_cast<const floatx4*>(g.bias + n);
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u) bv[u] = (n + u < g.N) ? g.bias[n + u] : 0.f;
                }
            }
#pragma unroll
            for (int j = 0; j < C::MB; ++j) {
                const int m = mw + 32 * j + c;
                if (m >= g.M) continue;
                if constexpr (ROWS_T) {  // stored above
                    const int mb = mw + 32 * j, nb = nw + 32 * i;
                    if (mb + 32 <= g.M && nb + 32 <= g.N && nb / g.seg_w == (nb + 31) / g.seg_w) continue;
                }
                floatx4 v;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    v[u] = acc[i][j][4 * q + u] + bv[u];

                if (VEC) {
                    if (n >= g.N) continue;
                    const int64_t off = (int64_t)(n / g.seg_w) * g.seg_stride + (int64_t)m * g.ldc + n % g.seg_w;
                    if (BF16OUT) {
                        bf16x4 o;
#pragma unroll
                        for (int u = 0; u < 4; ++u) o[u] = (__bf16)v[u];
                        *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(g.C) + off) = o;
                    } else {
                        *reinterpret_cast<floatx4*>(static_cast<float*>(g.C) + off) = v;
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int nn = n + u;
                        if (nn >= g.N) break;
                        const int64_t off = (int64_t)(nn / g.seg_w) * g.seg_stride + (int64_t)m * g.ldc + nn % g.seg_w;
                        if (BF16OUT)
                            static_cast<__bf16*>(g.C)[off] = (__bf16)v[u];
                        else
                            static_cast<float*>(g.C)[off] = v[u];
                    }
                }
            }
        }
    }
}

// KF: K is a multiple of GBK (16-byte path only), so no k-tile runs past K:
// the k offset of the loads rides in the buffer instruction's scalar offset
// and the per-element k mask goes away.
template <int BM, int BN, int WM, int WN, int GBK, bool VEC, bool BF16OUT, bool KF>
__device__ __forceinline__ void gemm_f32_tile(const GemmArgs& g, float* lds) {
    using C = Cfg<BM, BN, WM, WN, GBK>;
    constexpr int APITCH = C::APITCH;
    constexpr int ACPR = C::ACPR;
    constexpr int HS = GBK / 2;  // k-steps per tile (each step takes k = HS*h + s)

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int c = lane & 31, h = lane >> 5;
    const int tiles_n = (g.N + BN - 1) / BN;
    const int bid = g.by_xcd ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int tm = bid / tiles_n, tn = bid % tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    const int wm0 = (wave / C::WAVES_N) * WM;  // wave's rows within the tile
    const int wn0 = (wave % C::WAVES_N) * WN;  // wave's columns within the tile
    const int K = g.K;
    const int nkt = (K + GBK - 1) / GBK;

    // ---- global -> register staging of one k-tile ----
    floatx4 ar[C::A_PER], wr[C::W_PER];
    __amdgpu_buffer_rsrc_t ars, wrs;
    int aoff[C::A_PER], woff[C::W_PER];
    if constexpr (VEC) {
        const int rows = min(BM, g.M - m0);
        const int cols = min(BN, g.N - n0);
        ars = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.A + (int64_t)m0 * g.lda), 0,
                                                (int)(((int64_t)(rows - 1) * g.lda + K) * 4), kBufferFlags);
        wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.W + n0), 0,
                                                (int)(((int64_t)(K - 1) * g.ldw + cols) * 4), kBufferFlags);
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            const int f = tid + i * C::NT;
            aoff[i] = (int)(((f / ACPR) * g.lda + (f % ACPR) * 4) * 4);
        }
#pragma unroll
        for (int i = 0; i < C::W_PER; ++i) {
            const int f = tid + i * C::NT;
            const int kr = f / (BN / 4), nc = (f % (BN / 4)) * 4;
            // KF: columns past N re-read column n0 (in bounds; they only feed
            // outputs that are never stored), as the scalar k offset is outside
            // the buffer's range check
            woff[i] = (int)((kr * g.ldw + (KF && nc >= cols ? 0 : nc)) * 4);
        }
    }
    auto load = [&](int kt) {
        const int k0 = kt * GBK;
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            const int f = tid + i * C::NT;
            const int r = f / ACPR, kc = (f % ACPR) * 4;
            if constexpr (VEC && KF) {
                // rows past M read as zero (their voffset is past the range)
                ar[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ars, aoff[i], k0 * 4, 0));
            } else if constexpr (VEC) {
                // rows past M read as zero (buffer range); k past K is masked
                // here because it would read the next row's values
                const floatx4 v = __builtin_bit_cast(
                    floatx4, __builtin_amdgcn_raw_buffer_load_b128(ars, aoff[i] + k0 * 4, 0, 0));
                ar[i] = (k0 + kc < K) ? v : zero4();
            } else {
                const int m = m0 + r;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = k0 + kc + j;
                    ar[i][j] = (m < g.M && k < K) ? g.A[(int64_t)m * g.lda + k] : 0.f;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < C::W_PER; ++i) {
            const int f = tid + i * C::NT;
            const int kr = f / (BN / 4), nc = (f % (BN / 4)) * 4;
            if constexpr (VEC && KF) {
                wr[i] = __builtin_bit_cast(
                    floatx4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[i], (int)((int64_t)k0 * g.ldw * 4), 0));
            } else if constexpr (VEC) {
                // rows past K read as zero; columns past N only feed outputs
                // that are never stored
                wr[i] = __builtin_bit_cast(
                    floatx4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[i] + (int)((int64_t)k0 * g.ldw * 4), 0, 0));
            } else {
                const int k = k0 + kr;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int n = n0 + nc + j;
                    wr[i][j] = (k < K && n < g.N) ? g.W[(int64_t)k * g.ldw + n] : 0.f;
                }
            }
        }
    };
    auto store = [&](float* st) {
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            const int f = tid + i * C::NT;
            *reinterpret_cast<floatx4*>(st + (f / ACPR) * APITCH + (f % ACPR) * 4) = ar[i];
        }
        float* ws = st + C::A_ELEMS;
#pragma unroll
        for (int i = 0; i < C::W_PER; ++i) {
            const int f = tid + i * C::NT;
            *reinterpret_cast<floatx4*>(ws + C::wrow(f / (BN / 4)) + (f % (BN / 4)) * 4) = wr[i];
        }
    };

    floatx16 acc[C::NB][C::MB];
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
        for (int j = 0; j < C::MB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    auto compute = [&](const float* st) {
        const float* As = st + (wm0 + c) * APITCH + h * HS;
        const float* Ws = st + C::A_ELEMS + wn0 + c;
#pragma unroll
        for (int q = 0; q < HS / 4; ++q) {
            floatx4 av[C::MB];
#pragma unroll
            for (int j = 0; j < C::MB; ++j) av[j] = *reinterpret_cast<const floatx4*>(As + j * 32 * APITCH + 4 * q);
            float wv[C::NB][4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int row = C::wrow(h * HS + 4 * q + u);
#pragma unroll
                for (int i = 0; i < C::NB; ++i) wv[i][u] = Ws[row + 32 * i];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < C::NB; ++i)
#pragma unroll
                    for (int j = 0; j < C::MB; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[i][u], av[j][u], acc[i][j], 0, 0, 0);
        }
    };

    if (nkt > 0) {
        load(0);
        store(lds);
    }
    __syncthreads();
    // two k-tiles per iteration, so each stage buffer's address is a constant
    auto step = [&](int kt, auto stage_tag) {
        constexpr int SB = decltype(stage_tag)::value;
        if (kt + 1 < nkt) load(kt + 1);
        compute(lds + SB * C::STAGE);
        if (kt + 1 < nkt) store(lds + (1 - SB) * C::STAGE);
        __syncthreads();
    };
    for (int kt = 0; kt < nkt; kt += 2) {
        step(kt, std::integral_constant<int, 0>{});
        if (kt + 1 < nkt) step(kt + 1, std::integral_constant<int, 1>{});
    }

    store_tile<C, VEC, BF16OUT>(g, acc, lds, m0 + wm0, n0 + wn0, wave, lane);
}

// LDS of the tile on bf16 terms (one stage): three planes (terms) of the A tile
// [BM][32], pitch 40, each row's k in MFMA operand order, and three of the W
// tile [32][BN], row-major, pitch BN + 16.
template <int BM, int BN, int WM, int WN>
struct TermCfg : Cfg<BM, BN, WM, WN, 32> {
    static constexpr int AP = 40, WP = BN + 16;
    static constexpr int APL = BM * AP, WPL = 32 * WP;
    static constexpr int STAGE16 = 3 * (APL + WPL);  // 16-bit elements
    static constexpr int BYTES = STAGE16 * 2 + 16;   // and the not-finite flag
};

// The tile on operands split into three bf16 terms (terms.h).  One LDS stage:
// the next k-tile waits in registers while this one is multiplied, and two or
// three workgroups share a CU, one multiplying while another converts.  False,
// with nothing stored, where a result is not finite; the caller then runs the
// fp32 tile.
template <int BM, int BN, int WM, int WN, bool BF16OUT, bool KF>
__device__ __forceinline__ bool gemm_terms_tile(const GemmArgs& g, unsigned char* lds_raw) {
    using C = TermCfg<BM, BN, WM, WN>;
    typedef unsigned short u16;
    u16* const lds = reinterpret_cast<u16*>(lds_raw);
    int* const flag = reinterpret_cast<int*>(lds_raw + C::STAGE16 * 2);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 31, h = lane >> 5;
    const int tiles_n = (g.N + BN - 1) / BN;
    const int bid = g.by_xcd ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int m0 = bid / tiles_n * BM, n0 = bid % tiles_n * BN;
    const int wm0 = (wave / C::WAVES_N) * WM, wn0 = (wave % C::WAVES_N) * WN;
    const int K = g.K, nkt = (K + 31) / 32;
    const int rows = min(BM, g.M - m0), cols = min(BN, g.N - n0);

    floatx4 ar[C::A_PER], wr[C::W_PER];
    const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(g.A + (int64_t)m0 * g.lda), 0, (int)(((int64_t)(rows - 1) * g.lda + K) * 4), kBufferFlags);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(g.W + n0), 0, (int)(((int64_t)(K - 1) * g.ldw + cols) * 4), kBufferFlags);
    // chunk i: A row tid/8 + i*NT/8, k 4 (tid%8); W row tid/(BN/4) + i*NT/(BN/4), columns 4 (tid % (BN/4))
    const int kc = (tid & 7) * 4, nc = (tid % (BN / 4)) * 4;
    int aoff[C::A_PER], woff[C::W_PER];
#pragma unroll
    for (int i = 0; i < C::A_PER; ++i) aoff[i] = (int)(((tid / 8 + i * (C::NT / 8)) * g.lda + kc) * 4);
#pragma unroll
    for (int i = 0; i < C::W_PER; ++i)
        // columns past N re-read column n0: they feed outputs that are never stored
        woff[i] = (int)(((tid / (BN / 4) + i * (C::NT / (BN / 4))) * g.ldw + (nc >= cols ? 0 : nc)) * 4);
    // rows past M and k rows past K read as zero; a row's k past K is masked
    // (it would read the next row)
    auto load = [&](int kt) {
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            const floatx4 v =
                KF ? __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ars, aoff[i], kt * 128, 0))
                   : __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ars, aoff[i] + kt * 128, 0, 0));
            ar[i] = KF || kt * 32 + kc < K ? v : zero4();
        }
        const int off = (int)((int64_t)kt * 32 * g.ldw * 4);
#pragma unroll
        for (int i = 0; i < C::W_PER; ++i)
            wr[i] = KF ? __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[i], off, 0))
                       : __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[i] + off, 0, 0));
    };
    auto store = [&] {
        // k chunk q of a row holds k = 4q..4q+3; lane half h of step s takes
        // chunks 4s + h and 4s + h + 2 (the order W's transposed reads give)
        const int q = tid & 7;
        const int pos = (q >> 2) * 16 + (q & 1) * 8 + ((q >> 1) & 1) * 4;
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) store_terms(lds + (tid / 8 + i * (C::NT / 8)) * C::AP + pos, C::APL, ar[i]);
#pragma unroll
        for (int i = 0; i < C::W_PER; ++i)
            store_terms(lds + 3 * C::APL + (tid / (BN / 4) + i * (C::NT / (BN / 4))) * C::WP + nc, C::WPL, wr[i]);
    };

    // the small terms have sums of their own: an addition rounds at the size the
    // sum has, and these are 2^-8 of the others (M 8192 N 2304 K 768: 174 us and
    // 3.0e-7 in one sum, 173 and 1.2e-7 so)
    floatx16 acc[C::NB][C::MB], low[C::NB][C::MB];
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
        for (int j = 0; j < C::MB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.f;
    auto compute = [&] {
        const int r = c & 15;
        const u16* As = lds + (wm0 + c) * C::AP + h * 8;
        const u16* Ws = lds + 3 * C::APL + (4 * h + (r >> 2)) * C::WP + wn0 + (c & 16) + 4 * (r & 3);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Term8 a[C::MB], w[C::NB];
#pragma unroll
            for (int j = 0; j < C::MB; ++j)
#pragma unroll
                for (int t = 0; t < 3; ++t)
                    a[j].t[t] = *reinterpret_cast<const bf16x8*>(As + t * C::APL + j * 32 * C::AP + s * 16);
#pragma unroll
            for (int i = 0; i < C::NB; ++i)
#pragma unroll
                for (int t = 0; t < 3; ++t) w[i].t[t] = read_rows_tr(Ws + t * C::WPL + s * 16 * C::WP + i * 32, 8 * C::WP);
#pragma unroll
            for (int i = 0; i < C::NB; ++i)
#pragma unroll
                for (int j = 0; j < C::MB; ++j) {
                    low[i][j] = mfma_terms_small(w[i], a[j], low[i][j]);
                    acc[i][j] = mfma_bf16(w[i].t[0], a[j].t[0], acc[i][j]);
                }
        }
    };

    if (tid == 0) *flag = 0;  // ordered by the loop's barriers
    load(0);
    for (int kt = 0; kt < nkt; ++kt) {
        store();
        __syncthreads();
        if (kt + 1 < nkt) load(kt + 1);
        compute();
        __syncthreads();
    }

    unsigned top = 0;
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
        for (int j = 0; j < C::MB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] += low[i][j][r];
                top = top_bits(top, acc[i][j][r]);
                acc[i][j][r] *= kTermUnscale2;
            }
    if (top >= kInfBits) *flag = 1;
    __syncthreads();
    if (*flag) return false;
    store_tile<C, true, BF16OUT>(g, acc, reinterpret_cast<float*>(lds_raw), m0 + wm0, n0 + wn0, wave, lane);
    return true;
}

template <int BM, int BN, int WM, int WN, bool BF16OUT, bool KF>
__global__ __launch_bounds__(BM / WM * (BN / WN) * 64) void gemm_terms_kernel(GemmArgs g) {
    constexpr int FB = 2 * Cfg<BM, BN, WM, WN, 32>::STAGE * 4, TB = TermCfg<BM, BN, WM, WN>::BYTES;
    __shared__ __attribute__((aligned(16))) unsigned char lds[FB > TB ? FB : TB];
    if (gemm_terms_tile<BM, BN, WM, WN, BF16OUT, KF>(g, lds)) return;
    __syncthreads();
    gemm_f32_tile<BM, BN, WM, WN, 32, true, BF16OUT, KF>(g, reinterpret_cast<float*>(lds));
}

// Operands without 16-byte rows.
template <int BM, int BN, int WM, int WN, bool BF16OUT>
__global__ __launch_bounds__(BM / WM * (BN / WN) * 64) void gemm_f32_kernel(GemmArgs g) {
    __shared__ __attribute__((aligned(16))) float lds[2 * Cfg<BM, BN, WM, WN, 32>::STAGE];
    gemm_f32_tile<BM, BN, WM, WN, 32, false, BF16OUT, false>(g, lds);
}

template <int BM, int BN, int WM, int WN>
hipError_t launch_terms(const GemmArgs& g, hipStream_t s) {
    const int64_t tiles = (int64_t)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    if (tiles <= 0 || tiles > 0x7fffffff) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)tiles), block(BM / WM * (BN / WN) * 64);
    const bool kf = g.K % 32 == 0;
    if (g.out_bf16) {
        if (kf)
            hipLaunchKernelGGL((gemm_terms_kernel<BM, BN, WM, WN, true, true>), grid, block, 0, s, g);
        else
            hipLaunchKernelGGL((gemm_terms_kernel<BM, BN, WM, WN, true, false>), grid, block, 0, s, g);
    } else {
        if (kf)
            hipLaunchKernelGGL((gemm_terms_kernel<BM, BN, WM, WN, false, true>), grid, block, 0, s, g);
        else
            hipLaunchKernelGGL((gemm_terms_kernel<BM, BN, WM, WN, false, false>), grid, block, 0, s, g);
    }
    return hipGetLastError();
}

hipError_t launch_unaligned(const GemmArgs& g, hipStream_t s) {
    const int64_t tiles = (int64_t)((g.M + 63) / 64) * ((g.N + 127) / 128);
    if (tiles <= 0 || tiles > 0x7fffffff) return hipErrorInvalidConfiguration;
    if (g.out_bf16)
        hipLaunchKernelGGL((gemm_f32_kernel<64, 128, 32, 32, true>), dim3((unsigned)tiles), dim3(512), 0, s, g);
    else
        hipLaunchKernelGGL((gemm_f32_kernel<64, 128, 32, 32, false>), dim3((unsigned)tiles), dim3(512), 0, s, g);
    return hipGetLastError();
}

// Tile shapes by how many 128 x 128 tiles there are for the 256 CUs: 128 x 128
// (eight waves of 32 x 64, two workgroups per CU) where each CU gets one, 64 x 128
// (eight of 32 x 32) for half as many, 64 x 64 (four of 32 x 32) below.  us, in this order:
//   M 1024 N 768 K 256 (48 tiles of 128 x 128) 17.8, 12.3, 10.7; M 8192 N 256 K
//   256 (128) 17.4, 12.8, 13.3; M 1024 N 2304 K 768 (144) 41.6, 41.4, 40.4; M
//   2048 N 2304 K 768 (288) 63.3, 66.8, 65.2; M 8192 N 768 K 256 (384) 27.9,
//   27.8, 30.4; M 8192 N 2304 K 768 (1152) 174, 200, 216; M 8192 N 3072 K 1024
//   (1536) 280, 328, 352.
// Four waves of 64 x 64 on 128 x 128 187 at 1152 tiles, 256 x 128 201; two LDS
// stages, which leave one workgroup per CU, 216-266.
// Each XCD takes a contiguous range of tiles (by_xcd) while W is small enough
// to stay in its L2 beside the A rows.
hipError_t launch_vec(const GemmArgs& in, hipStream_t s) {
    GemmArgs g = in;
    g.by_xcd = (int64_t)g.K * g.N <= (int64_t)2 << 20;
    if (g.K <= 0) return launch_unaligned(g, s);  // bias alone
    const int64_t tiles = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
    if (tiles >= 256) return launch_terms<128, 128, 32, 64>(g, s);
    return tiles >= 128 ? launch_terms<64, 128, 32, 32>(g, s) : launch_terms<64, 64, 32, 32>(g, s);
}

}  // namespace

bool gemm_vec_ok(const GemmArgs& g) {
    auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    // 32-bit buffer offsets: W rows up to K + 64, A rows up to 128 past a tile's first row
    const int64_t wbytes = ((int64_t)(g.K + 64) * g.ldw + 128) * 4;
    const int64_t abytes = ((int64_t)128 * g.lda + g.K + 128) * 4;
    return al(g.A) && al(g.W) && al(g.C) && (!g.bias || al(g.bias)) && g.K % 4 == 0 && g.N % 4 == 0 &&
           g.lda % 4 == 0 && g.ldw % 4 == 0 && g.ldc % 4 == 0 && g.seg_w % 4 == 0 && g.seg_stride % 4 == 0 &&
           wbytes < ((int64_t)1 << 31) && abytes < ((int64_t)1 << 31);
}

hipError_t launch_gemm(const GemmArgs& g, hipStream_t s) {
    return gemm_vec_ok(g) ? launch_vec(g, s) : launch_unaligned(g, s);
}

}  // namespace hipgpt
