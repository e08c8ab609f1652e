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
// stores, 16-byte bias loads).  Operand staging: global -> registers -> LDS,
// double buffered, one barrier per k-tile; the next tile's global loads are in
// flight during the MFMAs.
//
// gemm_half_tile runs every problem with 16-byte rows on operands split into
// two fp16 terms (split.h; v_mfma_f32_32x32x16_f16, three per product): M 8192
// N 2304 K 768 222 -> 120 us, M 8192 N 768 K 256 30 -> 22.5; error against 64
// bits 4.9e-7 -> 3.1e-7 and 2.9e-7 -> 2.1e-7.  The matrix cores are busy 40% of
// the time, the LDS 57%, the vector ALUs 33% (the split).
//
// gemm_f32_tile (v_mfma_f32_32x32x2_f32) takes tiles whose data the split does
// not hold and operands without 16-byte rows:
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
#include "split.h"

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

// LDS of the split-operand tile (bytes of one stage): two planes (terms) of
// the A tile [BM][32], pitch 40, each row's k in MFMA operand order, and two
// of the W tile [32][BN], row-major, pitch BN + 16.
template <int BM, int BN, int WM, int WN>
struct HalfCfg : Cfg<BM, BN, WM, WN, 32> {
    static constexpr int AP = 40, WP = BN + 16;
    static constexpr int APL = BM * AP, WPL = 32 * WP;
    static constexpr int STAGE16 = 2 * (APL + WPL);  // 16-bit elements of a stage
    static constexpr int SCALES = BM + BN + (BM / WM) * (BN / WN) * BN;  // floats: 1 / row and column scales, column maxima
    static constexpr int BYTES = 2 * STAGE16 * 2 + SCALES * 4;
};

// The tile on split operands (split.h).  Every row of A and every column of W
// carries a power of two of its own, from its largest magnitude in the first
// k-tile (if that is zero there, in the first one where it is not); the
// accumulators are divided by both at the end.  A value more than 255 times
// that magnitude overflows and the result is not finite: false, and the caller
// runs the fp32 tile.
template <int BM, int BN, int WM, int WN, bool BF16OUT, bool KF>
__device__ __forceinline__ bool gemm_half_tile(const GemmArgs& g, unsigned char* lds_raw) {
    using C = HalfCfg<BM, BN, WM, WN>;
    typedef unsigned short u16;
    u16* const lds = reinterpret_cast<u16*>(lds_raw);
    float* const s_row = reinterpret_cast<float*>(lds_raw + 2 * C::STAGE16 * 2);
    float* const s_col = s_row + BM;
    float* const s_max = s_col + BN;
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
    auto load_a = [&](int kt) {
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            const floatx4 v =
                KF ? __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ars, aoff[i], kt * 128, 0))
                   : __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ars, aoff[i] + kt * 128, 0, 0));
            ar[i] = KF || kt * 32 + kc < K ? v : zero4();
        }
    };
    auto load_w = [&](int kt) {
        const int off = (int)((int64_t)kt * 32 * g.ldw * 4);
#pragma unroll
        for (int i = 0; i < C::W_PER; ++i)
            wr[i] = KF ? __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[i], off, 0))
                       : __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[i] + off, 0, 0));
    };

    // ---- scales ----
    float sa[C::A_PER];
    floatx4 sw;
    load_a(0);
    load_w(0);
    {
        float mx[C::A_PER];
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) mx[i] = 0.f;
        for (int kt = 0;;) {
            bool zero = false;
#pragma unroll
            for (int i = 0; i < C::A_PER; ++i) {
                float m = max4(ar[i]);
#pragma unroll
                for (int x = 1; x < 8; x <<= 1) m = fmaxf(m, __shfl_xor(m, x));
                if (mx[i] == 0.f) mx[i] = m;
                zero |= mx[i] == 0.f && tid / 8 + i * (C::NT / 8) < rows;
            }
            if (!__any(zero) || ++kt >= nkt) {
                if (kt > 0) load_a(0);
                break;
            }
            load_a(kt);
        }
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            const unsigned e = scale_exp(mx[i]);
            sa[i] = scale_of(e);
            if ((tid & 7) == 0) s_row[tid / 8 + i * (C::NT / 8)] = unscale_of(e);
        }
        floatx4 cm = zero4();
        for (int kt = 0;;) {
            floatx4 m = zero4();
#pragma unroll
            for (int i = 0; i < C::W_PER; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) m[u] = fmaxf(m[u], fabsf(wr[i][u]));
            if (BN / 4 < 64) {
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int x = BN / 4; x < 64; x <<= 1) m[u] = fmaxf(m[u], __shfl_xor(m[u], x));
            }
            *reinterpret_cast<floatx4*>(s_max + wave * BN + nc) = m;
            __syncthreads();
            bool zero = false;
#pragma unroll
            for (int w = 0; w < C::NW; ++w) {
                const floatx4 t = *reinterpret_cast<const floatx4*>(s_max + w * BN + nc);
#pragma unroll
                for (int u = 0; u < 4; ++u) m[u] = fmaxf(m[u], t[u]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (cm[u] == 0.f) cm[u] = m[u];
                zero |= cm[u] == 0.f && nc < cols;
            }
            // the same answer in every wave: each sees all columns
            if (!__any(zero) || ++kt >= nkt) {
                if (kt > 0) load_w(0);
                break;
            }
            __syncthreads();
            load_w(kt);
        }
        floatx4 us;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned e = scale_exp(cm[u]);
            sw[u] = scale_of(e);
            us[u] = unscale_of(e);
        }
        if (tid < BN / 4) *reinterpret_cast<floatx4*>(s_col + nc) = us;
    }

    auto store = [&](u16* st) {
        // k chunk q of a row holds k = 4q..4q+3; lane half h of step s takes
        // chunks 4s + h and 4s + h + 2 (the order W's transposed reads give)
        const int q = tid & 7;
        const int pos = (q >> 2) * 16 + (q & 1) * 8 + ((q >> 1) & 1) * 4;
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            uint2 t[2];
            half_pair(ar[i][0] * sa[i], ar[i][1] * sa[i], t[0].x, t[1].x);
            half_pair(ar[i][2] * sa[i], ar[i][3] * sa[i], t[0].y, t[1].y);
            u16* p = st + (tid / 8 + i * (C::NT / 8)) * C::AP + pos;
            *reinterpret_cast<uint2*>(p) = t[0];
            *reinterpret_cast<uint2*>(p + C::APL) = t[1];
        }
#pragma unroll
        for (int i = 0; i < C::W_PER; ++i) {
            uint2 t[2];
            half_pair(wr[i][0] * sw[0], wr[i][1] * sw[1], t[0].x, t[1].x);
            half_pair(wr[i][2] * sw[2], wr[i][3] * sw[3], t[0].y, t[1].y);
            u16* p = st + 2 * C::APL + (tid / (BN / 4) + i * (C::NT / (BN / 4))) * C::WP + nc;
            *reinterpret_cast<uint2*>(p) = t[0];
            *reinterpret_cast<uint2*>(p + C::WPL) = t[1];
        }
    };

    floatx16 acc[C::NB][C::MB];
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
        for (int j = 0; j < C::MB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto compute = [&](const u16* st) {
        const int r = c & 15;
        const u16* As = st + (wm0 + c) * C::AP + h * 8;
        const u16* Ws = st + 2 * C::APL + (4 * h + (r >> 2)) * C::WP + wn0 + (c & 16) + 4 * (r & 3);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Half8 a[C::MB], w[C::NB];
#pragma unroll
            for (int j = 0; j < C::MB; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    a[j].t[t] = *reinterpret_cast<const halfx8*>(As + t * C::APL + j * 32 * C::AP + s * 16);
#pragma unroll
            for (int i = 0; i < C::NB; ++i)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const u16* p = Ws + t * C::WPL + s * 16 * C::WP + i * 32;
                    w[i].t[t] = read_rows_tr(p, 8 * C::WP);
                }
#pragma unroll
            for (int i = 0; i < C::NB; ++i)
#pragma unroll
                for (int j = 0; j < C::MB; ++j) acc[i][j] = mfma_half(w[i], a[j], acc[i][j]);
        }
    };

    store(lds);
    __syncthreads();
    auto step = [&](int kt, auto stage_tag) {
        constexpr int SB = decltype(stage_tag)::value;
        if (kt + 1 < nkt) {
            load_a(kt + 1);
            load_w(kt + 1);
        }
        compute(lds + SB * C::STAGE16);
        if (kt + 1 < nkt) store(lds + (1 - SB) * C::STAGE16);
        __syncthreads();
    };
    for (int kt = 0; kt < nkt; kt += 2) {
        step(kt, std::integral_constant<int, 0>{});
        if (kt + 1 < nkt) step(kt + 1, std::integral_constant<int, 1>{});
    }

    unsigned top = 0;
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
        for (int j = 0; j < C::MB; ++j) {
            const float ua = s_row[wm0 + 32 * j + c];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const floatx4 uw = *reinterpret_cast<const floatx4*>(s_col + wn0 + 32 * i + 8 * q + 4 * h);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    top = max(top, __float_as_uint(acc[i][j][4 * q + u]) & 0x7fffffffu);
                    acc[i][j][4 * q + u] = acc[i][j][4 * q + u] * ua * uw[u];
                }
            }
        }
    int* const flag = reinterpret_cast<int*>(s_max);  // zero after the loop's barriers
    if (tid == 0) *flag = 0;
    __syncthreads();
    if (top >= 0x7f800000u) *flag = 1;  // inf or NaN
    __syncthreads();
    if (*flag) return false;
    store_tile<C, true, BF16OUT>(g, acc, reinterpret_cast<float*>(lds_raw), m0 + wm0, n0 + wn0, wave, lane);
    return true;
}

template <int BM, int BN, int WM, int WN, bool BF16OUT, bool KF>
__global__ __launch_bounds__(BM / WM * (BN / WN) * 64) void gemm_half_kernel(GemmArgs g) {
    constexpr int FB = 2 * Cfg<BM, BN, WM, WN, 32>::STAGE * 4, HB = HalfCfg<BM, BN, WM, WN>::BYTES;
    __shared__ __attribute__((aligned(16))) unsigned char lds[FB > HB ? FB : HB];
    if (gemm_half_tile<BM, BN, WM, WN, BF16OUT, KF>(g, lds)) return;
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
hipError_t launch_half(const GemmArgs& g, hipStream_t s) {
    const int64_t tiles = (int64_t)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    if (tiles <= 0 || tiles > 0x7fffffff) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)tiles), block(BM / WM * (BN / WN) * 64);
    const bool kf = g.K % 32 == 0;
    if (g.out_bf16) {
        if (kf)
            hipLaunchKernelGGL((gemm_half_kernel<BM, BN, WM, WN, true, true>), grid, block, 0, s, g);
        else
            hipLaunchKernelGGL((gemm_half_kernel<BM, BN, WM, WN, true, false>), grid, block, 0, s, g);
    } else {
        if (kf)
            hipLaunchKernelGGL((gemm_half_kernel<BM, BN, WM, WN, false, true>), grid, block, 0, s, g);
        else
            hipLaunchKernelGGL((gemm_half_kernel<BM, BN, WM, WN, false, false>), grid, block, 0, s, g);
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

// 128 x 128 outputs per workgroup (four waves of 64 x 64: the fewest LDS reads
// per MFMA that fit two workgroups on a CU) where those fill the CUs, else
// 64 x 128 (eight waves of 32 x 32).  us, 128 x 128 against 64 x 128, by 128 x
// 128 tiles: M 1024 N 768 K 256 (48) 16.8, 9.1; M 1024 N 2304 K 768 (144) 31.3,
// 26.4; M 2048 N 2304 K 768 (288) 41.5, 46.0; M 8192 N 768 K 256 (384) 23.6,
// 23.9; M 8192 N 2304 K 768 (1152) 122, 134.  256 x 128, 128 x 64, 64 x 64 and
// eight waves on 128 x 128 were level or slower.
// Each XCD takes a contiguous range of tiles (by_xcd) while W is small enough
// to stay in its L2 beside the A rows: 122 -> 120 us at W of 7 MB, 23.6 -> 22.5
// at 0.8 MB, level at 12 MB, 337 -> 356 at 50 MB.
hipError_t launch_vec(const GemmArgs& in, hipStream_t s) {
    GemmArgs g = in;
    g.by_xcd = (int64_t)g.K * g.N <= (int64_t)2 << 20;
    if (g.K <= 0) return launch_unaligned(g, s);  // bias alone
    const int64_t tiles = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
    return tiles >= 256 ? launch_half<128, 128, 64, 64>(g, s) : launch_half<64, 128, 32, 32>(g, s);
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
