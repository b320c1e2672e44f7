// Projections of T > 1 prompt rows on bf16 MFMA (v_mfma_f32_32x32x16_bf16), gfx950, and the row kernels around them.
//
// Y[t][n] (+)= sum_k X[t][k] W[n][k], replacing linear_ggml with PREC_F32 (text-decoder.cpp:83-90) and the RMSNorm,
// residual and SwiGLU ops beside it.  Every f32 value is the exact sum of three bf16 parts, v = hi + mid + lo
// (split3.hpp), so a product of two f32 values is a sum of bf16 products, each exact in f32, summed in f32 by the
// MFMAs: f32 products and f32 sums, as the reference's GEMM, in another order.
//   bf16-exact weights (WP 1, one part):  lo w, mid w, hi w                              3 MFMAs per 16 k
//   f32 weights (WP 3, three parts):      lo hi, hi lo, mid mid, mid hi, hi mid, hi hi   6 MFMAs per 16 k
// The products left out of the second form (mid lo, lo mid, lo lo) are within 2^-24 of the whole one, the rounding of
// one f32 sum, and of either sign, since hi and mid are rounded to nearest (split3.hpp).  Parts that are zero add exact
// zeros, and both forms follow one plan and one order, so f32 weights that hold bf16 values give the bits of their bf16
// copies.
//
// Sums.  The bf16 MFMA rounds a sum down more often than up, whatever its sign (products as large as the sum: 41% down,
// 31% up), and six MFMAs per 16 k on f32 weights add up to -1.1e-7 of the outputs' root mean square over 2048 k: the same
// for every token, so an average over tokens, as the attention takes, keeps it while it loses the signal.  X is therefore
// stored negated in blocks + - - + of 256 k (split_negated), and the accumulators turn round with it: 1e-9 remains.
// At 33 to 64 tokens (SUMS) every block of 256 k is a sum of its own, as short as the chains of the f32 kernel before,
// where a wave sums over more than one.
// Relative error against float64 (2-norm, N(0, 1) rows): q|k|v of 2048 k 1.9e-7 at 33 to 64 tokens (gemm_rows_kernel
// 2.0-2.2e-7), 3.5e-7 at 156 and 6.9e-7 from 700 on (sgemm 8.1e-7); a 1.7B layer whose residual is scaled away 0.72-0.77e-6
// (0.77-0.79e-6), 1.5e-6 at 156 and 2.3-2.6e-6 from 700 on (sgemm 2.8-3.0e-6; without the negation 2.9-4.2e-6).
//
// Layout.  X comes in MFMA fragment order (frag offset in split3.hpp): the operand of one MFMA, 32 rows x 16 k of
// one part, is 1 KB of consecutive memory, so a wave loads it from L2 straight into the operand registers with one
// 16-byte load per lane.  Each wave owns 32 token rows and all 128 columns of its workgroup, so no other wave of
// the workgroup needs its X and staging X in LDS would buy nothing; only W, which all its token tiles share, goes
// through LDS.  The kernels that produce X (RMSNorm, SwiGLU, the attention's split) write that order directly.
//
// Work split.  A workgroup is wm token tiles x kw K groups of waves over 128 columns and one of ks K slices
// (prompt_plan); K groups are summed through LDS, K slices are left as partial sums that the next row kernel adds
// up in slice order (prompt_norm, prompt_swiglu, the append), so no workgroup waits for another.
// What bounds it (us of a 1.7B layer's four GEMMs, traced in whole calls, weights from HBM): at T = 156 96 on bf16 weights,
// against 39 of MFMA time at 1.2 PFLOP/s and 16 for the 100 MB of weights; short K slices are chains of first loads, 4-16
// stages and a tail.  (The 128 x 256 tiles of gemm_split3.hip put 16-96 workgroups on 256 CUs: 436; at T = 52
// gemm_rows_kernel on f32 weights 294, now 59.)  f32 weights: T = 52 91 (gemm_rows_kernel 293), T = 156 166 (rocBLAS sgemm
// 259).  At T = 3913 it executes 1.16-1.21 PFLOP/s, the rate power allows (a library bf16 GEMM of random operands: 1.2),
// with the matrix cores busy for 0.5 to 0.64 of the cycles: 1065 on bf16 weights (gemm_split3.hip 1103), 2044 on f32 weights
// (sgemm 2892, at 98% of the f32 MFMA rate).
#include "ops.hpp"
#include "split3.hpp"
#include "wave.hpp"

#include <algorithm>
#include <cmath>

namespace qa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u4v __attribute__((ext_vector_type(4)));

constexpr int kPgCols = 128;               // columns per workgroup (256 with NT = 8)
constexpr int kMaxWaves = 8;

enum { kPgStore = 0, kPgAccumulate = 1, kPgSwiglu = 2, kPgPartial = 3 };
constexpr int kPgMaxSplitWgs = 320;        // workgroups of a plan with K slices: bounds the partial sums

struct PgParams {
    const uint16_t * Xf;     // fragment-ordered split of X (frag_index)
    const uint16_t * W;      // WP 1: [rows of W][K] bf16 bits; WP 3: fragment-ordered split of W (prompt_pack_launch)
    float * Y;               // [M][N] (store, accumulate) or the partials [ks][M][N]
    uint16_t * act;          // SwiGLU: fragment-ordered split of silu(gate) * up, [M][N]
    int32_t M, N, K;         // N output columns (SwiGLU: W has 2 N rows)
    int32_t m_tiles;         // ceil(M / 32)
    int32_t wm, kw;          // token tiles and K groups of a workgroup (wm kw waves)
    int32_t m_groups, n_groups, ks;
    int32_t per;             // stages of one K group of a slice, the same for all (kw ks per stages in all)
};

// WP: parts of W.  SK: 16-k MFMA steps per stage.  One stage of W per K group: WP 1: 128 rows x 128 B in 1 KB
// blocks of 8 rows, chunk c of row r in slot c ^ (r % 8); WP 3: SK x 4 tiles x 3 parts, 1 KB fragments.
template <int WP, int NT>
struct Stage {
    static constexpr int kSteps = WP == 1 ? 4 : 2;
    static constexpr int kBlocks = WP == 1 ? 4 * NT : kSteps * 3 * NT;   // 1 KB each
};

// NT: MFMA tiles of 32 columns per wave.  LPW: 1 KB blocks of a W stage that each wave loads, ceil(kBlocks / wm).
// SUMS: at most four waves per workgroup, which leaves each the registers for a second set of accumulators
template <int WP, int EPI, int NT, int LPW, bool SUMS>
__global__ __launch_bounds__(64 * (SUMS ? 4 : kMaxWaves)) void gemm_prefill_kernel(PgParams p) {
#pragma clang fp contract(off)
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    using St = Stage<WP, NT>;
    constexpr int kCols = 32 * NT;             // W rows per workgroup
    constexpr int SK = St::kSteps;
    constexpr int kStageBytes = St::kBlocks * 1024;
    constexpr bool kSwap = EPI == kPgSwiglu;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int wm = wave % p.wm, kg = wave / p.wm;

    // workgroup -> (slice, token group, column group)
    const int tiles = p.m_groups * p.n_groups;
    const int total = tiles * p.ks;
    int id = blockIdx.x;
    {
        const int q = total / 8, r = total % 8, x = id % 8, j = id / 8;
        id = x * q + min(x, r) + j;
    }
    const int sl = id / tiles;
    int t = id - sl * tiles;
    constexpr int kGm = 4;
    const int g0 = t / (kGm * p.n_groups) * kGm;
    const int gm = min(kGm, p.m_groups - g0);
    t -= g0 * p.n_groups;
    const int mg = g0 + t % gm, ng = t / gm;

    const int mt = mg * p.wm + wm;
    const bool live = mt < p.m_tiles;
    const int mtc = min(mt, p.m_tiles - 1);
    const int k16 = p.K / 16;
    const int my = p.per;
    const int s0 = (sl * p.kw + kg) * my;

    // element offset of 1 KB block blk of stage 0 of this K group of W, and of this lane's 16 bytes in any block (the
    // first is uniform for the wave, so the loads take a scalar base)
    auto w_block = [&](int blk) -> int64_t {
        if constexpr (WP == 1) {
            int64_t row;
            if constexpr (EPI == kPgSwiglu) {
                row = static_cast<int64_t>((blk >> 2) & 1) * p.N + ng * (kCols / 2) + 32 * (blk >> 3) + 8 * (blk & 3);
            } else {
                row = ng * kCols + blk * 8;
            }
            return row * p.K + static_cast<int64_t>(s0) * 64;
        } else {
            const int step = blk / (3 * NT), j = blk % (3 * NT) / 3, part = blk % 3;
            int tile;
            if constexpr (EPI == kPgSwiglu) tile = (j & 1) * (p.N / 32) + ng * (NT / 2) + (j >> 1);
            else tile = ng * NT + j;
            return ((static_cast<int64_t>(tile) * k16 + s0 * SK + step) * 3 + part) * 512;
        }
    };
    const uint32_t w_lane = WP == 1 ? (lane >> 3) * p.K + ((lane & 7) ^ (lane >> 3)) * 8 : lane * 8;
    constexpr int kStageElems = WP == 1 ? 64 : SK * 3 * 512;   // elements a source advances per stage
    unsigned char * ring = lds + kg * 2 * kStageBytes;

    const uint16_t * xbase = p.Xf + static_cast<int64_t>(mtc) * k16 * 3 * 512 + lane * 8;
    bf16x8 x[SK][3];
    auto load_x = [&](int s, int b) {
        const uint16_t * q = xbase + static_cast<int64_t>(min((s0 + s) * SK + b, k16 - 1)) * 3 * 512;
#pragma unroll
        for (int part = 0; part < 3; ++part) x[b][part] = *reinterpret_cast<const bf16x8 *>(q + part * 512);
    };

    v16f acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = v16f{};
    const int rr = lane & 31;
    // W fragments of half hf (4 tiles) of step b of the stage at st
    auto read_w = [&](const unsigned char * st, int b, int hf, bf16x8 (&w)[4][WP]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int tile = 4 * hf + j;
            if constexpr (WP == 1) {
                w[j][0] = *reinterpret_cast<const bf16x8 *>(st + (4 * tile + (rr >> 3)) * 1024 + 128 * (rr & 7) +
                                                            16 * ((2 * b + (lane >> 5)) ^ (rr & 7)));
            } else {
#pragma unroll
                for (int part = 0; part < 3; ++part)
                    w[j][part] = *reinterpret_cast<const bf16x8 *>(st + ((b * NT + tile) * 3 + part) * 1024 + lane * 16);
            }
        }
    };
    auto mma = [&](const bf16x8 & a, const bf16x8 & b, const v16f & c) {
        return kSwap ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, c, 0, 0, 0)
                     : __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    };

    // the MFMAs of stage s; the next step's W fragments are read from LDS, and the next stage's X fragments
    // loaded, around the MFMAs of a step (the scheduling barriers keep them there)
    auto compute = [&](const unsigned char * st, int s) {
        constexpr int kH = NT / 4;
        constexpr int kSets = LPW < 12 ? 2 : 1;    // (12 blocks per wave leave no registers for a second set)
        bf16x8 w[kSets][4][WP];
        if (kSets > 1) read_w(st, 0, 0, w[0]);
#pragma unroll
        for (int b = 0; b < SK; ++b) {
#pragma unroll
            for (int hf = 0; hf < kH; ++hf) {
                const int i = b * kH + hf;
                if (kSets == 1) read_w(st, b, hf, w[0]);
                else if (i + 1 < SK * kH) read_w(st, (i + 1) / kH, (i + 1) % kH, w[(i + 1) % kSets]);
                __builtin_amdgcn_sched_barrier(0);
                bf16x8 (&wb)[4][WP] = w[i % kSets];
                if constexpr (WP == 1) {
#pragma unroll
                    for (int part = 2; part >= 0; --part)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[4 * hf + j] = mma(x[b][part], wb[j][0], acc[4 * hf + j]);
                } else {
                    constexpr int px[6] = {2, 0, 1, 1, 0, 0}, pw[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                    for (int q = 0; q < 6; ++q)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[4 * hf + j] = mma(x[b][px[q]], wb[j][pw[q]], acc[4 * hf + j]);
                }
                if (hf + 1 == kH) load_x(s + 1, b);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // two LDS stages; stage s + 1 is loaded into registers while stage s computes, then written to LDS.  (Not
    // loaded straight into LDS: vector loads complete in issue order, and with LDS loads in flight the compiler
    // waits for every X load at once.)
    const uint16_t * src[LPW];
    int dst[LPW];
#pragma unroll
    for (int u = 0; u < LPW; ++u) {
        const int blk = min(wm + u * p.wm, St::kBlocks - 1);
        dst[u] = blk * 1024;
        src[u] = p.W + w_block(blk);
    }
    u4v wv[LPW];
    auto load_w = [&](int s) {
        const int64_t o = static_cast<int64_t>(min(s, my - 1)) * kStageElems;
#pragma unroll
        for (int u = 0; u < LPW; ++u) wv[u] = *reinterpret_cast<const u4v *>(src[u] + o + w_lane);
    };
    auto write_w = [&](int s) {
#pragma unroll
        for (int u = 0; u < LPW; ++u) *reinterpret_cast<u4v *>(ring + (s & 1) * kStageBytes + dst[u] + lane * 16) = wv[u];
    };
    load_w(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < SK; ++b) load_x(0, b);
    __builtin_amdgcn_sched_barrier(0);
    write_w(0);
    // stages in parts of at most kSplitSign k.  Where the sign of X changes the accumulators turn round with it; SUMS: each
    // part is added to a sum of its own and the accumulators start again (see the header)
    constexpr int kPart = kSplitSign / (16 * SK);
    v16f sums[SUMS ? NT : 1];
    if constexpr (SUMS) {
#pragma unroll
        for (int j = 0; j < NT; ++j) sums[j] = v16f{};
    }
    for (int s = 0; s < my;) {
        const int end = min(my, s + kPart - (s0 + s) % kPart);
        const bool minus = split_negated((s0 + s) * 16 * SK);
        for (; s < end; ++s) {
            __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): this wave's part of stage s is in LDS
            __builtin_amdgcn_s_barrier();          // and every wave's; nobody reads stage s - 1 any more
            __builtin_amdgcn_sched_barrier(0);
            load_w(s + 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(ring + (s & 1) * kStageBytes, s);
            write_w(s + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (SUMS) {
            const float sign = minus ? -1.0f : 1.0f;
            if (s < my) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) sums[j][e] = __builtin_fmaf(sign, acc[j][e], sums[j][e]);
                    acc[j] = v16f{};
                }
            } else {
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[j][e] = __builtin_fmaf(sign, acc[j][e], sums[j][e]);
            }
        } else if (s < my ? minus != split_negated((s0 + s) * 16 * SK) : minus) {
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[j] = -acc[j];
        }
    }
    // the K groups of the workgroup, in order, through LDS
    if (p.kw > 1) {
        __syncthreads();
        float * red = reinterpret_cast<float *>(lds);
        if (kg > 0) {
            float * o = red + ((kg - 1) * p.wm + wm) * (NT * 1024) + lane;
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[(j * 16 + e) * 64] = acc[j][e];
        }
        __syncthreads();
        if (kg > 0) return;
        for (int g = 1; g < p.kw; ++g) {
            const float * o = red + ((g - 1) * p.wm + wm) * (NT * 1024) + lane;
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[j][e] += o[(j * 16 + e) * 64];
        }
    }
    if (!live) return;
    const int h = lane >> 5;
    if constexpr (EPI == kPgSwiglu) {
        // D[W row][token]: token rr, W row 8 (e / 4) + 4 h + e % 4 of the tile; tiles 2 q, 2 q + 1 are gate and up
        const int n16 = p.N / 16;
#pragma unroll
        for (int q = 0; q < NT / 2; ++q) {
            const int c = ng * (kCols / 2) + 32 * q;
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float g = acc[2 * q][4 * o + e], u = acc[2 * q + 1][4 * o + e];
                    v[e] = (g / (1.0f + expf(-g))) * u;
                }
                store_frag4(p.act, n16, 32 * mtc + rr, c + 8 * o + 4 * h, v[0], v[1], v[2], v[3]);
            }
        }
    } else {
        // D[token][column]: column rr of the tile, token 8 (e / 4) + 4 h + e % 4
        float * y = p.Y + (EPI == kPgPartial ? static_cast<int64_t>(sl) * p.M * p.N : 0);
        const int tb = 32 * mt + 4 * h;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int col = ng * kCols + 32 * j + rr;
            if constexpr (EPI == kPgAccumulate) {
#pragma unroll
                for (int e0 = 0; e0 < 16; e0 += 8) {
                    float old[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        old[e] = y[static_cast<int64_t>(min(tb + 8 * ((e0 + e) >> 2) + (e & 3), p.M - 1)) * p.N + col];
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[j][e0 + e] = old[e] + acc[j][e0 + e];
                }
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = tb + 8 * (e >> 2) + (e & 3);
                if (row < p.M) y[static_cast<int64_t>(row) * p.N + col] = acc[j][e];
            }
        }
    }
}

// ---------------------------------------------------------------- row kernels
// 8 consecutive values (octet o) of row r of the ks partial sums [ks][rows][N], added to v in slice order
__device__ inline void add_partials(const float * part, int ks, int64_t rows, int64_t N, int64_t r, int64_t c, float (&v)[8]) {
    const float * q = part + r * N + c;
#pragma unroll 4
    for (int s = 0; s < ks; ++s, q += rows * N) {
        const v4f a = *reinterpret_cast<const v4f *>(q), b = *reinterpret_cast<const v4f *>(q + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] += a[e];
            v[4 + e] += b[e];
        }
    }
}

__device__ inline void load8(const float * q, float (&v)[8]) {
    const v4f a = *reinterpret_cast<const v4f *>(q), b = *reinterpret_cast<const v4f *>(q + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] = a[e];
        v[4 + e] = b[e];
    }
}

__device__ inline void store8(float * q, const float (&v)[8]) {
    *reinterpret_cast<v4f *>(q) = v4f{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<v4f *>(q + 4) = v4f{v[4], v[5], v[6], v[7]};
}

// x += the partial sums of the projection before it (ks > 0), then (Xf != null) the fragment-ordered split of
// RMSNorm(x) w, as rms_norm_row (text-decoder.cpp:542-557): squares summed in double, float scale, (x scale) w.  One
// pass: IT octets per thread stay in registers.  R rows per workgroup: a row's 16-byte piece of a fragment lies beside
// those of its neighbours, so with R = 8 the lanes of a store fill whole 128-byte lines (one row per workgroup: 40
// instead of 21 us for 3913 rows of 2048); with few rows R = 1 keeps more workgroups in flight.
template <int R, int IT>
__global__ __launch_bounds__(R == 1 ? 256 : 512) void prompt_norm_kernel(float * x, const float * part, int ks,
                                                                         const float * w, int rows, int dim, float eps,
                                                                         uint16_t * Xf) {
#pragma clang fp contract(off)
    constexpr int kThreads = R == 1 ? 256 : 512, G = kThreads / R;
    const int rl = threadIdx.x % R, g = threadIdx.x / R;
    const int row = blockIdx.x * R + rl;
    const bool live = row < rows;
    const int64_t r = min(row, rows - 1);
    float * xr = x + r * dim;
    const int oct = dim / 8;
    float v[IT][8], nw[IT][8];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int o = min(g + G * i, oct - 1);
        load8(xr + o * 8, v[i]);
        if (Xf) load8(w + o * 8, nw[i]);
    }
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int o = g + G * i;
        if (o >= oct) continue;
        if (ks > 0) {
            float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            add_partials(part, ks, rows, dim, r, o * 8, sum);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] += sum[e];
            if (live) store8(xr + o * 8, v[i]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += static_cast<double>(v[i][e]) * v[i][e];
    }
    if (!Xf) return;
    __shared__ double sp[kThreads / 64][R];
    double tot;
    if constexpr (R == 1) {
        ss = wave_sum_d_all(ss);
        if ((threadIdx.x & 63) == 0) sp[threadIdx.x >> 6][0] = ss;
        __syncthreads();
        tot = (sp[0][0] + sp[1][0]) + (sp[2][0] + sp[3][0]);
    } else {
#pragma unroll
        for (int off = R; off < 64; off *= 2) ss += __shfl_xor(ss, off, 64);
        if ((threadIdx.x & 63) < R) sp[threadIdx.x >> 6][rl] = ss;
        __syncthreads();
        tot = 0.0;
#pragma unroll
        for (int q = 0; q < kThreads / 64; ++q) tot += sp[q][rl];
    }
    const float scale = 1.0f / sqrtf(static_cast<float>(tot / static_cast<double>(dim)) + eps);
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int o = g + G * i;
        if (o >= oct || !live) continue;
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = v[i][e] * scale * nw[i][e];
        store_frag8<true>(Xf, dim / 16, static_cast<int>(r), o, y);
    }
}

// Thread = 8 consecutive values of one row; consecutive threads take 8 neighbouring rows, whose pieces of a fragment
// fill whole lines.  MODE 0: the split of src (3: of weights, without the signs of an input); 1: the split of silu(gate) up over the partial sums [ks][rows][2 dim]
// (rows gate | up); 2: the sum of the partial sums, stored to dst.
template <int MODE>
__global__ __launch_bounds__(256) void prompt_rows_kernel(const float * src, int ks, int rows, int dim, float * dst,
                                                          uint16_t * Xf) {
#pragma clang fp contract(off)
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int oct = dim / 8;
    const int64_t i8 = i >> 3;
    const int64_t rb = i8 / oct;
    const int64_t r = rb * 8 + (i & 7);
    const int o = static_cast<int>(i8 - rb * oct);
    if (r >= rows) return;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if constexpr (MODE == 0 || MODE == 3) {
        load8(src + r * dim + o * 8, v);
    } else if constexpr (MODE == 1) {
        float u[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        add_partials(src, ks, rows, 2 * static_cast<int64_t>(dim), r, o * 8, v);
        add_partials(src, ks, rows, 2 * static_cast<int64_t>(dim), r, dim + o * 8, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (v[e] / (1.0f + expf(-v[e]))) * u[e];
    } else {
        add_partials(src, ks, rows, dim, r, o * 8, v);
        store8(dst + r * dim + o * 8, v);
        return;
    }
    store_frag8<MODE != 3>(Xf, dim / 16, static_cast<int>(r), o, v);
}

template <int MODE>
int launch_rows(const float * src, int ks, int32_t rows, int32_t dim, float * dst, uint16_t * Xf, hipStream_t stream) {
    const int64_t blocks = (static_cast<int64_t>((rows + 7) / 8) * 8 * (dim / 8) + 255) / 256;
    hipLaunchKernelGGL((prompt_rows_kernel<MODE>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, src, ks,
                       rows, dim, dst, Xf);
    QA_LAUNCH_CHECK("prompt_rows_kernel");
    return QA_OK;
}

// ---------------------------------------------------------------- launch plan
struct Plan {
    int wm, kw, ks, nt;
    int m_groups;
    int per;          // 64-k units of one K group of a slice
};

// Token tiles per workgroup (wm), K groups (kw), K slices (ks) and column tiles per wave (nt), as the least of a model
// of the GEMM's time in us (bf16 weights):
//   a round of 256 workgroups takes 5 plus its stages; a stage takes 0.9 (the latency of the loads one stage ahead),
//   its MFMAs at 1 / 1.7 of their peak rate, or its bytes at 60 GB/s per CU, whichever is longest;
//   all workgroups together at most 12 TB/s from L2 and 1.1 PFLOP/s (nt 8, which moves less: 1.25);
//   K slices add 1, their partial sums at 6 TB/s, and for SwiGLU a launch of 4.
// Fitted to a sweep of (wm, kw, ks, nt) over 8 shapes and 20 to 3913 rows: the plan it picks is within 1% of the best
// one on average, 12% at worst.  Examples (1.7B q|k|v, us): 156 rows wm 2 kw 2 ks 2 15.5 (wm 5 ks 8 14.2 and more
// partial sums, wm 5 ks 4 20); 3913 rows wm 8 nt 8 157 (nt 4 170).
// It does not depend on the weights' parts, so that both forms sum in one order (nt does not change the order).
Plan prompt_plan(int32_t M, int64_t cols, int32_t units, bool swiglu) {
    const int tiles = (M + 31) / 32;
    const int mg0 = (tiles + kMaxWaves - 1) / kMaxWaves;
    Plan best{};
    double best_us = 0.0;
    auto consider = [&](int wm, int kw, int ks, int nt) {
        const int groups = (tiles + wm - 1) / wm, per = units / (kw * ks);
        const int64_t wgs = groups * (cols / (32 * nt)) * ks;
        const double bytes = 64.0 * kw * (wm * 32 * 6 + nt * 32 * 2);                       // per stage
        const double flops = 2.0 * 3.0 * wm * kw * 32 * (32 * nt) * 64;
        const double mfma_us = 0.64 * (nt / 4) * ((wm * kw + 3) / 4);
        const double stage_us = std::max({0.9, 1.7 * mfma_us, bytes / 60.0e3});
        double us = ((wgs + 255) / 256) * (5.0 + per * stage_us);
        us = std::max({us, wgs * per * bytes / 12.0e6, wgs * per * flops / (nt == 8 ? 1.25e9 : 1.1e9)});
        if (ks > 1) us += 1.0 + ks * 8.0 * M * cols / 6.0e6 + (swiglu ? 4.0 : 0.0);
        if (best_us == 0.0 || us < best_us) {
            best = Plan{wm, kw, ks, nt, groups, per};
            best_us = us;
        }
    };
    for (int mg = mg0; mg <= mg0 + 3 && mg <= tiles; ++mg) {
        const int wm = std::max(2, (tiles + mg - 1) / mg);   // one tile: the second wave repeats it
        const int64_t groups = (tiles + wm - 1) / wm;
        for (int kw = 1; kw <= 2 && wm * kw <= kMaxWaves; ++kw) {
            for (int ks = 1; ks <= 16; ++ks) {
                if (ks > 1 && groups * (cols / kPgCols) * ks > kPgMaxSplitWgs) break;
                if (units % (kw * ks) == 0) consider(wm, kw, ks, 4);
            }
        }
        if (wm == 8 && cols % (2 * kPgCols) == 0) consider(wm, 1, 1, 8);
    }
    return best;
}

template <int WP, int EPI, int NT, int LPW, bool SUMS = false>
int launch_one(const PgParams & p, hipStream_t stream) {
    const size_t lds = std::max(static_cast<size_t>(p.kw) * 2 * Stage<WP, NT>::kBlocks * 1024,
                                static_cast<size_t>(p.kw - 1) * p.wm * NT * 1024 * sizeof(float));
    if (lds > 64 * 1024) {
        QA_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_prefill_kernel<WP, EPI, NT, LPW, SUMS>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    }
    hipLaunchKernelGGL((gemm_prefill_kernel<WP, EPI, NT, LPW, SUMS>), dim3(static_cast<unsigned>(p.m_groups * p.n_groups * p.ks)),
                       dim3(static_cast<unsigned>(64 * p.wm * p.kw)), lds, stream, p);
    QA_LAUNCH_CHECK("gemm_prefill_kernel");
    return QA_OK;
}

template <int WP, int EPI>
int launch_wm(const PgParams & p, int nt, hipStream_t stream) {
    constexpr int B = Stage<WP, 4>::kBlocks;
    if constexpr (WP == 1 && EPI != kPgPartial) {
        if (nt == 8) return launch_one<WP, EPI, 8, 4>(p, stream);
    }
    switch (p.wm) {
        case 2:
            // Sums of blocks of 256 k where f32 weights had sums as short before, 33 to 64 tokens, and a wave's k reach over
            // more than one block (1.7B: gate|up 512 k, down 192; a length that divides 256 stays in one).  With more groups
            // of tokens one workgroup per CU, as their registers ask for, costs more than it brings (f32 weights, whole calls
            // of 4 layers: 100 tokens 899 / 912 us, 300 tokens 1451 / 1483).  Up to 32 tokens only bf16 weights come
            // here: without, 14 tokens are off by 0.60e-6 (with 0.55, f32 kernels 0.77; a 1.7B layer whose residual is scaled
            // away) and calls of 4 layers take 2% less (20 tokens, 0.6B: 366 us, with 373).
            if (p.m_tiles == 2 && p.m_groups == 1 && kSplitSign % (p.per * 16 * Stage<WP, 4>::kSteps) != 0) {
                return launch_one<WP, EPI, 4, B / 2, true>(p, stream);
            }
            return launch_one<WP, EPI, 4, B / 2>(p, stream);
        case 3: return launch_one<WP, EPI, 4, (B + 2) / 3>(p, stream);
        case 4: return launch_one<WP, EPI, 4, B / 4>(p, stream);
        case 5: return launch_one<WP, EPI, 4, (B + 4) / 5>(p, stream);
        case 6: return launch_one<WP, EPI, 4, (B + 5) / 6>(p, stream);
        case 7: return launch_one<WP, EPI, 4, (B + 6) / 7>(p, stream);
        default: return launch_one<WP, EPI, 4, B / 8>(p, stream);
    }
}

template <int WP>
int launch_epi(int epi, const PgParams & p, int nt, hipStream_t stream) {
    switch (epi) {
        case kPgStore: return launch_wm<WP, kPgStore>(p, nt, stream);
        case kPgAccumulate: return launch_wm<WP, kPgAccumulate>(p, nt, stream);
        case kPgSwiglu: return launch_wm<WP, kPgSwiglu>(p, nt, stream);
        default: return launch_wm<WP, kPgPartial>(p, nt, stream);
    }
}

}  // namespace

bool prompt_gemm_shape_ok(int32_t N, int32_t K, bool swiglu) {
    return N > 0 && K > 0 && K % 64 == 0 && N % (swiglu ? kPgCols / 2 : kPgCols) == 0;
}

size_t prompt_partial_bytes(int32_t rows) {
    const int tiles = std::min((rows + 31) / 32, kMaxWaves);
    return static_cast<size_t>(kPgMaxSplitWgs) * tiles * 32 * kPgCols * sizeof(float);
}

size_t prompt_frag_elems(int32_t rows, int32_t K) { return static_cast<size_t>((rows + 31) / 32) * 32 * K * 3; }

int prompt_gemm_launch(const PromptGemm & g, int32_t * slices, hipStream_t stream) {
    const bool swiglu = g.act != nullptr;
    if ((!g.W16 && !g.W3) || !g.Xf || !g.partial || !slices || g.M <= 0 || (!swiglu && !g.Y)) {
        return fail(QA_ERR_INVALID, "prompt_gemm: invalid arguments");
    }
    if (!prompt_gemm_shape_ok(g.N, g.K, swiglu)) return fail(QA_ERR_INVALID, "prompt_gemm: unsupported shape");
    const int32_t cols = swiglu ? 2 * g.N : g.N;
    const Plan pl = prompt_plan(g.M, cols, g.K / 64, swiglu);
    const int nt = g.W16 ? pl.nt : 4;      // three parts of W leave no registers for more
    PgParams p{};
    p.Xf = g.Xf;
    p.W = g.W16 ? g.W16 : g.W3;
    p.M = g.M;
    p.N = g.N;
    p.K = g.K;
    p.m_tiles = (g.M + 31) / 32;
    p.wm = pl.wm;
    p.kw = pl.kw;
    p.ks = pl.ks;
    p.m_groups = pl.m_groups;
    p.n_groups = cols / (32 * nt);
    p.per = pl.per * (64 / 16) / (g.W16 ? Stage<1, 4>::kSteps : Stage<3, 4>::kSteps);
    p.Y = g.Y;
    p.act = g.act;
    int epi = swiglu ? kPgSwiglu : g.accumulate ? kPgAccumulate : kPgStore;
    *slices = 0;
    if (pl.ks > 1) {
        if (g.partial_bytes < static_cast<size_t>(pl.ks) * g.M * cols * sizeof(float)) {
            return fail(QA_ERR_INVALID, "prompt_gemm: partial-sum buffer too small");
        }
        p.Y = g.partial;
        p.N = cols;                 // plain columns: gate rows, then up rows
        epi = kPgPartial;
        *slices = pl.ks;
    }
    return g.W16 ? launch_epi<1>(epi, p, nt, stream) : launch_epi<3>(epi, p, nt, stream);
}

int prompt_norm_launch(float * x, const float * partial, int32_t slices, const float * w, int32_t rows, int32_t dim,
                       float eps, uint16_t * Xf, hipStream_t stream) {
    if (!x || rows <= 0 || dim <= 0 || dim % 16 || dim > 8192 || (Xf && !w) || (slices > 0 && !partial)) {
        return fail(QA_ERR_INVALID, "prompt_norm: invalid arguments");
    }
    // R = 8 from 1024 rows (128 workgroups) on; below, one row per workgroup keeps more loads in flight.  us R 1 / R 8:
    // rows of 2048 156 6 / 9, 1000 14.0 / 14.1, 1200 15.6 / 13.3, 3913 40 / 21; rows of 1024 1000 9.6 / 10.9, 1200 9.6 / 9.4,
    // 1500 11.1 / 8.8
    const bool r8 = rows >= 1024 && dim <= 2048;
    const dim3 grid(static_cast<unsigned>(r8 ? (rows + 7) / 8 : rows)), block(r8 ? 512 : 256);
#define QA_NORM(R, IT) hipLaunchKernelGGL((prompt_norm_kernel<R, IT>), grid, block, 0, stream, x, partial, slices, w, rows, dim, eps, Xf)
    if (r8 && dim <= 1024) QA_NORM(8, 2);
    else if (r8) QA_NORM(8, 4);
    else if (dim <= 2048) QA_NORM(1, 1);
    else if (dim <= 4096) QA_NORM(1, 2);
    else QA_NORM(1, 4);
#undef QA_NORM
    QA_LAUNCH_CHECK("prompt_norm_kernel");
    return QA_OK;
}

int prompt_split_launch(const float * x, int32_t rows, int32_t dim, uint16_t * Xf, hipStream_t stream) {
    return launch_rows<0>(x, 0, rows, dim, nullptr, Xf, stream);
}

int prompt_pack_launch(const float * w, int32_t rows, int32_t dim, uint16_t * Wf, hipStream_t stream) {
    return launch_rows<3>(w, 0, rows, dim, nullptr, Wf, stream);
}

int prompt_swiglu_launch(const float * partial, int32_t slices, int32_t rows, int32_t dim, uint16_t * Xf,
                         hipStream_t stream) {
    return launch_rows<1>(partial, slices, rows, dim, nullptr, Xf, stream);
}

int prompt_sum_launch(const float * partial, int32_t slices, int32_t rows, int32_t dim, float * y, hipStream_t stream) {
    return launch_rows<2>(partial, slices, rows, dim, y, nullptr, stream);
}

}  // namespace qa
