// The decoder's projections for prompts and larger decode steps: fp32 rows times bf16
// weights on v_mfma_f32_16x16x32_bf16, every row value as three bf16 terms
// (bf16_terms.h), so the result is the fp32 product to within 2^-27 of |x|.
#include "proj.h"

#include <math.h>

#include <algorithm>

#include "bf16_terms.h"
#include "prefill_shared.h"

namespace sa {
namespace {

constexpr int kWaves = 8;
constexpr int kStep = 32;   // k per MFMA step

struct ProjArgs {
    const float* x;
    const uint16_t* w;
    float* out;
    int M, N, K, split;
};

// Workgroup tile: RW x CW x KW waves; a wave computes 16 MT rows by 16 CN
// columns over every KW-th part of the workgroup's k range.
template <int MT, int CN, int RW, int CW, int KW>
struct Tile {
    static_assert(RW * CW * KW == kWaves, "8 waves");
    static constexpr int ROWS = RW * 16 * MT;
    static constexpr int COLS = CW * 16 * CN;
    static constexpr int NB = MT * CN;                       // 16 x 16 blocks per wave
    static constexpr int NX = ROWS * KW * 4 / (kWaves * 64); // 8-float pieces a thread stages per stage
    static constexpr int TERM_BYTES = ROWS * kStep * 2;
    static constexpr int X_STAGE = KW * kTerms * TERM_BYTES;
    static constexpr int W_WAVE = 16 * CN * 2 * kStep * 2;   // two steps of the wave's columns
    static constexpr int STAGES_BYTES = 2 * X_STAGE + kWaves * W_WAVE;
    static constexpr int DUMP_BYTES = kWaves * NB * 1024;
    static constexpr int LDS = STAGES_BYTES > DUMP_BYTES ? STAGES_BYTES : DUMP_BYTES;
    static_assert(NX >= 1 && LDS <= 160 * 1024, "LDS");
};

// Per stage every wave takes one 32-wide k step of its k part: the rows of all
// KW parts are staged as bf16 terms (double-buffered, one barrier per stage);
// the wave's weights go through LDS it has to itself, two steps at a time, so
// that global loads cover whole 128-byte lines (an MFMA fragment loaded from
// global memory, 16 rows per 16 lanes, took 2.4 times as long per KiB).  PAIR:
// the first half of the column groups computes gate columns, the second the up
// columns beside them, and SwiGLU is applied where their sums meet.
//
// 64 x 64 per wave (32 x 64 for few rows) has the fewest LDS reads per MFMA, 16
// per 48, that leave the registers two waves per SIMD; the k parts let small
// grids keep it.  The row reads run one block ahead of their MFMAs and the
// split into terms runs between them.
//
// Bound: the serial course of a stage (weight store, first fragment reads,
// MFMAs, barrier, all waves in step) and of a workgroup's start and end; no
// unit is full.  Counters of the 4096 x 1024 launch at 512 rows, of 36,900 cycles per
// CU: MFMA 12,300, LDS 10,750 without bank conflicts, VALU 11,700.  A stage of 8
// wave steps measures 1.10 to 1.20 us against 0.64 us of MFMA.
//
// Measured (weights from HBM): 4096 x 1024 at 512 rows 17.2 us (64 x 64 tiles
// of 4 waves with weight fragments from global memory: 23.2), 1024 x 2048 12.0
// (17.8), 1024 x 3072 15.9 (17.8), gate and up with SwiGLU 27.8 (30.7 + 5.2);
// at 2048 rows 0.85 .. 1.05 PFLOP/s of bf16 products.
template <int MT, int CN, int RW, int CW, int KW, bool PAIR>
__global__ void __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
proj_kernel(ProjArgs a) {
    using T = Tile<MT, CN, RW, CW, KW>;
    constexpr int CWH = PAIR ? CW / 2 : CW;   // column groups of outputs
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int kq = wave % KW, cw = wave / KW % CW, rw = wave / KW / CW;
    const int M = a.M, N = a.N, K = a.K;
    const int m0 = blockIdx.z * T::ROWS;
    const int n0 = (blockIdx.x * CWH + cw % CWH) * 16 * CN;   // the wave's first output column
    const int nblk = (min(n0 + 16 * CN, N) - n0) / 16;        // its 16-column blocks (<= 0: none)

    // k steps of part q of this workgroup's split
    const int all = K / kStep;
    const int s_lo = all * (int)blockIdx.y / a.split, s_n = all * ((int)blockIdx.y + 1) / a.split - s_lo;
    auto q_first = [&](int q) { return s_lo + s_n * q / KW; };
    auto q_count = [&](int q) { return s_n * (q + 1) / KW - s_n * q / KW; };
    const int stages = (s_n + KW - 1) / KW;
    const int my_first = q_first(kq), my_count = q_count(kq);

    // ---- rows: thread piece i is 8 floats of row xr[i], part xq[i] ----
    const float* xbase = a.x + (size_t)m0 * K;
    int x_off[T::NX], x_first[T::NX], x_last[T::NX], x_dst[T::NX];
#pragma unroll
    for (int i = 0; i < T::NX; ++i) {
        const int q = __builtin_amdgcn_readfirstlane((i * kWaves * 64 + wave * 64) / (4 * T::ROWS));
        const int idx = i * kWaves * 64 + threadIdx.x;
        const int chunk = idx & 3, row = (idx >> 2) % T::ROWS;
        x_off[i] = min(row, M - 1 - m0) * K + 8 * chunk;
        x_first[i] = min(q_first(q), all - 1);
        x_last[i] = max(q_count(q) - 1, 0);
        x_dst[i] = q * kTerms * T::TERM_BYTES + row * 64 + ((chunk ^ ((row >> 1) & 3)) << 4);
    }
    f32x4_t xa[T::NX][2];
    auto load_x = [&](int j, int i) {
        const float* p = xbase + (size_t)(x_first[i] + min(j, x_last[i])) * kStep + x_off[i];
        xa[i][0] = *reinterpret_cast<const f32x4_t*>(p);
        xa[i][1] = *reinterpret_cast<const f32x4_t*>(p + 4);
    };
    auto store_x = [&](int buf, int i) {
        bf16x8_t t[kTerms];
        split_terms(xa[i][0], xa[i][1], t);
#pragma unroll
        for (int k = 0; k < kTerms; ++k)
            *reinterpret_cast<bf16x8_t*>(smem + buf * T::X_STAGE + x_dst[i] + k * T::TERM_BYTES) = t[k];
    };

    // ---- weights: load i takes columns 8 i .. 8 i + 7, 128 bytes (two steps) of each ----
    unsigned char* const wl = smem + 2 * T::X_STAGE + wave * T::W_WAVE;
    const int wn = min(n0, N - 16);   // a wave without columns loads the last ones and stores nothing
    const uint16_t* wbase = a.w + ((size_t)wn + (PAIR && cw >= CWH ? N : 0)) * K + (size_t)min(my_first, all - 1) * kStep;
    const int w_lane = (lane >> 3) * K + 8 * (lane & 7);
    const int w_lane1 = w_lane - ((lane & 4) ? kStep : 0);   // of a pair with one step
    u32x4_t wr[2 * CN];
    auto load_w = [&](int j) {   // steps j, j + 1
        const int at = max(min(j, (my_count - 1) & ~1), 0);
        const int off = (at + 1 < my_count ? w_lane : w_lane1) + at * kStep;
#pragma unroll
        for (int i = 0; i < 2 * CN; ++i) {
            const int blk = max(min(i >> 1, nblk - 1), 0);
            wr[i] = *reinterpret_cast<const u32x4_t*>(wbase + (size_t)(16 * blk + 8 * (i & 1)) * K + off);
        }
    };
    auto store_w = [&]() {
        unsigned char* p = wl + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
#pragma unroll
        for (int i = 0; i < 2 * CN; ++i) *reinterpret_cast<u32x4_t*>(p + i * 1024) = wr[i];
    };

    f32x4_t acc[MT][CN] = {};
    const int x_frag = kq * kTerms * T::TERM_BYTES + (rw * 16 * MT + r) * 64 + ((g ^ ((r >> 1) & 3)) << 4);

    load_w(0);
#pragma unroll
    for (int i = 0; i < T::NX; ++i) load_x(0, i);
#pragma unroll
    for (int i = 0; i < T::NX; ++i) store_x(0, i);
#pragma unroll
    for (int i = 0; i < T::NX; ++i) load_x(1, i);
    lds_barrier();
    auto stage = [&](int j, int h, bool on) {
        if (h == 0) store_w();
        const unsigned char* xs = smem + h * T::X_STAGE + x_frag;
        bf16x8_t wf[CN], xf[2][kTerms];
        auto read_x = [&](int mt) {
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
                xf[mt & 1][t] = *reinterpret_cast<const bf16x8_t*>(xs + t * T::TERM_BYTES + mt * 1024);
        };
#pragma unroll
        for (int c = 0; c < CN; ++c)
            wf[c] = *reinterpret_cast<const bf16x8_t*>(wl + (16 * c + r) * 128 + (((4 * h + g) ^ (r & 7)) << 4));
        read_x(0);
        // Kept in order: the row reads run one block ahead of the MFMAs that
        // use them, the term split of the next stage's rows between MFMAs.
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if (mt + 1 < MT) read_x(mt + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (on) {
#pragma unroll
                for (int t = 0; t < kTerms; ++t)
#pragma unroll
                    for (int c = 0; c < CN; ++c)
                        acc[mt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[c], xf[mt & 1][t], acc[mt][c], 0, 0, 0);
            }
            if (mt % (MT / T::NX) == 0) {
                const int i = mt / (MT / T::NX);
                store_x(h ^ 1, i);   // past the last stage: a buffer nobody reads
                load_x(j + 2, i);
#pragma unroll
                for (int u = 0; u < kTerms * CN; ++u) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, CN == 4 ? 4 : 8, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (h == 0) load_w(j + 2);
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // Stages in which every wave has a step carry no branch; the parts differ
    // by at most one step.
    const int full = s_n / KW;
    int j = 0;
    for (; j + 2 <= full; j += 2) {
        stage(j, 0, true);
        stage(j + 1, 1, true);
    }
    if (j < stages) stage(j, 0, j < my_count);
    if (j + 1 < stages) stage(j + 1, 1, j + 1 < my_count);

    // ---- sums of the k parts ----
    auto put = [&](int mt, int c, f32x4_t v) {
        const int row = m0 + rw * 16 * MT + 16 * mt + r;
        if (row < M && c < nblk)
            *reinterpret_cast<f32x4_t*>(a.out + ((size_t)blockIdx.y * M + row) * N + n0 + 16 * c + 4 * g) = v;
    };
    if constexpr (KW == 1 && !PAIR) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int c = 0; c < CN; ++c) put(mt, c, acc[mt][c]);
    } else {
        // Through LDS; every wave finishes SHARE-th blocks of its columns, of
        // which its own part stays in registers.
        f32x4_t(*dump)[T::NB][64] = reinterpret_cast<f32x4_t(*)[T::NB][64]>(smem);
        constexpr int SHARE = PAIR ? 2 * KW : KW, BLOCKS = T::NB / SHARE;
        static_assert(T::NB % SHARE == 0, "whole blocks per wave");
        const bool up = PAIR && cw >= CWH;
        const int part = up ? KW + kq : kq;
        const int w0 = (rw * CW + cw % CWH) * KW;   // first wave of the (gate) columns
#pragma unroll
        for (int b = 0; b < T::NB; ++b)
            if (b / BLOCKS != part) dump[wave][b][lane] = acc[b / CN][b % CN];
        lds_barrier();
        auto total = [&](int w, int b, f32x4_t own, int mine) {   // parts of waves w .. w + KW - 1, in order
            f32x4_t y = mine == 0 ? own : dump[w][b][lane];
#pragma unroll
            for (int q = 1; q < KW; ++q) y += mine == q ? own : dump[w + q][b][lane];
            return y;
        };
#pragma unroll
        for (int q = 0; q < SHARE; ++q) {
            if (q != part) continue;   // wave-uniform: the blocks' registers are known at compile time
#pragma unroll
            for (int b = q * BLOCKS; b < (q + 1) * BLOCKS; ++b) {
                const f32x4_t own = acc[b / CN][b % CN];
                if constexpr (PAIR) {
                    const f32x4_t gate = total(w0, b, own, q < KW ? q : -1);
                    const f32x4_t upv = total(w0 + CWH * KW, b, own, q < KW ? -1 : q - KW);
                    f32x4_t y;
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[e] = gate[e] * (1.0f / (1.0f + expf(-gate[e]))) * upv[e];
                    put(b / CN, b % CN, y);
                } else {
                    put(b / CN, b % CN, total(w0, b, own, q));
                }
            }
        }
    }
}

template <int MT, int CN, int RW, int CW, int KW, bool PAIR>
sa_status launch_tile(const ProjArgs& a, hipStream_t st) {
    using T = Tile<MT, CN, RW, CW, KW>;
    constexpr int cols = PAIR ? T::COLS / 2 : T::COLS;
    SA_TRY((pf::opt_in_lds<&proj_kernel<MT, CN, RW, CW, KW, PAIR>>(T::LDS)));
    const dim3 grid((a.N + cols - 1) / cols, a.split, (a.M + T::ROWS - 1) / T::ROWS);
    hipLaunchKernelGGL((proj_kernel<MT, CN, RW, CW, KW, PAIR>), grid, dim3(kWaves * 64), T::LDS, st, a);
    SA_CHECK_LAUNCH();
    return SA_OK;
}

template <bool PAIR>
sa_status launch(int tile, const ProjArgs& a, hipStream_t st) {
    switch (tile) {
        case 0: return launch_tile<4, 4, 1, 2, 4, PAIR>(a, st);
        case 1: return launch_tile<4, 4, 2, 2, 2, PAIR>(a, st);
        case 2: return launch_tile<4, 4, 2, 4, 1, PAIR>(a, st);
        default: return launch_tile<2, 4, 1, 2, 4, PAIR>(a, st);
    }
}

// The tiles of launch(): rows, columns, k parts, and measured us of a
// workgroup's start and end and of a stage.
struct TileCost { int rows, cols, kw; double fixed, stage; };
constexpr int kTiles = 4, kMaxSplit = 8;
constexpr TileCost kTileCost[kTiles] = {{64, 128, 4, 5.54, 1.18}, {128, 128, 2, 5.96, 1.20},
                                        {128, 256, 1, 6.37, 1.10}, {32, 128, 4, 4.19, 0.71}};

}  // namespace

// The tile and split of least estimated time.  The estimate is fitted to 486
// launches (the four projections of the Qwen3-0.6B shape, 17 .. 2048 rows, every
// tile and split, weights from HBM; 5 % rms): a workgroup's start and end, its
// stages (slower by up to 27 % when every CU runs one), a later round's start
// overlapped by 2 us with the end of the one before it, and the consumer's reads of
// the partial sums.  Its choice is the measured best in 67 of 68 shapes and
// within 1 % in the other.
ProjPlan plan_proj(int M, int N, int K, bool pair, int cus, int max_split) {
    ProjPlan best{N, K, pair, 0, 1};
    double best_us = 1e30;
    for (int t = 0; t < kTiles; ++t) {
        const TileCost& c = kTileCost[t];
        const int cols = pair ? c.cols / 2 : c.cols;
        const long long tiles = (long long)((N + cols - 1) / cols) * ((M + c.rows - 1) / c.rows);
        for (int s = 1; s <= kMaxSplit && s <= max_split; s *= 2) {
            if (s > 1 && (pair || K / kStep < kWaves * s)) break;
            const double stages = (K / kStep + s * c.kw - 1) / (s * c.kw);
            const double rounds = (double)((tiles * s + cus - 1) / cus);
            const double fill = std::min(1.0, (double)(tiles * s) / cus);
            double us = c.fixed + (rounds - 1) * (c.fixed - 2.0) + rounds * stages * c.stage * (1.0 + 0.27 * fill) +
                        0.63 * fill;
            if (s > 1) us += s * (4.0 / 3.0e6) * M * N;
            if (us < best_us) {
                best_us = us;
                best.tile = t;
                best.split = s;
            }
        }
    }
    return best;
}

sa_status project(const float* X, int M, const uint16_t* W, const ProjPlan& p, float* out, hipStream_t st) {
    const ProjArgs a{X, W, out, M, p.N, p.K, p.split};
    return p.pair ? launch<true>(p.tile, a, st) : launch<false>(p.tile, a, st);
}

}  // namespace sa
