// Dense fp32 operators of the Qwen3 decoder layer on gfx950: the linear
// projection (fp32 MFMA), RMSNorm, SwiGLU and the scaled add of residuals.
//
// They serve the reference's host-tensor layer API (tensor_cpp/src/ops.cpp
// linear :315-369, rms_norm :375-418, add :194-207, swiglu :493-509;
// tensor_cpp/src/qwen3_ops.cpp qwen3_mlp :265-296) with fp32 weights, so the
// layer keeps fp32 arithmetic end to end.  Every operator reads and writes
// HBM once per element; the linear is the only one with data reuse.
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "sa_internal.h"

namespace sa {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// y[M][N] = x[M][K] . w[N][K]^T (+ bias[N]), fp32 in and out.
//
// Workgroup (bx, by) owns the 64 x 64 output tile at rows 64 by, columns
// 64 bx; wave w computes its 32 x 32 quadrant (w >> 1, w & 1) as 2 x 2 tiles
// of v_mfma_f32_16x16x4_f32.  Per 32-wide k step the workgroup stages the
// 64 x 32 blocks of x and w through LDS, k-major, so that a fragment read
// (lane l: row l & 15 at k = l >> 4) is 16 consecutive floats per k.  Rows,
// columns and k past the matrix read as zero; stores are bounds-checked.
//
// VEC: K % 4 == 0 and 16-byte aligned x and w, so blocks load as float4; such
// calls take linear_f32_direct_kernel where launch_vec expects it to be faster.
// Here every step's 32 products per output are added up by themselves and then
// added to the sum, so no chain is longer than that kernel's: 1.5e-7 of the
// result in the 2-norm at K = 1024 (2.9e-7 there, 5.7e-7 in one chain over K).
// Eight workgroups share a CU and hide each other's staging; with the registers
// for five, 1024 rows times 6144 x 1024 take 174 us instead of 147.
// ---------------------------------------------------------------------------
constexpr int kLinTile = 64;
constexpr int kLinK = 32;
constexpr int kLinStride = kLinTile + 4;   // floats per LDS k row

template <bool VEC>
__device__ __forceinline__ void stage_block(const float* __restrict__ src, int rows, int K, int r0, int k0,
                                            float (*dst)[kLinStride]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int slot = threadIdx.x + i * 256;   // 512 slots of 4 floats: 64 rows x 8
        const int r = slot >> 3, kq = (slot & 7) * 4;
        const int row = r0 + r, k = k0 + kq;
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
        if (row < rows) {
            const float* p = src + (size_t)row * K + k;
            if constexpr (VEC) {
                if (k < K) v = *reinterpret_cast<const f32x4_t*>(p);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (k + j < K) v[j] = p[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[kq + j][r] = v[j];
    }
}

template <bool VEC>
__global__ void __launch_bounds__(256, VEC ? 8 : 1)
linear_f32_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                  float* __restrict__ y, int M, int N, int K) {
    __shared__ float xs[kLinK][kLinStride];
    __shared__ float ws[kLinK][kLinStride];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m0 = blockIdx.y * kLinTile, n0 = blockIdx.x * kLinTile;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int c = lane & 15, kl = lane >> 4;
    f32x4_t sum[2][2] = {}, acc[2][2] = {};
    for (int k0 = 0; k0 < K; k0 += kLinK) {
        stage_block<VEC>(x, M, K, m0, k0, xs);
        stage_block<VEC>(w, N, K, n0, k0, ws);
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < kLinK; ks += 4) {
            const int kk = ks + kl;
            const float a0 = xs[kk][wm + c], a1 = xs[kk][wm + 16 + c];
            const float b0 = ws[kk][wn + c], b1 = ws[kk][wn + 16 + c];
            acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b1, acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, acc[1][1], 0, 0, 0);
        }
        if constexpr (VEC) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    sum[i][j] += acc[i][j];
                    acc[i][j] = f32x4_t{};
                }
        }
        __syncthreads();
    }
    // Output fragment: lane l holds column l & 15 of rows 4 (l >> 4) + r.
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int col = n0 + wn + 16 * j + c;
        if (col >= N) continue;
        const float b = bias ? bias[col] : 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wm + 16 * i + 4 * kl + r;
                if (row < M) y[(size_t)row * N + col] = (VEC ? sum : acc)[i][j][r] + b;
            }
    }
}

// ---------------------------------------------------------------------------
// The same product for K % 4 == 0 and 16-byte aligned x and w, without LDS in
// the k loop.  A workgroup owns a TM x TN output tile; its W waves each take a
// contiguous range of the 32-wide k steps for the whole tile and add up in
// LDS at the end, in wave order.  A lane loads two 16-byte pieces of a row per
// step (lane (r, g): k0 + 4 g .. + 3 and k0 + 16 + 4 g .. + 3 of row r, a whole
// 128-byte line per row between them, issued together) and uses element j in
// MFMA j of the piece: any assignment of the k values to the MFMAs' k slots
// gives the same sum as long as both operands share it.  kLinRing steps of
// loads are in flight per wave, all issued unconditionally (steps past the
// last re-read it), so no wait drains them.  Rows and columns past the matrix
// re-read the last one; their outputs are not stored.  k past K (a last step
// that is cut) enters as zero from both operands.
//
// Bound: HBM / L2 on w for few rows, fp32 MFMA for many.
// ---------------------------------------------------------------------------
constexpr int kLinRing = 2;
// Cost rule of launch_vec: bytes per cycle a CU loads with 16 rows per
// 16-lane group (measured: one such 1 KiB wave load per 64 cycles), and cycles
// a tile costs besides (LDS sum, stores).
constexpr double kLinLoadBytes = 15, kLinTileCycles = 1000;

template <int TM, int TN, int W>
__global__ void __launch_bounds__(W * 64)
linear_f32_direct_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                         float* __restrict__ y, int M, int N, int K, int vec_out) {
    constexpr int MB = TM / 16, NB = TN / 16, STRIDE = TN + 4;
    __shared__ __align__(16) float sh[W][TM][STRIDE];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * TN, m0 = blockIdx.y * TM;
    const int steps = (K - 1) / 32 + 1;
    const int s0 = (int)((long long)steps * wave / W), s1 = (int)((long long)steps * (wave + 1) / W);

    f32x4_t acc[MB][NB] = {};
    if (s0 < s1) {   // wave-uniform
        const float* xp[MB];
        const float* wp[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i) xp[i] = x + (size_t)min(m0 + 16 * i + r, M - 1) * K;
#pragma unroll
        for (int i = 0; i < NB; ++i) wp[i] = w + (size_t)min(n0 + 16 * i + r, N - 1) * K;
        f32x4_t xr[kLinRing][MB][2], wr[kLinRing][NB][2];
        auto load = [&](int step, int slot) {
            const int k0 = 32 * min(step, s1 - 1) + 4 * g;
            const int ka = min(k0, K - 4), kb = min(k0 + 16, K - 4);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                wr[slot][i][0] = *reinterpret_cast<const f32x4_t*>(wp[i] + ka);
                wr[slot][i][1] = *reinterpret_cast<const f32x4_t*>(wp[i] + kb);
            }
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                xr[slot][i][0] = *reinterpret_cast<const f32x4_t*>(xp[i] + ka);
                xr[slot][i][1] = *reinterpret_cast<const f32x4_t*>(xp[i] + kb);
            }
        };
        auto compute = [&](int slot) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int a = 0; a < MB; ++a)
#pragma unroll
                        for (int b = 0; b < NB; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[slot][b][h][j], xr[slot][a][h][j],
                                                                             acc[a][b], 0, 0, 0);
        };
        // A step that runs past K: the lanes whose 4 values lie there hold a
        // re-read of the row's end instead.
        auto cut = [&](int step, int slot) {
            if (32 * step + 32 > K) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool on = 32 * step + 16 * h + 4 * g < K;
#pragma unroll
                    for (int i = 0; i < NB; ++i) wr[slot][i][h] = on ? wr[slot][i][h] : f32x4_t{};
#pragma unroll
                    for (int i = 0; i < MB; ++i) xr[slot][i][h] = on ? xr[slot][i][h] : f32x4_t{};
                }
            }
        };
#pragma unroll
        for (int u = 0; u < kLinRing; ++u) load(s0 + u, u);
        int s = s0;
        // Whole groups that end before the wave's last step, so no step of
        // theirs can run past K.
        for (; s + kLinRing < s1; s += kLinRing) {
#pragma unroll
            for (int u = 0; u < kLinRing; ++u) {
                compute(u);
                load(s + kLinRing + u, u);
            }
        }
#pragma unroll
        for (int u = 0; u < kLinRing; ++u) {
            if (s + u < s1) {
                cut(s + u, u);
                compute(u);
            }
        }
    }
    // acc[a][b]: element i is row 16 a + r, column 16 b + 4 g + i.
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) *reinterpret_cast<f32x4_t*>(&sh[wave][16 * a + r][16 * b + 4 * g]) = acc[a][b];
    __syncthreads();
    for (int e = threadIdx.x; e < TM * TN / 4; e += W * 64) {
        const int m = e / (TN / 4), n = e % (TN / 4) * 4;
        if (m0 + m >= M || n0 + n >= N) continue;
        f32x4_t v = *reinterpret_cast<const f32x4_t*>(&sh[0][m][n]);
#pragma unroll
        for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4_t*>(&sh[k][m][n]);
        float* out = y + (size_t)(m0 + m) * N + n0 + n;
        if (vec_out) {   // N % 4 == 0: the four columns are all inside
            if (bias) v += f32x4_t{bias[n0 + n], bias[n0 + n + 1], bias[n0 + n + 2], bias[n0 + n + 3]};
            *reinterpret_cast<f32x4_t*>(out) = v;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n0 + n + i < N) out[i] = v[i] + (bias ? bias[n0 + n + i] : 0.f);
        }
    }
}

// ---------------------------------------------------------------------------
// Row RMSNorm, one workgroup per row: y = (x / sqrt(sum(x^2) / n + eps)) * w.
// y may alias x (each element is read before it is written, by one thread).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
rms_norm_f32_kernel(const float* x, int n, const float* __restrict__ w, float eps, float* y) {
    __shared__ float red[4];
    const float* xr = x + (size_t)blockIdx.x * n;
    float* yr = y + (size_t)blockIdx.x * n;
    float ss = 0.f;
    for (int i = threadIdx.x; i < n; i += 256) ss = fmaf(xr[i], xr[i], ss);
    ss = group_reduce<OpSum, 1, kWave>(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float total = (red[0] + red[1]) + (red[2] + red[3]);
    const float rms = sqrtf(total / (float)n + eps);
    for (int i = threadIdx.x; i < n; i += 256) {
        const float v = xr[i] / rms;
        yr[i] = w ? v * w[i] : v;
    }
}

// out = up * (gate * sigmoid(gate)), sigmoid(g) = 1 / (1 + exp(-g)).
__global__ void __launch_bounds__(256)
swiglu_f32_kernel(const float* gate, const float* up, size_t n, float* out) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float g = gate[i];
        const float silu = g * (1.0f / (1.0f + expf(-g)));
        out[i] = up[i] * silu;
    }
}

// out = a x + b y (y == NULL: out = a x).
__global__ void __launch_bounds__(256)
axpby_f32_kernel(const float* x, float a, const float* y, float b, size_t n, float* out) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        out[i] = y ? fmaf(a, x[i], b * y[i]) : a * x[i];
}

template <int TM, int TN, int W>
void launch_tile(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, hipStream_t st) {
    const dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
    hipLaunchKernelGGL((linear_f32_direct_kernel<TM, TN, W>), grid, dim3(W * 64), 0, st, x, w, bias, y, M, N, K,
                       N % 4 == 0 && aligned16(y) ? 1 : 0);
}

// K % 4 == 0, 16-byte aligned x and w.  Of the direct kernel's tiles, the one
// with the smallest estimated time per CU: tiles per CU times the larger of a
// tile's MFMA cycles (its waves share the CU's four SIMDs, 32 cycles per
// 16x16x4) and its load cycles, plus a tile's fixed cycles.  That tile or
// linear_f32_kernel, whichever has the smaller estimated microseconds (direct_us,
// lds_us: fitted to 1684 sizes, M 1 .. 4096, N 16 .. 151936, K 32 .. 8192).  A
// direct tile is one workgroup's serial course; the LDS kernel's workgroups
// share a CU, so it is ahead where a CU has many tiles of a short K.
//
// Measured us, tiles 16x16 / 16x32 / 32x32 / 32x64 / 64x64 against the LDS
// kernel.  N, K = 3072, 1024 (weights rotated over 75 MB): M = 1 4.8 / 6.6 / 8.6
// / 13.7 / 22.5 against 48; M = 128 24 / 18.5 / 18.7 / 15.7 / 27 against 53;
// M = 1024 170 / 130 / 103 / 93 / 81 against 81; M = 4096 64x64 304 against 250.
// M = 1024, N = 4096: K = 32 19 / 22 / 17 / 14 / 20 against 8.8, K = 256 115 / 90 /
// 59 / 35 / 36 against 28, K = 2048 64x64 171 against 185.  N, K = 151936, 1024:
// M = 64 64x64 279 against 252, M = 512 2068 against 1638.
struct DirectTile { int rows, cols, waves; double us, us_k; };   // us of a tile: us + us_k K
constexpr DirectTile kDirectTiles[] = {{16, 16, 8, 0.24, 0.0034}, {16, 32, 8, 0.6, 0.00514}, {32, 32, 8, 0.85, 0.00733},
                                       {32, 64, 4, 1.1, 0.0105}, {64, 64, 4, 3.6, 0.0168}};

void launch_vec(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, hipStream_t st) {
    const long long cus = device_cu_count();
    int best = 4;
    double best_t = INFINITY, direct_us = 0;
    for (int i = 0; i < 5; ++i) {
        const DirectTile& d = kDirectTiles[i];
        const long long rows = ((long long)M + d.rows - 1) / d.rows, cols = ((long long)N + d.cols - 1) / d.cols;
        if (i < 4 && (rows > 65535 || cols * d.waves * 64 > 0xffffffffLL)) continue;   // grid limits
        const long long per_cu = (rows * cols + cus - 1) / cus;
        const double mfma = (double)(d.rows * d.cols) / 256 * K / 16 * 32;
        const double load = (double)(d.rows + d.cols) * K * 4 / kLinLoadBytes;
        const double both = d.waves == 4 ? 0.5 * std::min(mfma, load) : 0.0;   // one wave per SIMD: partly serial
        const double t = per_cu * (std::max(mfma, load) + both + kLinTileCycles);
        if (t < best_t) {
            best = i;
            best_t = t;
            double us = d.us + d.us_k * K;
            if (i == 4) us += std::min(4.4, std::max(0.0036 * K, 0.009 * (K - 256)));   // beyond the loads in flight
            if (i >= 3 && (double)N * K * 4 > 202e6) us *= 1.08;   // w not kept in the 256 MB cache
            direct_us = per_cu * us;
        }
    }
    const dim3 grid((N + kLinTile - 1) / kLinTile, (M + kLinTile - 1) / kLinTile);
    const double tiles = (double)grid.x * grid.y / cus;   // of the LDS kernel per CU
    const double lds_us = 1.0 + 0.5 * tiles +
                          K * std::max({0.0645, 0.044 + 0.012 * tiles, 0.0295 + 0.0155 * tiles, 0.0197 * tiles});
    if (lds_us < direct_us) best = 5;
    switch (best) {
        case 0: return launch_tile<16, 16, 8>(x, w, bias, y, M, N, K, st);
        case 1: return launch_tile<16, 32, 8>(x, w, bias, y, M, N, K, st);
        case 2: return launch_tile<32, 32, 8>(x, w, bias, y, M, N, K, st);
        case 3: return launch_tile<32, 64, 4>(x, w, bias, y, M, N, K, st);
        case 4: return launch_tile<64, 64, 4>(x, w, bias, y, M, N, K, st);
        default:
            hipLaunchKernelGGL(linear_f32_kernel<true>, grid, dim3(256), 0, st, x, w, bias, y, M, N, K);
    }
}

// Enough workgroups to cover n once, at most 8 per CU (grid-stride beyond).
dim3 elementwise_grid(size_t n) {
    const size_t want = (n + 255) / 256;
    const size_t cap = (size_t)device_cu_count() * 8;
    return dim3((unsigned)(want < cap ? (want ? want : 1) : cap));
}

}  // namespace
}  // namespace sa

using namespace sa;

extern "C" sa_status sa_linear_f32(const float* x, int M, int K, const float* w, int N, const float* bias,
                                   float* y, sa_stream_t stream) {
    clear_error();
    if (!y || (K > 0 && (!x || !w))) return fail(SA_EINVAL, "null pointer");
    if (M < 0 || N < 0 || K < 0) return fail(SA_EINVAL, "M, N and K must be >= 0");
    if (M == 0 || N == 0) return SA_OK;
    const dim3 grid((N + kLinTile - 1) / kLinTile, (M + kLinTile - 1) / kLinTile);
    if (grid.y > 65535u) return fail(SA_EINVAL, "M too large for one launch");
    hipStream_t st = as_stream(stream);
    if (K > 0 && K <= (1 << 30) && K % 4 == 0 && aligned16(x) && aligned16(w))
        launch_vec(x, w, bias, y, M, N, K, st);
    else
        hipLaunchKernelGGL(linear_f32_kernel<false>, grid, dim3(256), 0, st, x, w, bias, y, M, N, K);
    SA_CHECK_LAUNCH();
    return SA_OK;
}

extern "C" sa_status sa_rms_norm_f32(const float* x, int rows, int n, const float* w, float eps, float* y,
                                     sa_stream_t stream) {
    clear_error();
    if (!x || !y) return fail(SA_EINVAL, "null pointer");
    if (rows < 0 || n <= 0) return fail(SA_EINVAL, "rows must be >= 0 and n > 0");
    if (rows == 0) return SA_OK;
    hipLaunchKernelGGL(rms_norm_f32_kernel, dim3(rows), dim3(256), 0, as_stream(stream), x, n, w, eps, y);
    SA_CHECK_LAUNCH();
    return SA_OK;
}

extern "C" sa_status sa_swiglu_f32(const float* gate, const float* up, size_t n, float* out,
                                   sa_stream_t stream) {
    clear_error();
    if (!gate || !up || !out) return fail(SA_EINVAL, "null pointer");
    if (n == 0) return SA_OK;
    hipLaunchKernelGGL(swiglu_f32_kernel, elementwise_grid(n), dim3(256), 0, as_stream(stream), gate, up, n,
                       out);
    SA_CHECK_LAUNCH();
    return SA_OK;
}

extern "C" sa_status sa_axpby_f32(const float* x, float a, const float* y, float b, size_t n, float* out,
                                  sa_stream_t stream) {
    clear_error();
    if (!x || !out) return fail(SA_EINVAL, "null pointer");
    if (n == 0) return SA_OK;
    hipLaunchKernelGGL(axpby_f32_kernel, elementwise_grid(n), dim3(256), 0, as_stream(stream), x, a, y, b, n,
                       out);
    SA_CHECK_LAUNCH();
    return SA_OK;
}
