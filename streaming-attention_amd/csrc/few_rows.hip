// The decoder's projections for a decode step of at most 16 token rows.
//
// Bound: HBM on the weights (8 MB per projection at the Qwen3-0.6B shape, 1.3
// us at the read rate), but a launch of a few microseconds is mostly latency:
// its start, one memory round trip for what the previous launch wrote, one
// for the weights, and the reduction.  So the design saves launches and round
// trips: the residual sum and RMSNorm run in the prologue of the projection
// that consumes them, SwiGLU in the epilogue of gate_up, and every wave
// issues all its weight loads before it waits for its input.  A decode layer
// is qkv, attention, o, gate_up, down: no separate norm or activation launch.
//
// Reference: the same lines as model.hip (tensor_cpp/src/qwen3_ops.cpp:265-296,
// :620-934; ops.cpp:278-417).
#include "few_rows.h"

#include <math.h>

#include <type_traits>

#include "bf16_terms.h"
#include "prefill_shared.h"

namespace sa {
namespace {

constexpr int kStep = 32;               // k per MFMA step
constexpr int kChunk = 4;               // steps a wave holds in registers at a time
constexpr int kXStride = kChunk * kStep + 4;   // floats per staged row: conflict-free 16-byte reads

enum { kPlain = 0, kNorm = 1 };
enum { kOut = 0, kSwiglu = 1 };

struct FewArgs {
    FewInput in;
    const uint16_t* w;   // [N or 2 N][K]
    float* out;          // [split][M][N]
    int M, K, N;
    DecodeParts parts;   // NS > 0: partials of heads of 1 << d_log2 columns
    int d_log2;
};

// Workgroup (bx, by) owns 16 output columns (kSwiglu: 16 gate and the 16 up
// columns beside them) for all rows and K split by; its W waves split that k
// range again and add up in LDS.  v_mfma_f32_16x16x32_bf16 with the weights as
// A (16 columns) and the rows as B, in three bf16 terms (bf16_terms.h).
//
// Weights and rows reach the MFMA layout through LDS the wave has to itself
// (no barrier): a load instruction covers 256 consecutive bytes of 4 weight
// rows, or 512 of 2 input rows.  Loaded as MFMA fragments, 16 rows per 16
// lanes, a 1 KiB load takes 64 cycles of address processing instead of 16.
// The rows go first; their fragments are in registers when the weights, whose
// loads were issued before, take their place.
//
// kNorm: the norm's division by the row's rms is applied to the sums instead of
// the rows, so the waves exchange sums of squares together with the outputs,
// and no barrier precedes the MFMAs.
//
// NS > 0: the rows are attention outputs left as up to NS split-KV partials,
// merged here; their (m, l) and O are all loaded before the first use, in the
// round trip that would load the merged rows.  The merge launch this saves
// took 4.0 us of a layer; these loads add 0.5 (3 partials) to 1.6 (5; 2.3
// in the 8-partial form) to the projection's 4.4.
template <int W, int RP, int PRO, int EPI, int NS = 0>
__global__ void __launch_bounds__(W * 64)
few_rows_kernel(FewArgs a) {
    constexpr int NC = EPI == kSwiglu ? 2 : 1;
    constexpr int kWaveBytes = 2 * RP * kXStride * 4 > NC * 4096 ? 2 * RP * kXStride * 4 : NC * 4096;
    __shared__ __align__(16) unsigned char stage[W][kWaveBytes];
    __shared__ __align__(16) float so[W][NC][kFewRows][20];
    __shared__ float ss_sh[W][kFewRows];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int M = a.M, K = a.K;
    const int n0 = blockIdx.x * 16;
    const int steps = K / kStep;
    const int part = blockIdx.y * W + wave, parts = gridDim.y * W;
    const int s_begin = steps * part / parts, s_end = steps * (part + 1) / parts;
    const bool write_x = PRO == kNorm && a.in.x_out && blockIdx.x == 0 && blockIdx.y == 0;
    float(*sx)[kXStride] = reinterpret_cast<float(*)[kXStride]>(stage[wave]);
    // Weight rows of 16 16-byte chunks; chunk c of row i sits at place c ^ i, so
    // that writes (one row per 16 lanes) and fragment reads (16 rows, one
    // chunk) both cover all banks.
    u32x4_t(*sw)[16][16] = reinterpret_cast<u32x4_t(*)[16][16]>(stage[wave]);

    const int xrow = r & (2 * RP - 1);   // columns of the MFMA past the staged rows repeat them
    f32x4_t acc[NC] = {};
    float ss = 0.f;
    for (int s0 = s_begin; s0 < s_end; s0 += kChunk) {
        const int ns = min(kChunk, s_end - s0), last = s_end - 1;
        // The chunk's weights: lane l takes 16 bytes of row 4 i + l / 16 (lanes
        // past a short chunk repeat its last 16).
        u32x4_t wr[NC][4];
        {
            const uint16_t* p = a.w + (size_t)(n0 + g) * K + (size_t)s0 * kStep + 8 * min(r, 4 * ns - 1);
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    wr[c][i] = *reinterpret_cast<const u32x4_t*>(p + ((size_t)c * a.N + 4 * i) * K);
        }
        f32x4_t nw[kChunk][2];
        if constexpr (PRO == kNorm) {
#pragma unroll
            for (int j = 0; j < kChunk; ++j) {
                const float* p = a.in.norm_w + min(s0 + j, last) * kStep + 8 * g;
                nw[j][0] = *reinterpret_cast<const f32x4_t*>(p);
                nw[j][1] = *reinterpret_cast<const f32x4_t*>(p + 4);
            }
        }
        // Rows 2 i and 2 i + 1: lane l loads floats 4 (l & 31) .. + 3 of row
        // 2 i + l / 32; all loads are issued before the first use.
        const int half = lane >> 5, kk = 4 * (lane & 31);
        const bool on = kk < ns * kStep;
        const size_t k = (size_t)s0 * kStep + (on ? kk : 0);
        f32x4_t v[RP];
        size_t at[RP];
#pragma unroll
        for (int i = 0; i < RP; ++i) at[i] = (size_t)min(2 * i + half, M - 1) * K + k;
        if constexpr (NS > 0) {
            const int D = 1 << a.d_log2, head = (int)k >> a.d_log2, d = (int)k & (D - 1);
#pragma unroll
            for (int i = 0; i < RP; ++i) {
                const int m = min(2 * i + half, M - 1), n = a.parts.n_act[m];
                const int p0 = (m * (K >> a.d_log2) + head) * a.parts.n_split;
                // One partial or none: the row itself, with weight 1.
                const float* o = n > 1 ? a.parts.o + ((size_t)p0 << a.d_log2) + d : a.in.x + at[i];
                const float2* ml = reinterpret_cast<const float2*>(a.parts.ml) + p0;
                f32x4_t y[NS];
                float2 w[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int c = s < n ? s : 0;
                    w[s] = ml[c];
                    y[s] = *reinterpret_cast<const f32x4_t*>(o + (c << a.d_log2));
                }
                float mx = w[0].x;
#pragma unroll
                for (int s = 1; s < NS; ++s) mx = fmaxf(mx, w[s].x);
                f32x4_t sum = {};
                float l = 0.f;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const float e = s < n ? __builtin_amdgcn_exp2f((w[s].x - mx) * 1.4426950408889634f) : 0.f;
                    l = fmaf(e, w[s].y, l);
#pragma unroll
                    for (int j = 0; j < 4; ++j) sum[j] = fmaf(e, y[s][j], sum[j]);
                }
                v[i] = n > 1 ? sum * (1.0f / l) : y[0];
            }
        } else {
#pragma unroll
            for (int i = 0; i < RP; ++i) v[i] = *reinterpret_cast<const f32x4_t*>(a.in.x + at[i]);
        }
        if constexpr (PRO == kNorm) {
            if (a.in.n_y) {
                f32x4_t y[RP][kFewSplit];
#pragma unroll
                for (int i = 0; i < RP; ++i)
#pragma unroll
                    for (int s = 0; s < kFewSplit; ++s)
                        y[i][s] = *reinterpret_cast<const f32x4_t*>(a.in.y + (size_t)s * M * K + at[i]);
#pragma unroll
                for (int i = 0; i < RP; ++i)
#pragma unroll
                    for (int s = 0; s < kFewSplit; ++s) v[i] += y[i][s];
            }
            if (write_x) {
#pragma unroll
                for (int i = 0; i < RP; ++i)
                    if (on && 2 * i + half < M) *reinterpret_cast<f32x4_t*>(a.in.x_out + at[i]) = v[i];
            }
        }
        // The wave's own LDS accesses complete in order: only the compiler is
        // kept from moving them across the changes of the stage's contents.
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < RP; ++i)
            if (on) *reinterpret_cast<f32x4_t*>(&sx[2 * i + half][kk]) = v[i];
        asm volatile("" ::: "memory");
        bf16x8_t t[kChunk][kTerms];
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
            f32x4_t xa = *reinterpret_cast<const f32x4_t*>(&sx[xrow][kStep * j + 8 * g]);
            f32x4_t xb = *reinterpret_cast<const f32x4_t*>(&sx[xrow][kStep * j + 8 * g + 4]);
            if constexpr (PRO == kNorm) {
                if (j < ns) {   // wave-uniform
#pragma unroll
                    for (int e = 0; e < 4; ++e) ss = fmaf(xa[e], xa[e], fmaf(xb[e], xb[e], ss));
                }
                xa *= nw[j][0];
                xb *= nw[j][1];
            }
            split_terms(xa, xb, t[j]);
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) sw[c][4 * i + g][r ^ (4 * i + g)] = wr[c][i];
        asm volatile("" ::: "memory");
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
            if (j < ns) {   // wave-uniform
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const bf16x8_t wf = __builtin_bit_cast(bf16x8_t, sw[c][r][(4 * j + g) ^ r]);
#pragma unroll
                    for (int i = 0; i < kTerms; ++i)
                        acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, t[j][i], acc[c], 0, 0, 0);
                }
            }
        }
        asm volatile("" ::: "memory");
    }
    // Element e of acc: row r, column 4 g + e.
#pragma unroll
    for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4_t*>(&so[wave][c][r][4 * g]) = acc[c];
    if constexpr (PRO == kNorm) {
        ss += swz_xor16(ss);
        ss += xor32(ss);
        if (g == 0) ss_sh[wave][r] = ss;
    }
    __syncthreads();
    const int m = threadIdx.x >> 4, n = threadIdx.x & 15;
    if (m >= M) return;   // threads past 16 rows too
    float y[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        y[c] = so[0][c][m][n];
#pragma unroll
        for (int w = 1; w < W; ++w) y[c] += so[w][c][m][n];
    }
    if constexpr (PRO == kNorm) {
        float t = ss_sh[0][m];
#pragma unroll
        for (int w = 1; w < W; ++w) t += ss_sh[w][m];
        const float rms = sqrtf(t / (float)K + a.in.eps);
#pragma unroll
        for (int c = 0; c < NC; ++c) y[c] /= rms;
    }
    float* out = a.out + ((size_t)blockIdx.y * M + m) * a.N + n0 + n;
    if constexpr (EPI == kSwiglu) *out = y[0] * (1.0f / (1.0f + expf(-y[0]))) * y[1];
    else *out = y[0];
}

// ---------------------------------------------------------------------------
// lm_head: a persistent grid; every workgroup keeps all rows in LDS as bf16
// terms, and each of its waves streams whole 16-column weight tiles with
// kHeadRing steps in flight across tile boundaries: no barrier after the
// prologue.  Consecutive steps of a row share its 128-byte lines and are
// loaded together.  The greedy maximum is kept per lane on the way.
// ---------------------------------------------------------------------------
constexpr int kHeadWaves = 8;
constexpr int kHeadRing = 8;            // steps in flight per wave
constexpr int kHeadLds = 150 * 1024;    // bytes of staged rows
constexpr int head_row_bytes(int K) { return 2 * (K + 8); }   // conflict-free 16-byte reads

struct HeadArgs {
    FewInput in;
    const uint16_t* w;
    float* logits;
    float* am_val;
    int32_t* am_idx;
    int M, K, N;
};

__global__ void __launch_bounds__(kHeadWaves * 64)
few_head_kernel(HeadArgs a) {
    extern __shared__ __align__(16) unsigned char terms[];   // [kTerms][kFewRows][K + 8] bf16
    __shared__ float sv[kHeadWaves][kFewRows];
    __shared__ int si[kHeadWaves][kFewRows];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int M = a.M, K = a.K;
    const int tiles = a.N / 16, groups = K / (kStep * kHeadRing);
    const int t0 = blockIdx.x * kHeadWaves + wave, t_step = gridDim.x * kHeadWaves;
    const int row_bytes = head_row_bytes(K), term_bytes = kFewRows * row_bytes;

    bf16x8_t ring[kHeadRing];
    auto load = [&](int tile, int group) {
        const uint16_t* p = a.w + (size_t)(min(tile, tiles - 1) * 16 + r) * K + (size_t)group * kHeadRing * kStep + 8 * g;
#pragma unroll
        for (int u = 0; u < kHeadRing; ++u)
            ring[u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(p + u * kStep));
    };
    load(t0, 0);
    // Rows wave, wave + kHeadWaves, ...: residual sum, RMSNorm, terms.
    for (int m = wave; m < M; m += kHeadWaves) {
        f32x4_t v[6];   // K <= 1536: 6 pieces of 256
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int k = 256 * i + 4 * lane;
            if (256 * i < K) {
                v[i] = *reinterpret_cast<const f32x4_t*>(a.in.x + (size_t)m * K + k);
                if (a.in.norm_w)
                    for (int s = 0; s < a.in.n_y; ++s)
                        v[i] += *reinterpret_cast<const f32x4_t*>(a.in.y + ((size_t)s * M + m) * K + k);
#pragma unroll
                for (int e = 0; e < 4; ++e) ss = fmaf(v[i][e], v[i][e], ss);
            }
        }
        float rms = 1.f;
        if (a.in.norm_w) rms = sqrtf(group_reduce<OpSum, 1, 64>(ss) / (float)K + a.in.eps);
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int k = 256 * i + 4 * lane;
            if (256 * i < K) {
                if (a.in.norm_w) v[i] = v[i] / rms * *reinterpret_cast<const f32x4_t*>(a.in.norm_w + k);
                bf16x8_t t[kTerms];
                split_terms(v[i], f32x4_t{}, t);
#pragma unroll
                for (int j = 0; j < kTerms; ++j) {
                    const u32x4_t b = __builtin_bit_cast(u32x4_t, t[j]);
                    *reinterpret_cast<uint2*>(terms + j * term_bytes + m * row_bytes + 2 * k) = make_uint2(b[0], b[1]);
                }
            }
        }
    }
    __syncthreads();
    float best = -INFINITY;
    int best_n = 0x7fffffff;
    const unsigned char* xr = terms + r * row_bytes + 16 * g;
    for (int tile = t0; tile < tiles; tile += t_step) {
        f32x4_t acc[kTerms] = {};   // one chain per term
        for (int group = 0; group < groups; ++group) {
            const bool wrap = group + 1 == groups;
#pragma unroll
            for (int u = 0; u < kHeadRing; u += 2) {
                const bf16x8_t wf[2] = {ring[u], ring[u + 1]};
                // the same two slots of the next group, both halves of the lines together
                const uint16_t* p = a.w + (size_t)(min(wrap ? tile + t_step : tile, tiles - 1) * 16 + r) * K +
                                    (size_t)((wrap ? 0 : group + 1) * kHeadRing + u) * kStep + 8 * g;
                ring[u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(p));
                ring[u + 1] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(p + kStep));
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < kTerms; ++i) {
                        const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(
                            xr + i * term_bytes + 2 * (group * kHeadRing + u + h) * kStep);
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h], x, acc[i], 0, 0, 0);
                    }
            }
        }
        const f32x4_t y = acc[0] + (acc[1] + acc[2]);
        if (r < M) {
            const int n = tile * 16 + 4 * g;
            *reinterpret_cast<f32x4_t*>(a.logits + (size_t)r * a.N + n) = y;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (better(y[e], n + e, best, best_n)) { best = y[e]; best_n = n + e; }
        }
    }
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
        const float ov = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(best_n, off, 64);
        if (better(ov, oi, best, best_n)) { best = ov; best_n = oi; }
    }
    if (g == 0) { sv[wave][r] = best; si[wave][r] = best_n; }
    __syncthreads();
    const int m = threadIdx.x;
    if (m >= M) return;
    best = sv[0][m];
    best_n = si[0][m];
    for (int w = 1; w < kHeadWaves; ++w)
        if (better(sv[w][m], si[w][m], best, best_n)) { best = sv[w][m]; best_n = si[w][m]; }
    a.am_val[(size_t)m * gridDim.x + blockIdx.x] = best;
    a.am_idx[(size_t)m * gridDim.x + blockIdx.x] = best_n;
}

// One wave per row over the workgroups' maxima.
__global__ void __launch_bounds__(64)
few_argmax_kernel(const float* pv, const int32_t* pi, int nb, int32_t* out) {
    const int m = blockIdx.x;
    float v = -INFINITY;
    int idx = 0x7fffffff;
    for (int b = threadIdx.x; b < nb; b += 64) {
        const float ov = pv[(size_t)m * nb + b];
        const int oi = pi[(size_t)m * nb + b];
        if (better(ov, oi, v, idx)) { v = ov; idx = oi; }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(v, off, 64);
        const int oi = __shfl_xor(idx, off, 64);
        if (better(ov, oi, v, idx)) { v = ov; idx = oi; }
    }
    if (threadIdx.x == 0) out[m] = idx == 0x7fffffff ? 0 : idx;
}

}  // namespace

bool few_rows_fit(int rows, int hidden) {
    return rows <= kFewRows && hidden % (kStep * kHeadRing) == 0 &&
           kTerms * kFewRows * head_row_bytes(hidden) <= kHeadLds;
}

namespace {

// One instantiation per power of two of row pairs: the row loads are
// unconditional.  Merged rows: at most kPartsMax partials over a wave's row
// pairs (more spill the 128 registers that 16 waves leave), as parts_limit says.
template <int W, int PRO, int EPI, int NS = 0>
sa_status launch_rows(const FewArgs& a, dim3 grid, hipStream_t st) {
    auto launch = [&](auto rp) -> sa_status {
        constexpr int RP = decltype(rp)::value;
        if constexpr (RP * NS <= kPartsMax) {
            hipLaunchKernelGGL((few_rows_kernel<W, RP, PRO, EPI, NS>), grid, dim3(W * 64), 0, st, a);
            SA_CHECK_LAUNCH();
            return SA_OK;
        } else {
            return fail(SA_EINVAL, "no launch merges this many partials of this many rows");
        }
    };
    switch (row_pairs(a.M)) {
        case 1: return launch(std::integral_constant<int, 1>{});
        case 2: return launch(std::integral_constant<int, 2>{});
        case 4: return launch(std::integral_constant<int, 4>{});
        default: return launch(std::integral_constant<int, 8>{});
    }
}

}  // namespace

sa_status few_project_norm(const FewInput& in, int M, int K, const uint16_t* W, int N, float* out, hipStream_t st) {
    return launch_rows<8, kNorm, kOut>(FewArgs{in, W, out, M, K, N, {}, 0}, dim3(N / 16), st);
}

sa_status few_gate_up(const FewInput& in, int M, int K, const uint16_t* W, int I, float* out, hipStream_t st) {
    return launch_rows<8, kNorm, kSwiglu>(FewArgs{in, W, out, M, K, I, {}, 0}, dim3(I / 16), st);
}

sa_status few_project_split(const float* x, int M, int K, const uint16_t* W, int N, float* out, hipStream_t st,
                            const DecodeParts* parts, int D) {
    FewArgs a{{x, nullptr, 0, nullptr, 0.f, nullptr}, W, out, M, K, N, {}, 0};
    const dim3 grid(N / 16, kFewSplit);
    if (!parts || parts->n_split <= 1) return launch_rows<16, kPlain, kOut>(a, grid, st);
    if (parts->n_split > parts_limit(M)) return fail(SA_EINVAL, "more partials than the rows can merge");
    a.parts = *parts;
    a.d_log2 = __builtin_ctz(D);
    switch (parts_form(parts->n_split)) {
        case 2: return launch_rows<16, kPlain, kOut, 2>(a, grid, st);
        case 4: return launch_rows<16, kPlain, kOut, 4>(a, grid, st);
        case 6: return launch_rows<16, kPlain, kOut, 6>(a, grid, st);
        default: return launch_rows<16, kPlain, kOut, kPartsMax>(a, grid, st);
    }
}

sa_status few_head(const FewInput& in, int M, int K, const uint16_t* W, int N, float* logits, float* am_val,
                   int32_t* am_idx, int32_t* next, hipStream_t st) {
    const int bytes = kTerms * kFewRows * head_row_bytes(K);
    SA_TRY((pf::opt_in_lds<&few_head_kernel>(kHeadLds)));
    hipLaunchKernelGGL(few_head_kernel, dim3(kFewHeadBlocks), dim3(kHeadWaves * 64), bytes, st,
                       HeadArgs{in, W, logits, am_val, am_idx, M, K, N});
    SA_CHECK_LAUNCH();
    return few_argmax(am_val, am_idx, kFewHeadBlocks, M, next, st);
}

sa_status few_argmax(const float* pv, const int32_t* pi, int nb, int M, int32_t* next, hipStream_t st) {
    hipLaunchKernelGGL(few_argmax_kernel, dim3(M), dim3(64), 0, st, pv, pi, nb, next);
    SA_CHECK_LAUNCH();
    return SA_OK;
}

}  // namespace sa
