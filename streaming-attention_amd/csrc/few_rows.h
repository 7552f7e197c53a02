// The decoder's projections for at most kFewRows token rows (few_rows.hip).
#pragma once

#include "sa_internal.h"

namespace sa {

constexpr int kFewRows = 16;      // token rows one launch covers
constexpr int kFewSplit = 2;      // K splits of the o and down projections
constexpr int kFewHeadBlocks = 256;   // lm_head workgroups (argmax partials per row)

// The rows a projection starts from.
struct FewInput {
    const float* x;          // [M][K]
    // With norm_w: the rows are v = x + sum over s of y[s] (y: n_y partials
    // [n_y][M][K], n_y 0 or kFewSplit), enter as rms_norm(v) * norm_w, and v goes to
    // x_out (if given; not x).
    const float* y;
    int n_y;
    const float* norm_w;
    float eps;
    float* x_out;
};

// Whether rows x hidden size of a model can take these launches (the head keeps 16
// rows of terms in LDS: hidden a multiple of 256 up to 1536).  Others take
// proj.hip: 12 layers of hidden 2048 at 1 / 16 rows 970 / 1022 us.
bool few_rows_fit(int rows, int hidden);

// out[M][N] = input . W^T (input with norm_w).
sa_status few_project_norm(const FewInput& in, int M, int K, const uint16_t* W, int N, float* out, hipStream_t st);
// out[M][I] = silu(gate) * up of input . W^T, W [2 I][K] (gate rows, then up).
sa_status few_gate_up(const FewInput& in, int M, int K, const uint16_t* W, int I, float* out, hipStream_t st);
// out[kFewSplit][M][N]: the K splits of x . W^T.  With parts (n_split > 0) rows of
// several partials are merged from them instead of read from x: K = heads of
// D columns (D a power of two, 4 or more), at most parts_limit(M) partials.
sa_status few_project_split(const float* x, int M, int K, const uint16_t* W, int N, float* out, hipStream_t st,
                            const DecodeParts* parts = nullptr, int D = 0);
// next[m] = the greedy index of row m's nb workgroup maxima pv / pi [M][nb].
sa_status few_argmax(const float* pv, const int32_t* pi, int nb, int M, int32_t* next, hipStream_t st);
// logits[M][N] = input . W^T and next[m] = the lowest index of row m's maximum;
// am_val / am_idx: [M][kFewHeadBlocks] scratch.
sa_status few_head(const FewInput& in, int M, int K, const uint16_t* W, int N, float* logits, float* am_val,
                   int32_t* am_idx, int32_t* next, hipStream_t st);

}  // namespace sa
