// The decoder's projections of prompts and of decode steps that few_rows.hip does
// not take (proj.hip).
#pragma once

#include "sa_internal.h"

namespace sa {

// One projection: [M][K] fp32 rows times a bf16 weight [N][K] (pair: [2 N][K],
// gate rows then up rows, N activations out).
struct ProjPlan {
    int N, K;
    bool pair;
    int tile;    // index of the workgroup tile (proj.hip)
    int split;   // K splits: partial sums per output (1 with pair)
};

// The plan of an M-row projection on cus compute units with at most max_split
// K splits.
ProjPlan plan_proj(int M, int N, int K, bool pair, int cus, int max_split);

// out[split][M][N]: the K splits of X . W^T; with pair out[M][N] =
// silu(X . gate^T) * (X . up^T).  N % 16 == 0, K % 32 == 0.
sa_status project(const float* X, int M, const uint16_t* W, const ProjPlan& p, float* out, hipStream_t st);

}  // namespace sa
