// Host-only planning of launches (no HIP): plain integers, so that it is
// tested without a GPU.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace sa {

// The split-KV partials of a decode launch whose consumer merges them: row m's
// query head h has n_act[m] of them (one or none: its output was written as
// usual), partial i's (m, l) at ml[((m n_q + h) n_split + i) 2] and its D floats
// O, relative to that m, at o[((m n_q + h) n_split + i) D].
constexpr int kPartsRows = 8, kPartsMax = 8;
struct DecodeParts {
    const float* ml;
    const float* o;
    int n_split;             // 0: nothing to merge, n_act unset
    int n_act[kPartsRows];
};

// The most partials per row that M rows' consumer holds in registers.
constexpr int parts_limit(int M) { return M <= 2 ? 8 : M <= 4 ? 4 : M <= kPartsRows ? 2 : 1; }
// The forms of that consumer: row pairs it has registers for, and partials
// per row.  A form exists where the two multiply to at most kPartsMax.
constexpr int row_pairs(int M) { return M <= 2 ? 1 : M <= 4 ? 2 : M <= 8 ? 4 : 8; }
constexpr int parts_form(int n) { return n <= 2 ? 2 : n <= 4 ? 4 : n <= 6 ? 6 : kPartsMax; }

// The partials that a launch of n_seq rows in n_split chunks leaves to its
// consumer: those of at most parts_limit chunks, so of at most kPartsRows rows.
// Row i holds tokens 0 .. pos[i] of at most capacity.
inline DecodeParts plan_parts(const float* ml, const float* o, int n_seq, int n_split, int chunk, int capacity,
                              const int32_t* pos) {
    DecodeParts p{ml, o, 0, {}};
    if (n_split <= 1 || n_split > parts_limit(n_seq)) return p;
    p.n_split = n_split;
    for (int i = 0; i < n_seq; ++i) p.n_act[i] = (std::min(pos[i] + 1, capacity) + chunk - 1) / chunk;
    return p;
}

// Tokens that one launch of rows head rows per token takes, lanes threads each:
// at most 2^31 threads (a launch has fewer than 2^32).
inline int tokens_per_launch(int rows, int lanes) {
    return (int)std::max<long long>(1, (1LL << 31) / ((long long)rows * lanes));
}

}  // namespace sa
