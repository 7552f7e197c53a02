// CPU unit test of the host-side launch planning (csrc/host_plan.h; no GPU, no
// HIP): the partials a decode launch leaves to its consumer, the tokens of an
// append's launch.
#include "host_plan.h"

#include <cstdio>
#include <cstring>
#include <vector>

static int g_fail = 0;

#define EXPECT(cond)                                                       \
    do {                                                                   \
        if (!(cond)) {                                                     \
            std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond);    \
            ++g_fail;                                                      \
        }                                                                  \
    } while (0)

// A plan of n rows, row i of lens[i] tokens, between guard words.
struct Guarded {
    int32_t before[16];
    sa::DecodeParts p;
    int32_t after[16];
};

static void check_rows(int n, int longest, int chunk, int capacity) {
    std::vector<int32_t> pos;   // the longest row last, the others shorter
    for (int i = 0; i < n; ++i) pos.push_back(i + 1 == n ? longest - 1 : (longest - 1) * i / n);
    const int n_split = (std::min(longest, capacity) + chunk - 1) / chunk;
    Guarded g;
    std::memset(&g, 0x5a, sizeof g);
    static const float ml = 0.f, o = 0.f;
    g.p = sa::plan_parts(&ml, &o, n, n_split, chunk, capacity, pos.data());
    for (int i = 0; i < 16; ++i) EXPECT(g.before[i] == 0x5a5a5a5a && g.after[i] == 0x5a5a5a5a);
    EXPECT(g.p.ml == &ml && g.p.o == &o);
    const int limit = n <= 2 ? 8 : n <= 4 ? 4 : n <= 8 ? 2 : 1;
    const bool merged = n_split > 1 && n_split <= limit;
    EXPECT(g.p.n_split == (merged ? n_split : 0));
    for (int i = 0; i < sa::kPartsRows; ++i) {
        const int len = i < n ? std::min(pos[i] + 1, capacity) : 0;
        EXPECT(g.p.n_act[i] == (merged ? (len + chunk - 1) / chunk : 0));
    }
}

int main() {
    for (int n = 1; n <= 16; ++n) {
        EXPECT(sa::parts_limit(n) >= 1 && sa::parts_limit(n) <= sa::kPartsMax);
        EXPECT(n <= sa::kPartsRows || sa::parts_limit(n) == 1);
        // every count up to the limit has a form that holds it
        EXPECT(2 * sa::row_pairs(n) >= n);
        for (int s = 2; s <= sa::parts_limit(n); ++s)
            EXPECT(sa::parts_form(s) >= s && sa::parts_form(s) * sa::row_pairs(n) <= sa::kPartsMax);
        for (int chunk : {64, 128, 256, 4096})
            for (int chunks = 1; chunks <= 10; ++chunks)
                for (int longest : {chunk * (chunks - 1) + 1, chunk * chunks}) {
                    check_rows(n, longest, chunk, 1 << 20);
                    check_rows(n, longest, chunk, longest - 1 > 0 ? longest - 1 : 1);   // a full table row
                }
    }
    for (int lanes : {1, 2, 4, 8, 16, 32, 64})
        for (int rows : {2, 3, 24, 32, 48, 64, 1000, 1 << 20}) {
            const long long t = sa::tokens_per_launch(rows, lanes);
            EXPECT(t >= 1 && t * rows * lanes <= 1LL << 31);          // threads of a launch
            EXPECT((t + 1) * rows * lanes > 1LL << 31);               // as many as fit
        }
    if (g_fail) return 1;
    std::printf("all checks passed\n");
    return 0;
}
