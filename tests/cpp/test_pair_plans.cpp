// The plans of a backward's two products (plan.h), host code only: where both fit
// one launch without a split over K they pair (a split of 128x128 tiles would make
// three or four launches), and products too large for that keep their own plans.
#include <cstdio>

#include "plan.h"

using namespace seera;

int main() {
    struct Case {
        int M, N, K;
        bool pair;
    };
    int bad = 0;
    for (const Case c : {Case{3584, 2752, 128, true},    // one launch 27 us, four 41
                         Case{4288, 4288, 64, true},     // 31 / 41
                         Case{2048, 3072, 128, true},    // on 64x64 tiles: 27 / 31
                         Case{64, 784, 128, true}, Case{4096, 4096, 4096, false}, Case{2304, 2304, 2304, false}}) {
        Plan a, b;  // dA = dC . B^T (M x K over N), dB = A^T . dC (K x N over M)
        const bool pair = pair_plans(c.M, c.K, c.N, c.K, c.N, c.M, a, b);
        if (pair != c.pair || (pair && (a.splits != 1 || b.splits != 1))) {
            std::printf("%d x %d x %d: pair %d, splits %d %d\n", c.M, c.N, c.K, pair, a.splits, b.splits);
            ++bad;
        }
    }
    if (!bad) std::puts("all checks passed");
    return bad != 0;
}
