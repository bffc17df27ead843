// The sums behind a decision of the direction search (csrc/opt_decide.hpp),
// every thread's share run on the host: no store may leave P[n_cells] or
// sums[kScanThreads], and the powers are the sums over the groups.
#include <cmath>
#include <cstdio>
#include <vector>

#include "opt_decide.hpp"

using namespace bfhip;

static int check(int n_cells, int groups) {
    const int padded = (n_cells + 15) / 16 * 16;
    std::vector<double> part((size_t)groups * padded);
    for (size_t i = 0; i < part.size(); ++i) part[i] = 1.0 + (double)((i * 2654435761u) % 1000u);
    const float kUnwritten = -1.0f;
    std::vector<float> P(n_cells + 64, kUnwritten);
    std::vector<double> sums(kScanThreads + 64, kUnwritten);
    const DecideSplit d = decide_split(n_cells, groups);
    for (int t = 0; t < kScanThreads; ++t)
        decide_sum(d, t, n_cells, groups, part.data(), P.data(), sums.data());
    if (d.ways > 1)
        for (int t = 0; t < kScanThreads; ++t)
            decide_fold(d, t, n_cells, sums.data(), P.data());
    int bad = 0;
    for (int i = 0; i < 64; ++i)
        bad += P[n_cells + i] != kUnwritten || sums[kScanThreads + i] != kUnwritten;
    for (int c = 0; c < n_cells; ++c) {
        double want = 0.0;
        for (int q = 0; q < groups; ++q) want += part[(size_t)q * padded + c];
        bad += P[c] != (float)want;  // whole numbers: exact in any order
    }
    if (bad) std::printf("cells %d groups %d: %d wrong\n", n_cells, groups, bad);
    return bad;
}

int main() {
    int bad = check(9, 1) + check(9, 84) + check(9, 16384);
    for (int G = 2; G <= 64; ++G)
        for (int groups : {1, 7, 42}) bad += check(G * G, groups);
    if (bad) return 1;
    std::puts("OK");
    return 0;
}
