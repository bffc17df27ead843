// opt_decide.hpp -- the sums behind one decision of the direction search: a
// scan launch leaves part[group][cell], the powers of every cell summed over
// each group's channels; the next launch's workgroups each fold the groups
// into P[cell].  Shared with a host test, which runs every thread's share
// with bounds checks.
#pragma once

#include <cstddef>

#ifdef __HIPCC__
#define BF_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define BF_HOST_DEVICE inline
#endif

namespace bfhip {

constexpr int kScanWaves = 8;
constexpr int kScanThreads = 64 * kScanWaves;

// Rows of `part` hold whole tiles of 16 cells.  `ways` threads share a cell,
// each `per` groups, as long as the tiles leave threads over.
struct DecideSplit {
    int padded, ways, per;
};
BF_HOST_DEVICE DecideSplit decide_split(int n_cells, int groups) {
    DecideSplit d;
    d.padded = (n_cells + 15) & ~15;
    d.ways = d.padded < kScanThreads ? kScanThreads / d.padded : 1;
    d.per = (groups + d.ways - 1) / d.ways;
    return d;
}

// Thread `tid`'s sums, in FP64 and a fixed order: with several ways into
// sums[kScanThreads], else into P[n_cells], which holds no padding.
BF_HOST_DEVICE void decide_sum(const DecideSplit& d, int tid, int n_cells, int groups,
                               const double* part, float* P, double* sums) {
    for (int i = tid; i < d.padded * d.ways; i += kScanThreads) {
        const int cell = i % d.padded, way = i / d.padded;
        const int last = (way + 1) * d.per;
        const int end = last < groups ? last : groups;
        double sum = 0.0;
#pragma unroll 8
        for (int q = way * d.per; q < end; ++q) sum += part[(size_t)q * d.padded + cell];
        if (d.ways > 1)
            sums[i] = sum;
        else if (cell < n_cells)
            P[cell] = (float)sum;
    }
}

// Where several ways shared a cell (after a barrier): thread `tid`'s cells.
BF_HOST_DEVICE void decide_fold(const DecideSplit& d, int tid, int n_cells, const double* sums,
                                float* P) {
    for (int cell = tid; cell < n_cells; cell += kScanThreads) {
        double sum = 0.0;
        for (int way = 0; way < d.ways; ++way) sum += sums[way * d.padded + cell];
        P[cell] = (float)sum;
    }
}

}  // namespace bfhip
