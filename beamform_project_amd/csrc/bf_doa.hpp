// bf_doa.hpp -- DOA kernel launchers (internal).
#pragma once

#include "bf_common.hpp"

namespace bfhip {

// Exact smoothed integer covariance of snapshots t0 .. t0+K-1 as `parts`
// partial sums rs [parts][F][M][M][2] over disjoint snapshot ranges (their
// sum is the covariance), parts = doa_covariance_parts(K, max_parts), one
// with r_full, which then also receives the full [F][A][A][2] covariance.
// Returns parts.
size_t doa_covariance_parts(size_t K, size_t max_parts);
size_t launch_doa_covariance(hipStream_t stream, const uint8_t* x, size_t T, size_t F,
                             size_t A, size_t t0, size_t K, size_t M, int* rs, int* r_full,
                             size_t max_parts = 1);

// The same for `n` consecutive windows of K snapshots from t0, the last one
// cut short by T: rs [n][F][M][M][2], one part each.
void launch_doa_covariance_windows(hipStream_t stream, const uint8_t* x, size_t T, size_t F,
                                   size_t A, size_t t0, size_t K, size_t n, size_t M, int* rs);

// FP64 fold, Cholesky, inverse and Bartlett/Capon scans per channel; rs
// holds `parts` partial covariances, summed here.
void launch_doa_fold_scan(hipStream_t stream, const int* rs, size_t parts, double* state,
                          bool first,
                          size_t F, size_t M, size_t K, size_t L, double alpha, double load,
                          const float* freqs, double x_step, size_t n_theta,
                          const double* sin_theta, double* capon, double* bartlett,
                          int* chol_ok);

// Broadband spectra and the strongest local maxima with parabolic refinement.
void launch_doa_estimate(hipStream_t stream, const double* capon, const double* bartlett,
                         size_t F, size_t n_theta, const double* theta, size_t max_peaks,
                         double* broadband, double* peaks, int* n_peaks);

// ----------------------------------------------- planar direction search
// Device state of one search: the centre of the window's coarse grid (the
// previous window's estimate) and the running centre of the refinement.
struct OptSearch {
    float prev[3];
    float centre[3];
};

struct OptGridArgs {
    int G;         // coarse cells per axis
    int M;         // sub-array size (steered antennas 0 .. M-1)
    float fov_l;   // half-extent of the coarse grid
    float fov_m;
    int coplanar;  // steer at nominal lattice points (every |z| <= 1e-6)
    int interp;    // quadratic peak interpolation
};

// Windows whose operands are prepared together at most.
inline constexpr int kOptBatch = 8;

// Scan operands of `n` <= kOptBatch consecutive windows, per channel:
// operand_bytes each, the trace, and the form (1: R^-1 in FP64; 0: R in
// FP32).
struct OptWindows {
    size_t n = 0;
    char* operand = nullptr;
    double* trace = nullptr;
    int* mode = nullptr;
};
size_t opt_operand_bytes(size_t M, bool capon);
// Doubles of launch_opt_scan's scratch.
size_t opt_part_count(size_t F, size_t n_cells);

// Per channel and window, in order: R_block = Rs / (K L) (forward-backward
// averaged when fb; K_last snapshots in the last window), diagonal load
// (Capon), forgetting fold into state [F][M][M][2] FP64, and the scan
// operand: R, or Capon's R^-1, or R where its factorisation fails.
void launch_opt_fold(hipStream_t stream, const OptWindows& b, const int* rs, double* state,
                     bool first, size_t F, size_t M, size_t K, size_t K_last, size_t L, bool fb,
                     bool capon, float load, float lambda);

// The chain of scan launches of one run.  A launch reads state[n & 1], takes
// the decision on launch n - 1 from part[(n - 1) & 1], leaves the new state in
// state[(n + 1) & 1] and its own sums in part[n & 1].
struct OptScan {
    OptSearch* state = nullptr;          // [2]; state[0] set before the first launch
    double* part[2] = {nullptr, nullptr};  // opt_part_count doubles each
    unsigned launches = 0;               // of this run
    int level = 0;                       // the last launch's
    size_t cells = 0, groups = 0, window = 0;
};

// One level of the search of window `index` of the batch: every channel's
// power at the cells (0: the G x G grid around the state's prev, else the 3 x
// 3 refinement candidates), after the decision on the launch before, which
// at last_level writes its window's direction to dirs[window][3].  With
// n_cells = 0 only that decision is taken.
void launch_opt_scan(hipStream_t stream, OptScan& q, const OptWindows& b, size_t index,
                     const float* pos, const float* freqs, const OptGridArgs& g, int level,
                     int last_level, size_t window, size_t F, size_t n_cells, bool capon,
                     float* dirs);

}  // namespace bfhip
