// k_opt_tracker.hip -- adaptive planar direction search for gfx950: the
// searching path of the reference's CpuOptBeamTracker::run_into
// (src/cpu_opt_beam_tracker.cpp:1619-2457), one integration window at a time.
//
// All stages are stream-ordered, nothing returns to the host.  For a batch of
// windows at once:
//   covariance      launch_doa_covariance (k_doa.hip): exact int32 sums of
//                   x x^H over each window's snapshots, forward smoothing over
//                   L = A - M + 1 sub-arrays (:559-636).
//   opt_fold        per channel, FP64: R_block = Rs / (K L), forward-backward
//                   average when smoothing (:637-656, without the in-place
//                   read of already-averaged entries), diagonal load for
//                   Capon (:244-253, before the fold, :1803-1804), forgetting
//                   fold R = lambda R + (1 - lambda) R_block (:1880-1892)
//                   window by window, trace.
//   opt_factor      Capon only: R^-1 by Gauss-Jordan, whose pivots are those
//                   of the Cholesky factorisation (:398-421).
// Then per window and level, one launch:
//   opt_scan        per (channel, cell): the steering vector
//                   a_j = exp(-j k p_j . d) (:96-106) and the Bartlett power
//                   tr(R) + 2 Re sum_{r<c} conj(a_r) R_rc a_c (:287-306) or
//                   the Capon power 1 / (a^H R^-1 a), on the matrix cores,
//                   summed over a workgroup's channels.  Every workgroup of
//                   the next launch first adds those sums up and takes the
//                   level's decision for itself: argmax, the next centre,
//                   quadratic peak interpolation (:830-853), and at the last
//                   level the window's direction.  (A launch of its own for
//                   the decision costs two more gaps per level; letting the
//                   last workgroup decide costs each one a fence across the
//                   XCDs, 105 us instead of 23 for 144 cells.)
// Level 0 scans the G x G grid centred on the previous estimate
// (build_centred_grid, :798-828); each refinement level scans the 3 x 3
// neighbourhood of the running centre at half the previous pitch
// (:2179-2388).
//
// Steering directions follow the reference's two cases.  For a coplanar
// array (every |z| <= 1e-6) the reference multiplies a centre phasor by a
// tabulated relative phasor, i.e. it steers at the nominal lattice point
// centre + offset in FP64 (:1971-2013, :1216-1296); a lattice point outside
// l^2 + m^2 <= 0.999 and every point of a non-coplanar array steers at the
// clamped float direction instead.  Here the FP64 phase of that direction is
// evaluated directly, so the steering vector equals the reference's up to
// the rounding of its phasor product.
#include <algorithm>

#include "bf_doa.hpp"
#include "gauss_jordan.hpp"
#include "opt_decide.hpp"
#include "steering.hpp"

namespace bfhip {
namespace {

constexpr int kFoldThreads = 512;

struct cd {
    double re, im;
};

// ------------------------------------------------------- search geometry
// Coarse cell (u, v) of the grid centred on `c` (build_centred_grid,
// src/cpu_opt_beam_tracker.cpp:798-828): its clamped float direction, and
// the direction the scan steers at.
__device__ void coarse_cell(const OptGridArgs& g, const float c[3], int u, int v, float dir[3],
                            double st[3]) {
    const int G = g.G;
    const float step_l = G == 1 ? 0.0f : (2.0f * g.fov_l) / (float)(G - 1);
    const float step_m = G == 1 ? 0.0f : (2.0f * g.fov_m) / (float)(G - 1);
    float l = (c[0] - g.fov_l) + (float)u * step_l;
    float m = (c[1] - g.fov_m) + (float)v * step_m;
    const float r2 = l * l + m * m;
    if (r2 > 0.999f) {
        const float s = sqrtf(0.999f / r2);
        l *= s;
        m *= s;
    }
    dir[0] = l;
    dir[1] = m;
    dir[2] = sqrtf(1.0f - (l * l + m * m));
    st[0] = (double)dir[0];
    st[1] = (double)dir[1];
    st[2] = (double)dir[2];
    if (g.coplanar) {
        // nominal lattice point (:1971-1993)
        const double sl = G == 1 ? 0.0 : (2.0 * (double)g.fov_l) / (double)(G - 1);
        const double sm = G == 1 ? 0.0 : (2.0 * (double)g.fov_m) / (double)(G - 1);
        const double mid = (double)(G - 1) * 0.5;
        const double nl = (double)c[0] + ((double)u - mid) * sl;
        const double nm = (double)c[1] + ((double)v - mid) * sm;
        if (!(nl * nl + nm * nm > 0.999)) {
            st[0] = nl;
            st[1] = nm;
            st[2] = 0.0;
        }
    }
}

// Candidate i = (dv + 1) * 3 + (du + 1) of refinement level `level` >= 1
// around centre `c` (:2179-2203, :2219-2233).
__device__ void refine_cell(const OptGridArgs& g, const float c[3], int level, int i,
                            float dir[3], double st[3]) {
    const int du = i % 3 - 1, dv = i / 3 - 1;
    float hl = g.fov_l / (float)g.G, hm = g.fov_m / (float)g.G;
    for (int k = 0; k < level; ++k) {
        hl *= 0.5f;
        hm *= 0.5f;
    }
    float l = c[0] + (float)du * hl;
    float m = c[1] + (float)dv * hm;
    const float r2 = l * l + m * m;
    const bool clamped = r2 > 0.999f;
    if (clamped) {
        const float s = sqrtf(0.999f / r2);
        l *= s;
        m *= s;
    }
    dir[0] = l;
    dir[1] = m;
    dir[2] = sqrtf(1.0f - (l * l + m * m));
    if (g.coplanar && !clamped) {
        st[0] = (double)c[0] + (double)du * (double)hl;
        st[1] = (double)c[1] + (double)dv * (double)hm;
        st[2] = 0.0;
    } else {
        st[0] = (double)dir[0];
        st[1] = (double)dir[1];
        st[2] = (double)dir[2];
    }
}

__device__ void cell_direction(const OptGridArgs& g, const OptSearch& s, int level, int cell,
                               float dir[3], double st[3]) {
    if (level == 0)
        coarse_cell(g, s.prev, cell % g.G, cell / g.G, dir, st);
    else
        refine_cell(g, s.centre, level, cell, dir, st);
}

// quadratic_interp (:830-853): offsets applied only where the 3-point
// curvature is positive, clamped to half a cell.
__device__ void quadratic_interp(float pc, float p_up, float p_down, float p_vp, float p_vm,
                                 float* du, float* dv) {
    *du = 0.0f;
    *dv = 0.0f;
    const float den_u = p_down - 2.0f * pc + p_up;
    if (den_u > 0.0f) {
        float d = (0.5f * (p_up - p_down)) / den_u;
        d = d > 0.5f ? 0.5f : d;
        d = d < -0.5f ? -0.5f : d;
        *du = d;
    }
    const float den_v = p_vm - 2.0f * pc + p_vp;
    if (den_v > 0.0f) {
        float d = (0.5f * (p_vp - p_vm)) / den_v;
        d = d > 0.5f ? 0.5f : d;
        d = d < -0.5f ? -0.5f : d;
        *dv = d;
    }
}

// direction_from_lm of (l, m) after the 0.999 horizon clamp (:2350-2357).
__device__ void clamp_direction(float l, float m, float out[3]) {
    const float r2 = l * l + m * m;
    if (r2 > 0.999f) {
        const float s = sqrtf(0.999f / r2);
        l *= s;
        m *= s;
    }
    out[0] = l;
    out[1] = m;
    out[2] = sqrtf(1.0f - (l * l + m * m));
}

// ------------------------------------------------------------------ fold
// The scan's operand of one channel: the Hermitian form H = X + iY (R, or
// R^-1) without its diagonal, which the trace carries, as two real planes
// [Mp][Mp], Mp = M rounded up to 16, zero outside M.  Only the 16 x 16 blocks
// (I, J) with J >= I are read; a block on the diagonal is read whole, so its
// X is halved (exactly): the scan doubles every sum.  FP64 planes keep the
// columns of a block in the order c -> 4 (c % 4) + c / 4, so that a lane's
// four values of a block row are contiguous in both precisions.
__device__ __forceinline__ int plane_column64(int c) {
    return (c & ~15) | (4 * (c & 3) + ((c & 15) >> 2));
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// The windows of one batch, in order.
struct FoldArgs {
    const int2* rs;  // [n][F][M][M]
    double2* state;  // [F][M][M]
    char* operand;   // [n][F] operands of operand_bytes
    double* trace;   // [n][F]
    int* mode;       // [n][F]
    size_t operand_bytes;
    int n, first, M, Mp, K, K_last, L, fb, capon;
    float load, lambda;
};

// One workgroup per channel: each thread carries its covariance entries
// through the batch's windows: R_block = Rs / (K L), forward-backward averaged
// when fb (the mirrored entry is read from Rs directly), diagonal load for
// Capon, and the fold.  Bartlett writes the scan's FP32 planes, for the
// entries of the blocks that are read; Capon the folded R, [M][M] complex FP64
// in the operand's place, for opt_factor_kernel.  Bound by memory latency: an
// entry's loads of all windows are issued together.
__global__ __launch_bounds__(kFoldThreads) void opt_fold_kernel(FoldArgs a) {
    __shared__ double s_eps[kOptBatch];
    const int f = blockIdx.x;
    const int F = gridDim.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int M = a.M, MM = M * M;
    const bool copy_all = a.lambda >= 1.0f;
    const double lam = (double)a.lambda;
    const double comp = (double)(1.0f - a.lambda);
    // R_block of entry (r, c) in every window of the batch
    auto blocks = [&](int r, int c, cd (&v)[kOptBatch]) {
        int2 p[kOptBatch], m[kOptBatch];
#pragma unroll
        for (int w = 0; w < kOptBatch; ++w) {
            const int2* rf = a.rs + ((size_t)min(w, a.n - 1) * F + f) * MM;
            p[w] = rf[r * M + c];
            if (a.fb) m[w] = rf[(M - 1 - r) * M + (M - 1 - c)];
        }
#pragma unroll
        for (int w = 0; w < kOptBatch; ++w) {
            const double scale = 1.0 / ((double)(w + 1 == a.n ? a.K_last : a.K) * (double)a.L);
            v[w] = cd{(double)p[w].x * scale, (double)p[w].y * scale};
            if (a.fb) {
                // (R + J conj(R) J) / 2
                v[w].re = 0.5 * (v[w].re + (double)m[w].x * scale);
                v[w].im = 0.5 * (v[w].im - (double)m[w].y * scale);
            }
        }
    };
    double2* st = a.state + (size_t)f * MM;
    if (wave == 0) {  // traces (M <= 64: one lane per diagonal entry)
        cd v[kOptBatch];
        const int i = min(lane, M - 1);
        blocks(i, i, v);
        // of the folded R, by the recursion below on the diagonal
        double d = a.first || copy_all ? 0.0 : st[i * M + i].x;
#pragma unroll
        for (int w = 0; w < kOptBatch; ++w) {
            if (w >= a.n) break;
            const double tr = wave_sum_f64(lane < M ? v[w].re : 0.0);
            d = copy_all || (a.first && w == 0) ? v[w].re : lam * d + comp * v[w].re;
            const double folded = wave_sum_f64(lane < M ? d : 0.0);
            if (lane == 0) {
                s_eps[w] = (a.capon && a.load > 0.0f) ? (double)a.load * tr / (double)M : 0.0;
                if (!a.capon) {
                    a.trace[(size_t)w * F + f] = folded;
                    a.mode[(size_t)w * F + f] = 0;
                }
            }
        }
    }
    __syncthreads();  // and the diagonal's old state has been read
    const int Mp = a.Mp;
    // thread = column c of rows r0, r0 + step, ...
    const int c = tid & 63, step = kFoldThreads / 64;
    if (c >= Mp) return;
    for (int r = tid >> 6; r < Mp; r += step) {
        if (!a.capon && (r >> 4) > (c >> 4)) continue;
        const bool in = r < M && c < M;
        const int es = in ? r * M + c : 0;
        cd v[kOptBatch];
        blocks(min(r, M - 1), min(c, M - 1), v);
        const double2 old = a.first || copy_all ? make_double2(0.0, 0.0) : st[es];
        cd prev{old.x, old.y};
#pragma unroll
        for (int w = 0; w < kOptBatch; ++w) {
            if (w >= a.n) break;
            if (r == c) v[w].re += s_eps[w];
            if (!copy_all && !(a.first && w == 0)) {
                v[w].re = lam * prev.re + comp * v[w].re;
                v[w].im = lam * prev.im + comp * v[w].im;
            }
            prev = v[w];
            char* const op = a.operand + ((size_t)w * F + f) * a.operand_bytes;
            if (a.capon) {
                if (in) reinterpret_cast<double2*>(op)[es] = make_double2(prev.re, prev.im);
            } else {
                float* const X = reinterpret_cast<float*>(op) + r * Mp + c;
                const bool zero = !in || r == c;
                X[0] = zero ? 0.0f : ((r >> 4) == (c >> 4) ? 0.5f : 1.0f) * (float)prev.re;
                X[Mp * Mp] = zero ? 0.0f : (float)prev.im;
            }
        }
        if (in) st[es] = make_double2(prev.re, prev.im);
    }
}

// ---------------------------------------------------------------- factor
constexpr int kGjBlock = 4;                                     // 4 x 4 blocks
constexpr int kFactorThreads = (64 / kGjBlock) * (64 / kGjBlock);  // 256
// Capon operand: Q = R^-1 of the folded covariance by in-place Gauss-Jordan
// elimination in FP64 (gauss_jordan.hpp), one workgroup per (channel,
// window).  The reference's factorisation test (d_k > 1e-12, :398-421) is
// applied to the pivots; a failed channel falls back to the Bartlett form on
// the folded R (:354-375).  Bound by the chain of M pivots, each a barrier
// and an FP64 division: a batch of windows in one launch keeps several
// workgroups per CU in flight (10 windows of 64 antennas, 336 channels: 1.48
// ms one window at a time).
__global__ __launch_bounds__(kFactorThreads) void opt_factor_kernel(
    char* __restrict__ operand, size_t operand_bytes, int M, int Mp, double* __restrict__ trace,
    int* __restrict__ mode) {
    __shared__ GjShared<cd> sh;
    __shared__ double s_diag[64];
    const size_t f = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    const int tid = threadIdx.x;
    const int i0 = gj_row0<kGjBlock>(tid), j0 = gj_col0<kGjBlock>(tid);
    char* const op = operand + f * operand_bytes;
    const double* R = reinterpret_cast<const double*>(op);
    cd a[kGjBlock][kGjBlock];
    gj_load<kGjBlock>(a, R, M, M, tid);
    const bool ok = gj_invert<kGjBlock>(a, M, 1e-12, sh, tid);
    if (!ok) gj_load<kGjBlock>(a, R, M, M, tid);  // R again, in place
    __syncthreads();  // R has been read by all before the planes replace it
#pragma unroll
    for (int u = 0; u < kGjBlock; ++u)
#pragma unroll
        for (int v = 0; v < kGjBlock; ++v) {
            const int i = i0 + u, j = j0 + v;
            if (i >= Mp || j >= Mp) continue;
            const bool in = i < M && j < M && i != j;
            const double half = (i >> 4) == (j >> 4) ? 0.5 : 1.0;
            const double re = in ? half * a[u][v].re : 0.0, im = in ? a[u][v].im : 0.0;
            if (ok) {
                double* const X = reinterpret_cast<double*>(op);
                X[i * Mp + plane_column64(j)] = re;
                X[(Mp + i) * Mp + plane_column64(j)] = im;
            } else {
                float* const X = reinterpret_cast<float*>(op);
                X[i * Mp + j] = (float)re;
                X[(Mp + i) * Mp + j] = (float)im;
            }
            if (i == j) s_diag[i] = i < M ? a[u][v].re : 0.0;
        }
    __syncthreads();
    if (tid < 64) {
        const double tr = wave_sum_f64(tid < M ? s_diag[tid] : 0.0);
        if (tid == 0) {
            trace[f] = tr;
            mode[f] = ok ? 1 : 0;
        }
    }
}

// ------------------------------------------------------------------ scan
// With a = u + iv and H = X + iY (X symmetric, Y antisymmetric, both without
// the diagonal), a^H H a = tr H + 2 sum_{r<c} Re(conj(a_r) H_rc a_c).  By 16 x
// 16 blocks that is 2 sum_I [u_I . (U - Z) + v_I . (V + W)] with U, V =
// sum_{J >= I} X_IJ u_J, X_IJ v_J, W = sum_{J >= I} Y_IJ u_J and Z =
// sum_{J > I} Y_IJ v_J (a diagonal block needs no Z: v . Y u counts both of its
// triangles).  A wave evaluates 16 cells of one channel, a column each:
// the four sums are 16x16x4 MFMAs (FP32, or FP64 for Capon, where the large
// entries of R^-1 cancel), with H's rows as the A operand straight from L2.
// Lane l holds cell l % 16 and a quarter of the antennas (g = l / 16):
// slot 4 J + r is antenna 16 J + 4 g + r in FP32 and 16 J + 4 r + g in FP64, the
// rows its MFMA results hold, so u, v meet U, V, W, Z without moving.
typedef double bf_double4 __attribute__((ext_vector_type(4)));

template <typename T>
struct ScanTypes;
template <>
struct ScanTypes<float> {
    typedef bf_float4 vec;
    __device__ static vec mfma(float a, float b, vec c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static int antenna(int j, int r, int g) { return 16 * j + 4 * g + r; }
};
template <>
struct ScanTypes<double> {
    typedef bf_double4 vec;
    __device__ static vec mfma(double a, double b, vec c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static int antenna(int j, int r, int g) { return 16 * j + 4 * r + g; }
};

// This lane's part of sum_I [...] over the block rows I whose bit is set in
// `rows`, for the cell whose phase per metre (in turns) is d.
template <typename T>
__device__ __forceinline__ T scan_form(const T* __restrict__ X, int Mp, const double* s_pos,
                                       const double (&d)[3], unsigned rows, int lane) {
    using ST = ScanTypes<T>;
    typedef typename ST::vec vec;
    const int g = lane >> 4;
    const int nb = Mp >> 4;
    T u[16], v[16];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double* const p = s_pos + 3 * ST::antenna(j, r, g);
            const double t = fma(p[2], d[2], fma(p[1], d[1], p[0] * d[0]));
            const double2 cs = cos_sin_turns64(t);
            u[4 * j + r] = (T)cs.x;
            v[4 * j + r] = (T)-cs.y;
        }
    const T* const row = X + (size_t)(lane & 15) * Mp + 4 * g;  // + 16 I Mp + 16 J
    T sum = (T)0;
#pragma unroll
    for (int I = 0; I < 4; ++I) {
        if (I >= nb || !((rows >> I) & 1u)) continue;  // uniform
        vec U = {0, 0, 0, 0}, V = {0, 0, 0, 0}, W = {0, 0, 0, 0}, Z = {0, 0, 0, 0};
#pragma unroll
        for (int J = I; J < 4; ++J) {
            if (J >= nb) continue;
            const vec x = *reinterpret_cast<const vec*>(row + (size_t)16 * I * Mp + 16 * J);
            const vec y = *reinterpret_cast<const vec*>(row + (size_t)(Mp + 16 * I) * Mp + 16 * J);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                U = ST::mfma(x[r], u[4 * J + r], U);
                V = ST::mfma(x[r], v[4 * J + r], V);
                W = ST::mfma(y[r], u[4 * J + r], W);
                if (J > I) Z = ST::mfma(y[r], v[4 * J + r], Z);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            sum += u[4 * I + r] * (U[r] - Z[r]) + v[4 * I + r] * (V[r] + W[r]);
    }
    return sum;
}

struct ScanArgs {
    const char* operand;  // the window's [F] operands
    const double* trace;  // [F]
    const int* mode;      // [F]
    size_t operand_bytes;
    const float* pos;
    const float* freqs;
    const OptSearch* search;  // the state before that launch's decision
    OptGridArgs g;
    int level, n_cells, F, Mp;
    double* part;  // [groups][16 tiles] sums over the channels of a workgroup
    // the launch before this one, whose decision is taken here
    int last_level, before_level, before_cells, before_groups, before_window;
    const double* before_part;  // null: no launch before
    OptSearch* next;  // the state after that decision
    float* dirs;
};

// The decision on the launch before, by the whole workgroup: its powers summed
// over the channel groups (opt_decide.hpp), then thread 0's serial part; the
// new state goes to *out.  LDS scratch: P[before_cells], sums[kScanThreads].
__device__ void decide(const ScanArgs& a, float* P, double* sums, OptSearch* out) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int n_cells = a.before_cells;
    const DecideSplit d = decide_split(n_cells, a.before_groups);
    const int level = a.before_level, last_level = a.last_level;
    const OptGridArgs& g = a.g;
    decide_sum(d, tid, n_cells, a.before_groups, a.before_part, P, sums);
    __syncthreads();
    if (d.ways > 1) {
        decide_fold(d, tid, n_cells, sums, P);
        __syncthreads();
    }
    if (tid >= 64) return;
    // argmax with the reference's rule (strict >, so the first maximum):
    // each lane scans its cells in increasing order, then the lanes combine
    // preferring the larger value and, on a tie, the lower index
    float bv = -__builtin_huge_valf();
    int bi = n_cells;  // none yet
    for (int i = lane; i < n_cells; i += 64)
        if (bi == n_cells || P[i] > bv) {
            bv = P[i];
            bi = i;
        }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (oi < n_cells && (bi == n_cells || ov > bv || (ov == bv && oi < bi))) {
            bv = ov;
            bi = oi;
        }
    }
    if (lane != 0) return;
    OptSearch s = *a.search;
    float dir[3];
    double st[3];
    const int best = bi;
    cell_direction(g, s, level, best, dir, st);
    float c[3] = {dir[0], dir[1], dir[2]};
    if (g.interp) {
        float du = 0.0f, dv = 0.0f;
        if (level == 0 && last_level == 0) {
            // coarse-grid interpolation when there is no refinement (:2362-2396)
            const int G = g.G, bu = best % G, bv = best / G;
            auto at = [&](int u, int v) -> float {
                const int uu = bu + u, vv = bv + v;
                return (uu < 0 || uu >= G || vv < 0 || vv >= G) ? 0.0f : P[vv * G + uu];
            };
            quadratic_interp(P[best], at(1, 0), at(-1, 0), at(0, 1), at(0, -1), &du, &dv);
            const float step_l = G == 1 ? 0.0f : (2.0f * g.fov_l) / (float)(G - 1);
            const float step_m = G == 1 ? 0.0f : (2.0f * g.fov_m) / (float)(G - 1);
            clamp_direction(c[0] + du * step_l, c[1] + dv * step_m, c);
        } else if (level > 0) {
            quadratic_interp(P[4], P[5], P[3], P[7], P[1], &du, &dv);
            float hl = g.fov_l / (float)g.G, hm = g.fov_m / (float)g.G;
            for (int k = 0; k < level; ++k) {
                hl *= 0.5f;
                hm *= 0.5f;
            }
            clamp_direction(c[0] + du * hl, c[1] + dv * hm, c);
        }
    }
    s.centre[0] = c[0];
    s.centre[1] = c[1];
    s.centre[2] = c[2];
    if (level == last_level) {
        s.prev[0] = c[0];
        s.prev[1] = c[1];
        s.prev[2] = c[2];
        if (blockIdx.x == 0 && blockIdx.y == 0)
            for (int i = 0; i < 3; ++i) a.dirs[3 * a.before_window + i] = c[i];
    }
    *out = s;
    if (blockIdx.x == 0 && blockIdx.y == 0) *a.next = s;
}

// Grid (channel groups, tiles of 16 cells).  A workgroup's eight waves take
// eight channels; with HALVES (the nine refinement cells, where the time of
// one wave is what counts) four, and each wave two of the four block rows:
// {0, 3} or {1, 2}, 72 MFMAs either way.  A launch without cells only takes the
// decision on the one before.
template <bool CAPON, bool HALVES>
__global__ __launch_bounds__(kScanThreads) void opt_scan_kernel(ScanArgs a) {
    constexpr int kChannels = HALVES ? kScanWaves / 2 : kScanWaves;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ double s_sums[kScanThreads];
    __shared__ double s_pos[3 * 64];
    __shared__ double s_form[kScanWaves][16];
    __shared__ OptSearch s_search;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int f0 = blockIdx.x * kChannels;
    const int f = f0 + (HALVES ? wave >> 1 : wave);
    for (int i = tid; i < 3 * 64; i += kScanThreads)
        s_pos[i] = i < 3 * a.g.M ? (double)a.pos[i] : 0.0;
    if (a.before_part != nullptr) {
        decide(a, reinterpret_cast<float*>(smem), s_sums, &s_search);
    } else if (tid == 0) {
        s_search = *a.search;
        if (blockIdx.x == 0 && blockIdx.y == 0) *a.next = s_search;
    }
    __syncthreads();
    if (a.n_cells == 0) return;
    float dir[3];
    double st[3];
    const int cell = min((int)blockIdx.y * 16 + (lane & 15), a.n_cells - 1);
    cell_direction(a.g, s_search, a.level, cell, dir, st);
    if (f < a.F) {
        const double per_metre = turns_per_metre(a.freqs[f]);
        const double d[3] = {st[0] * per_metre, st[1] * per_metre, st[2] * per_metre};
        const char* const op = a.operand + (size_t)f * a.operand_bytes;
        const unsigned rows = HALVES ? ((wave & 1) ? 0x6u : 0x9u) : 0xFu;
        double form;
        if (CAPON && a.mode[f] == 1)
            form = scan_form<double>(reinterpret_cast<const double*>(op), a.Mp, s_pos, d, rows,
                                     lane);
        else
            form = (double)scan_form<float>(reinterpret_cast<const float*>(op), a.Mp, s_pos, d,
                                            rows, lane);
        form += __shfl_xor(form, 16);
        form += __shfl_xor(form, 32);
        if (lane < 16) s_form[wave][lane] = form;
    }
    __syncthreads();
    if (tid < 16) {
        double sum = 0.0;
        for (int i = 0; i < kChannels && f0 + i < a.F; ++i) {
            const double form = HALVES ? s_form[2 * i][tid] + s_form[2 * i + 1][tid]
                                       : s_form[i][tid];
            const double q = a.trace[f0 + i] + 2.0 * form;
            float p;
            if (CAPON && a.mode[f0 + i] == 1)
                p = q > 1.0e-12 ? (float)(1.0 / q) : 0.0f;
            else
                p = (float)q;
            if (!isfinite(p)) p = 0.0f;
            sum += (double)p;
        }
        a.part[((size_t)blockIdx.x * gridDim.y + blockIdx.y) * 16 + tid] = sum;
    }
}

}  // namespace

size_t opt_operand_bytes(size_t M, bool capon) {
    const size_t Mp = 16 * ceil_div(M, 16);
    return 2 * Mp * Mp * (capon ? sizeof(double) : sizeof(float));
}

size_t opt_part_count(size_t F, size_t n_cells) {
    return 16 * ceil_div(n_cells, 16) * ceil_div(F, kScanWaves / 2);
}

void launch_opt_fold(hipStream_t stream, const OptWindows& b, const int* rs, double* state,
                     bool first, size_t F, size_t M, size_t K, size_t K_last, size_t L, bool fb,
                     bool capon, float load, float lambda) {
    FoldArgs a{};
    a.rs = reinterpret_cast<const int2*>(rs);
    a.state = reinterpret_cast<double2*>(state);
    a.operand = b.operand;
    a.trace = b.trace;
    a.mode = b.mode;
    a.operand_bytes = opt_operand_bytes(M, capon);
    a.n = (int)b.n;
    a.first = first ? 1 : 0;
    a.M = (int)M;
    a.Mp = 16 * (int)ceil_div(M, 16);
    a.K = (int)K;
    a.K_last = (int)K_last;
    a.L = (int)L;
    a.fb = fb ? 1 : 0;
    a.capon = capon ? 1 : 0;
    a.load = load;
    a.lambda = lambda;
    hipLaunchKernelGGL(opt_fold_kernel, dim3((unsigned)F), dim3(kFoldThreads), 0, stream, a);
    hip_check(hipGetLastError(), "opt_fold_kernel launch");
    if (!capon) return;
    hipLaunchKernelGGL(opt_factor_kernel, dim3((unsigned)F, (unsigned)b.n), dim3(kFactorThreads),
                       0, stream, b.operand, a.operand_bytes, a.M, a.Mp, b.trace, b.mode);
    hip_check(hipGetLastError(), "opt_factor_kernel launch");
}

void launch_opt_scan(hipStream_t stream, OptScan& q, const OptWindows& b, size_t index,
                     const float* pos, const float* freqs, const OptGridArgs& g, int level,
                     int last_level, size_t window, size_t F, size_t n_cells, bool capon,
                     float* dirs) {
    ScanArgs a{};
    a.operand_bytes = opt_operand_bytes((size_t)g.M, capon);
    a.operand = b.operand + index * F * a.operand_bytes;
    a.trace = b.trace + index * F;
    a.mode = b.mode + index * F;
    a.pos = pos;
    a.freqs = freqs;
    a.g = g;
    a.level = level;
    a.n_cells = (int)n_cells;
    a.F = (int)F;
    a.Mp = 16 * (int)ceil_div((size_t)g.M, 16);
    a.last_level = last_level;
    const unsigned now = q.launches & 1u;
    a.part = q.part[now];
    a.search = q.state + now;
    a.next = q.state + (now ^ 1u);
    a.dirs = dirs;
    if (q.launches > 0) {
        a.before_part = q.part[now ^ 1u];
        a.before_level = q.level;
        a.before_cells = (int)q.cells;
        a.before_groups = (int)q.groups;
        a.before_window = (int)q.window;
    }
    // one tile cannot fill the chip: half the work per wave
    const size_t tiles = ceil_div(n_cells, 16);
    const bool halves = tiles <= 1;
    const size_t groups = n_cells == 0 ? 1 : ceil_div(F, halves ? kScanWaves / 2 : kScanWaves);
    const dim3 grid((unsigned)groups, (unsigned)std::max<size_t>(tiles, 1));
    const size_t smem = std::max<size_t>(q.cells, 1) * sizeof(float);
#define BF_SCAN(C_, H_) \
    hipLaunchKernelGGL((opt_scan_kernel<C_, H_>), grid, dim3(kScanThreads), smem, stream, a)
    if (capon && halves)
        BF_SCAN(true, true);
    else if (capon)
        BF_SCAN(true, false);
    else if (halves)
        BF_SCAN(false, true);
    else
        BF_SCAN(false, false);
#undef BF_SCAN
    hip_check(hipGetLastError(), "opt_scan_kernel launch");
    ++q.launches;
    q.level = level;
    q.cells = n_cells;
    q.groups = groups;
    q.window = window;
}

}  // namespace bfhip
