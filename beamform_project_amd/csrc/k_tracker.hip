// k_tracker.hip -- dynamic beam tracker for gfx950: the one-beam stream
// kernel, the streaming server's kernels and the dispatch.  The multi-beam
// body is in tracker_wave.hpp (instantiated per antenna count in
// k_tracker_a*.hip), geometry and steering weights in steering.hpp.
//
// The tracker files are compiled without FMA contraction so that the
// direction (float) arithmetic rounds exactly like the reference's ISO C++
// build; sums use explicit fma.
#include <algorithm>

#include "bf_serve.hpp"
#include "tracker_wave.hpp"

namespace bfhip {
namespace {

using namespace wave_detail;

// ------------------------------------------------------------ serving loop
// Plan: one thread per request slot reads the step's head, finds the
// windows from the slot's cursor whose last spectrum is at or before the
// head (a slot admitted with a start behind the previous head gets all its
// windows held by the ring at once) and the work they make; block scans
// turn the counts into offsets.  Each thread advances only its own slot's
// cursor; the step's head is recorded as the processed head.
__global__ __launch_bounds__(kServeMaxSlots) void serve_plan_kernel(
    ServeSlot* __restrict__ slots, ServeCtrl* __restrict__ ctrl,
    ServeWork* __restrict__ work, const long long* heads, int F) {
    __shared__ int scan[kServeMaxSlots];
    const int s = threadIdx.x;
    const long long step = ctrl->step;
    // system-scope load: the host wrote this entry just before the launch
    const long long H = __hip_atomic_load(heads + (step & (kServeHeadRing - 1)),
                                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    ServeSlot& sl = slots[s];
    int n_win = 0;
    int w_lo = 0;
    int n_tasks = 0;
    if (sl.active) {
        const long long S = sl.S;
        const long long t0 = sl.t0;
        const long long te = sl.t_end;
        const long long W = (te - t0 + S - 1) / S;
        // windows from the slot's cursor up to the last one ending at or
        // before H (the last window may be partial and end at te)
        const long long lo = sl.w_next;
        const long long h = H >= te ? W : (H < t0 ? 0 : (H - t0) / S);
        const long long hi = h > lo ? h : lo;
        sl.w_next = hi;
        if (hi > lo) {
            n_win = (int)(hi - lo);
            w_lo = (int)lo;
            n_tasks = F * ((sl.B + kServeTaskBeams - 1) / kServeTaskBeams) *
                      ((n_win + sl.wpi - 1) / sl.wpi);
        }
    }
    scan[s] = n_tasks;
    __syncthreads();
    for (int d = 1; d < kServeMaxSlots; d <<= 1) {
        const int v = s >= d ? scan[s - d] : 0;
        __syncthreads();
        scan[s] += v;
        __syncthreads();
    }
    work->off[s] = scan[s] - n_tasks;
    work->w_lo[s] = w_lo;
    work->n_win[s] = n_win;
    if (s == kServeMaxSlots - 1) {
        work->off[kServeMaxSlots] = scan[s];
        ctrl->processed = H;
        ctrl->step = step + 1;
    }
}

// Last slot s with off[s] <= i (off non-decreasing, off[0] = 0 <= i < off[n]).
__device__ __forceinline__ int owner_slot(const int* off, int i) {
    int lo = 0;
    int hi = kServeMaxSlots;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= i)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// The step's wave tasks (run of windows, block of beams, channel), dealt out
// to a persistent grid.  A task is the multi-beam tracker's own body, so
// results are bit-identical to it.  Two workgroups per CU (the persistent
// grid) need at most 256 registers.
template <int A, int PARTS, bool MASKED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void serve_tasks_kernel(
    const uint8_t* __restrict__ ring, const uint8_t* __restrict__ valid, long long ring_mask,
    int F, Geom geo, const ServeSlot* __restrict__ slots, const ServeWork* __restrict__ work) {
    __shared__ int off[kServeMaxSlots + 1];
    __shared__ Positions<A> pos;
    for (int i = threadIdx.x; i <= kServeMaxSlots; i += kThreads) off[i] = work->off[i];
    stage_positions<A>(geo, pos);
    __syncthreads();
    const int n_tasks = off[kServeMaxSlots];
    // XCD-aware order: blockIdx.x % 8 names the XCD; consecutive tasks
    // (blocks of one channel, neighbouring channels) go to one XCD.
    const int lin = gridDim.x % kXcds == 0
                        ? (int)(blockIdx.x % kXcds) * (int)(gridDim.x / kXcds) + (int)(blockIdx.x / kXcds)
                        : (int)blockIdx.x;
    Channel<A> ch{pos, {0.0f, 0.0f, 0.0f}, 0.0};
    geometry_reach<A>(geo, threadIdx.x & (kWaveSize - 1), ch.reach);
    const int first =
        __builtin_amdgcn_readfirstlane(lin * kWaves + (int)(threadIdx.x / kWaveSize));
    for (int task = first; task < n_tasks; task += gridDim.x * kWaves) {
        const int sidx = __builtin_amdgcn_readfirstlane(owner_slot(off, task));
        const ServeSlot* sl = slots + sidx;
        const int local = task - __builtin_amdgcn_readfirstlane(off[sidx]);
        const int blocks = (sl->B + kServeTaskBeams - 1) / kServeTaskBeams;
        const int block = local % blocks;
        const int rest = local / blocks;
        const int f = rest % F;
        const int w_first = work->w_lo[sidx];
        const int w_last = w_first + work->n_win[sidx];
        const int w_begin = w_first + rest / F * sl->wpi;
        const int w_end = w_begin + sl->wpi < w_last ? w_begin + sl->wpi : w_last;
        const DirArgs da{nullptr, &sl->traj[0][0], {}, 0L, sl->S, sl->B};
        const RowSource rs{ring + (size_t)f * A, (unsigned)(F * A), (long)ring_mask,
                           (long)sl->t0, (long)sl->t_end, MASKED ? valid + f : nullptr,
                           (size_t)F};
        const OutTarget ot{sl->out, (long)sl->out_windows, F, f};
        ch.per_metre = turns_per_metre(channel_frequency(geo, f));
        // masked long windows in a body of their own, with their loads ahead (8
        // requests of 64 beams, windows of 320, 64 antennas: 141 -> 108 us a step)
        if (MASKED && sl->S >= kDirectWeightMinSpectra)
            wave_windows<A, kServeTaskBeams / 8, PARTS, true, false, MASKED>(
                rs, ch, da, ot, w_begin, w_end, block * kServeTaskBeams);
        else
            wave_windows<A, kServeTaskBeams / 8, PARTS, true, true, MASKED>(
                rs, ch, da, ot, w_begin, w_end, block * kServeTaskBeams);
    }
}

// Single-beam per-spectrum tracker as an HBM stream (FP32 VALU).  Every
// lane holds 32 antennas of one channel, LPC = A / 32 lanes per channel,
// so a wave covers 64 / LPC adjacent channels and reads, per spectrum, one
// contiguous 2 KB run of packed rows (two 16-byte loads per lane, with the
// next kB1Depth - 1 spectra in flight while one is summed).  A unit is (window,
// channel group, time chunk); its weights (steering.hpp) stay in 64 registers for the whole chunk.  The complex sum runs
// over the lane's antennas in order in two interleaved accumulator pairs,
// then across the LPC lanes of the channel by xor shuffles.
constexpr int kB1WavesPerBlock = 4;
constexpr int kB1Depth = 4;  // spectra in flight per lane

template <int A>
__global__ __launch_bounds__(kB1WavesPerBlock * 64) void beam1_stream_kernel(
    const uint8_t* __restrict__ x, float* __restrict__ out, int T, int F, int S, int n_windows,
    int groups, int chunks, Geom geo, DirArgs da) {
#pragma clang fp contract(off)
    constexpr int LPC = A / 32;
    constexpr int CPW = 64 / LPC;  // channels per wave
    const int lane = threadIdx.x & 63;
    const long unit = (long)blockIdx.x * kB1WavesPerBlock + (threadIdx.x >> 6);
    if (unit >= (long)n_windows * groups * chunks) return;  // whole waves
    const int c = (int)(unit % chunks);
    const long r = unit / chunks;
    const int g = (int)(r % groups);
    const int w = (int)(r / groups);
    const int f = g * CPW + lane / LPC;
    const int part = lane % LPC;  // antennas 32 part .. 32 part + 31
    const bool live = f < F;
    const int fl = live ? f : F - 1;  // loads stay in bounds; nothing is stored
    const int tw0 = w * S;
    const int tw1 = min(tw0 + S, T);
    const int per = (tw1 - tw0 + chunks - 1) / chunks;
    const int t0 = min(tw0 + c * per, tw1);
    const int t1 = min(t0 + per, tw1);
    float d[3];
    beam_direction(da, beam_row(da, 0), w, 0, d);
    float reach[3];
    geometry_reach<A>(geo, lane, reach);
    const Steer st = make_steer(d, turns_per_metre(channel_frequency(geo, fl)), reach);
    float wr[32], wi[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        float p[3];
        antenna_position(geo, 32 * part + j, p);
        const double pd[3] = {(double)p[0], (double)p[1], (double)p[2]};
        const float2 v = steering_weight_any(pd, st);
        wr[j] = v.x;
        wi[j] = v.y;
    }
    const uint8_t* base = x + (size_t)fl * A + 32 * part;
    const size_t row = (size_t)F * A;
    // a ring of kB1Depth spectra in flight: slot u holds spectrum tb + u and
    // is refilled with spectrum tb + u + kB1Depth once it has been summed
    uint4 ring[kB1Depth][2];
#pragma unroll
    for (int u = 0; u < kB1Depth; ++u)
        if (t0 + u < t1) {
            const uint4* q = reinterpret_cast<const uint4*>(base + (size_t)(t0 + u) * row);
            ring[u][0] = q[0];
            ring[u][1] = q[1];
        }
    for (int tb = t0; tb < t1; tb += kB1Depth) {
#pragma unroll
        for (int u = 0; u < kB1Depth; ++u) {
            const int t = tb + u;
            if (t >= t1) break;  // uniform
            float re[2] = {0.0f, 0.0f}, im[2] = {0.0f, 0.0f};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const unsigned wd[4] = {ring[u][h].x, ring[u][h].y, ring[u][h].z, ring[u][h].w};
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int j = 16 * h + q;
                    const int byte = (int)((wd[q >> 2] >> (8 * (q & 3))) & 0xFFu);
                    const float xr = (float)((byte << 28) >> 28);
                    const float xi = (float)((byte << 24) >> 28);
                    const int e = q & 1;
                    re[e] = fmaf(wr[j], xr, re[e]);
                    re[e] = fmaf(-wi[j], xi, re[e]);
                    im[e] = fmaf(wr[j], xi, im[e]);
                    im[e] = fmaf(wi[j], xr, im[e]);
                }
            }
            if (t + kB1Depth < t1) {
                const uint4* q = reinterpret_cast<const uint4*>(base + (size_t)(t + kB1Depth) * row);
                ring[u][0] = q[0];
                ring[u][1] = q[1];
            }
            float sr = re[0] + re[1], si = im[0] + im[1];
#pragma unroll
            for (int o = 1; o < LPC; o <<= 1) {
                sr += __shfl_xor(sr, o);
                si += __shfl_xor(si, o);
            }
            if (live && part == 0) out[(size_t)t * F + f] = sr * sr + si * si;
        }
    }
}

// Units (window, channel group, time chunk) for about four waves per SIMD,
// chunks of at least 8 spectra.
void launch_beam1_stream(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da) {
    const size_t cpw = 64 / (L.A / 32);
    const size_t groups = ceil_div(L.F, cpw);
    const size_t target = 4096;
    size_t chunks = std::max<size_t>(1, ceil_div(target, L.n_windows * groups));
    chunks = std::min(chunks, std::max<size_t>(1, L.S / 8));
    const size_t n_units = L.n_windows * groups * chunks;
    const size_t blocks = ceil_div(n_units, kB1WavesPerBlock);
    if (blocks > (size_t)UINT32_MAX) fail(BF_ERR_OVERFLOW, "tracker grid exceeds the supported size");
#define BF_B1(A_)                                                                              \
    hipLaunchKernelGGL((beam1_stream_kernel<A_>), dim3((unsigned)blocks),               \
                       dim3(kB1WavesPerBlock * 64), 0, stream, L.x, L.out, (int)L.T, (int)L.F, \
                       (int)L.S, (int)L.n_windows, (int)groups, (int)chunks, L.geo, da)
    switch (L.A) {
    case 32: BF_B1(32); break;
    case 64: BF_B1(64); break;
    case 128: BF_B1(128); break;
    case 256: BF_B1(256); break;
    default: invalid("n_ant must be 32, 64, 128, or 256");
    }
#undef BF_B1
}

}  // namespace

void launch_tracker(hipStream_t stream, const TrackerLaunch& L) {
    if (L.T == 0 || L.F == 0 || L.B == 0 || L.S == 0 || L.n_windows == 0) return;
    if (L.T > (size_t)INT32_MAX / 2 || L.S > (size_t)INT32_MAX / 2 || L.F > 65535 ||
        L.n_windows > (size_t)INT32_MAX / 2)
        fail(BF_ERR_OVERFLOW, "tracker grid exceeds the supported size");
    const bool table = L.dir_source == kDirTable;
    const float* const q = L.trajectory;
    const DirArgs da{table ? L.dir_table : nullptr, table ? nullptr : L.trajectories,
                     {q[0], q[1], q[2], q[3]}, table ? 0L : (long)L.window_offset, (int)L.S,
                     (int)L.B};
    if (!table && L.trajectories == nullptr && L.B != 1)
        invalid("a trajectory by value is for one beam");
    // One beam, per-spectrum output: the FP32 stream kernel (AUTO and FP32).
    if (L.B == 1 && !L.integrate &&
        (L.kernel == BF_KERNEL_AUTO || L.kernel == BF_KERNEL_FP32)) {
        launch_beam1_stream(stream, L, da);
    } else {
        const int parts = L.kernel == BF_KERNEL_F16 ? 1 : (L.kernel == BF_KERNEL_FP32 ? 3 : 2);
        switch (L.A) {
        case 32: launch_tracker_a32(stream, L, da, parts); break;
        case 64: launch_tracker_a64(stream, L, da, parts); break;
        case 128: launch_tracker_a128(stream, L, da, parts); break;
        case 256: launch_tracker_a256(stream, L, da, parts); break;
        default: invalid("n_ant must be 32, 64, 128, or 256");
        }
    }
    hip_check(hipGetLastError(), "tracker kernel launch");
}

void launch_serve_step(hipStream_t stream, const ServeLaunch& L) {
    hipLaunchKernelGGL(serve_plan_kernel, dim3(1), dim3(kServeMaxSlots), 0, stream, L.slots,
                       L.ctrl, L.work, L.heads, (int)L.F);
#define BF_SERVE(A_, SPLIT_)                                                                  \
    do {                                                                                      \
        if (L.valid != nullptr)                                                               \
            hipLaunchKernelGGL((serve_tasks_kernel<A_, SPLIT_ ? 2 : 1, true>), dim3((unsigned)L.grid), \
                               dim3(kThreads), 0, stream, L.ring, L.valid, L.ring_mask,       \
                               (int)L.F, L.geo, L.slots, L.work);                             \
        else                                                                                  \
            hipLaunchKernelGGL((serve_tasks_kernel<A_, SPLIT_ ? 2 : 1, false>),                       \
                               dim3((unsigned)L.grid), dim3(kThreads), 0, stream, L.ring,     \
                               L.valid, L.ring_mask, (int)L.F, L.geo, L.slots, L.work);       \
    } while (0)
    if (L.A == 32 && L.split)
        BF_SERVE(32, true);
    else if (L.A == 32)
        BF_SERVE(32, false);
    else if (L.A == 64 && L.split)
        BF_SERVE(64, true);
    else if (L.A == 64)
        BF_SERVE(64, false);
    else
        invalid("the serving loop supports 32 or 64 antennas");
#undef BF_SERVE
    hip_check(hipGetLastError(), "serve step launch");
}

}  // namespace bfhip
