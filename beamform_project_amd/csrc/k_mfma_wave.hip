// k_mfma_wave.hip -- the fixed-grid beamformer for 256 antennas and windows of
// a multiple of 64 spectra: one wave, 8 beams, no LDS.
//
// Staged through LDS (mfma_fused.hpp), 256 antennas leave registers for 8
// beams per wave, so every wave reads all of every tile: 16 KB of LDS per 32
// MFMAs, at four waves the whole LDS bandwidth, and beams past the last of a
// 32-beam group idle while their group stages.  Here each wave loads its own
// MFMA operand (the scheme of tracker_wave.hpp: a lane's operand of a tile is
// 64 contiguous packed bytes of one row) and converts it in registers beside
// the MFMAs, 9 instructions per two; the waves of a workgroup take
// neighbouring blocks of 8 beams of one channel and share the rows in cache.
// A = 256, T = 4100, B = 45, S = 320: 383 -> 336 us, 0.38 PFLOP/s
// counted once, bound by instruction issue.
#include "mfma_fused.hpp"
#include "tracker_wave.hpp"

namespace bfhip {
namespace {

using namespace wave_detail;

constexpr int kA = 256;
constexpr int kSteps = kA / 16;

// The 8 beams' weights as the B operand (element order of tracker_wave.hpp).
template <int PARTS>
__device__ __forceinline__ void load_block_weights(const float2* __restrict__ w, int F, int B,
                                                   int f, int beam0, int lane,
                                                   bf_uint4v (&bw)[PARTS][kSteps]) {
    const int c = lane & 15;
    const bool odd = (c & 1) != 0;
    // columns past the last beam repeat it; they are not stored
    const int b = min(beam0 + (c >> 1), B - 1);
    const float2* const p = w + ((size_t)b * F + f) * kA + (lane >> 4) * (kA / 4);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        float2 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = p[4 * s + j];
        // Re column (wr, -wi), Im column (wi, wr)
        unsigned e[4][PARTS];
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // antennas h, h + 2
            const float2 a = v[h], z = v[h + 2];
            slice_pair<PARTS>(odd ? a.y : a.x, odd ? z.y : z.x, e[2 * h]);
            slice_pair<PARTS>(odd ? a.x : -a.y, odd ? z.x : -z.y, e[2 * h + 1]);
        }
#pragma unroll
        for (int q = 0; q < PARTS; ++q)
            bw[q][s] = bf_uint4v{e[0][q], e[1][q], e[2][q], e[3][q]};
    }
}

// One tile in flight.  With a loss mask the row's byte travels beside its
// voltages and clears them where they are used, so that neither load waits for
// the other.
template <bool MASKED>
struct Tile {
    TileBytes<kA> bytes;
};
template <>
struct Tile<true> {
    TileBytes<kA> bytes;
    uint8_t valid;
};

// Windows [w_begin, w_end) of one channel for 8 beams per wave.
template <int PARTS, bool MASKED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void frame_wave_kernel(const uint8_t* __restrict__ x, const float2* __restrict__ w,
                       float* __restrict__ out, const uint8_t* __restrict__ mask, int T, int F,
                       int B, int S, int W, int run, int blocks, long n_tasks, int per_xcd) {
    const long group = (long)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    const long task = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWaveSize)) +
                      group * kWaves;
    if (task >= n_tasks) return;  // whole wave; no barriers
    const int block = (int)(task % blocks);
    const long rest = task / blocks;
    const int f = (int)(rest % F);
    const int w_begin = (int)(rest / F) * run;
    const int w_end = w_begin + run < W ? w_begin + run : W;
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int col = lane & 15;
    const int G = lane >> 4;
    const int beam0 = block * 8;
    bf_uint4v bw[PARTS][kSteps];
    load_block_weights<PARTS>(w, F, B, f, beam0, lane, bw);

    const unsigned row_stride = (unsigned)(F * kA);
    const unsigned lane_off = (unsigned)col * row_stride + (unsigned)(G * (kA / 4));
    const uint8_t* const x_f = x + (size_t)f * kA;
    const int tile_begin = w_begin * (S >> 4);
    const int tile_last = min(w_end * (S >> 4), (T + 15) >> 4);  // exclusive
    const int per_window = S >> 4;
    // Tile i: rows 16 i .. 16 i + 15; rows at or after T read as zero.
    auto load_tile = [&](int i) -> Tile<MASKED> {
        const uint8_t* const p = x_f + (size_t)i * 16 * row_stride;
        const int t = 16 * i + col;
        Tile<MASKED> r;
        if constexpr (MASKED) r.valid = t < T ? mask[(size_t)t * F + f] : 0;
        if (16 * (i + 1) <= T) {
            r.bytes = load_bytes<kA>(p + lane_off);
            return r;
        }
#pragma unroll
        for (int s = 0; s < kSteps; ++s) r.bytes.w[s] = 0u;
        if (t < T) r.bytes = load_bytes<kA>(p + lane_off);
        return r;
    };
    float win = 0.0f;
    auto use_tile = [&](const Tile<MASKED>& t) {
        unsigned keep = ~0u;
        if constexpr (MASKED) keep = t.valid != 0 ? ~0u : 0u;
        bf_float4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const bf_uint4v av = int4_slots<PARTS>(t.bytes.w[s] & keep);
            // large and small slices in sums of their own: two chains
#pragma unroll
            for (int q = 0; q < PARTS; ++q) acc[q] = mfma<PARTS>(av, bw[q][s], acc[q]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float y = PARTS == 2 ? acc[0][r] + acc[1][r] : acc[0][r];
            win = fmaf(y, y, win);
        }
    };
    auto close = [&](int i) {  // after tile i
        if ((i + 1) % per_window != 0 && i + 1 != tile_last) return;  // uniform
        float v = win;
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        v += dpp_swap_pairs(v);
        const int b = beam0 + (col >> 1);
        if (G == 0 && (col & 1) == 0 && b < B)
            out[((size_t)(i / per_window) * F + f) * B + b] = v;
        win = 0.0f;
    };
    // two tiles in flight; a window is a multiple of four tiles, so only the
    // run's end can be odd
    Tile<MASKED> buf[2];
    buf[0] = load_tile(tile_begin);
    if (tile_begin + 1 < tile_last) buf[1] = load_tile(tile_begin + 1);
#pragma unroll 1
    for (int i = tile_begin; i < tile_last; i += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (i + u >= tile_last) break;
            use_tile(buf[u]);
            if (i + u + 2 < tile_last) buf[u] = load_tile(i + u + 2);
            close(i + u);
        }
    }
}

template <int PARTS>
void launch_parts(hipStream_t stream, const MfmaLaunch& L, int resident) {
    const int W = (int)ceil_div((size_t)L.T, (size_t)L.S);
    const size_t blocks = ceil_div((size_t)L.B, 8);
    // windows per task: the weights of one (16 KB) are worth reading once for
    // several, as long as three rounds of the resident waves remain
    const size_t all = (size_t)W * L.F * blocks;
    const size_t run =
        std::max<size_t>(1, std::min<size_t>(16, all / (3 * kWaves * (size_t)resident)));
    const size_t n_tasks = ceil_div((size_t)W, run) * L.F * blocks;
    const size_t per_xcd = ceil_div(ceil_div(n_tasks, kWaves), kXcds);
    if (per_xcd * kXcds > (size_t)INT32_MAX)
        fail(BF_ERR_OVERFLOW, "MFMA beamformer grid exceeds the supported size");
#define BF_LAUNCH(MASKED_)                                                                     \
    hipLaunchKernelGGL((frame_wave_kernel<PARTS, MASKED_>), dim3((unsigned)(per_xcd * kXcds)), \
                       dim3(kThreads), 0, stream, L.x, reinterpret_cast<const float2*>(L.w),   \
                       L.out, L.mask, L.T, L.F, L.B, L.S, W, (int)run, (int)blocks,            \
                       (long)n_tasks, (int)per_xcd)
    if (L.mask != nullptr)
        BF_LAUNCH(true);
    else
        BF_LAUNCH(false);
#undef BF_LAUNCH
}

}  // namespace

// Up to six blocks: with more, a channel's blocks no longer run together, the
// rows are read again from HBM, and sharing them through LDS pays (T = 4096, S =
// 320: B = 48 438 us staged, 362 here; B = 64 452, 442; B = 96 577, 687).  A mask
// changes nothing in that, so that a masked frame sums as the plain one does
// (T = 4100, B = 45, S = 320, masked: 766 us staged, 406 here).
bool frame_wave_supported(const MfmaLaunch& L, int A) {
    return A == kA && L.S > 0 && L.S % 64 == 0 && L.B <= 48 && L.parts <= 2 && !L.tiled;
}

void launch_frame_wave(hipStream_t stream, const MfmaLaunch& L, int resident) {
    if (L.parts == 2)
        launch_parts<2>(stream, L, resident);
    else
        launch_parts<1>(stream, L, resident);
}

}  // namespace bfhip
