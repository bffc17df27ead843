// mfma_fused.hpp -- FP16-MFMA fused fixed-grid beamformer for gfx950
// (kernel template; instantiated per antenna count in k_mfma_a*.hip).
//
// Per frequency f the contraction y[t][b] = sum_a W[b][f][a] * X[t][f][a]
// (reference src/cpu_beamformer.cpp:56-78, no conjugate) is a real GEMM
//   [xr0 xi0 xr1 xi1 ...] (1 x 2A)  *  B (2A x 2B),
// where output column 2b holds Re(y_b) (weights (wr, -wi) per antenna) and
// column 2b+1 holds Im(y_b) (weights (wi, wr)).  int4 samples are exact in
// FP16 (and in bfloat16), so the only rounding in the products comes from
// the weights, which are held in PARTS slices: one fp16; hi = fp16(w) plus
// lo = fp16(w - hi), ~22 significant bits; or three bfloat16, the float
// itself.  The K loop runs over every slice with the same A operand
// (products are exact in the FP32 accumulator).
//
// Instruction: v_mfma_f32_16x16x32_f16.  A workgroup of WV waves owns one
// frequency, one chunk of time and WV*NT*8 beams; each wave keeps the
// weights of NT N-tiles (8 beams each, re/im interleaved) in VGPRs for the
// whole chunk.  The packed int4 rows of a stage (ST tiles of 16 spectra)
// are loaded once per workgroup with coalesced dword loads, converted to
// FP16 pairs (byte permute, xor, one packed subtraction) and written to LDS
// in the MFMA A-operand layout, so each lane reads its operand with one
// 16-byte LDS load per k-step.  Every staging address is a per-thread
// constant plus a wave-uniform (scalar) stage offset.  The next stage's
// global loads are in flight while the current stage is computed.  With
// DB the LDS holds two stages and the conversion and stores of the next
// stage, and the loads of the one after, are spread over the tiles of the
// current stage, inside the same (fully unrolled) block as its MFMAs, so
// this VALU work issues between MFMAs; a stage costs one barrier.  The
// window bookkeeping of a tile is static in the unrolled stage, and the
// two lanes of a re/im pair split each window's stores.
//
// Output layout of a 16x16 MFMA: lane l holds column l%16 for rows
// 4*(l/16)+r, r = 0..3.  Tile rows are mapped to time so that row group
// G = l/16 of a super-tile covers consecutive spectra: each lane then
// accumulates whole integration windows in registers.
//   MODE 0 (no integration): tile i, row 4G+r -> t = 16i + 4G + r
//   MODE 1 (S == 10): super-tile of 5 tiles, G covers 20 spectra (2 windows)
//   MODE 2 (S % 4 == 0): super-tile of S/4 tiles, G covers one window
//   MODE 3 (S % 64 == 0, few windows): tiles as in MODE 0; the row groups
//     share every window and are folded by two shuffles where it closes.
//     Windows are this long that a stage of 4 tiles lies inside one, and the
//     work is whole windows, not groups of four
// Re and im of a beam sit in adjacent lanes; a quad-permute DPP adds the
// two squared sums.
#pragma once

#include <algorithm>
#include <type_traits>

#include "bf_kernels.hpp"
#include "mfma_stage.hpp"

namespace bfhip {

struct MfmaLaunch {
    const uint8_t* x = nullptr;
    const float* w = nullptr;
    float* out = nullptr;
    const uint8_t* mask = nullptr;  // [T][F] frame validity (0 = lost), or null
    int T = 0, F = 0, B = 0, S = 0;
    int parts = 2;       // weight slices: 1 fp16, 2 fp16 hi + lo, 3 bfloat16 (the float itself)
    bool tiled = false;  // weights [F][B/32][A][32] instead of [B][F][A]
    // windows of a multiple of 64 spectra one after another, not four side by
    // side: these sum in another order, so this follows from the problem alone
    // (windows_one_by_one), never from a tile shape or a mask
    bool one_by_one = false;
};

// Launch the kernel of `cfg` for one antenna count; false when `cfg` is
// not an instantiated shape (k_mfma_a32/64/128/256.hip).
bool launch_mfma_a32(hipStream_t stream, const MfmaLaunch& L, const MfmaConfig& cfg);
bool launch_mfma_a64(hipStream_t stream, const MfmaLaunch& L, const MfmaConfig& cfg);
bool launch_mfma_a128(hipStream_t stream, const MfmaLaunch& L, const MfmaConfig& cfg);
bool launch_mfma_a256(hipStream_t stream, const MfmaLaunch& L, const MfmaConfig& cfg);

namespace mfma_detail {

constexpr int kWaveSize = 64;
constexpr int kXcds = 8;

__device__ __forceinline__ float dpp_swap_pairs(float v) {
    // quad_perm [1,0,3,2]: lane i <- lane i^1.
    return __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}

// PARTS names how a weight reaches the matrix unit: 1 = fp16(w); 2 = fp16
// hi + lo, about 22 bits; 3 = three bfloat16 slices of 8 bits each, which
// together are the float weight itself (bfloat16 has float's exponent), so
// every product with an int4 sample is exact and only the FP32 accumulation
// rounds.
template <int PARTS>
__device__ __forceinline__ bf_float4 mfma_16x16x32(bf_half8 a, bf_half8 b, bf_float4 c) {
    if constexpr (PARTS == 3)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf_bfloat8, a),
                                                       __builtin_bit_cast(bf_bfloat8, b), c, 0, 0,
                                                       0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The three bfloat16 slices of the weight component e, as the 16 bits of
// their operand elements: cut off, not rounded, 8 + 8 + 8 bits hold all 24 of
// a float.  Infinities and NaN stay whole in slice 0.
__device__ __forceinline__ void weight_slices(float e, _Float16 (&out)[3]) {
    auto top = [](float v) { return __builtin_bit_cast(unsigned, v) & 0xFFFF0000u; };
    auto bits = [](unsigned u) { return __builtin_bit_cast(_Float16, (unsigned short)(u >> 16)); };
    unsigned h = top(e);
    float r = e - __builtin_bit_cast(float, h);
    if (!isfinite(e)) {
        r = 0.0f;
        if (isnan(e)) h |= 0x00400000u;  // a NaN of low payload bits only stays a NaN
    }
    const unsigned m = top(r);
    out[0] = bits(h);
    out[1] = bits(m);
    out[2] = bits(top(r - __builtin_bit_cast(float, m)));
}

// Loads the B operand (weights) of one wave into registers, from canonical
// [B][F][A]: fp16 weights, whole vectors of both slices at a time.
template <int A, int NT, int PARTS>
__device__ __forceinline__ void load_weights(const float2* __restrict__ w, int F, int B, int f,
                                             int beam0, int lane, bf_half8 (&bhi)[NT][A / 16],
                                             bf_half8 (&blo)[NT][A / 16]) {
    static_assert(PARTS <= 2, "fp16 slices");
    constexpr int KS = A / 16;
    const int c = lane & 15;
    const int g = lane >> 4;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int b = beam0 + nt * 8 + (c >> 1);
        const bool comp_im = (c & 1) != 0;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            bf_half8 h, l;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int a = g * (A / 4) + 4 * s + j;
                float2 v = make_float2(0.0f, 0.0f);
                if (b < B) v = w[((size_t)b * F + f) * A + a];
                // column re: (wr, -wi); column im: (wi, wr)
                const float e0 = comp_im ? v.y : v.x;
                const float e1 = comp_im ? v.x : -v.y;
                const _Float16 h0 = (_Float16)e0;
                const _Float16 h1 = (_Float16)e1;
                h[2 * j] = h0;
                h[2 * j + 1] = h1;
                if (PARTS == 2) {
                    l[2 * j] = (_Float16)(e0 - (float)h0);
                    l[2 * j + 1] = (_Float16)(e1 - (float)h1);
                }
            }
            bhi[nt][s] = h;
            if (PARTS == 2) blo[nt][s] = l;
        }
    }
}

// The same of float weights, canonical or tiled [F][B/32][A][32], as three
// bfloat16 slices, element by element into one array: with whole vectors in
// three arrays the compiler keeps more loads in flight than the registers
// carry (A = 128 134 -> 202 VGPRs, T = 4100, B = 33, S = 10 232 -> 303 us).
template <int A, int NT>
__device__ __forceinline__ void load_float_weights(const float2* __restrict__ w, bool tiled, int F,
                                                   int B, int f, int beam0, int lane,
                                                   bf_half8 (&bw)[3][NT][A / 16]) {
    constexpr int KS = A / 16;
    const int c = lane & 15;
    const int g = lane >> 4;
    const int tiles = (B + 31) / 32;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int b = beam0 + nt * 8 + (c >> 1);
        const bool comp_im = (c & 1) != 0;
        const float2* const wb = tiled ? w + ((size_t)f * tiles + b / 32) * A * 32 + b % 32
                                       : w + ((size_t)b * F + f) * A;
        const int step = tiled ? 32 : 1;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int a = g * (A / 4) + 4 * s + j;
                float2 v = make_float2(0.0f, 0.0f);
                if (b < B) v = wb[a * step];
                _Float16 e0[3], e1[3];
                weight_slices(comp_im ? v.y : v.x, e0);
                weight_slices(comp_im ? v.x : -v.y, e1);
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    bw[q][nt][s][2 * j] = e0[q];
                    bw[q][nt][s][2 * j + 1] = e1[q];
                }
            }
        }
    }
}

// Float weights may be infinite, and the zero samples past T turn that into a
// NaN in a last window cut short by T.  Where such a window ended as a NaN, its
// power is summed again over the rows it has, a row per lane (the result is an
// infinity or a NaN: any order of sums gives it).  After the stages, by the
// waves that stored the window: clearing the rows in the stage itself cost the
// common path 10 registers and with them a wave per SIMD (A = 64, S = 10).
template <int A, int NT>
__device__ __noinline__ void repair_short_window(const uint8_t* __restrict__ x,
                                                 const float2* __restrict__ w, bool tiled,
                                                 float* out, int T, int F, int B,
                                                 int S, int W, int f, int beam0, int lane) {
    __threadfence_block();  // the window's stores, by other lanes of this wave
    float* const o = out + ((size_t)(W - 1) * F + f) * B + beam0;
    const int live = B - beam0 < NT * 8 ? B - beam0 : NT * 8;
    unsigned long long bad = __ballot(lane < live && isnan(o[lane < live ? lane : 0]));
    const int tiles = (B + 31) / 32;
    while (bad != 0) {
        const int i = __builtin_ctzll(bad);
        bad &= bad - 1;
        const int b = beam0 + i;
        const float2* const wb = tiled ? w + ((size_t)f * tiles + b / 32) * A * 32 + b % 32
                                       : w + ((size_t)b * F + f) * A;
        float sum = 0.0f;
        for (int t = (W - 1) * S + lane; t < T; t += kWaveSize) {
            const uint8_t* const row = x + ((size_t)t * F + f) * A;
            float re = 0.0f, im = 0.0f;
            for (int a = 0; a < A; ++a) {
                const float2 v = wb[a * (tiled ? 32 : 1)];
                const float xr = (float)bf_nibble(row[a], 0), xi = (float)bf_nibble(row[a], 4);
                re = fmaf(-v.y, xi, fmaf(v.x, xr, re));
                im = fmaf(v.y, xr, fmaf(v.x, xi, im));
            }
            sum += re * re + im * im;
        }
#pragma unroll
        for (int k = 32; k >= 1; k >>= 1) sum += __shfl_xor(sum, k);
        if (lane == 0) o[i] = sum;
    }
}

// At least two waves per SIMD (at most 256 registers per lane): the
// unrolled stage otherwise keeps several tiles' accumulators in flight.
// SHORT: float weights and a last window cut short by T (a kernel of its own:
// the check alone cost whole windows 2 %).
template <int A, int NT, int WV, int PARTS, int MODE, int ST, bool DB, bool MASKED = false,
          bool SHORT = false>
__global__ __launch_bounds__(WV * kWaveSize) __attribute__((amdgpu_waves_per_eu(2)))
void mfma_fused_kernel(
    const uint8_t* __restrict__ x, const float2* __restrict__ w, bool tiled,
    float* __restrict__ out, const uint8_t* __restrict__ mask, int T, int F, int B, int S, int W,
    int tiles_total, int tiles_per_chunk, int n_items, int per_xcd) {
    constexpr int kThreads = WV * kWaveSize;
    constexpr int KS = A / 16;                      // k-steps of 32 (16 antennas x re/im)
    using Map = StageMap<A, kThreads>;
    constexpr int TILE_BYTES = Map::TILE_BYTES;     // LDS bytes per 16-row tile
    constexpr int STAGE_BYTES = ST * TILE_BYTES;
    constexpr int DW_TILE = Map::DW_TILE;           // packed dwords per tile
    constexpr int DW_STAGE = ST * DW_TILE;
    constexpr int DW_THREAD = (DW_STAGE + kThreads - 1) / kThreads;
    constexpr bool ALL_VALID = DW_STAGE % kThreads == 0;
    // MODE 1 stages hold whole super-tiles of 5 tiles
    static_assert(MODE != 1 || ST % 5 == 0, "S = 10 stages are whole super-tiles");
    static_assert(kThreads % DW_TILE == 0 || DW_TILE % kThreads == 0, "power-of-two staging");
    __shared__ __attribute__((aligned(16))) unsigned char lds[(DB ? 2 : 1) * STAGE_BYTES];

    const int tid = threadIdx.x;
    const int lane = tid & (kWaveSize - 1);
    const int wave = tid / kWaveSize;
    // XCD-aware order: workgroups are dispatched round-robin over the 8
    // XCDs, so blockIdx.x % 8 names the XCD.  Each XCD takes a contiguous
    // range of frequency-major items: all time chunks of a channel run on
    // one XCD back to back (its weights stay in that L2) and the
    // neighbouring channel, which shares the 128-byte lines of every packed
    // row, follows on the same XCD.
    const int item = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (item >= n_items) return;  // whole workgroup
    const int n_chunks = n_items / F;
    const int f = item / n_chunks;
    const int chunk = item - f * n_chunks;
    const int beam0 = (blockIdx.y * WV + wave) * NT * 8;
    const bool has_beams = beam0 < B;

    // the slices, largest first: fp16 in bhi and blo, bfloat16 in bw
    bf_half8 bhi[NT][KS];
    bf_half8 blo[NT][KS];
    bf_half8 bw[3][NT][KS];
    if (has_beams) {
        if constexpr (PARTS == 3)
            load_float_weights<A, NT>(w, tiled, F, B, f, beam0, lane, bw);
        else
            load_weights<A, NT, PARTS>(w, F, B, f, beam0, lane, bhi, blo);
    }

    const int tile_begin = chunk * tiles_per_chunk;
    int tile_end = tile_begin + tiles_per_chunk;
    tile_end = tile_end < tiles_total ? tile_end : tiles_total;
    const size_t row_stride = (size_t)F * A;
    // tiles per super-tile (MODE 3: per window)
    const int tps = MODE == 2 ? (S >> 2) : (MODE == 3 ? (S >> 4) : 5);
    const int pitch = MODE == 0 || MODE == 3 ? 4 : (MODE == 1 ? 20 : S);  // spectra between row groups

    // Per-thread staging constants (StageMap: rows fastest within 16 lanes).
    const int tl0 = Map::tile0(wave);  // uniform per wave
    const int rem0 = Map::rem0(tid);
    const int rho = rem0 & 15;
    const int j0 = rem0 >> 4;
    // spectrum of this thread's row within its tile's row group pattern
    const int prow = (rho >> 2) * pitch + (rho & 3);
    const uint8_t* xs = x + (size_t)f * A + (size_t)prow * row_stride + 4 * j0;
    const int lds_mine = Map::lds_offset(tl0, rem0);

    // First spectrum of the stage starting at tile st0, and offset of tile
    // tl of a stage from it (row group 0, row 0).
    auto stage_time = [&](int st0) -> int {
        if (MODE != 2) return 16 * st0;  // MODE 1: 80 per super-tile
        return 4 * S * (st0 / tps) + 4 * (st0 % tps);
    };
    auto tile_rows = [&](int tl) -> int {
        if (MODE == 0 || MODE == 3) return 16 * tl;
        if (MODE == 1) return ST == 5 ? 4 * tl : 80 * (tl / 5) + 4 * (tl % 5);
        return 4 * tl;
    };
    // Whether every row of the stage at st0 lies before T.
    auto stage_full = [&](int st0) -> bool {
        return stage_time(st0) + tile_rows(ST - 1) + 3 * pitch + 3 < T;
    };
    auto dword_valid = [&](int k) -> bool {
        return ALL_VALID || tl0 + Map::tld(k) < ST;
    };
    unsigned pre[DW_THREAD];
    // Global load of dword k of the stage whose first spectrum is t_stage;
    // GUARD: rows at or after t_lim, and with MASKED rows of lost frames
    // (mask byte 0), read as zero.  MASKED kernels always take this path.
    auto load_dword = [&](auto guard, int k, int t_stage, int t_lim) {
        constexpr bool GUARD = decltype(guard)::value;
        const int rel = t_stage + tile_rows(tl0 + Map::tld(k));
        const uint8_t* p = xs + (size_t)rel * row_stride + Map::byte_delta(k);
        unsigned v = 0u;
        if (GUARD) {
            const int t = prow + rel;
            if (dword_valid(k) && t < t_lim && (!MASKED || mask[(size_t)t * F + f] != 0))
                v = *reinterpret_cast<const unsigned*>(p);
        } else if (dword_valid(k)) {
            v = *reinterpret_cast<const unsigned*>(p);
        }
        pre[k] = v;
    };
    auto store_dword = [&](int k, unsigned char* buf) {
        if (!dword_valid(k)) return;
        unsigned h2[4];
        if (PARTS == 3)
            bf_int4x4_to_bfloat2x4(pre[k], h2);
        else
            bf_int4x4_to_half2x4(pre[k], h2);
        bf_uint4v u = {h2[0], h2[1], h2[2], h2[3]};
        *reinterpret_cast<bf_uint4v*>(buf + lds_mine + Map::lds_delta(k)) = u;
    };
    auto load_stage = [&](int st0) {
        const int ts = stage_time(st0);
        if (!MASKED && stage_full(st0)) {
#pragma unroll
            for (int k = 0; k < DW_THREAD; ++k) load_dword(std::false_type{}, k, ts, T);
        } else {
#pragma unroll
            for (int k = 0; k < DW_THREAD; ++k) load_dword(std::true_type{}, k, ts, T);
        }
    };

    float win[NT][2];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) win[nt][0] = win[nt][1] = 0.0f;
    const int col = lane & 15;
    const int G = lane >> 4;
    const int odd = col & 1;
    // Output pointer of this lane at window (or spectrum) group 0.  Lanes
    // 2c and 2c+1 hold the same power after the pair swap, so they split
    // the stores: MODE 1 by window of the pair (q = odd), MODE 2 by N-tile
    // (nt + odd), MODE 0 by row (r = odd + 2m).
    const int bl = beam0 + (col >> 1);
    float* const out_lane =
        MODE == 1 ? out + ((size_t)(2 * G + odd) * F + f) * B + bl
        : MODE == 2 ? out + ((size_t)G * F + f) * B + bl + (NT >= 2 ? 8 * odd : 0)
        : MODE == 3 ? out + (size_t)f * B + bl
                    : out + ((size_t)(4 * G + odd) * F + f) * B + bl;
    const size_t group_stride = (size_t)F * B;  // floats between consecutive windows

    // Powers and window sums of tile tl (global tile i) from acc.
    auto epilogue = [&](int tl, int i, const bf_float4 (&acc)[NT]) {
        if (MODE == 0) {
            float* const o = out_lane + (size_t)(16 * i) * group_stride;
            const int t0 = 16 * i + 4 * G + odd;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float sq = acc[nt][r] * acc[nt][r];
                    p[r] = sq + dpp_swap_pairs(sq);
                }
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const float v = odd ? p[2 * m + 1] : p[2 * m];
                    if (bl + nt * 8 < B && t0 + 2 * m < T)
                        o[(size_t)(2 * m) * group_stride + nt * 8] = v;
                }
            }
            return;
        }
        if (MODE == 1 && tl % 5 == 2) {
            // spectra 8, 9 close window 0; 10, 11 open window 1
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                win[nt][0] = fmaf(acc[nt][0], acc[nt][0], win[nt][0]);
                win[nt][0] = fmaf(acc[nt][1], acc[nt][1], win[nt][0]);
                win[nt][1] = fmaf(acc[nt][2], acc[nt][2], win[nt][1]);
                win[nt][1] = fmaf(acc[nt][3], acc[nt][3], win[nt][1]);
            }
            return;
        }
        const int q = (MODE == 1 && tl % 5 > 2) ? 1 : 0;  // static once the tile loop is unrolled
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float a = acc[nt][0] * acc[nt][0];
#pragma unroll
            for (int r = 1; r < 4; ++r) a = fmaf(acc[nt][r], acc[nt][r], a);
            if (q == 0)
                win[nt][0] += a;
            else
                win[nt][1] += a;
        }
    };
    // Stores and resets the windows of the super-tile (MODE 1) or stage
    // (MODE 2) that starts at tile i0.
    auto close_windows = [&](int i0) {
        if (MODE == 1) {
            const int super = i0 / 5;
            float* const o = out_lane + (size_t)(8 * super) * group_stride;
            const bool ok = 8 * super + 2 * G + odd < W;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const float p0 = win[nt][0] + dpp_swap_pairs(win[nt][0]);
                const float p1 = win[nt][1] + dpp_swap_pairs(win[nt][1]);
                if (ok && bl + nt * 8 < B) o[nt * 8] = odd ? p1 : p0;
                win[nt][0] = win[nt][1] = 0.0f;
            }
        } else if (MODE == 2) {
            const int super = i0 / tps;
            float* const o = out_lane + (size_t)(4 * super) * group_stride;
            const bool ok = 4 * super + G < W;
            float p[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                p[nt] = win[nt][0] + dpp_swap_pairs(win[nt][0]);
                win[nt][0] = 0.0f;
            }
            if (NT == 1) {
                if (ok && !odd && bl < B) o[0] = p[0];
            } else {
#pragma unroll
                for (int nt = 0; nt < NT; nt += 2)
                    if (ok && bl + (nt + odd) * 8 < B) o[nt * 8] = odd ? p[nt + 1] : p[nt];
            }
        } else if (MODE == 3) {
            float* const o = out_lane + (size_t)(i0 / tps) * group_stride;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                float p = win[nt][0];
                p += __shfl_xor(p, 16);
                p += __shfl_xor(p, 32);
                p += dpp_swap_pairs(p);
                win[nt][0] = 0.0f;
                if (G == nt % 4 && !odd && bl + nt * 8 < B) o[nt * 8] = p;
            }
        }
    };
    // MODE 2, 3: whether the stage at st0 ends a super-tile or window (MODE
    // 1 closes its windows inside the stage, after every fifth tile).  The
    // last window may be cut short by T.
    auto closes_window = [&](int st0) -> bool {
        if (MODE == 3) return (st0 % tps) + ST == tps || st0 + ST >= tiles_total;
        return MODE == 2 && (st0 % tps) + ST == tps;
    };

    // MFMAs and epilogues of the stage held at `cur`; with DB, the dwords
    // of the next stage (in pre) are converted into `nxt` and the loads of
    // the stage after it are issued, spread over the tiles so that this
    // VALU and memory work interleaves with the MFMAs.
    auto stage = [&](auto mf, auto guard, const unsigned char* cur, unsigned char* nxt, int st0,
                     int t_load, int t_lim) {
        constexpr bool MF = decltype(mf)::value;
        // Up to 64 antennas the next tile's A operands are read while this
        // tile's MFMAs run; wider tiles read them per k-step (a second
        // tile of operands would not fit in registers).
        constexpr bool PREFETCH = KS <= 4;
        bf_half8 av[KS];
        if (MF && PREFETCH) {
#pragma unroll
            for (int s = 0; s < KS; ++s)
                av[s] = *reinterpret_cast<const bf_half8*>(cur + (s * kWaveSize + lane) * 16);
        }
#pragma unroll
        for (int tl = 0; tl < ST; ++tl) {
            bf_half8 an[KS];
            bf_float4 acc[NT];
            if (MF) {
                if (PREFETCH && tl + 1 < ST) {
#pragma unroll
                    for (int s = 0; s < KS; ++s)
                        an[s] = *reinterpret_cast<const bf_half8*>(
                            cur + (tl + 1) * TILE_BYTES + (s * kWaveSize + lane) * 16);
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[nt] = bf_float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const bf_half8 a_s =
                        PREFETCH ? av[s]
                                 : *reinterpret_cast<const bf_half8*>(
                                       cur + tl * TILE_BYTES + (s * kWaveSize + lane) * 16);
                    if constexpr (PARTS == 3) {
#pragma unroll
                        for (int q = 0; q < 3; ++q)
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
                                acc[nt] = mfma_16x16x32<PARTS>(a_s, bw[q][nt][s], acc[nt]);
                    } else {
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt)
                            acc[nt] = mfma_16x16x32<PARTS>(a_s, bhi[nt][s], acc[nt]);
                        if (PARTS == 2) {
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
                                acc[nt] = mfma_16x16x32<PARTS>(a_s, blo[nt][s], acc[nt]);
                        }
                    }
                }
            }
            if (DB) {
#pragma unroll
                for (int k = tl * DW_THREAD / ST; k < (tl + 1) * DW_THREAD / ST; ++k) {
                    store_dword(k, nxt);
                    load_dword(guard, k, t_load, t_lim);
                }
            }
            if (MF) {
                epilogue(tl, st0 + tl, acc);
                if (MODE == 1 && tl % 5 == 4) close_windows(st0 + tl - 4);
                if (PREFETCH && tl + 1 < ST) {
#pragma unroll
                    for (int s = 0; s < KS; ++s) av[s] = an[s];
                }
            }
            // Wide tiles: keep the scheduler from hoisting the next tile's
            // operand reads into this one (registers).
            if (!PREFETCH) __builtin_amdgcn_sched_barrier(0);
        }
    };

    if (DB) {
        if (tile_begin < tile_end) {
            load_stage(tile_begin);
#pragma unroll
            for (int k = 0; k < DW_THREAD; ++k) store_dword(k, lds);
        }
        if (tile_begin + ST < tile_end) load_stage(tile_begin + ST);
        __syncthreads();
        int buf = 0;
        for (int st0 = tile_begin; st0 < tile_end; st0 += ST) {
            const unsigned char* cur = lds + buf * STAGE_BYTES;
            unsigned char* nxt = lds + (buf ^ 1) * STAGE_BYTES;
            // The other buffer was last read before the previous barrier.
            // Loads of the stage after next: unguarded when it exists and
            // lies before T; otherwise guarded (t_lim 0 when it does not exist).
            const int st2 = st0 + 2 * ST;
            const int t_load = stage_time(st2);
            if (!MASKED && st2 < tile_end && stage_full(st2)) {
                if (has_beams)
                    stage(std::true_type{}, std::false_type{}, cur, nxt, st0, t_load, T);
                else
                    stage(std::false_type{}, std::false_type{}, cur, nxt, st0, t_load, T);
            } else {
                const int t_lim = st2 < tile_end ? T : 0;
                if (has_beams)
                    stage(std::true_type{}, std::true_type{}, cur, nxt, st0, t_load, t_lim);
                else
                    stage(std::false_type{}, std::true_type{}, cur, nxt, st0, t_load, t_lim);
            }
            if (has_beams && closes_window(st0)) close_windows(st0);
            __syncthreads();
            buf ^= 1;
        }
    } else {
        if (tile_begin < tile_end) load_stage(tile_begin);
        for (int st0 = tile_begin; st0 < tile_end; st0 += ST) {
            __syncthreads();  // previous stage fully consumed
#pragma unroll
            for (int k = 0; k < DW_THREAD; ++k) store_dword(k, lds);
            if (st0 + ST < tile_end) load_stage(st0 + ST);  // in flight during compute
            __syncthreads();  // stage visible to all waves
            if (has_beams) {
                stage(std::true_type{}, std::false_type{}, lds, lds, st0, 0, 0);
                if (closes_window(st0)) close_windows(st0);
            }
        }
    }
    if constexpr (SHORT)
        if (has_beams && tile_end == tiles_total)
            repair_short_window<A, NT>(x, w, tiled, out, T, F, B, S, W, f, beam0, lane);
}

struct Plan {
    int mode, st, tiles_total, tiles_per_chunk, n_items, per_xcd, beam_blocks, W;
    double cost;  // modelled time, in tiles
};

// Whether windows of a multiple of 20 spectra (and not of 16) stage five tiles
// at a time instead of one: fewer barriers per tile, five times the LDS.  Up
// to 64 antennas that is free (split, S = 20, T = 4100, B = 33: A = 32 69 -> 38
// us, A = 64 73 -> 61 us).  Above it leaves two workgroups to a CU, which
// costs nothing where no more were launched and there are stages to overlap
// (A = 128, T = 512, B = 9, S = 20, 336 workgroups of 35 tiles: 32 -> 27 us; S = 40,
// 672 of them: 35 -> 41 us; A = 256, S = 100, T = 65, B = 20, 25 tiles: 34 -> 31 us; but
// S = 60, T = 200, 15 tiles 25 -> 29 us, and A = 128, S = 20, T = 70, B = 40, 5 tiles 12.8
// -> 13.7 us).  Beyond those it pays at 128 for two N-tiles of split weights (T =
// 4100, B = 33, S = 100: 180 -> 141 us; but B = 2 87 -> 112 us, F16 98 -> 106 us) and
// at 256 in long calls (T = 4100, S = 100, B = 33: 510 -> 448 us; T = 1024, B = 20: 71
// -> 80 us), for single weights with one block of beams (T = 4100, S = 20: B = 9
// 0.88 of the time, B = 33 1.05).  Float weights were measured with five tiles only.
inline bool five_tile_stages(int A, int parts, int nt, int T, int B, long workgroups, int tiles) {
    if (A <= 64 || parts == 3) return true;
    if (A == 128) return tiles > 5 && (workgroups <= 512 || (parts == 2 && nt >= 2));
    return (workgroups <= 512 && tiles >= 25) || (T >= 4096 && (parts == 2 || B <= 32));
}

inline Plan make_plan(int A, int parts, int T, int F, int B, int S, bool one_by_one,
                      const MfmaConfig& cfg) {
    Plan p{};
    p.mode = S == 0 ? 0 : (S == 10 ? 1 : (one_by_one ? 3 : 2));
    int tiles_per_super = 1;
    if (p.mode == 0) {
        p.st = 4;
        p.W = T;
    } else if (p.mode == 1) {
        p.st = 5;
        tiles_per_super = 5;
        p.W = (int)ceil_div((size_t)T, 10);
    } else if (p.mode == 3) {
        p.st = 4;
        tiles_per_super = S / 16;
        p.W = (int)ceil_div((size_t)T, (size_t)S);
    } else {
        tiles_per_super = S / 4;
        p.st = tiles_per_super % 4 == 0 ? 4 : 1;
        p.W = (int)ceil_div((size_t)T, (size_t)S);
    }
    const int rows_super = 16 * tiles_per_super;
    const int n_super = (int)ceil_div((size_t)T, (size_t)rows_super);
    p.tiles_total = n_super * tiles_per_super;
    // tiles in time order: whole stages up to T
    if (p.mode == 0 || p.mode == 3) p.tiles_total = 4 * (int)ceil_div((size_t)T, 64);
    p.beam_blocks = (int)ceil_div((size_t)B, (size_t)(cfg.waves * cfg.nt * 8));
    // Chunk length: a whole number of super-tiles and stages, chosen to
    // minimise (rounds of resident workgroups) x (tiles per workgroup + a
    // fixed start-up cost for loading the weights).
    int unit = tiles_per_super;
    while (unit % p.st) unit += tiles_per_super;
    const long resident = cfg.resident, startup_tiles = 12;
    long best_cost = -1;
    int per_chunk = unit;
    for (int c = unit; c <= 640 && c <= p.tiles_total + unit; c += unit) {
        const long chunks = (long)ceil_div((size_t)p.tiles_total, (size_t)c);
        const long rounds =
            (long)ceil_div((size_t)(chunks * F * p.beam_blocks), (size_t)resident);
        // A chunk of whole windows may reach past the last tile.  Counted in
        // full it gives way to more and shorter ones, which measured faster
        // but for 256 antennas, whose weights weigh more (F16, T = 1024, B =
        // 128, S = 320: 171 us in two chunks, 142 in one).
        const long tiles = A == 256 ? std::min(c, p.tiles_total) : c;
        const long cost = rounds * (tiles + startup_tiles);
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            per_chunk = c;
            // the end of a window that runs alone costs about 0.8 tiles
            p.cost = (double)cost + (p.mode == 3 ? rounds * tiles * 0.8 * 16 / S : 0.0);
        }
    }
    p.tiles_per_chunk = per_chunk;
    const int n_chunks = (int)ceil_div((size_t)p.tiles_total, (size_t)per_chunk);
    p.n_items = n_chunks * F;
    p.per_xcd = (int)ceil_div((size_t)p.n_items, kXcds);
    if (p.mode == 2 && p.st == 1 && tiles_per_super % 5 == 0 &&
        five_tile_stages(A, parts, cfg.nt, T, B, (long)p.n_items * p.beam_blocks, per_chunk))
        p.st = 5;
    return p;
}

// Whether windows of a multiple of 64 spectra run one after another (MODE 3)
// instead of four side by side (MODE 2), for the problem's untuned shape
// `cfg`.  Side by side pads the time axis to whole groups of four windows; one
// by one costs the folds and stores at the end of every window, 1.5 tiles (24
// spectra) a window at most.  So one by one where the padding is the larger
// part: A = 64, split, B = 64, S = 320, T = 512 (2.5 times its length padded) 29
// -> 16 us, T = 4100 (1.25) 123 -> 102 us; but S = 64, T = 16384 (no padding) 251
// -> 271 us, and A = 32, B = 2 there 82 -> 108 us.  For 64 and 128 antennas also
// where shorter chunks fill the chip (A = 64, T = 1024, B = 9, S = 64, 336
// workgroups against 1008: 24 -> 17 us) or the two are modelled alike (A =
// 128, T = 8192, B = 9, S = 128: 265 -> 212 us; within 5 %, the least that keeps
// these); the other counts gain nothing there (A = 32, T = 8192, B = 9, S = 64: 1.16).
inline bool windows_one_by_one(int A, int parts, int T, int F, int B, int S,
                               const MfmaConfig& cfg) {
    if (S == 0 || S % 64 != 0) return false;
    const long group = 4L * S;
    const long padding = (T + group - 1) / group * group - T;
    if (padding * S > 24L * T) return true;
    if (A != 64 && A != 128) return false;
    const Plan side = make_plan(A, parts, T, F, B, S, false, cfg);
    const Plan one = make_plan(A, parts, T, F, B, S, true, cfg);
    if ((long)side.n_items * side.beam_blocks < cfg.resident && one.n_items > side.n_items)
        return true;
    return one.cost < 1.05 * side.cost;
}

template <int A, int NT, int WV, int PARTS, bool DB, bool MASKED = false>
void launch_shape(hipStream_t stream, const MfmaLaunch& L, const MfmaConfig& cfg) {
    const Plan p = make_plan(A, PARTS, L.T, L.F, L.B, L.S, L.one_by_one, cfg);
    const dim3 grid((unsigned)(p.per_xcd * kXcds), (unsigned)p.beam_blocks);
    const dim3 block(WV * kWaveSize);
    const float2* w2 = reinterpret_cast<const float2*>(L.w);
#define BF_LAUNCH_SHORT(MODE_, ST_, SHORT_)                                                     \
    hipLaunchKernelGGL((mfma_fused_kernel<A, NT, WV, PARTS, MODE_, ST_, DB, MASKED, SHORT_>),   \
                       grid, block, 0, stream, L.x, w2, L.tiled, L.out, L.mask, L.T, L.F, L.B,  \
                       L.S, p.W, p.tiles_total, p.tiles_per_chunk, p.n_items, p.per_xcd)
#define BF_LAUNCH(MODE_, ST_)                                     \
    do {                                                          \
        if (PARTS == 3 && MODE_ != 0 && L.T % L.S != 0)           \
            BF_LAUNCH_SHORT(MODE_, ST_, PARTS == 3 && MODE_ != 0); \
        else                                                      \
            BF_LAUNCH_SHORT(MODE_, ST_, false);                   \
    } while (0)
    if (p.mode == 0) {
        BF_LAUNCH(0, 4);
    } else if (p.mode == 1) {
        BF_LAUNCH(1, 5);
    } else if (p.mode == 3) {
        BF_LAUNCH(3, 4);
    } else if (p.st == 4) {
        BF_LAUNCH(2, 4);
    } else if (p.st == 5) {
        BF_LAUNCH(2, 5);
    } else {
        BF_LAUNCH(2, 1);
    }
#undef BF_LAUNCH
#undef BF_LAUNCH_SHORT
}

template <int A, int NT, int WV>
void launch_split_db(hipStream_t stream, const MfmaLaunch& L, const MfmaConfig& cfg) {
    if (L.parts == 2) {
        if (cfg.db)
            launch_shape<A, NT, WV, 2, true>(stream, L, cfg);
        else
            launch_shape<A, NT, WV, 2, false>(stream, L, cfg);
    } else {
        if (cfg.db)
            launch_shape<A, NT, WV, 1, true>(stream, L, cfg);
        else
            launch_shape<A, NT, WV, 1, false>(stream, L, cfg);
    }
}

}  // namespace mfma_detail

// The kernel of k_mfma_wave.hip, where it takes the problem.  `resident`: the
// workgroups assumed to run at once, which sizes a task's run of windows.
bool frame_wave_supported(const MfmaLaunch& L, int A);
void launch_frame_wave(hipStream_t stream, const MfmaLaunch& L, int resident);

// Launches the kernel with float weights (PARTS = 3) for `A` antennas
// (k_mfma_exact.hip): `L.tiled` chooses the weight layout.
void launch_mfma_exact(hipStream_t stream, const MfmaLaunch& L, int A);

// Instantiated shapes per antenna count: (NT, waves) pairs whose split
// weights fit in at most 128 VGPRs per lane and that compile without
// register spills for the common modes.
#define BF_MFMA_SHAPES_32_64(A_)                                            \
    BF_SHAPE(A_, 4, 4) BF_SHAPE(A_, 2, 8) BF_SHAPE(A_, 2, 4) BF_SHAPE(A_, 1, 8) \
    BF_SHAPE(A_, 1, 4)
#define BF_MFMA_SHAPES_128 BF_SHAPE(128, 2, 4) BF_SHAPE(128, 1, 8) BF_SHAPE(128, 1, 4)
#define BF_MFMA_SHAPES_256 BF_SHAPE(256, 1, 4)

// A launch with a loss mask runs the one masked instantiation per antenna
// count: 8 beams per wave, 4 waves, one LDS stage (any beam count).
#define BF_DEFINE_MFMA_FOR_A(A_, SHAPES)                                                   \
    bool launch_mfma_a##A_(hipStream_t stream, const MfmaLaunch& L, const MfmaConfig& cfg) { \
        if (L.mask != nullptr) {                                                           \
            MfmaConfig m = cfg;                                                            \
            m.nt = 1;                                                                      \
            m.waves = 4;                                                                   \
            m.db = 0;                                                                      \
            if (L.parts == 2)                                                              \
                mfma_detail::launch_shape<A_, 1, 4, 2, false, true>(stream, L, m);      \
            else                                                                           \
                mfma_detail::launch_shape<A_, 1, 4, 1, false, true>(stream, L, m);         \
            return true;                                                                   \
        }                                                                                  \
        SHAPES                                                                             \
        return false;                                                                      \
    }
#define BF_SHAPE(A_, NT_, WV_)                                               \
    if (cfg.nt == NT_ && cfg.waves == WV_) {                                 \
        mfma_detail::launch_split_db<A_, NT_, WV_>(stream, L, cfg);          \
        return true;                                                         \
    }

}  // namespace bfhip
