// tracker_wave.hpp -- the tracker's matrix-core body: one wave re-points its
// beams at every window and contracts the window's spectra.
//
// The tracker re-points every beam once per integration window: window w
// uses the direction of its first spectrum (reference
// src/beam_tracker.cpp:166-190) and the steering weights of steering.hpp,
// then contracts like the fixed grid (src/cpu_beamformer.cpp:56-78).  Weights
// live in registers only, never in memory.
//
// A wave owns one channel, NT * 8 beams and a run of windows, and works
// alone: no LDS staging and no barrier.  A tile is 16 consecutive spectra of
// one window; in the A operand of v_mfma_f32_16x16x32 lane l holds row l % 16
// and the antennas g (A / 4) .. of group g = l / 16, which is one contiguous
// run of A / 4 packed bytes of that row, so a lane loads its own operand
// straight from HBM and converts it in registers.  The beams a wave holds
// share that operand, so a channel's rows are loaded and converted once for
// 8 NT beams.  Staged through LDS with 8 beams on each of four waves, as
// before, every wave read the whole tile, as many LDS bytes per clock as
// there are.  What bounds it now is instruction issue: per tile 8 NT MFMAs of
// 16 cycles and some 53 other instructions, and the weights, about 43 a piece
// (64 antennas, 672 channels, 65536 spectra, 32 beams, windows of 320: 1.85 ->
// 1.34 ms, 0.54 PFLOP/s counted once; 13 beams, windows of 10, 4003 spectra,
// 336 channels: 0.33 -> 0.20 ms; float weights there, 2.35 ms on FP32 FMAs,
// 0.41 ms).  Wave tasks run block, then channel fastest: a workgroup's four waves
// read neighbouring channels (or the same one) of the same spectra, which share
// 128-byte lines.
//
// Element order within a lane's 8 contraction slots: (re0, re2, im0, im2,
// re1, re3, im1, im3) of antennas 0..3 of a dword; output column 2b holds
// Re(y_b) (weights wr, -wi), column 2b + 1 Im(y_b) (weights wi, wr).
//
// PARTS: weights as one fp16, as fp16 hi + lo (about 22 bits), or as three
// bfloat16 slices that add up to the float (the FP32 selector), which then
// comes from its own FP64 phase in every window.  Sums run from the smallest
// slice to the largest.
#pragma once

#include <type_traits>

#include "steering.hpp"

namespace bfhip {
namespace wave_detail {

constexpr int kWaveSize = 64;
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWaveSize;
constexpr int kXcds = 8;

__device__ __forceinline__ unsigned dpp_swap_pairs_u(unsigned v) {
    // quad_perm [1,0,3,2]: lane i <- lane i^1.
    return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);
}
// quad_perm [0,0,2,2] and [1,1,3,3]: the even or odd lane's value in both
// lanes of a pair (these fold into the select that uses them).
__device__ __forceinline__ unsigned dpp_even(unsigned v) {
    return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xA0, 0xF, 0xF, true);
}
__device__ __forceinline__ unsigned dpp_odd(unsigned v) {
    return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xF5, 0xF, 0xF, true);
}
__device__ __forceinline__ float dpp_swap_pairs(float v) {
    return __builtin_bit_cast(float, dpp_swap_pairs_u(__builtin_bit_cast(unsigned, v)));
}

// Positions of all antennas in LDS (read many times per window): as doubles
// for the phase, as floats for the rotation between windows.
template <int A>
struct Positions {
    double d[3 * A];
    float s[3 * A];
};

// By the whole workgroup; visible after a barrier.
template <int A>
__device__ __forceinline__ void stage_positions(const Geom& geo, Positions<A>& pos) {
    for (int a = threadIdx.x; a < A; a += blockDim.x) {
        float p[3];
        antenna_position(geo, a, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            pos.s[3 * a + i] = p[i];
            pos.d[3 * a + i] = (double)p[i];
        }
    }
}

// The 4 packed bytes of `d` (4 antennas) as 8 exact halves in the slot order
// above.  With the sign bit flipped a nibble is n = x + 8; it is put in place
// under the exponent of 1024 (low nibble, unit 1) or of 64 (high nibble,
// unit 1/16), so one packed subtraction of 1032 or 72 leaves x.
__device__ __forceinline__ void int4_slots_half(unsigned d, unsigned (&out)[4]) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const unsigned d1 = d >> 8;
    // (sign flip and exponent in one xor: one three-input bit operation each)
    const unsigned w[4] = {(d & 0x000F000Fu) ^ 0x64086408u, (d & 0x00F000F0u) ^ 0x54805480u,
                           (d1 & 0x000F000Fu) ^ 0x64086408u, (d1 & 0x00F000F0u) ^ 0x54805480u};
    const h2 re_bias = {(_Float16)1032.0f, (_Float16)1032.0f};
    const h2 im_bias = {(_Float16)72.0f, (_Float16)72.0f};
#pragma unroll
    for (int j = 0; j < 4; ++j)
        out[j] = __builtin_bit_cast(unsigned, (h2)(__builtin_bit_cast(h2, w[j]) -
                                                   ((j & 1) ? im_bias : re_bias)));
}
// The same as bfloat16: the upper halves of the exact floats.
__device__ __forceinline__ void int4_slots_bfloat(unsigned d, unsigned (&out)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int bit = 8 * (j >> 1) + 4 * (j & 1);
        const float a = (float)bf_nibble(d, bit);
        const float b = (float)bf_nibble(d, bit + 16);
        out[j] = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, b),
                                       __builtin_bit_cast(unsigned, a), 0x07060302u);
    }
}
template <int PARTS>
__device__ __forceinline__ bf_uint4v int4_slots(unsigned d) {
    unsigned o[4];
    if (PARTS == 3)
        int4_slots_bfloat(d, o);
    else
        int4_slots_half(d, o);
    return bf_uint4v{o[0], o[1], o[2], o[3]};
}

template <int PARTS>
__device__ __forceinline__ bf_float4 mfma(bf_uint4v a, bf_uint4v b, bf_float4 c) {
    if constexpr (PARTS == 3)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf_bfloat8, a),
                                                       __builtin_bit_cast(bf_bfloat8, b), c, 0, 0,
                                                       0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(bf_half8, a),
                                                      __builtin_bit_cast(bf_half8, b), c, 0, 0, 0);
}

// Slices of two weight components, each packed (a in the low half).
template <int PARTS>
__device__ __forceinline__ void slice_pair(float a, float b, unsigned (&out)[PARTS]) {
    if constexpr (PARTS == 3) {
        auto top = [](float v) {
            return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) & 0xFFFF0000u);
        };
        auto pack = [](float u, float v) {
            return __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, v),
                                         __builtin_bit_cast(unsigned, u), 0x07060302u);
        };
        const float ra = a - top(a), rb = b - top(b);
        out[0] = pack(a, b);
        out[1] = pack(ra, rb);
        out[2] = pack(ra - top(ra), rb - top(rb));
    } else {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        const h2 h = __builtin_convertvector((f2{a, b}), h2);
        out[0] = __builtin_bit_cast(unsigned, h);
        if constexpr (PARTS == 2) {
            const f2 r = {a - (float)h[0], b - (float)h[1]};
            out[1] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, h2));
        }
    }
}

// Windows of at least this many spectra evaluate every window's weights from
// its own phase.  Shorter windows, where weight generation dominates, use
// anchored weights: every kAnchorWindows-th window (by window index) is an
// anchor evaluated that way, and window w rotates the anchor's phasor by the
// phase change delta = k (p . (d_w - d_anchor)), formed in FP32 from the
// small direction difference (some 15 instructions instead of 38).  A beam
// whose phases may have moved by 1/8 or more since its anchor is evaluated
// from its own phase again.  On trajectories the index is the absolute one
// (an anchor may lie before the launch's first window), so a window's weights
// never depend on how windows are grouped into launches; a table holds the
// launch's own windows only, and its anchors count from the launch's first.
constexpr int kDirectWeightMinSpectra = 64;
constexpr int kAnchorWindows = 16;  // a power of two

// Anchor phasors of this lane's own weights and the anchor's directions.
template <int A, int NT>
struct WeightAnchor {
    float2 own[NT][A / 16][2];
    float dir[NT][3];
};

// (cos, sin)(phi + delta) from z = (cos, sin)(phi), |delta| <= 1/8: the next
// terms of the series are below 2^-27 of the result.
__device__ __forceinline__ float2 rotate_phasor(float2 z, float delta) {
    const float d2 = delta * delta;
    const float sd = fmaf(delta * d2, fmaf(d2, 1.0f / 120.0f, -1.0f / 6.0f), delta);
    const float cm = d2 * fmaf(d2, 1.0f / 24.0f, -0.5f);  // cos(delta) - 1
    return make_float2(fmaf(z.x, cm, fmaf(-z.y, sd, z.x)), fmaf(z.y, cm, fmaf(z.x, sd, z.y)));
}

// What a wave's weights depend on besides the window: one channel.
template <int A>
struct Channel {
    const Positions<A>& pos;
    float reach[3];
    double per_metre;  // f / c
};

// B operand of one wave for window w, `since` windows after its anchor (`fresh`:
// the anchor is not the one in `anc`).  Lane c holds column c of each 8-beam
// N-tile (Re of beam c/2 for even c, Im for odd c) over the antennas
// g (A/4) + 4 s + j.  Lanes c and c^1 need the same complex weights, so the
// even lane evaluates j = 0, 2 and the odd lane j = 1, 3; each slices its own
// and takes the partner's by DPP.
template <int A, int NT, int PARTS, bool ANCHORED>
__device__ __forceinline__ void window_operands(const DirArgs& da, const BeamRow (&rows)[NT],
                                                const Channel<A>& ch, int w, int since, bool fresh,
                                                int beam0, int lane, bool direct,
                                                WeightAnchor<A, NT>& anc,
                                                bf_uint4v (&bw)[PARTS][NT][A / 16]) {
    constexpr int KS = A / 16;
    const int c = lane & 15;
    const int g = lane >> 4;
    const bool odd = (c & 1) != 0;
    const unsigned flip = odd ? 0u : 0x80008000u;
    const int a0 = g * (A / 4) + (odd ? 1 : 0);  // own antennas a0 + 4 s + 2 jj
    const bool anchored = ANCHORED && !direct;
    const int wa = w - since;
    // Direction of column c's beam.  Columns past the last beam hold the
    // weights of direction 0; they are not stored.
    auto direction = [&](int nt, int window, float (&d)[3]) {
        const int b = beam0 + nt * 8 + (c >> 1);
        d[0] = d[1] = d[2] = 0.0f;
        if (b < da.B) beam_direction(da, rows[nt], window, b, d);
    };
    if (anchored && fresh) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float d[3];
            direction(nt, wa, d);
#pragma unroll
            for (int i = 0; i < 3; ++i) anc.dir[nt][i] = d[i];
            const Steer st = make_steer(d, ch.per_metre, ch.reach);
            auto fill = [&](auto weight) {
#pragma unroll
                for (int s = 0; s < KS; ++s)
#pragma unroll
                    for (int jj = 0; jj < 2; ++jj)
                        anc.own[nt][s][jj] = weight(ch.pos.d + 3 * (a0 + 4 * s + 2 * jj), st);
            };
            if (__all(st.in_range))
                fill(steering_weight_near);
            else
                fill(steering_weight_any);
        }
    }
    const float kf = (float)(kTwoPi * ch.per_metre);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        float d[3];
        direction(nt, w, d);
        float dk[3] = {0.0f, 0.0f, 0.0f};
        bool rotate = anchored;  // this lane's beam, from its anchor
        if (anchored) {
            float bound = 0.0f;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                // (0 at the anchor itself: the rotation leaves it as it is)
                dk[i] = kf * (d[i] - anc.dir[nt][i]);
                bound += ch.reach[i] * fabsf(dk[i]);
            }
            rotate = bound < 0.125f || since == 0;
            if (since == 0) dk[0] = dk[1] = dk[2] = 0.0f;
        }
        // k-steps one after another, each with its weights from `make`; only
        // LDS reads may move across, which hides their latency (13 beams,
        // windows of 10, 64 antennas: 232 -> 201 us); at 256 antennas there
        // are no registers for that
        auto steps = [&](auto make) {
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                float2 v[2];
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) v[jj] = make(s, jj);
                unsigned re[PARTS], im[PARTS];
                slice_pair<PARTS>(v[0].x, v[1].x, re);
                slice_pair<PARTS>(v[0].y, v[1].y, im);
#pragma unroll
                for (int q = 0; q < PARTS; ++q) {
                    // (read by all lanes, outside the selects)
                    const unsigned er = dpp_even(re[q]), ei = dpp_even(im[q]);
                    const unsigned pr = dpp_odd(re[q]), pi = dpp_odd(im[q]);
                    bw[q][nt][s] = bf_uint4v{odd ? ei : re[q], odd ? er : im[q] ^ flip,
                                             odd ? im[q] : pr, (odd ? re[q] : pi) ^ flip};
                }
                __builtin_amdgcn_sched_barrier(A <= 128 ? 0x100 : 0);
            }
        };
        auto rotated = [&](int s, int jj) {
            const float* p = ch.pos.s + 3 * (a0 + 4 * s + 2 * jj);
            const float t = fmaf(p[2], dk[2], fmaf(p[1], dk[1], p[0] * dk[0]));
            return rotate_phasor(anc.own[nt][s][jj], t);
        };
        if (ANCHORED && __all(rotate)) {
            steps(rotated);
            continue;
        }
        const Steer st = make_steer(d, ch.per_metre, ch.reach);
        if (PARTS == 3) {  // float weights: as exact as they are held
            steps([&](int s, int jj) {
                return steering_weight_exact(ch.pos.d + 3 * (a0 + 4 * s + 2 * jj), st);
            });
        } else if (!anchored && __all(st.in_range)) {
            steps([&](int s, int jj) {
                return steering_weight_near(ch.pos.d + 3 * (a0 + 4 * s + 2 * jj), st);
            });
        } else {
            steps([&](int s, int jj) {
                float2 v = steering_weight_any(ch.pos.d + 3 * (a0 + 4 * s + 2 * jj), st);
                if (ANCHORED && rotate) v = rotated(s, jj);
                return v;
            });
        }
    }
}

// Time rows of one channel.  Spectrum t (absolute) lives at
// x_f + (t & ring_mask) * row_stride: a linear [T][F][A] array uses
// ring_mask = -1, a ring of 2^k spectra uses 2^k - 1.  Window w covers
// spectra [t_base + w*S, t_base + (w+1)*S) clipped to t_limit.
// With a loss mask, frame (t, f) is valid when valid_f[(t & ring_mask) * F]
// is non-zero; a lost frame's row reads as zero.
struct RowSource {
    const uint8_t* x_f;  // x + f * A, a multiple of A / 4 bytes
    unsigned row_stride;  // F * A bytes
    long ring_mask;
    long t_base;
    long t_limit;
    const uint8_t* valid_f = nullptr;  // mask + f, [t][F] bytes (MASKED only)
    size_t mask_stride = 0;             // F
};

// Output of one channel: integrated [slot][F][B] with slot = w mod
// out_windows (0: slot = w), or per-spectrum [t - t_base][F][B].
struct OutTarget {
    float* out;
    long out_windows;
    int F;
    int f;
};

// A lane's operand of one tile: A / 4 packed bytes.
template <int A>
struct TileBytes {
    unsigned w[A / 16];
};
template <int A>
__device__ __forceinline__ TileBytes<A> load_bytes(const uint8_t* p) {
    constexpr int KS = A / 16;
    TileBytes<A> r;
    if constexpr (KS >= 4) {
#pragma unroll
        for (int i = 0; i < KS / 4; ++i) {
            const bf_uint4v v = reinterpret_cast<const bf_uint4v*>(p)[i];
#pragma unroll
            for (int j = 0; j < 4; ++j) r.w[4 * i + j] = v[j];
        }
    } else {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        r.w[0] = v.x;
        r.w[1] = v.y;
    }
    return r;
}

// Tiles whose loads are in flight; A = 256 has no registers for more.
template <int A>
constexpr int kDepth = A <= 64 ? 4 : (A == 128 ? 2 : 1);
// Whether the conversion of a tile runs beside the MFMAs of the one before
// (two converted operands in registers).  Masked short windows, which never
// have a whole group of tiles, leave the code out: with it they ran 11 % slower.
template <int A, bool ANCHORED, bool MASKED>
constexpr bool kPipelined = A <= 128 && !(MASKED && ANCHORED);

// Windows [w_begin, w_end) of one channel for the beams beam0 ..
// beam0 + NT*8 - 1, by one wave (every argument wave-uniform).  The loads of
// a window's first tiles are issued before its weights are generated.
template <int A, int NT, int PARTS, bool INTEGRATE, bool ANCHORED, bool MASKED = false>
__device__ __forceinline__ void wave_windows(const RowSource& rs, const Channel<A>& ch,
                                             const DirArgs& da, const OutTarget& ot, int w_begin,
                                             int w_end, int beam0) {
    constexpr int KS = A / 16;
    constexpr int D = kDepth<A>;
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int col = lane & 15;
    const int G = lane >> 4;
    const int odd = col & 1;
    const int S = da.S;
    const int B = da.B;
    const int tpw = (S + 15) >> 4;
    const bool direct = S >= kDirectWeightMinSpectra;
    const int bl = beam0 + (col >> 1);
    // operand row of this lane: col; its bytes start at G (A / 4)
    const unsigned lane_off = (unsigned)col * rs.row_stride + (unsigned)(G * (A / 4));

    bf_uint4v bw[PARTS][NT][KS];
    WeightAnchor<A, NT> anc;
    BeamRow rows[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) rows[nt] = beam_row(da, min(bl + 8 * nt, B - 1));
    int since = ((int)da.window_offset + w_begin) & (kAnchorWindows - 1);
#pragma unroll 1
    for (int w = w_begin; w < w_end; ++w, since = (since + 1) & (kAnchorWindows - 1)) {
        const long t_win = rs.t_base + (long)w * S;
        auto load_tile = [&](int jt) -> TileBytes<A> {
            const long t0 = t_win + 16 * jt;
            const long row0 = t0 & rs.ring_mask;
            // all 16 rows belong to the window and do not wrap the ring
            if (!MASKED && 16 * (jt + 1) <= S && t0 + 16 <= rs.t_limit &&
                (rs.ring_mask < 0 || row0 + 16 <= rs.ring_mask + 1))
                return load_bytes<A>(rs.x_f + (size_t)row0 * rs.row_stride + lane_off);
            TileBytes<A> r;
#pragma unroll
            for (int i = 0; i < KS; ++i) r.w[i] = 0u;
            const long t = t0 + col;
            const size_t row = (size_t)(t & rs.ring_mask);
            if (16 * jt + col < S && t < rs.t_limit &&
                (!MASKED || rs.valid_f[row * rs.mask_stride] != 0))
                r = load_bytes<A>(rs.x_f + row * rs.row_stride + G * (A / 4));
            return r;
        };
        float win[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) win[nt] = 0.0f;
        auto epilogue = [&](int jt, const bf_float4 (&acc)[NT]) {
            if (INTEGRATE) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) win[nt] = fmaf(acc[nt][r], acc[nt][r], win[nt]);
                return;
            }
            // the two lanes of a Re/Im pair split the rows
            const int in_win = 16 * jt + 4 * G + odd;
            const long t = (long)w * S + in_win;
            float* const o = ot.out + ((size_t)t * ot.F + ot.f) * B + bl;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                auto power = [&](float y) { return y * y + dpp_swap_pairs(y * y); };
                const float p0 = power(acc[nt][0]), p1 = power(acc[nt][1]);
                const float p2 = power(acc[nt][2]), p3 = power(acc[nt][3]);
                const bool ok = bl + 8 * nt < B;
                if (ok && in_win < S && rs.t_base + t < rs.t_limit) o[8 * nt] = odd ? p1 : p0;
                if (ok && in_win + 2 < S && rs.t_base + t + 2 < rs.t_limit)
                    o[(size_t)2 * ot.F * B + 8 * nt] = odd ? p3 : p2;
            }
        };
        auto convert = [&](const TileBytes<A>& x, bf_uint4v (&av)[KS]) {
#pragma unroll
            for (int s = 0; s < KS; ++s) av[s] = int4_slots<PARTS>(x.w[s]);
        };
        auto contract = [&](const bf_uint4v (&av)[KS], bf_float4 (&acc)[NT]) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[nt] = bf_float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int q = PARTS - 1; q >= 0; --q)
#pragma unroll
                for (int s = 0; s < KS; ++s)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        acc[nt] = mfma<PARTS>(av[s], bw[q][nt][s], acc[nt]);
        };
        // Tiles [0, n_fast): whole groups of D full tiles that do not wrap the
        // ring.  They run as straight code, each tile's conversion written
        // between the MFMAs of the tile before, where it costs no time.
        int n_fast = 0;
        const long row0 = t_win & rs.ring_mask;
        if (kPipelined<A, ANCHORED, MASKED>) {
            long full = S >> 4;
            const long room = (rs.t_limit - t_win) >> 4;
            full = full < room ? full : room;
            if (rs.ring_mask >= 0) {
                const long left = (rs.ring_mask + 1 - row0) >> 4;
                full = full < left ? full : left;
            }
            n_fast = full > 0 ? (int)full / D * D : 0;
        }
        const uint8_t* x_next = rs.x_f + (size_t)row0 * rs.row_stride;
        const size_t tile_stride = (size_t)16 * rs.row_stride;
        // With a loss mask a row's byte travels beside its voltages and clears
        // them where they are converted: neither load waits for the other.
        const uint8_t* valid_next =
            MASKED ? rs.valid_f + (size_t)(row0 + col) * rs.mask_stride : nullptr;
        TileBytes<A> buf[D];
        uint8_t valid[D];
        auto load_next = [&](int u) {
            if (MASKED) valid[u] = valid_next[(size_t)(16 * u) * rs.mask_stride];
            buf[u] = load_bytes<A>(x_next + u * tile_stride + lane_off);
        };
        auto convert_next = [&](int u, bf_uint4v (&av)[KS]) {
            TileBytes<A> x = buf[u];
            if (MASKED) {
                const unsigned keep = valid[u] != 0 ? ~0u : 0u;
#pragma unroll
                for (int s = 0; s < KS; ++s) x.w[s] &= keep;
            }
            convert(x, av);
        };
        if (n_fast > 0) {
#pragma unroll
            for (int u = 0; u < D; ++u) load_next(u);
        } else {
#pragma unroll
            for (int u = 0; u < D; ++u)
                if (u < tpw) buf[u] = load_tile(u);
        }
        window_operands<A, NT, PARTS, ANCHORED>(da, rows, ch, w, since,
                                                 since == 0 || w == w_begin, beam0, lane, direct,
                                                 anc, bw);
        if (n_fast > 0) {
            bf_uint4v av[2][KS];
            auto group = [&](auto more, int j0) {
                constexpr bool MORE = decltype(more)::value;
                x_next += D * tile_stride;
                if (MASKED) valid_next += (size_t)(16 * D) * rs.mask_stride;
#pragma unroll
                for (int u = 0; u < D; ++u) {
                    bf_float4 acc[NT];
                    contract(av[u & 1], acc);
                    if (MORE) load_next(u);
                    if (MORE || u + 1 < D) convert_next((u + 1) % D, av[(u + 1) & 1]);
                    epilogue(j0 + u, acc);
                    if (INTEGRATE) {
#pragma unroll
                        for (int i = 0; i < PARTS * KS * NT; ++i) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
                        }
                    }
                }
            };
            convert_next(0, av[0]);
            int j0 = 0;
#pragma unroll 1
            for (; j0 + D < n_fast; j0 += D) group(std::true_type{}, j0);
            group(std::false_type{}, j0);
        }
#pragma unroll 1
        for (int j0 = n_fast; j0 < tpw; j0 += D) {
            if (j0 > 0) {
#pragma unroll
                for (int u = 0; u < D; ++u)
                    if (j0 + u < tpw) buf[u] = load_tile(j0 + u);
            }
#pragma unroll
            for (int u = 0; u < D; ++u) {
                if (j0 + u >= tpw) break;  // uniform
                bf_float4 acc[NT];
                if constexpr (KS <= 8) {
                    bf_uint4v av[KS];
                    convert(buf[u], av);
                    contract(av, acc);
                } else {
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) acc[nt] = bf_float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        const bf_uint4v av = int4_slots<PARTS>(buf[u].w[s]);
#pragma unroll
                        for (int q = PARTS - 1; q >= 0; --q)
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
                                acc[nt] = mfma<PARTS>(av, bw[q][nt][s], acc[nt]);
                    }
                }
                epilogue(j0 + u, acc);
            }
        }
        if (INTEGRATE) {
            const long slot = ot.out_windows > 0 ? (long)w % ot.out_windows : (long)w;
            float* const o = ot.out + ((size_t)slot * ot.F + ot.f) * B + bl;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                float v = win[nt];
                v += __shfl_xor(v, 16);
                v += __shfl_xor(v, 32);
                v += dpp_swap_pairs(v);
                if (G == 0 && !odd && bl + 8 * nt < B) o[8 * nt] = v;
            }
        }
    }
}

// Two waves per SIMD, or three where they almost fit by themselves (one
// N-tile, few antennas: windows of 10, 320 spectra, 64 antennas 16 against 19 us).
constexpr int min_waves(int A, int NT, int PARTS) {
    return NT == 1 && A <= 64 && PARTS <= 2 ? 3 : 2;
}

template <int A, int NT, int PARTS, bool INTEGRATE, bool ANCHORED>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(min_waves(A, NT, PARTS))))
void tracker_wave_kernel(const uint8_t* __restrict__ x, Geom geo, DirArgs da,
                         float* __restrict__ out, int T, int F, int n_windows, int run, int blocks,
                         long n_tasks, int per_xcd) {
    __shared__ Positions<A> pos;
    // Workgroups are dealt round-robin to the 8 XCDs; each XCD takes a
    // contiguous range of tasks.
    const long group = (long)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    const long task = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWaveSize)) +
                      group * kWaves;
    stage_positions<A>(geo, pos);
    __syncthreads();
    if (task >= n_tasks) return;  // whole wave, after the only barrier
    const int block = (int)(task % blocks);
    const long rest = task / blocks;
    const int f = (int)(rest % F);
    const int w_begin = (int)(rest / F) * run;
    const int w_end = w_begin + run < n_windows ? w_begin + run : n_windows;
    Channel<A> ch{pos, {0.0f, 0.0f, 0.0f}, turns_per_metre(channel_frequency(geo, f))};
    geometry_reach<A>(geo, threadIdx.x & (kWaveSize - 1), ch.reach);
    const RowSource rs{x + (size_t)f * A, (unsigned)(F * A), -1L, 0L, (long)T};
    const OutTarget ot{out, 0L, F, f};
    wave_windows<A, NT, PARTS, INTEGRATE, ANCHORED>(rs, ch, da, ot, w_begin, w_end,
                                                    block * NT * 8);
}

template <int A, int NT, int PARTS, bool INTEGRATE, bool ANCHORED>
void launch_nt(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da) {
    const size_t tpw = ceil_div(L.S, 16);
    const size_t blocks = ceil_div(L.B, (size_t)(NT * 8));
    // Windows per task: about 32 tiles, or an anchor's 16 windows; short windows
    // as long as two waves per SIMD remain (float weights, 32 antennas, 17
    // channels, 200 spectra, 3 beams, windows of 10: 32 tiles 32 us, this 10 us).
    size_t run = ANCHORED ? kAnchorWindows : ceil_div(32, tpw);
    if (L.S < (size_t)kDirectWeightMinSpectra)
        while (run > 1 && ceil_div(L.n_windows, run) * L.F * blocks < 2048) run /= 2;
    const size_t n_tasks = ceil_div(L.n_windows, run) * L.F * blocks;
    const size_t per_xcd = ceil_div(ceil_div(n_tasks, kWaves), kXcds);
    if (per_xcd * kXcds > (size_t)INT32_MAX)
        fail(BF_ERR_OVERFLOW, "tracker grid exceeds the supported size");
    hipLaunchKernelGGL((tracker_wave_kernel<A, NT, PARTS, INTEGRATE, ANCHORED>),
                       dim3((unsigned)(per_xcd * kXcds)), dim3(kThreads), 0, stream, L.x, L.geo,
                       da, L.out, (int)L.T, (int)L.F, (int)L.n_windows, (int)run, (int)blocks,
                       (long)n_tasks, (int)per_xcd);
}

// Beams per wave: as many 8-beam N-tiles as the beams need and the registers
// hold (A PARTS NT / 4 for the weights and A NT / 4 for the anchors), as long as
// about two waves per SIMD remain.
template <int A, int PARTS, bool INTEGRATE>
void launch_parts(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da) {
    constexpr int kMax = A * PARTS <= 128 ? 4 : (A * PARTS <= 256 ? 2 : 1);
    constexpr int kMax2 = kMax < 2 ? kMax : 2;
    auto tasks = [&](size_t nt) { return ceil_div(L.B, nt * 8) * L.F * L.n_windows; };
    const bool two = kMax >= 2 && L.B > 8 && tasks(2) >= 2048;
    if constexpr (PARTS <= 2) {  // float weights are never rotated
        if (L.S < (size_t)kDirectWeightMinSpectra) {
            constexpr int kMaxAnchored = A * (PARTS + 1) <= 256 ? kMax2 : 1;
            if (two && kMaxAnchored == 2)
                launch_nt<A, kMaxAnchored, PARTS, INTEGRATE, true>(stream, L, da);
            else
                launch_nt<A, 1, PARTS, INTEGRATE, true>(stream, L, da);
            return;
        }
    }
    if (kMax >= 4 && L.B > 16 && tasks(4) >= 2048)
        launch_nt<A, kMax, PARTS, INTEGRATE, false>(stream, L, da);
    else if (two)
        launch_nt<A, kMax2, PARTS, INTEGRATE, false>(stream, L, da);
    else
        launch_nt<A, 1, PARTS, INTEGRATE, false>(stream, L, da);
}

template <int A>
void launch_a(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da, int parts) {
#define BF_PARTS(P_)                                             \
    L.integrate ? launch_parts<A, P_, true>(stream, L, da)       \
                : launch_parts<A, P_, false>(stream, L, da)
    if (parts == 1)
        BF_PARTS(1);
    else if (parts == 2)
        BF_PARTS(2);
    else
        BF_PARTS(3);
#undef BF_PARTS
}

}  // namespace wave_detail

// The tracker for one antenna count (k_tracker_a*.hip); `parts`: weight
// slices 1, 2 or 3.
void launch_tracker_a32(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da, int parts);
void launch_tracker_a64(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da, int parts);
void launch_tracker_a128(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da, int parts);
void launch_tracker_a256(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da, int parts);

#define BF_DEFINE_TRACKER_FOR_A(A_)                                                        \
    void launch_tracker_a##A_(hipStream_t stream, const TrackerLaunch& L, const DirArgs& da, \
                              int parts) {                                                 \
        wave_detail::launch_a<A_>(stream, L, da, parts);                                   \
    }

}  // namespace bfhip
