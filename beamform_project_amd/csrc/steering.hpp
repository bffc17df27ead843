// steering.hpp -- array geometry and steering weights of the tracker
// kernels: w = (float)cos(phi), (float)sin(phi) with phi = (2 pi f / c)
// (p . d) (reference src/weights.cpp:37-55), evaluated for many (beam,
// antenna) pairs per window inside the kernels.
//
// The phase in turns, (p . d) f / c, is summed in FP64 onto 1.5 * 2^20, whose
// last place is 2^-32: the low word of the sum is the fraction of a turn as a
// 32-bit integer, right to 2^-31 of a turn, after three FP64 FMAs.  Integer
// operations then split off the quadrant, and the rest, |x| <= pi/4 carried
// as a float and its remainder, goes through polynomials for sin and cos (to
// x^7 and x^8: least-maximum fits, off by 2.2e-9 and 1.7e-9).  Over random
// geometries the result is off by at most 8.2e-8 and 1.84e-8 rms, in some 36
// instructions; a reduced FP64 phase and sincosf took about 90 and were off by
// 1.00e-7 and 2.14e-8.  Where the caller asks for float weights (the tracker's
// FP32 selector with several beams or integration) the phase stays in FP64 and
// the weight is rounded once, off by 2^-25 (cos_sin_turns64).
#pragma once

#include "bf_tracker.hpp"

namespace bfhip {

struct DirArgs {
    const float* table;  // directions [n_windows_table][B][3], or null for
    const float* traj;   // trajectories [B][4] = l0, m0, rate_l, rate_m, or null for
    float row[4];        // the only beam's trajectory
    long window_offset;  // absolute index of local window 0; 0 with a table
    int S;
    int B;
};

// What a beam's direction is made of besides the window: its trajectory's row
// (kept in registers over a run of windows), or nothing with a table.
struct BeamRow {
    float q[4];
};
__device__ __forceinline__ BeamRow beam_row(const DirArgs& da, int b) {
    BeamRow r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        r.q[i] = da.table != nullptr ? 0.0f
                                     : (da.traj != nullptr ? da.traj[(size_t)b * 4 + i] : da.row[i]);
    return r;
}

// Direction of beam b in local window w: the table's, or
// l = l0 + (float)t * rate_l, n = sqrt(1 - l^2 - m^2)
// (src/beam_tracker.cpp:166-179, src/geometry.cpp:97-106).
__device__ __forceinline__ void beam_direction(const DirArgs& da, const BeamRow& row, int w, int b,
                                               float d[3]) {
    if (da.table != nullptr) {
        const float* p = da.table + ((size_t)w * da.B + b) * 3;
        d[0] = p[0];
        d[1] = p[1];
        d[2] = p[2];
    } else {
        const float* q = row.q;
        const float tf = (float)((da.window_offset + w) * (long)da.S);
        const float l = q[0] + tf * q[2];
        const float m = q[1] + tf * q[3];
        const float t2 = l * l + m * m;
        d[0] = l;
        d[1] = m;
        d[2] = __builtin_sqrtf(1.0f - t2);
    }
}

// Antenna position: a device table, or the reference's regular grid
// (src/geometry.cpp:33-67: x = column * spacing, y = row * spacing).
__device__ __forceinline__ void antenna_position(const Geom& geo, int a, float p[3]) {
    if (geo.pos != nullptr) {
        p[0] = geo.pos[3 * a];
        p[1] = geo.pos[3 * a + 1];
        p[2] = geo.pos[3 * a + 2];
    } else {
        p[0] = (float)(a % geo.cols) * geo.spacing;
        p[1] = (float)(a / geo.cols) * geo.spacing;
        p[2] = 0.0f;
    }
}

// Channel frequency: a device table, or src/geometry.cpp:79-95.
__device__ __forceinline__ float channel_frequency(const Geom& geo, int f) {
    if (geo.freqs != nullptr) return geo.freqs[f];
    const float step = (float)f * geo.f_step;
    return geo.f_start + step;
}

// sin and cos of the angle whose fraction of a turn is i 2^-32.
__device__ __forceinline__ float2 cos_sin_turns(unsigned i) {
    const unsigned u = i + 0x20000000u;
    const unsigned quad = u >> 30;
    const int rem = (int)(u & 0x3FFFFFFFu) - 0x20000000;  // [-1/8, 1/8) turn
    const float rh = (float)rem;
    const float rl = (float)(rem - (int)rh);  // |rh| <= 2^29
    constexpr float kHi = 0x1.921fb6p-30f;            // 2 pi 2^-32 as a float
    constexpr float kLo = -0x1.777a5cp-55f;           // and its remainder
    const float x = rh * kHi;
    const float xl = fmaf(rl, kHi, fmaf(rh, kLo, fmaf(rh, kHi, -x)));
    const float z = x * x;
    float p = fmaf(z, -0x1.98da36p-13f, 0x1.1105b4p-7f);
    p = fmaf(z, p, -0x1.555540p-3f);
    float q = fmaf(z, 2.439040872559417e-05f, -0.0013886763481423259f);
    q = fmaf(z, q, 0.04166662320494652f);
    q = fmaf(z, q, -0.5f);
    const float s0 = fmaf(x * z, p, x);
    const float c0 = fmaf(z, q, 1.0f);
    const float s = fmaf(xl, c0, s0);
    const float c = fmaf(-xl, s0, c0);
    const bool swap = (quad & 1u) != 0;
    const unsigned cs = __builtin_bit_cast(unsigned, swap ? s : c) ^ (((quad + 1u) << 30) & 0x80000000u);
    const unsigned sn = __builtin_bit_cast(unsigned, swap ? c : s) ^ ((quad << 30) & 0x80000000u);
    return make_float2(__builtin_bit_cast(float, cs), __builtin_bit_cast(float, sn));
}

// cos and sin of v turns in FP64, any finite v (else NaN): the quadrant split
// off exactly, then the Taylor series on |x| <= pi/4 (to x^17 and x^16: the
// next terms are below 2^-56).
__device__ __forceinline__ double2 cos_sin_turns64(double v) {
    const double v4 = 4.0 * (v - rint(v));  // exact
    const double n = rint(v4);
    const double x = (v4 - n) * (0.25 * kTwoPi);
    const double z = x * x;
    double p = 1.0 / 355687428096000.0;
    p = fma(z, p, -1.0 / 1307674368000.0);
    p = fma(z, p, 1.0 / 6227020800.0);
    p = fma(z, p, -1.0 / 39916800.0);
    p = fma(z, p, 1.0 / 362880.0);
    p = fma(z, p, -1.0 / 5040.0);
    p = fma(z, p, 1.0 / 120.0);
    p = fma(z, p, -1.0 / 6.0);
    double q = 1.0 / 20922789888000.0;
    q = fma(z, q, -1.0 / 87178291200.0);
    q = fma(z, q, 1.0 / 479001600.0);
    q = fma(z, q, -1.0 / 3628800.0);
    q = fma(z, q, 1.0 / 40320.0);
    q = fma(z, q, -1.0 / 720.0);
    q = fma(z, q, 1.0 / 24.0);
    q = fma(z, q, -0.5);
    const double s = fma(x * z, p, x);
    const double c = fma(z, q, 1.0);
    const int quad = (int)n & 3;  // n = -2 .. 2
    const double cs = (quad & 1) ? s : c;
    const double sn = (quad & 1) ? c : s;
    return make_double2((quad == 1 || quad == 2) ? -cs : cs, (quad & 2) ? -sn : sn);
}

// Turns per metre of a channel.
__device__ __forceinline__ double turns_per_metre(float f_hz) {
    return (double)f_hz / kSpeedOfLight;
}

// Steering direction of one beam and channel: the direction times f / c, and
// whether every antenna's phase fits the integer form (below 2^18 turns; no
// infinity or NaN anywhere).
struct Steer {
    double d[3];
    bool in_range;
};

// `reach`: per axis the largest |p|, as reach_max forms it.
__device__ __forceinline__ Steer make_steer(const float d[3], double per_metre,
                                            const float reach[3]) {
    Steer s;
    float bound = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        s.d[i] = (double)d[i] * per_metre;
        bound += reach[i] * fabsf((float)s.d[i]);
    }
    s.in_range = bound < 262144.0f;
    return s;
}

// Larger of two magnitudes by their bits (a NaN counts as the largest), and
// the largest |p| per axis over the A antennas, by a whole wave.
__device__ __forceinline__ float reach_max(float a, float b) {
    const unsigned x = __builtin_bit_cast(unsigned, a) & 0x7FFFFFFFu;
    const unsigned y = __builtin_bit_cast(unsigned, b) & 0x7FFFFFFFu;
    return __builtin_bit_cast(float, x > y ? x : y);
}

template <int A>
__device__ __forceinline__ void geometry_reach(const Geom& geo, int lane, float (&reach)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) reach[i] = 0.0f;
    for (int a = lane; a < A; a += 64) {
        float p[3];
        antenna_position(geo, a, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) reach[i] = reach_max(reach[i], p[i]);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) reach[i] = reach_max(reach[i], __shfl_xor(reach[i], o));
}

// The weight where the phase fits the integer form.
__device__ __forceinline__ float2 steering_weight_near(const double* p, const Steer& st) {
    double t = fma(p[0], st.d[0], 0x1.8p20);
    t = fma(p[1], st.d[1], t);
    t = fma(p[2], st.d[2], t);
    return cos_sin_turns((unsigned)__builtin_bit_cast(unsigned long long, t));
}

// The weight of any phase: outside that range it is reduced in FP64 first,
// and one that is not finite gives NaN.
__device__ __forceinline__ float2 steering_weight_any(const double* p, const Steer& st) {
    if (st.in_range) return steering_weight_near(p, st);
    const double t = fma(p[2], st.d[2], fma(p[1], st.d[1], p[0] * st.d[0]));
    const double r = t - rint(t);
    const float nan = (float)(r * 0.0);  // 0, or NaN
    const float2 v =
        cos_sin_turns((unsigned)__builtin_bit_cast(unsigned long long, r + 0x1.8p20));
    return make_float2(v.x + nan, v.y + nan);
}

// The weight in FP64, rounded once; a phase that is not finite gives NaN.
__device__ __forceinline__ float2 steering_weight_exact(const double* p, const Steer& st) {
    const double t = fma(p[2], st.d[2], fma(p[1], st.d[1], p[0] * st.d[0]));
    const double2 v = cos_sin_turns64(t);
    return make_float2((float)v.x, (float)v.y);
}

}  // namespace bfhip
