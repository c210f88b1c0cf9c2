// Device functions shared by the tree kernels: path keys and exact moments.
#pragma once
#include "engine_internal.h"

namespace gfa2 {

__device__ __forceinline__ int lcp_levels(unsigned long long a, unsigned long long b) {
    unsigned long long x = a ^ b;
    return x == 0ull ? kKeyLevels : (__clzll((long long)x) >> 1);
}

// A body's path: 32 quadrant digits (bit 0: x, bit 1: y), obtained by replaying the reference's
// float centre arithmetic (src/RPBHKernels.cu:217-241, :292-308).
__device__ __forceinline__ unsigned long long path_key(float2 p, float rootx, float rooty, float radius) {
    float r = radius * 0.5f;
    bool bx = rootx < p.x, by = rooty < p.y;
    float x = rootx + (bx ? r : -r);
    float y = rooty + (by ? r : -r);
    unsigned long long key = (unsigned long long)((unsigned)bx | ((unsigned)by << 1)) << 62;
#pragma unroll
    for (int l = 1; l < kKeyLevels; ++l) {
        r *= 0.5f;
        bx = x < p.x;
        by = y < p.y;
        key |= (unsigned long long)((unsigned)bx | ((unsigned)by << 1)) << (62 - 2 * l);
        x += bx ? r : -r;
        y += by ? r : -r;
    }
    return key;
}

// Exact moments (integer-mass path). Sums are taken modulo 2^128 on two 64-bit limbs.
using u128 = unsigned __int128;

// Fixed-point exponent of a graph whose root radius is R < 2^e: a coordinate relative to the
// root centre lies within a few R (the centre and radius are rounded floats), so scaled by
// 2^(58-e) it stays below 2^61 in magnitude. R = 0 (one point) gives coordinates 0.
__device__ __forceinline__ int moment_shift(float radius) {
    int e = 0;
    (void)frexpf(radius, &e);
    return 58 - e;
}

__device__ __forceinline__ long long fixed_coord(float p, float c, int s) {
    double t = ldexp((double)p - (double)c, s);
    t = fmin(fmax(t, -0x1p62), 0x1p62);
    return (long long)rint(t);
}

// The signed 128-bit value hi*2^64 + lo as a double (magnitude converted, so small negative
// values keep their precision).
__device__ __forceinline__ double i128_to_double(unsigned long long lo, unsigned long long hi) {
    u128 v = ((u128)hi << 64) | lo;
    const bool neg = (long long)hi < 0;
    if (neg) v = (u128)0 - v;
    const unsigned long long vh = (unsigned long long)(v >> 64), vl = (unsigned long long)v;
    const double mag = vh == 0ull ? (double)vl : (double)vh * 0x1p64 + (double)vl;
    return neg ? -mag : mag;
}

// Prefix moments over sorted bodies: q = fixed-point coordinate = 2^31 h + l with 0 <= l < 2^31, so
// the sums of m h and m l stay within 64 bits for integer masses of under 2^30 together, and
// 2^31 sum(m h) + sum(m l) is the exact 128-bit moment.
// (Sums wrap: a difference of two prefix sums is exact if it is within 64 bits itself.)
template <typename M>
struct SplitOf {
    long long xh, xl, yh, yl;
    M m;
};

__device__ __forceinline__ long long wrap_add(long long a, long long b) {
    return (long long)((unsigned long long)a + (unsigned long long)b);
}

__device__ __forceinline__ long long wrap_sub(long long a, long long b) {
    return (long long)((unsigned long long)a - (unsigned long long)b);
}

template <typename M>
__device__ __forceinline__ SplitOf<M> split_of(float4 b, float4 c) {
    const int s = moment_shift(c.z);
    const long long m = (long long)b.z;
    const long long qx = fixed_coord(b.x, c.x, s), qy = fixed_coord(b.y, c.y, s);
    return SplitOf<M>{m * (qx >> 31), m * (qx & 0x7fffffff), m * (qy >> 31), m * (qy & 0x7fffffff), (M)m};
}

template <typename M>
__device__ __forceinline__ SplitOf<M> operator+(const SplitOf<M>& a, const SplitOf<M>& b) {
    return SplitOf<M>{wrap_add(a.xh, b.xh), wrap_add(a.xl, b.xl), wrap_add(a.yh, b.yh), wrap_add(a.yl, b.yl), a.m + b.m};
}

template <typename M>
__device__ __forceinline__ SplitOf<M> operator-(const SplitOf<M>& a, const SplitOf<M>& b) {
    return SplitOf<M>{wrap_sub(a.xh, b.xh), wrap_sub(a.xl, b.xl), wrap_sub(a.yh, b.yh), wrap_sub(a.yl, b.yl), a.m - b.m};
}

// One step of a wave-wide scan by a data-parallel move (no LDS): the value of the lane the control
// word names, 0 where there is none or the row mask leaves the lane out.
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned int moved(unsigned int v) {
    return (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, true);
}

template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long moved(unsigned long long v) {
    const unsigned int lo = moved<CTRL, ROWS>((unsigned int)v);
    const unsigned int hi = moved<CTRL, ROWS>((unsigned int)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// Inclusive scan over the wave: within rows of 16 lanes (shifts by 1, 2, 4, 8), then lane 15 of a
// row into the next, then lane 31 into the upper half.
template <typename T>
__device__ __forceinline__ T wave_scan(T v) {
    v += moved<0x111, 0xf>(v);
    v += moved<0x112, 0xf>(v);
    v += moved<0x114, 0xf>(v);
    v += moved<0x118, 0xf>(v);
    v += moved<0x142, 0xa>(v);
    v += moved<0x143, 0xc>(v);
    return v;
}

template <typename M>
__device__ __forceinline__ SplitOf<M> wave_scan(const SplitOf<M>& v) {
    return SplitOf<M>{(long long)wave_scan((unsigned long long)v.xh), (long long)wave_scan((unsigned long long)v.xl),
                      (long long)wave_scan((unsigned long long)v.yh), (long long)wave_scan((unsigned long long)v.yl),
                      wave_scan(v.m)};
}

// The value of one lane (uniform).
__device__ __forceinline__ unsigned int from_lane(unsigned int v, int l) {
    return (unsigned)__builtin_amdgcn_readlane((int)v, l);
}

__device__ __forceinline__ unsigned long long from_lane(unsigned long long v, int l) {
    const unsigned int lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, l);
    const unsigned int hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l);
    return ((unsigned long long)hi << 32) | lo;
}

template <typename M>
__device__ __forceinline__ SplitOf<M> from_lane(const SplitOf<M>& v, int l) {
    return SplitOf<M>{(long long)from_lane((unsigned long long)v.xh, l), (long long)from_lane((unsigned long long)v.xl, l),
                      (long long)from_lane((unsigned long long)v.yh, l), (long long)from_lane((unsigned long long)v.yl, l),
                      from_lane(v.m, l)};
}

// The 128-bit moments.
template <typename M>
__device__ __forceinline__ u128 moment_x(const SplitOf<M>& v) {
    return ((u128)(__int128)v.xh << 31) + (u128)(__int128)v.xl;
}

template <typename M>
__device__ __forceinline__ u128 moment_y(const SplitOf<M>& v) {
    return ((u128)(__int128)v.yh << 31) + (u128)(__int128)v.yl;
}

}  // namespace gfa2
