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

}  // namespace gfa2
