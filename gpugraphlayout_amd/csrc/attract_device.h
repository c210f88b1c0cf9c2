// Device functions of the attraction and gravity shared by its kernels.
#pragma once
#include "engine_internal.h"

namespace gfa2 {

// What the attraction reads and writes.
struct AttractArgs {
    const float2* pos;
    const float* mass;
    int n;
    const float2* pos_rank;
    const int* rowptr;
    const int* col;              // ranks
    const int* lists;
    int nlight, nmedium;
    int strong;
    float k_g;
    float2* fga;
    int linlog;
    const float* ew;
};

__device__ __forceinline__ float2 gravity(float2 p, float m, int strong, float k_g) {
    float fg;
    if (strong) fg = k_g * m;
    else if (p.x != 0.0f || p.y != 0.0f) fg = k_g * m * rsqrtf(p.x * p.x + p.y * p.y);
    else fg = 0.0f;
    return make_float2(-p.x * fg, -p.y * fg);
}

// One edge's attraction term on node p from neighbour q. Linear: q - p. With linlog (the
// reference's CPU rule, src/RPCPUForceAtlas2.cpp:63-67): (q - p) * log(1 + d) / d, and 0 at
// d = 0 (the reference multiplies the zero vector by FLT_MAX there). With edge weights:
// times w^delta.
template <bool GEN>
__device__ __forceinline__ void attract_term(float2 p, float2 q, int linlog, const float* __restrict__ ew, int e,
                                             float& ax, float& ay) {
    const float dx = q.x - p.x;
    const float dy = q.y - p.y;
    if constexpr (!GEN) {
        ax += dx;
        ay += dy;
    } else {
        float fa = 1.0f;
        if (linlog) {
            const float d = sqrtf(dx * dx + dy * dy);
            fa = d == 0.0f ? 0.0f : logf(1.0f + d) / d;
        }
        if (ew) fa *= ew[e];
        ax += dx * fa;
        ay += dy * fa;
    }
}

// The terms of CSR entries e, e + S, e + 2S, ... below e1, added in that order. Four entries at
// a time: their index and position loads are all issued before the first term is added (the
// loads past e1 read node 0 and are not added), so a row's tail costs no more round trips to
// memory than a full group of four.
// With HUB, the positions of the kHubCache highest-degree nodes come from the block's LDS copy
// (hub), which spares the L2 the most requested lines.
constexpr int kHubCache = 2048;

template <bool GEN, int S, bool HUB>
__device__ __forceinline__ void gather_terms(float2 p, const float2* __restrict__ pos_rank,
                                             const float2* hub, const int* __restrict__ col, int e, int e1,
                                             int linlog, const float* __restrict__ ew, float& ax, float& ay) {
    for (; e < e1; e += 4 * S) {
        int j[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) j[u] = e + u * S < e1 ? col[e + u * S] : 0;
        float2 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (HUB && j[u] < kHubCache) q[u] = hub[j[u]];
            else q[u] = pos_rank[j[u]];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (e + u * S < e1) attract_term<GEN>(p, q[u], linlog, ew, e + u * S, ax, ay);
    }
}

// Light row k of the list (one thread): gravity + the row's entries in order.
template <bool GEN, bool HUB>
__device__ __forceinline__ void attract_light(int k, const AttractArgs& A, const float2* hub) {
    if (k >= A.nlight) return;
    const int v = A.lists[k];
    const float2 p = A.pos[v];
    float ax = 0.0f, ay = 0.0f;
    gather_terms<GEN, 1, HUB>(p, A.pos_rank, hub, A.col, A.rowptr[v], A.rowptr[v + 1], A.linlog, A.ew, ax, ay);
    const float2 g = gravity(p, A.mass[v], A.strong, A.k_g);
    A.fga[v] = make_float2(g.x + ax, g.y + ay);
}

// Medium row k (one wave): lane-strided sums, then a butterfly.
template <bool GEN, bool HUB>
__device__ __forceinline__ void attract_medium(int k, int lane, const AttractArgs& A, const float2* hub) {
    if (k >= A.nmedium) return;      // uniform per wave
    const int v = A.lists[A.nlight + k];
    const float2 p = A.pos[v];
    float ax = 0.0f, ay = 0.0f;
    gather_terms<GEN, 64, HUB>(p, A.pos_rank, hub, A.col, A.rowptr[v] + lane, A.rowptr[v + 1], A.linlog, A.ew, ax, ay);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ax += __shfl_xor(ax, o, 64);
        ay += __shfl_xor(ay, o, 64);
    }
    if (lane == 0) {
        const float2 g = gravity(p, A.mass[v], A.strong, A.k_g);
        A.fga[v] = make_float2(g.x + ax, g.y + ay);
    }
}

}  // namespace gfa2
