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

// A node's force from its position, mass and attraction: gravity added. Here and in the other terms
// every fused multiply-add is written out: left to the compiler, which product of a sum of two is
// fused differs from kernel to kernel, and with it the last bit.
__device__ __forceinline__ float2 add_gravity(float2 p, float m, int strong, float k_g, float ax, float ay) {
    float fg;
    if (strong) fg = k_g * m;
    else if (p.x != 0.0f || p.y != 0.0f) fg = k_g * m * rsqrtf(fmaf(p.x, p.x, p.y * p.y));
    else fg = 0.0f;
    return make_float2(fmaf(-p.x, fg, ax), fmaf(-p.y, fg, ay));
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
            const float d = sqrtf(fmaf(dx, dx, dy * dy));
            fa = d == 0.0f ? 0.0f : logf(1.0f + d) / d;
        }
        if (ew) fa *= ew[e];
        ax = fmaf(dx, fa, ax);
        ay = fmaf(dy, fa, ay);
    }
}

// One row, or a part of one: len CSR entries from first.
struct Row {
    const int* col;
    const float* ew;
    int len;
    __device__ __forceinline__ Row(const AttractArgs& A, int first, int end)
        : col(A.col + first), ew(A.ew ? A.ew + first : nullptr), len(end - first) {}
};

// Entries i, i + S, i + 2S, i + 3S of the row (0 past its end) ...
template <int S>
__device__ __forceinline__ void load_four(const Row& R, int i, int (&j)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) j[u] = i + u * S < R.len ? R.col[i + u * S] : 0;
}

// ... and their terms, added in that order. The position loads are all issued before the first
// term is added (those past the end read node 0 and are not added), so a row's tail costs no more
// round trips to memory than a full group of four.
// The positions of the HUB highest-degree nodes (HUB > 0) come from the block's LDS copy (hub),
// which spares the L2 the most requested lines.
template <int HUB>
__device__ __forceinline__ void load_positions(const float2* __restrict__ pos_rank, const float2* hub,
                                               const int (&j)[4], float2 (&q)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if (j[u] < HUB) q[u] = hub[j[u]];
        else q[u] = pos_rank[j[u]];
    }
}

template <bool GEN, int S>
__device__ __forceinline__ void add_four(float2 p, const Row& R, int i, const float2 (&q)[4], int linlog, float& ax,
                                         float& ay) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (i + u * S < R.len) attract_term<GEN>(p, q[u], linlog, R.ew, i + u * S, ax, ay);
}

// The terms of entries i, i + S, i + 2S, ... of the row, four at a time.
template <bool GEN, int S, int HUB>
__device__ __forceinline__ void gather_terms(float2 p, const AttractArgs& A, const float2* hub, const Row& R, int i,
                                             float& ax, float& ay) {
    for (; i < R.len; i += 4 * S) {
        int j[4];
        load_four<S>(R, i, j);
        float2 q[4];
        load_positions<HUB>(A.pos_rank, hub, j, q);
        add_four<GEN, S>(p, R, i, q, A.linlog, ax, ay);
    }
}

// Light row k of the list (one thread): gravity + the row's entries in order.
template <bool GEN, int HUB>
__device__ __forceinline__ void attract_light(int k, const AttractArgs& A, const float2* hub) {
    if (k >= A.nlight) return;
    const int v = A.lists[k];
    const float2 p = A.pos[v];
    float ax = 0.0f, ay = 0.0f;
    gather_terms<GEN, 1, HUB>(p, A, hub, Row(A, A.rowptr[v], A.rowptr[v + 1]), 0, ax, ay);
    A.fga[v] = add_gravity(p, A.mass[v], A.strong, A.k_g, ax, ay);
}

// Medium rows k0 to k0 + rows - 1 (one wave, rows <= kMediumBatch): lane-strided sums, then a
// butterfly. What bounds a row of some hundred entries is its chain of dependent loads (id, bounds,
// indices, positions). So the rows' ids, bounds and positions are read by a lane each, and the
// next row's first 256 indices are under way while this row's positions arrive. R-MAT 2^22 (64M
// entries, 278k such rows): the attraction 462 -> 424 us with the blocks' order in k_attract; batches
// of 8 are slower where long rows follow one another (BA, 1M bodies: 663 -> 702 us an iteration).
constexpr int kMediumBatch = 4;

template <bool GEN, int HUB>
__device__ __forceinline__ void attract_medium(int k0, int rows, int lane, const AttractArgs& A, const float2* hub) {
    k0 = __builtin_amdgcn_readfirstlane(k0);
    const int nb = min(rows, A.nmedium - k0);
    if (nb <= 0) return;             // uniform per wave
    int v = 0, e0 = 0, e1 = 0;
    float2 p = make_float2(0.0f, 0.0f), sum = p;
    if (lane < nb) {
        v = A.lists[A.nlight + k0 + lane];
        e0 = A.rowptr[v];
        e1 = A.rowptr[v + 1];
        p = A.pos[v];
    }
    int j[4];
    load_four<64>(Row(A, __builtin_amdgcn_readlane(e0, 0), __builtin_amdgcn_readlane(e1, 0)), lane, j);
    for (int r = 0; r < nb; ++r) {
        const Row R(A, __builtin_amdgcn_readlane(e0, r), __builtin_amdgcn_readlane(e1, r));
        const float2 pr = make_float2(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(p.x), r)),
                                      __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p.y), r)));
        float2 q[4];
        load_positions<HUB>(A.pos_rank, hub, j, q);
        if (r + 1 < nb)
            load_four<64>(Row(A, __builtin_amdgcn_readlane(e0, r + 1), __builtin_amdgcn_readlane(e1, r + 1)), lane, j);
        float ax = 0.0f, ay = 0.0f;
        add_four<GEN, 64>(pr, R, lane, q, A.linlog, ax, ay);
        gather_terms<GEN, 64, HUB>(pr, A, hub, R, lane + 256, ax, ay);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            ax += __shfl_xor(ax, o, 64);
            ay += __shfl_xor(ay, o, 64);
        }
        if (lane == r) sum = make_float2(ax, ay);
    }
    if (lane < nb) A.fga[v] = add_gravity(p, A.mass[v], A.strong, A.k_g, sum.x, sum.y);
}

// Block i of the light and medium ones, which take turns in proportion (256 threads).
template <bool GEN, int HUB>
__device__ __forceinline__ void attract_rows(int i, int light_blocks, int medium_blocks, int medium_rows, int tid,
                                             const AttractArgs& A, const float2* hub) {
    const unsigned int t = light_blocks + medium_blocks;
    const int m0 = (int)((unsigned long long)i * medium_blocks / t);          // medium blocks before i
    const int m1 = (int)((i + 1ull) * medium_blocks / t);
    if (m1 > m0) attract_medium<GEN, HUB>((m0 * 4 + (tid >> 6)) * medium_rows, medium_rows, tid & 63, A, hub);
    else attract_light<GEN, HUB>((i - m0) * 256 + tid, A, hub);
}

// red[0] = the sum over 256 threads. red[0] is written again only by thread 0, and every other
// entry only after the barriers here, so thread 0 may read it after the call.
__device__ __forceinline__ void sum_chunk(float2* red, int tid, float ax, float ay) {
    red[tid] = make_float2(ax, ay);
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            const float2 a = red[tid], b = red[tid + o];
            red[tid] = make_float2(a.x + b.x, a.y + b.y);
        }
        __syncthreads();
    }
}

// Chunk c of a heavy row (a block of 256 threads): thread-strided sums, then an LDS tree.
template <bool GEN, int HUB>
__device__ __forceinline__ void attract_chunk(int c, const int2* __restrict__ chunks, float2* __restrict__ part, int tid,
                                              const AttractArgs& A, const float2* hub, float2* red) {
    const int2 ch = chunks[c];
    const int v = A.lists[A.nlight + A.nmedium + ch.x];
    const float2 p = A.pos[v];
    float ax = 0.0f, ay = 0.0f;
    const int len = min(kAttrChunk, A.rowptr[v + 1] - ch.y);
    gather_terms<GEN, 256, HUB>(p, A, hub, Row(A, ch.y, ch.y + len), tid, ax, ay);
    sum_chunk(red, tid, ax, ay);
    if (tid == 0) part[c] = red[0];
}

// What a launch of the attraction covers: chunks, then light and medium blocks (256 threads each).
struct AttractPlan {
    int light_blocks, medium_blocks, medium_rows, chunks;
    int total;
};

// One of a plan's blocks, without a copy of the hubs.
template <bool GEN>
__device__ __forceinline__ void attract_block(int vb, const AttractPlan& w, const int2* __restrict__ chunks,
                                              float2* __restrict__ part, const AttractArgs& A, float2* red) {
    if (vb < w.chunks) attract_chunk<GEN, 0>(vb, chunks, part, threadIdx.x, A, nullptr, red);
    else attract_rows<GEN, 0>(vb - w.chunks, w.light_blocks, w.medium_blocks, w.medium_rows, threadIdx.x, A, nullptr);
}

AttractPlan attract_plan(const Bufs& b);
AttractArgs attract_args(const Bufs& b, const Params& p);
void launch_attract_heavy(const Bufs& b, const Params& p, hipStream_t s);

}  // namespace gfa2
