// ForceAtlas2 force, speed and displacement kernels for gfx950 (FP32 VALU throughout).
#include "attract_device.h"
#include "engine_internal.h"

#include <algorithm>

namespace gfa2 {
namespace {

// ---------------------------------------------------------------------------------------
// Gravity + attraction, one pass over the symmetric CSR.
// Reference: GravityKernel (src/RPFA2Kernels.cu:35-73) and AttractiveForceKernel
// (:75-109). The reference adds each edge's p_t - p_s to F_s and its negation to F_t with
// four float atomics per edge, in no fixed order; here each node gathers
// sum_j (p_j - p_i) over its own row, which holds exactly the same terms, in a fixed
// order and without atomics. Nodes are pre-sorted into degree classes:
//   light (deg <= 32): one thread per node, sequential sum
//   medium (deg <= 2048): one wave per node, lane-strided sums + butterfly reduction
//   heavy: a 256-thread block per 4,096 entries, thread-strided sums + LDS tree reduction
// ---------------------------------------------------------------------------------------
// col_rank[e] = rank[col[e]] (once per graph).
__global__ __launch_bounds__(256) void k_gather_rank(const int* __restrict__ col, const int* __restrict__ rank,
                                                     long long nnz, int* __restrict__ col_rank) {
    for (long long e = blockIdx.x * 256ll + threadIdx.x; e < nnz; e += (long long)gridDim.x * 256)
        col_rank[e] = rank[col[e]];
}

// Attraction + gravity, fga[v] = gravity(v) + sum over CSR entries of v (in entry order for the
// light rows; lane-strided then a shuffle tree for medium rows; see below for heavy rows).
// Degree classes: light rows (<= 32 entries) one thread each, entries four at a time;
// medium rows (<= 2,048) one wave each, or up to kMediumBatch to a wave; heavy rows in chunks of kAttrChunk entries, one block
// per chunk writing its partial (thread-strided, then an LDS tree), added per row in chunk order
// by k_attract_heavy. Neighbour positions come from the degree-ranked copy. The work is a list
// of virtual blocks that the grid strides over: one launch block per virtual block by default, or
// a smaller grid that leaves room on every compute unit for kernels running beside it on another
// stream. Every row's sum is the same whatever the grid. The chunks come first, being longest;
// light and medium blocks then take turns in proportion, since the light rows wait on their
// serial loads and the medium ones on the L2 (1M bodies, 32M entries, half of them in either: 919 us
// an iteration with the light blocks first, 934 with them last, 888 in turns).
constexpr int kHubCache = 2048;      // hubs' positions in LDS: 16 KB, so that 8 blocks fit a CU

template <bool GEN, int HUB>
__global__ __launch_bounds__(256) void k_attract(const AttractArgs A, const int2* __restrict__ chunks, int nchunks,
                                                 int light_blocks, int medium_blocks, int medium_rows,
                                                 float2* __restrict__ part) {
    __shared__ float2 red[256];
    __shared__ float2 hub[HUB > 0 ? HUB : 1];
    const int tid = threadIdx.x;
    if constexpr (HUB > 0) {
        for (int i = tid; i < HUB && i < A.n; i += 256) hub[i] = A.pos_rank[i];
        __syncthreads();
    }
    const int total = light_blocks + medium_blocks + nchunks;
    for (int vb = blockIdx.x; vb < total; vb += gridDim.x) {   // uniform per block
        if (vb >= nchunks) {
            attract_rows<GEN, HUB>(vb - nchunks, light_blocks, medium_blocks, medium_rows, tid, A, hub);
            continue;
        }
        attract_chunk<GEN, HUB>(vb, chunks, part, tid, A, hub, red);
    }
}

// The same sums on one stream where many entries are of hubs: blocks of kWideThreads that stay on
// the chip, two to a compute unit, with the positions of the kWideHubs highest-degree nodes in
// 64 KB of LDS. The gathers are bound by the L2, which each serves as a request of its own, and by
// the lines it misses; the copy takes a third of the requests away (R-MAT 2^22: 33% of 64M
// entries). There 424 -> 368 us.
constexpr int kWideThreads = 1024, kWideSubs = kWideThreads / 256;

template <bool GEN>
__global__ __launch_bounds__(kWideThreads) void k_attract_wide(const AttractArgs A, const int2* __restrict__ chunks,
                                                               int nchunks, int light_blocks, int medium_blocks,
                                                               int medium_rows, float2* __restrict__ part) {
    __shared__ float2 hub[kWideHubs];
    __shared__ float2 red_all[kWideThreads];
    const int tid = threadIdx.x & 255, sub = threadIdx.x >> 8;
    float2* red = red_all + sub * 256;
    for (int i = threadIdx.x; i < kWideHubs && i < A.n; i += kWideThreads) hub[i] = A.pos_rank[i];
    __syncthreads();
    // chunks: one to each of the block's quarters at a time (the loop is uniform per block)
    for (int base = blockIdx.x * kWideSubs; base < nchunks; base += gridDim.x * kWideSubs) {
        const int c = base + sub;
        float ax = 0.0f, ay = 0.0f;
        if (c < nchunks) {
            const int2 ch = chunks[c];
            const int v = A.lists[A.nlight + A.nmedium + ch.x];
            const int len = min(kAttrChunk, A.rowptr[v + 1] - ch.y);
            gather_terms<GEN, 256, kWideHubs>(A.pos[v], A, hub, Row(A, ch.y, ch.y + len), tid, ax, ay);
        }
        sum_chunk(red, tid, ax, ay);
        if (tid == 0 && c < nchunks) part[c] = red[0];
    }
    // rows: no barriers, the quarters go on by themselves
    for (int i = blockIdx.x * kWideSubs + sub; i < light_blocks + medium_blocks; i += gridDim.x * kWideSubs)
        attract_rows<GEN, kWideHubs>(i, light_blocks, medium_blocks, medium_rows, tid, A, hub);
}

// Heavy rows: gravity + the row's chunk partials in chunk order.
__global__ __launch_bounds__(256) void k_attract_heavy(const float2* __restrict__ pos, const float* __restrict__ mass,
                                                       const int* __restrict__ heavy, int nheavy,
                                                       const int* __restrict__ c0, const float2* __restrict__ part,
                                                       int strong, float k_g, float2* __restrict__ fga) {
    const int h = blockIdx.x * 256 + threadIdx.x;
    if (h >= nheavy) return;
    const int v = heavy[h];
    float ax = 0.0f, ay = 0.0f;
    for (int c = c0[h]; c < c0[h + 1]; ++c) {
        ax += part[c].x;
        ay += part[c].y;
    }
    fga[v] = add_gravity(pos[v], mass[v], strong, k_g, ax, ay);
}

// A body's swing and traction terms (SpeedKernel, src/RPFA2Kernels.cu:111-161) from its total
// force F and previous force P: m |F - P| and m |F + P| / 2. The squared norms are written as
// explicit fmaf so that every kernel that forms them (walk, combine, exact) rounds alike.
__device__ __forceinline__ void swing_traction(float mi, float2 F, float2 P, float& sw, float& tr) {
    float dx = F.x - P.x, dy = F.y - P.y;
    sw = mi * sqrtf(fmaf(dx, dx, dy * dy));
    dx = F.x + P.x;
    dy = F.y + P.y;
    tr = mi * (sqrtf(fmaf(dx, dx, dy * dy)) * 0.5f);
}

// The end of a body's force evaluation in the exact kernel: total force
// F = F_ga + F_r, optional repulsion capture, and the group's swing/traction/interaction sums
// (SpeedKernel's per-body terms, src/RPFA2Kernels.cu:111-161), reduced within the G lanes.
template <int G>
__device__ __forceinline__ void group_finish(bool active, bool group_ok, int gl, int gidx, unsigned int id, float mi,
                                             float ax, float ay, unsigned int inter,
                                             const float2* __restrict__ fga, const float2* __restrict__ fprev,
                                             float2* __restrict__ f, float2* __restrict__ rep,
                                             WalkPart* __restrict__ part) {
    float sw = 0.0f, tr = 0.0f;
    if (active) {
        const float2 a = fga[id];
        const float2 F = make_float2(a.x + ax, a.y + ay);
        f[id] = F;
        if (rep) rep[id] = make_float2(ax, ay);
        swing_traction(mi, F, fprev[id], sw, tr);
    }
    // Reduce within the group (xor offsets below G stay inside it).
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        sw += __shfl_xor(sw, o, 64);
        tr += __shfl_xor(tr, o, 64);
        inter += __shfl_xor(inter, o, 64);
    }
    if (group_ok && gl == 0) {
        WalkPart wp;
        wp.swing = sw;
        wp.traction = tr;
        wp.interactions = inter;
        wp.pad = 0;
        part[gidx] = wp;
    }
}

// XCD-aware block order: consecutive logical blocks stay on one XCD's L2 (blocks are
// dealt to the 8 XCDs round-robin by hardware block id).
__device__ __forceinline__ int xcd_block() {
    const int nb = gridDim.x;
    const int xcd = blockIdx.x & 7;
    const int per = (nb + 7) >> 3;
    const int full = nb & 7;
    if (full == 0) return xcd * per + (blockIdx.x >> 3);
    return (xcd < full ? xcd * per : full * per + (xcd - full) * (per - 1)) + (blockIdx.x >> 3);
}

// ---------------------------------------------------------------------------------------
// Barnes-Hut repulsion walk. Reference: ForceCalculationKernel, src/RPBHKernels.cu:566-693.
//
// Groups of G consecutive bodies of a graph's sorted (in-order) permutation walk that graph's
// pre-order record array together; groups start at the graph's first sorted position, as the
// reference's warps start at position 0 (a graph in a batch is walked as it is alone). G = 32
// reproduces the reference's 32-lane warp vote; G = 64 votes over the whole wave. One
// wavefront walks one group in two parts:
//
//  traversal  records are tested 64 at a time, one per lane, taken from a stack of pending
//             record indices in LDS. A body record is always accepted. A cell at level L is accepted when every active body b of the group
//             has d2(b, c) >= dq[L-1] (the reference's all-lanes vote, :661), with
//             d2 = fma(dx, dx, fma(dy, dy, eps)) and dq[d] = (2 radius)^2 itolsq 0.25^d + eps
//             (:576-590, formed with ldexp, exact for the power-of-4 scaling). Most cells are
//             decided without the bodies one by one: d2 is monotone in |dx| and |dy|, so the
//             distance from the cell's centroid to the group's bounding box gives a float lower
//             bound of every body's d2 (accept when it clears dq), and the first, middle or
//             last body's own d2 below dq rejects. Only the cells left are voted on, body by
//             body, all lanes at once (lanes = bodies, as in the reference). An accepted record
//             is appended {x, y, k_r m} to an LDS list; an opened cell pushes all its 1-4
//             children at once (their record indices, listed per cell when the tree is
//             built), so a cell's children are tested in the same round (a cell of level 32 holds
//             any number of bodies: those past the fourth go to the list directly). The children go on
//             top, so the traversal runs depth-first in blocks of up to 64 records (one record
//             per round near the stack's capacity, where a depth-first walk adds at most three
//             entries per tree level).
//  sums       when the list is nearly full, and at the end, every body adds the list's terms
//             (k_r m_n) d / d2 (k_r m_n formed once per record as it is listed; hardware
//             reciprocal, where the reference divides) and multiplies the sum by its own mass
//             m_i at the end (the reference's k_r d m_i m_n / d2 per term, an ulp or two apart);
//             lanes 0-31 take the even entries and lanes 32-63 the odd ones when G = 32, added
//             together before the multiply.
// The accepted set is the reference's; the order of the terms is the traversal's (fixed for a
// given tree, so every launch shape and a graph alone or in a batch give the same bits).
// The epilogue adds gravity + attraction, writes the total force, and forms the group's
// swing/traction sums (SpeedKernel, src/RPFA2Kernels.cu:111-161).
// ---------------------------------------------------------------------------------------
// LDS per wave: 448 * 4 + (256 + 8) * 12 = 4,960 bytes, so that eight waves fit per SIMD
// (eight 256-thread blocks of 19,840 bytes in the CU's 160 KiB); full 64-entry rounds need
// top <= 128, far above the stacks the walks reach
constexpr int kWalkStack = 448;     // stack entries (record indices) per wave
constexpr int kWalkSlack = 128;     // the depth-first rounds' headroom: at most 3 per tree level
constexpr int kWalkList = 256;      // accepted records buffered per wave
static_assert(kWalkSlack >= 3 * (kMaxLevels + 1) + 4, "a depth-first descent must fit the headroom");
static_assert(kWalkStack - kWalkSlack >= 64 * 3 + 128, "a full round must fit above a stack of 128");

__device__ __forceinline__ float vote_d2(float px, float py, float cx, float cy, float epssq) {
    const float dx = px - cx, dy = py - cy;
    return fmaf(dx, dx, fmaf(dy, dy, epssq));
}

// Orders this wave's LDS writes before its later LDS reads by other lanes.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int G, int BT>
__global__ __launch_bounds__(BT) void k_walk(const float4* __restrict__ rec, const int4* __restrict__ kids,
                                              const float4* __restrict__ sbody,
                                              const unsigned int* __restrict__ perm, const int2* __restrict__ groups,
                                              int ngroups, const int* __restrict__ node_off,
                                              const int* __restrict__ rec_begin, const float4* __restrict__ seg_root,
                                              const float2* __restrict__ fga, const float2* __restrict__ fprev,
                                              float2* __restrict__ f, float2* __restrict__ rep,
                                              WalkPart* __restrict__ part, float k_r, float itolsq, float epssq,
                                              const DevState* __restrict__ st) {
    static_assert(G == 32 || G == 64, "vote group of 32 or 64 lanes");
    constexpr int W = BT / 64;
    constexpr int kStride = (G == 32) ? 2 : 1;     // list entries per drain step (one per half-wave for G = 32)
    constexpr int kUnroll = 4;                     // drain steps per loop trip
    constexpr int kPad = kStride * kUnroll;
    __shared__ int stk_all[W][kWalkStack];
    __shared__ float3 lst_all[W][kWalkList + kPad];
    if (st->err != 0) return;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: one group per wave
    int* stk = stk_all[wv];
    float3* lst = lst_all[wv];
    const int gidx = xcd_block() * W + wv;
    if (gidx >= ngroups) return;                  // uniform per wave; no block barriers below
    const int2 grp = groups[gidx];
    const int g = grp.y;
    const int nact = min(G, node_off[g + 1] - grp.x);
    const int bl = (G == 32) ? (lane & 31) : lane;    // this lane's body within the group
    const bool bact = bl < nact;
    const int k = grp.x + min(bl, nact - 1);          // inactive lanes duplicate the last body
    const float4 me = sbody[k];     // = the body's record, read without the record-index hop
    const float px = me.x, py = me.y, mi = me.z;
    const unsigned int id = perm[k];
    // the group's bounding box (inactive lanes duplicate an active body) and its first body
    float mnx = px, mny = py, mxx = px, mxy = py;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        mnx = fminf(mnx, __shfl_xor(mnx, o, 64));
        mny = fminf(mny, __shfl_xor(mny, o, 64));
        mxx = fmaxf(mxx, __shfl_xor(mxx, o, 64));
        mxy = fmaxf(mxy, __shfl_xor(mxy, o, 64));
    }
    const float b0x = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(px)));
    const float b0y = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(py)));
    // its middle and last bodies
    const int jm = __builtin_amdgcn_readfirstlane((nact - 1) >> 1), jl = __builtin_amdgcn_readfirstlane(nact - 1);
    const float bmx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(px), jm));
    const float bmy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(py), jm));
    const float blx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(px), jl));
    const float bly = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(py), jl));
    // the lanes whose bodies vote: the group's active bodies (for G = 32 in both half-waves,
    // which hold the same bodies; each half is read as its own 32-bit vote)
    const unsigned long long voters = __builtin_amdgcn_ballot_w64(bact);
    // each half-wave's voters (G = 32), and the byte offset that selects a half-wave's own cell
    const unsigned long long vlo = voters & __builtin_amdgcn_ballot_w64(lane < 32);
    const unsigned long long vhi = voters & __builtin_amdgcn_ballot_w64(lane >= 32);
    const int upper4 = (lane >> 5) << 2;    // 4 in the upper half-wave, else 0 (j2 >= j)
    const float two_r = seg_root[g].z * 2;
    const float base = two_r * two_r * itolsq;
    const bool deep = st->max_level >= kKeyLevels;     // the tree has a level-32 cell
    // the root's children start the walk (a graph of one body has no cell records)
    const int root = rec_begin[g];
    const bool has_root = root + 1 < rec_begin[g + 1];
    int top = 0;                  // stack size (uniform)
    int nlist = 0;                // buffered accepted records (uniform)
    unsigned int naccepted = 0;   // accepted records of the whole walk (uniform)
    if (has_root) {
        const int4 k0 = kids[root];
        if (lane == 0) {
            stk[0] = k0.x;
            stk[1] = k0.y;
            stk[2] = k0.z;
            stk[3] = k0.w;
        }
        top = 1 + (k0.y >= 0) + (k0.z >= 0) + (k0.w >= 0);
    }
    wave_lds_sync();
    float ax = 0.0f, ay = 0.0f;
    const int half = (G == 32) ? (lane >> 5) : 0;
    auto drain = [&]() {
        // pad to whole loop trips with massless entries (their terms are exactly 0)
        const int padded = (nlist + kPad - 1) / kPad * kPad;
        if (nlist + lane < padded) lst[nlist + lane] = make_float3(0.0f, 0.0f, 0.0f);
        wave_lds_sync();
        for (int q0 = 0; q0 < padded; q0 += kPad) {
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const float3 e = lst[q0 + u * kStride + half];
                const float dx = px - e.x, dy = py - e.y;
                const float w = e.z * __builtin_amdgcn_rcpf(fmaf(dx, dx, fmaf(dy, dy, epssq)));
                ax = fmaf(dx, w, ax);
                ay = fmaf(dy, w, ay);
            }
        }
        nlist = 0;
        wave_lds_sync();
    };
    while (top > 0) {
        // a round takes up to 64 entries; each may push up to 4 children (net +3), so near the
        // capacity the rounds shrink to depth-first steps, whose growth the slack bounds
        int take = top < 64 ? top : 64;
        const int room = (kWalkStack - kWalkSlack - top) / 3;
        if (room < take) take = room > 1 ? room : 1;
        top -= take;
        const bool live = lane < take;
        const unsigned long long livem = take >= 64 ? ~0ull : (1ull << take) - 1ull;
        // lanes past `take` repeat the last entry (in bounds) and take no part below
        const int r = stk[top + min(lane, take - 1)];
        const float4 c = rec[r];
        const int4 kd = kids[r];      // read with the record; used only if the cell is opened
        const unsigned int info = __float_as_uint(c.w);
        const bool body = info == 0xffffffffu;
        const float thr = ldexpf(base, -2 * (int)(info & 31u)) + epssq;
        // distance from the group's box (mnx <= mxx: at most one term is positive)
        const float ex = fmaxf(fmaxf(mnx - c.x, c.x - mxx), 0.0f);
        const float ey = fmaxf(fmaxf(mny - c.y, c.y - mxy), 0.0f);
        // lane masks: bodies; cells every body clears (d2 >= thr); cells the first, middle and
        // last bodies all clear (any of them below thr rejects)
        const unsigned long long bodym = __builtin_amdgcn_ballot_w64(body);
        const unsigned long long clearm = __builtin_amdgcn_ballot_w64(fmaf(ex, ex, fmaf(ey, ey, epssq)) >= thr);
        const unsigned long long p3m = __builtin_amdgcn_ballot_w64(vote_d2(b0x, b0y, c.x, c.y, epssq) >= thr) &
                                       __builtin_amdgcn_ballot_w64(vote_d2(bmx, bmy, c.x, c.y, epssq) >= thr) &
                                       __builtin_amdgcn_ballot_w64(vote_d2(blx, bly, c.x, c.y, epssq) >= thr);
        // the remaining cells, voted on by the group's bodies (lanes = bodies); with G = 32 the
        // two half-waves hold the same bodies and vote on two cells at once
        unsigned long long okm = livem & (bodym | clearm);
        unsigned long long um = livem & p3m & ~(bodym | clearm);
        while (um) {
            const int j = __builtin_ctzll(um);
            um &= um - 1;
            int j2 = j;
            if constexpr (G == 32) {
                if (um) {
                    j2 = __builtin_ctzll(um);
                    um &= um - 1;
                }
            }
            float cx, cy, tj;
            if constexpr (G == 32) {
                // each half-wave fetches its own cell's values (the upper half: the second cell)
                const int src = (j << 2) + upper4 * (j2 - j);
                cx = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(c.x)));
                cy = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(c.y)));
                tj = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(thr)));
            } else {
                cx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.x), j));
                cy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.y), j));
                tj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(thr), j));
            }
            const unsigned long long fails = __builtin_amdgcn_ballot_w64(!(vote_d2(px, py, cx, cy, epssq) >= tj));
            if constexpr (G == 32) {
                if ((fails & vlo) == 0ull) okm |= 1ull << j;
                if ((fails & vhi) == 0ull) okm |= 1ull << j2;
            } else {
                if ((fails & voters) == 0ull) okm |= 1ull << j;
            }
        }
        // opened cells push their 1-4 children, in four planes (every opened cell's first
        // child, then every second child, ...); okm holds live lanes only
        const unsigned long long am = okm;
        const unsigned long long m0 = livem & ~bodym & ~okm;
        const unsigned long long m1 = m0 & __builtin_amdgcn_ballot_w64(kd.y >= 0);
        const unsigned long long m2 = m0 & __builtin_amdgcn_ballot_w64(kd.z >= 0);
        const unsigned long long m3 = m0 & __builtin_amdgcn_ballot_w64(kd.w >= 0);
        const bool accept = (okm >> lane) & 1ull;
        const bool open = live && !body && !accept;
        const int p1 = top + __popcll(m0), p2 = p1 + __popcll(m1), p3 = p2 + __popcll(m2);
        const int na = __popcll(am);
        if (open) {
            stk[top + __builtin_amdgcn_mbcnt_hi((unsigned)(m0 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m0, 0u))] =
                kd.x;
            if (kd.y >= 0)
                stk[p1 + __builtin_amdgcn_mbcnt_hi((unsigned)(m1 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m1, 0u))] =
                    kd.y;
            if (kd.z >= 0)
                stk[p2 + __builtin_amdgcn_mbcnt_hi((unsigned)(m2 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m2, 0u))] =
                    kd.z;
            if (kd.w >= 0)
                stk[p3 + __builtin_amdgcn_mbcnt_hi((unsigned)(m3 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m3, 0u))] =
                    kd.w;
        }
        if (accept) {
            const int ra =
                __builtin_amdgcn_mbcnt_hi((unsigned)(am >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)am, 0u));
            lst[nlist + ra] = make_float3(c.x, c.y, k_r * c.z);
        }
        top = p3 + __popcll(m3);
        nlist += na;
        naccepted += (unsigned int)na;
        if (deep) {
            // opened cells of level 32 (info level 31) have any number of bodies: those past the fourth
            // follow it in the records
            unsigned long long mb = m3 & __builtin_amdgcn_ballot_w64((info & 31u) == 31u);
            while (mb != 0ull) {
                const int j = __builtin_ctzll(mb);
                mb &= mb - 1;
                const int cell = __builtin_amdgcn_readlane(r, j);
                const int end = cell + (int)((unsigned int)__builtin_amdgcn_readlane((int)info, j) >> kInfoLevelBits);
                for (int q = cell + 5; q < end; q += 64) {
                    if (nlist > kWalkList - 64) drain();
                    const int more = min(end - q, 64);
                    if (lane < more) {
                        const float4 b = rec[q + lane];
                        lst[nlist + lane] = make_float3(b.x, b.y, k_r * b.z);
                    }
                    nlist += more;
                    naccepted += (unsigned int)more;
                }
            }
        }
        if (nlist > kWalkList - 64 || top == 0) drain();
        wave_lds_sync();
    }
    if constexpr (G == 32) {
        // even entries (lanes 0-31) + odd entries (lanes 32-63)
        ax += __shfl_down(ax, 32, 64);
        ay += __shfl_down(ay, 32, 64);
    }
    ax *= mi;   // the body's own mass, taken out of every term
    ay *= mi;
    const bool own = bact && lane < G;
    if (!fga) {
        // split: the repulsion alone goes to f and the group's interaction count to its
        // partial; k_combine adds F_ga and forms the swing/traction sums once the
        // attraction, run concurrently on another stream, is done
        if (own) f[id] = make_float2(ax, ay);
        if (lane == 0) {
            WalkPart wp;
            wp.swing = 0.0f;
            wp.traction = 0.0f;
            wp.interactions = naccepted * (unsigned int)nact;   // = the sum over the group's bodies
            wp.pad = 0;
            part[gidx] = wp;
        }
        return;
    }
    // epilogue: total force, repulsion capture, the group's swing/traction/interaction sums
    float sw = 0.0f, tr = 0.0f;
    unsigned int inter = own ? naccepted : 0u;
    if (own) {
        const float2 a = fga[id];
        const float2 F = make_float2(a.x + ax, a.y + ay);
        f[id] = F;
        if (rep) rep[id] = make_float2(ax, ay);
        swing_traction(mi, F, fprev[id], sw, tr);
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        sw += __shfl_xor(sw, o, 64);
        tr += __shfl_xor(tr, o, 64);
        inter += __shfl_xor(inter, o, 64);
    }
    if (lane == 0) {
        WalkPart wp;
        wp.swing = sw;
        wp.traction = tr;
        wp.interactions = inter;
        wp.pad = 0;
        part[gidx] = wp;
    }
}

// The walk's epilogue for a split walk (k_walk with fga == nullptr): F = F_ga + F_r per body,
// the optional repulsion capture, and the group's swing/traction sums, with the arithmetic and
// the reduction order of the fused epilogue, so both give the same bits. Groups of G = 32 take
// half a wave each (the xor offsets of the reduction stay inside a half).
template <int G>
__global__ __launch_bounds__(256) void k_combine(const float4* __restrict__ sbody,
                                                 const unsigned int* __restrict__ perm, const int2* __restrict__ groups,
                                                 int ngroups, const int* __restrict__ node_off,
                                                 const float2* __restrict__ fga, const float2* __restrict__ fprev,
                                                 float2* __restrict__ f, float2* __restrict__ rep,
                                                 WalkPart* __restrict__ part, const DevState* __restrict__ st) {
    if (st->err != 0) return;
    const int lane = threadIdx.x & 63;
    const int gidx = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 / G) + lane / G;
    const int bl = lane % G;
    const bool gok = gidx < ngroups;
    bool own = false;
    unsigned int id = 0;
    float mi = 0.0f;
    if (gok) {
        const int2 grp = groups[gidx];
        own = bl < node_off[grp.y + 1] - grp.x;
        if (own) {
            const int k = grp.x + bl;
            id = perm[k];
            mi = sbody[k].z;
        }
    }
    float sw = 0.0f, tr = 0.0f;
    if (own) {
        const float2 r = f[id];
        const float2 a = fga[id];
        const float2 F = make_float2(a.x + r.x, a.y + r.y);
        f[id] = F;
        if (rep) rep[id] = r;
        swing_traction(mi, F, fprev[id], sw, tr);
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        sw += __shfl_xor(sw, o, 64);
        tr += __shfl_xor(tr, o, 64);
    }
    if (gok && bl == 0) {
        part[gidx].swing = sw;
        part[gidx].traction = tr;
    }
}

// ---------------------------------------------------------------------------------------
// Speed update and displacement.
//
// Speed. Reference: SpeedKernel's last block, src/RPFA2Kernels.cu:167-219 (Gephi's adaptive
// speed). The graph's group partials are summed in double in a fixed order: 1,024 strided sums,
// then a halving tree over them, the same for a graph alone or inside a batch and whatever the
// threads of the block that sums them. The update itself is the reference's float arithmetic,
// including its double literals. Graph 0 is mirrored into DevState.
//
// Displacement. Reference: DisplacementKernel, src/RPFA2Kernels.cu:223-251:
// factor = gs/(1.0 + sqrtf(gs*swg)) (double, because of the literal), p += F*factor, F' = F.
// The new position also goes to the degree-ranked copy that the next attraction gathers from,
// and the new bounding box (or its partials) is left for the next tree.
//
// Three forms of the pair, with the same results:
//   k_advance      one graph of up to kAdvanceGroups walk groups: every block sums the partials
//                  itself (a few tens of KB from L2) and displaces its nodes, one launch
//   k_advance_seg  a batch of graphs of up to kSegSortMax nodes: one block per graph
//   k_speed, k_displace   larger graphs
// Each launch on a small graph costs 4-5 us however little it does: with the attraction's
// position copy the three launches were 13.9 us of 107 on 10,000 nodes.
// ---------------------------------------------------------------------------------------
constexpr int kSpeedSums = 1024;
constexpr int kAdvanceGroups = 2048;

struct GroupSums {
    double s, t;
    unsigned long long it;
};

// The graph's group partials [g0, g1) summed by a block of NT threads; thread 0 gets the result.
template <int NT>
__device__ __forceinline__ GroupSums sum_groups(const WalkPart* __restrict__ part, int g0, int g1) {
    constexpr int V = kSpeedSums / NT;            // strided sums per thread
    static_assert(V == 1 || V == 2 || V == 4, "a thread folds its sums with the tree's own offsets");
    __shared__ double rs[NT], rt[NT];
    __shared__ unsigned long long ri[NT];
    const int tid = threadIdx.x;
    double s[V], t[V];
    unsigned long long it = 0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        s[v] = 0.0;
        t[v] = 0.0;
        // 8 partials are loaded before they are added, keeping 8 loads in flight per thread
        constexpr int kAhead = 8;
        int k = g0 + tid + v * NT;
        for (; k + (kAhead - 1) * kSpeedSums < g1; k += kAhead * kSpeedSums) {
            WalkPart p[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) p[j] = part[k + j * kSpeedSums];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                s[v] += (double)p[j].swing;
                t[v] += (double)p[j].traction;
                it += p[j].interactions;
            }
        }
        for (; k < g1; k += kSpeedSums) {
            const WalkPart p = part[k];
            s[v] += (double)p.swing;
            t[v] += (double)p.traction;
            it += p.interactions;
        }
    }
    // the halving tree over the 1,024 sums: offsets 512 and 256 first, as far as a thread holds
    // both halves itself, then through LDS, then within the first wave
    double a = s[0], c = t[0];
    if constexpr (V == 4) {
        a = (s[0] + s[2]) + (s[1] + s[3]);
        c = (t[0] + t[2]) + (t[1] + t[3]);
    } else if constexpr (V == 2) {
        a = s[0] + s[1];
        c = t[0] + t[1];
    }
    rs[tid] = a;
    rt[tid] = c;
    ri[tid] = it;
    __syncthreads();
    for (int o = NT / 2; o >= 64; o >>= 1) {
        if (tid < o) {
            rs[tid] += rs[tid + o];
            rt[tid] += rt[tid + o];
            ri[tid] += ri[tid + o];
        }
        __syncthreads();
    }
    GroupSums r{0.0, 0.0, 0ull};
    if (tid < 64) {
        r = GroupSums{rs[tid], rt[tid], ri[tid]};
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            r.s += __shfl_down(r.s, o, 64);
            r.t += __shfl_down(r.t, o, 64);
            r.it += __shfl_down(r.it, o, 64);
        }
    }
    return r;
}

// The adaptive speed after an iteration with these sums, from the graph's state q of n nodes.
__device__ __forceinline__ SegState speed_update(SegState q, const GroupSums& r, int n) {
    q.swing = r.s;
    q.traction = r.t;
    q.interactions = r.it;
    const float swg = (float)r.s, etra = (float)r.t;
    float gs = q.global_speed, se = q.speed_efficiency;
    const float jitter = q.jitter_tolerance, ksmax = q.k_s_max;
    const float eojt = (float)(0.05 * sqrtf((float)n));
    const float minjt = sqrtf(eojt);
    float jt = jitter * fmaxf(minjt, fminf(ksmax, eojt * etra / powf((float)n, 2.0f)));
    const float min_se = (float)0.05;
    if (swg / etra > 2.0) {
        if (se > min_se) se = (float)(se * 0.5);
        jt = fmaxf(jt, jitter);
    }
    const float target = jt * se * etra / swg;
    if (swg > jt * etra) {
        if (se > min_se) se = (float)(se * 0.7);
    } else if (gs < 1000) {
        se = (float)(se * 1.3);
    }
    gs += fminf(target - gs, (float)0.5 * gs);
    q.global_speed = gs;
    q.speed_efficiency = se;
    q.iteration += 1;
    q.interactions_total += r.it;
    return q;
}

// The tree's largest cell at level 4, 8, ..., 32, from the blocks of k_tile and k_cross (the small
// tree: its one block), into rm
// (8 words of LDS; followed by a barrier).
template <int NT>
__device__ __forceinline__ void max_runs(const int* __restrict__ kids_part, int kids_blocks, int* rm) {
    const int tid = threadIdx.x;
    if (tid < 8) rm[tid] = 0;
    __syncthreads();
    // thread t reads level slot t & 7 (the stride keeps the slot), eight loads in flight
    int m = 0;
    const int nq = kids_blocks * 8;
    int q = tid;
    for (; q + 7 * NT < nq; q += 8 * NT) {
        int v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = kids_part[q + u * NT];
#pragma unroll
        for (int u = 0; u < 8; ++u) m = max(m, v[u]);
    }
    for (; q < nq; q += NT) m = max(m, kids_part[q]);
    if (m > 0) atomicMax(&rm[tid & 7], m);
    __syncthreads();
}

// Graph 0's part of the instance state (one thread).
__device__ __forceinline__ void mirror_state(DevState* st, const SegState& q, const int* rm) {
    st->swing = q.swing;
    st->traction = q.traction;
    st->interactions = q.interactions;
    st->global_speed = q.global_speed;
    st->speed_efficiency = q.speed_efficiency;
    // the next path-key sort: p 8-bit passes order the bodies by their top 4p levels,
    // and the pairs left tied are the bodies of one 4p-level cell, which the fix-up
    // orders; take the fewest passes whose cells (in this tree) hold at most
    // kSortRunMax bodies each
    int p = 1;
    while (p < 8 && rm[p - 1] > kSortRunMax) ++p;
    if (st->full_sorts > 0) {
        st->full_sorts -= 1;      // still settling after new positions
        p = 8;
    }
    st->sort_skip = 8 - p;
    for (int k = 0; k < 8; ++k) st->runmax[k] = rm[k];
}

// One node's new position.
__device__ __forceinline__ float2 displaced(float2 p, float2 F, float2 P, float gs) {
    const float dx = F.x - P.x, dy = F.y - P.y;
    const float swg = sqrtf(fmaf(dx, dx, dy * dy));
    const float factor = (float)((double)gs / (1.0 + (double)sqrtf(gs * swg)));
    p.x = fmaf(F.x, factor, p.x);
    p.y = fmaf(F.y, factor, p.y);
    return p;
}

__device__ __forceinline__ float4 box_add(float4 acc, float2 p) {
    return make_float4(fminf(acc.x, p.x), fminf(acc.y, p.y), fmaxf(acc.z, p.x), fmaxf(acc.w, p.y));
}

// The block's box {min x, min y, max x, max y}; thread 0 gets it.
template <int NT>
__device__ __forceinline__ float4 box_reduce(float4 acc) {
    __shared__ float4 red[NT / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        acc = make_float4(fminf(acc.x, __shfl_xor(acc.x, o, 64)), fminf(acc.y, __shfl_xor(acc.y, o, 64)),
                          fmaxf(acc.z, __shfl_xor(acc.z, o, 64)), fmaxf(acc.w, __shfl_xor(acc.w, o, 64)));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < NT / 64; ++w) {
            const float4 v = red[w];
            acc = make_float4(fminf(acc.x, v.x), fminf(acc.y, v.y), fmaxf(acc.z, v.z), fmaxf(acc.w, v.w));
        }
    return acc;
}

constexpr int kSpeedThreads = 1024;

__global__ __launch_bounds__(kSpeedThreads) void k_speed(const WalkPart* __restrict__ part,
                                                         const int* __restrict__ grp_first,
                                                         const int* __restrict__ node_off, SegState* __restrict__ seg,
                                                         DevState* st, const int* __restrict__ kids_part,
                                                         int kids_blocks) {
    __shared__ int rm[8];
    if (st->err != 0) return;
    const int g = blockIdx.x;
    if (g == 0) max_runs<kSpeedThreads>(kids_part, kids_blocks, rm);
    const GroupSums r = sum_groups<kSpeedThreads>(part, grp_first[g], grp_first[g + 1]);
    if (threadIdx.x == 0) {
        // per graph (one block each): no word shared by the blocks of a batch
        const SegState q = speed_update(seg[g], r, node_off[g + 1] - node_off[g]);
        seg[g] = q;
        if (g == 0) mirror_state(st, q, rm);
    }
}

__global__ __launch_bounds__(256) void k_displace(float2* __restrict__ pos, const float2* __restrict__ f,
                                                  float2* __restrict__ fprev, int n, const int* __restrict__ rank,
                                                  float2* __restrict__ pos_rank, const int* __restrict__ seg_of,
                                                  const SegState* __restrict__ seg, float4* __restrict__ part,
                                                  DevState* st) {
    const int tid = threadIdx.x;
    const bool live = st->err == 0;
    const float gs0 = seg[0].global_speed;
    float4 acc = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (int i = blockIdx.x * 256 + tid; i < n; i += gridDim.x * 256) {
        float2 p = pos[i];
        if (live) {
            const float gs = seg_of ? seg[seg_of[i]].global_speed : gs0;
            const float2 F = f[i];
            p = displaced(p, F, fprev[i], gs);
            pos[i] = p;
            pos_rank[rank[i]] = p;
            fprev[i] = F;
        }
        acc = box_add(acc, p);
    }
    if (part == nullptr) {
        if (blockIdx.x == 0 && tid == 0 && live) st->iteration += 1;
        return;
    }
    acc = box_reduce<256>(acc);
    if (tid == 0) {
        part[blockIdx.x] = acc;
        if (blockIdx.x == 0) {
            st->nbbox = gridDim.x;
            if (live) st->iteration += 1;
        }
    }
}

// One graph: speed and displacement in one launch. Every block forms the new speed from seg_cur,
// the state before the iteration (copied from seg by the iteration's first kernel); block 0
// alone writes the new state, to seg, which no block of this launch reads.
__global__ __launch_bounds__(256) void k_advance(float2* __restrict__ pos, const float2* __restrict__ f,
                                                 float2* __restrict__ fprev, int n, const int* __restrict__ rank,
                                                 float2* __restrict__ pos_rank, const WalkPart* __restrict__ wpart,
                                                 int ngroups, const SegState* __restrict__ seg_cur,
                                                 SegState* __restrict__ seg, const int* __restrict__ kids_part,
                                                 int kids_blocks, float4* __restrict__ part, DevState* st) {
    __shared__ int rm[8];
    __shared__ float new_speed;
    const int tid = threadIdx.x;
    const bool live = st->err == 0;               // nothing in this launch changes it
    // the block's first nodes are loaded beside the sums
    const int i0 = blockIdx.x * 256 + tid;
    float2 p0 = make_float2(0.0f, 0.0f), F0 = p0, P0 = p0;
    int r0 = 0;
    if (i0 < n) {
        p0 = pos[i0];
        F0 = f[i0];
        P0 = fprev[i0];
        r0 = rank[i0];
    }
    if (live) {
        if (blockIdx.x == 0) max_runs<256>(kids_part, kids_blocks, rm);
        const GroupSums r = sum_groups<256>(wpart, 0, ngroups);
        if (tid == 0) {
            const SegState q = speed_update(*seg_cur, r, n);
            new_speed = q.global_speed;
            if (blockIdx.x == 0) {
                seg[0] = q;
                mirror_state(st, q, rm);
            }
        }
        __syncthreads();
    }
    const float gs = live ? new_speed : 0.0f;
    float4 acc = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (int i = i0; i < n; i += gridDim.x * 256) {
        if (i != i0) {
            p0 = pos[i];
            F0 = f[i];
            P0 = fprev[i];
            r0 = rank[i];
        }
        float2 p = p0;
        if (live) {
            p = displaced(p0, F0, P0, gs);
            pos[i] = p;
            pos_rank[r0] = p;
            fprev[i] = F0;
        }
        acc = box_add(acc, p);
    }
    acc = box_reduce<256>(acc);
    if (tid == 0) {
        part[blockIdx.x] = acc;
        if (blockIdx.x == 0) {
            st->nbbox = gridDim.x;
            if (live) st->iteration += 1;
        }
    }
}

// A batch, one block per graph (largest first): the graph's speed, its nodes' displacement and
// the root of its next tree (as k_seg_bbox sets it).
constexpr int kAdvanceSegThreads = 512;

__global__ __launch_bounds__(kAdvanceSegThreads) void k_advance_seg(
    float2* __restrict__ pos, const float2* __restrict__ f, float2* __restrict__ fprev, const int* __restrict__ rank,
    float2* __restrict__ pos_rank, const WalkPart* __restrict__ wpart, const int* __restrict__ grp_first,
    const int* __restrict__ node_off, const int* __restrict__ order, SegState* __restrict__ seg,
    const int* __restrict__ kids_part, int kids_blocks, float4* __restrict__ seg_root, DevState* st) {
    constexpr int NT = kAdvanceSegThreads;
    __shared__ int rm[8];
    __shared__ float new_speed;
    if (st->err != 0) return;
    const int g = order[blockIdx.x], tid = threadIdx.x;
    const int a = node_off[g], e = node_off[g + 1];
    if (g == 0) max_runs<NT>(kids_part, kids_blocks, rm);
    const GroupSums r = sum_groups<NT>(wpart, grp_first[g], grp_first[g + 1]);
    if (tid == 0) {
        const SegState q = speed_update(seg[g], r, e - a);
        new_speed = q.global_speed;
        seg[g] = q;
        if (g == 0) {
            mirror_state(st, q, rm);
            st->iteration += 1;
        }
    }
    __syncthreads();
    const float gs = new_speed;
    float4 acc = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
#pragma unroll 2
    for (int i = a + tid; i < e; i += NT) {
        const float2 F = f[i];
        const float2 p = displaced(pos[i], F, fprev[i], gs);
        pos[i] = p;
        pos_rank[rank[i]] = p;
        fprev[i] = F;
        acc = box_add(acc, p);
    }
    acc = box_reduce<NT>(acc);
    if (tid == 0) {
        // no ordered coordinate at all (every one NaN): the box k_seg_bbox would form
        if (!(acc.x <= acc.z)) acc.x = acc.z = NAN;
        if (!(acc.y <= acc.w)) acc.y = acc.w = NAN;
        seg_root[g] = make_float4((acc.x + acc.z) * 0.5f, (acc.y + acc.w) * 0.5f,
                                  fmaxf(acc.z - acc.x, acc.w - acc.y) * 0.5f, 0.0f);
    }
}

// ---------------------------------------------------------------------------------------
// Exact repulsion (no counterpart in the reference's GPU path). Each lane is one node and runs
// over nodes j of its graph in ascending order, reading the packed {x, y, mass} of node j, with
// the walk's term k_r m_i m_j (p_i - p_j) / (|p_i - p_j|^2 + eps^2) (node i itself adds 0).
// Every body interacts with every body of its graph, so the interaction count is the sum of n_g^2.
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_pack(const float2* __restrict__ pos, const float* __restrict__ mass, int n,
                                              float4* __restrict__ body, const SegState* __restrict__ seg,
                                              SegState* __restrict__ seg_cur) {
    if (seg_cur && blockIdx.x == 0 && threadIdx.x == 0) *seg_cur = seg[0];   // for k_advance
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float2 p = pos[i];
        body[i] = make_float4(p.x, p.y, mass[i], 0.0f);
    }
}

// A block takes 64 bodies and cuts their graph's nodes into kExactSlices runs, one per wave; the
// runs' sums are added in run order through LDS. The cut depends on the graph's size alone, so a
// graph in a batch gets the bits it gets alone. The wave's lanes all read the same node, which
// goes through the scalar cache.
//
// Bound by FP32 VALU issue (7 vector instructions and a quarter-rate reciprocal per term) once
// there are waves enough: with one lane per body and no cut, 12,345 bodies were 193 waves on
// 1,024 SIMDs, each waiting for one load per term, 1,238 us; with the cut 70 us (the issue alone:
// 44 cycles per term and wave, 51 us on the 193 compute units that hold a block).
constexpr int kExactSlices = 16;

template <int G>
__global__ __launch_bounds__(64 * kExactSlices) void k_exact(const float4* __restrict__ body,
                                                             const int2* __restrict__ groups, int ngroups,
                                                             const int* __restrict__ node_off,
                                                             const float2* __restrict__ fga,
                                                             const float2* __restrict__ fprev,
                                                             float2* __restrict__ f, float2* __restrict__ rep,
                                                             WalkPart* __restrict__ part, float k_r, float epssq,
                                                             const DevState* __restrict__ st) {
    __shared__ float2 red[kExactSlices][64];
    if (st->err != 0) return;
    const int lane = threadIdx.x & 63;
    const int slice = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = xcd_block() * (64 / G);       // the block's first group
    const int gidx = first + lane / G;
    const bool group_ok = gidx < ngroups;
    const int2 grp = groups[min(gidx, ngroups - 1)];
    const int g = grp.y;
    const int k = grp.x + lane % G;
    const bool active = group_ok && k < node_off[g + 1];
    float px = 0.0f, py = 0.0f, mi = 0.0f;
    if (active) {
        const float4 me = body[k];
        px = me.x;
        py = me.y;
        mi = me.z;
    }
    float ax = 0.0f, ay = 0.0f;
    // the one or (a block of two groups of 32) two graphs of the block's bodies
#pragma unroll
    for (int q = 0; q < 64 / G; ++q) {
        const int gq = __builtin_amdgcn_readlane(g, q * G);
        if (q > 0 && gq == __builtin_amdgcn_readlane(g, 0)) break;      // uniform
        const int j0 = node_off[gq], m = node_off[gq + 1] - j0;
        const int run = (m + kExactSlices - 1) / kExactSlices;
        const int ja = __builtin_amdgcn_readfirstlane(j0 + min(m, slice * run));
        const int jb = __builtin_amdgcn_readfirstlane(j0 + min(m, (slice + 1) * run));
        if (g != gq) continue;
#pragma unroll 8
        for (int j = ja; j < jb; ++j) {
            const float4 c = body[j];
            const float dx = px - c.x;
            const float dy = py - c.y;
            const float w = c.z * __builtin_amdgcn_rcpf(fmaf(dx, dx, fmaf(dy, dy, epssq)));
            ax = fmaf(dx, w, ax);
            ay = fmaf(dy, w, ay);
        }
    }
    red[slice][lane] = make_float2(ax, ay);
    __syncthreads();
    if (slice != 0) return;
#pragma unroll
    for (int q = 1; q < kExactSlices; ++q) {
        ax += red[q][lane].x;
        ay += red[q][lane].y;
    }
    const float kmi = k_r * mi;                     // taken out of every term
    const unsigned int inter = active ? (unsigned int)(node_off[g + 1] - node_off[g]) : 0u;
    group_finish<G>(active, group_ok, lane % G, gidx, (unsigned int)k, mi, kmi * ax, kmi * ay, inter, fga, fprev, f,
                    rep, part);
}

// All-pairs repulsion into out, one thread per node, FP32 or FP64 arithmetic; the graph of
// node i is found from node_off by binary search.
template <typename T>
__global__ __launch_bounds__(256) void k_exact_only(const float4* __restrict__ body, int n, int nseg,
                                                    const int* __restrict__ node_off, float k_r, float epssq,
                                                    double2* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int lo = 0, hi = nseg;           // node_off[lo] <= i < node_off[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (node_off[mid] <= i) lo = mid;
        else hi = mid;
    }
    const float4 me = body[i];
    const T px = me.x, py = me.y, kmi = (T)k_r * (T)me.z, eps = epssq;
    T ax = 0, ay = 0;
    for (int j = node_off[lo]; j < node_off[lo + 1]; ++j) {
        const float4 c = body[j];
        const T dx = px - (T)c.x;
        const T dy = py - (T)c.y;
        const T d2 = dx * dx + dy * dy + eps;
        const T w = kmi * (T)c.z / d2;
        ax += dx * w;
        ay += dy * w;
    }
    out[i] = make_double2((double)ax, (double)ay);
}

// w^delta per CSR entry (delta = 0 gives 1).
__global__ __launch_bounds__(256) void k_edge_pow(const float* __restrict__ w, long long nnz, float delta,
                                                  float* __restrict__ out) {
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < nnz;
         e += (long long)gridDim.x * blockDim.x)
        out[e] = delta == 0.0f ? 1.0f : (delta == 1.0f ? w[e] : powf(w[e], delta));
}

}  // namespace

namespace {

template <int G, int BT>
void walk_launch(const Bufs& b, const Params& p, bool split, hipStream_t s) {
    constexpr int W = BT / 64;     // one group per wave
    const int blocks = (b.ngroups + W - 1) / W;
    k_walk<G, BT><<<blocks < 1 ? 1 : blocks, BT, 0, s>>>(b.rec, b.kids, b.sbody, b.sort.vals[0], b.groups, b.ngroups,
                                                          b.node_off, b.rec_begin, b.seg_root, split ? nullptr : b.fga,
                                                          b.fprev, b.f, split ? nullptr : b.rep, b.grp_part, p.k_r,
                                                          p.itolsq, p.epssq, b.st);
}

template <int G>
void walk_dispatch(const Bufs& b, const Params& p, bool split, hipStream_t s) {
    switch (p.walk_bt) {
        case 64: walk_launch<G, 64>(b, p, split, s); break;
        case 128: walk_launch<G, 128>(b, p, split, s); break;
        case 512: walk_launch<G, 512>(b, p, split, s); break;
        default: walk_launch<G, 256>(b, p, split, s); break;
    }
}

}  // namespace

void launch_col_rank(const Bufs& b, hipStream_t s) {
    if (b.nnz > 0) k_gather_rank<<<(int)std::min<long long>((b.nnz + 255) / 256, 16384), 256, 0, s>>>(b.col, b.rank, b.nnz, b.col_rank);
}

AttractPlan attract_plan(const Bufs& b) {
    AttractPlan a;
    a.light_blocks = (b.nlight + 255) / 256;
    // several medium rows to a wave once one each would more than fill the card (8 waves on each
    // of 1,024 SIMDs): with one each, R-MAT 2^18 at 4M entries took 182 us an iteration against 176
    a.medium_rows = std::max(1, std::min(kMediumBatch, b.nmedium / 8192));
    a.medium_blocks = (b.nmedium + 4 * a.medium_rows - 1) / (4 * a.medium_rows);
    a.chunks = b.nattr_chunks;
    a.total = a.light_blocks + a.medium_blocks + a.chunks;
    return a;
}

AttractArgs attract_args(const Bufs& b, const Params& p) {
    return AttractArgs{b.pos,    b.mass,    b.n,              b.pos_rank, b.rowptr, b.col_rank, b.node_lists,
                       b.nlight, b.nmedium, p.strong_gravity, p.k_g,      b.fga,    p.linlog,   b.ew};
}

// The wide blocks stay until all rows are done, which pays where their staging and their uneven
// ends are small beside the work and hubs hold many entries (R-MAT on one stream: 8M entries 252 us
// an iteration without, 265 with; 17M 292 either way; 20M 398, 400; 64M 1,245, 1,207; BA with 1M
// bodies, 20M entries, 9% of them of hubs: 667, 753), and nothing is to run beside them.
bool attract_wide(const Bufs& b) {
    return b.attr_grid == 0 && b.nnz >= kWideEntries && b.hub_entries >= b.nnz / 4;
}

void launch_attract_heavy(const Bufs& b, const Params& p, hipStream_t s) {
    if (b.nheavy > 0)
        k_attract_heavy<<<(b.nheavy + 255) / 256, 256, 0, s>>>(b.pos, b.mass, b.node_lists + b.nlight + b.nmedium,
                                                               b.nheavy, b.attr_c0, b.attr_part, p.strong_gravity,
                                                               p.k_g, b.fga);
}

void launch_attraction(const Bufs& b, const Params& p, bool alone, hipStream_t s) {
    const AttractPlan w = attract_plan(b);
    const AttractArgs A = attract_args(b, p);
    const bool gen = p.linlog || b.ew;
    if (alone && attract_wide(b)) {
        const int blocks = std::min(2 * b.cus, (w.total + kWideSubs - 1) / kWideSubs);
        if (gen)
            k_attract_wide<true><<<blocks, kWideThreads, 0, s>>>(A, b.attr_chunks, w.chunks, w.light_blocks,
                                                                 w.medium_blocks, w.medium_rows, b.attr_part);
        else
            k_attract_wide<false><<<blocks, kWideThreads, 0, s>>>(A, b.attr_chunks, w.chunks, w.light_blocks,
                                                                  w.medium_blocks, w.medium_rows, b.attr_part);
    } else if (w.total > 0) {
        const int blocks = b.attr_grid > 0 ? std::min(w.total, b.attr_grid) : w.total;
        // a grid smaller than the work (beside other kernels): every block stages the hubs'
        // positions once and uses them for several virtual blocks
        const bool hub = b.attr_grid > 0 && w.total > 2 * blocks;
#define GFA2_ATTRACT(G, H) \
    k_attract<G, H><<<blocks, 256, 0, s>>>(A, b.attr_chunks, w.chunks, w.light_blocks, w.medium_blocks, w.medium_rows, b.attr_part)
        if (gen) {
            if (hub) GFA2_ATTRACT(true, kHubCache);
            else GFA2_ATTRACT(true, 0);
        } else {
            if (hub) GFA2_ATTRACT(false, kHubCache);
            else GFA2_ATTRACT(false, 0);
        }
#undef GFA2_ATTRACT
    }
    launch_attract_heavy(b, p, s);
}

void launch_walk(const Bufs& b, const Params& p, bool split, hipStream_t s) {
    if (p.group == 64) walk_dispatch<64>(b, p, split, s);
    else walk_dispatch<32>(b, p, split, s);
}

void launch_combine(const Bufs& b, const Params& p, hipStream_t s) {
    const int per_block = 4 * (64 / p.group);
    const int blocks = (b.ngroups + per_block - 1) / per_block;
    if (p.group == 64)
        k_combine<64><<<blocks < 1 ? 1 : blocks, 256, 0, s>>>(b.sbody, b.sort.vals[0], b.groups, b.ngroups,
                                                              b.node_off, b.fga, b.fprev, b.f, b.rep, b.grp_part, b.st);
    else
        k_combine<32><<<blocks < 1 ? 1 : blocks, 256, 0, s>>>(b.sbody, b.sort.vals[0], b.groups, b.ngroups,
                                                              b.node_off, b.fga, b.fprev, b.f, b.rep, b.grp_part, b.st);
}

namespace {

// How a graph or batch takes speed and displacement (see above k_speed).
bool advance_one(const Bufs& b) { return b.nseg == 1 && b.ngroups <= kAdvanceGroups; }

}  // namespace

bool advance_seg(const Bufs& b) { return b.nseg > 1 && b.max_seg <= kSegSortMax; }

void launch_speed(const Bufs& b, hipStream_t s) {
    if (advance_one(b) || advance_seg(b)) return;          // done with the displacement
    k_speed<<<b.nseg, kSpeedThreads, 0, s>>>(b.grp_part, b.grp_first, b.node_off, b.seg_st, b.st, b.kids_part,
                                              b.kids_blocks);
}

void launch_displacement(const Bufs& b, hipStream_t s) {
    if (advance_seg(b)) {
        k_advance_seg<<<b.nseg, kAdvanceSegThreads, 0, s>>>(b.pos, b.f, b.fprev, b.rank, b.pos_rank, b.grp_part,
                                                            b.grp_first, b.node_off, b.seg_order, b.seg_st,
                                                            b.kids_part, b.kids_blocks, b.seg_root, b.st);
    } else if (advance_one(b)) {
        k_advance<<<displacement_blocks(b), 256, 0, s>>>(b.pos, b.f, b.fprev, b.n, b.rank, b.pos_rank, b.grp_part,
                                                         b.ngroups, b.seg_cur, b.seg_st, b.kids_part, b.kids_blocks,
                                                         b.bbox_part, b.st);
    } else {
        k_displace<<<displacement_blocks(b), 256, 0, s>>>(b.pos, b.f, b.fprev, b.n, b.rank, b.pos_rank,
                                                           b.nseg > 1 ? b.seg_of : nullptr, b.seg_st,
                                                           b.nseg > 1 ? nullptr : b.bbox_part, b.st);
    }
}

void launch_exact(const Bufs& b, const Params& p, hipStream_t s) {
    int pb = (b.n + 255) / 256;
    if (pb > 4096) pb = 4096;
    k_pack<<<pb, 256, 0, s>>>(b.pos, b.mass, b.n, b.sbody, b.seg_st, b.seg_cur);
    const int per_block = 64 / p.group;
    const int blocks = (b.ngroups + per_block - 1) / per_block;
    if (p.group == 64)
        k_exact<64><<<blocks, 64 * kExactSlices, 0, s>>>(b.sbody, b.groups, b.ngroups, b.node_off, b.fga, b.fprev, b.f,
                                                         b.rep, b.grp_part, p.k_r, p.epssq, b.st);
    else
        k_exact<32><<<blocks, 64 * kExactSlices, 0, s>>>(b.sbody, b.groups, b.ngroups, b.node_off, b.fga, b.fprev, b.f,
                                                         b.rep, b.grp_part, p.k_r, p.epssq, b.st);
}

void launch_exact_only(const Bufs& b, const Params& p, bool fp64, double2* out, hipStream_t s) {
    int pb = (b.n + 255) / 256;
    if (pb > 4096) pb = 4096;
    k_pack<<<pb, 256, 0, s>>>(b.pos, b.mass, b.n, b.sbody, nullptr, nullptr);
    const int blocks = (b.n + 255) / 256;
    if (fp64)
        k_exact_only<double><<<blocks, 256, 0, s>>>(b.sbody, b.n, b.nseg, b.node_off, p.k_r, p.epssq, out);
    else
        k_exact_only<float><<<blocks, 256, 0, s>>>(b.sbody, b.n, b.nseg, b.node_off, p.k_r, p.epssq, out);
}

void launch_edge_weights(const Bufs& b, float delta, hipStream_t s) {
    if (!b.ew_raw || !b.ew || b.nnz == 0) return;
    long long blocks = (b.nnz + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    k_edge_pow<<<(int)blocks, 256, 0, s>>>(b.ew_raw, b.nnz, delta, b.ew);
}

}  // namespace gfa2
