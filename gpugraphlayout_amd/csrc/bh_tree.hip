// Barnes-Hut quadtree construction for gfx950, deterministic and lock-free.
//
// The reference builds its quadtree by concurrent insertion with CAS locks and then
// summarises and sorts it with spin-waiting kernels (src/RPBHKernels.cu:184-559). Here
// the same tree is derived from sorted path keys instead:
//  1. bounding box (the reference's BoundingBoxKernel, src/RPBHKernels.cu:70-157), from
//     per-block partials every key block reduces redundantly;
//  2. per body a 64-bit key of 32 quadrant digits (bit0: x, bit1: y), obtained by
//     replaying the reference's float centre arithmetic along the body's path
//     (r *= 0.5f, x += +/-r; src/RPBHKernels.cu:217-241, :292-308). A quadrant tree is
//     fixed by the bodies' paths, whatever the insertion order;
//  3. radix sort of the keys: the sorted order is the reference's in-order body
//     permutation (SortKernel, src/RPBHKernels.cu:513-559);
//  4. with lcp_i the common digits of sorted neighbours i and i+1, the cells are exactly
//     the prefixes of length <= lcp_i; the cells starting at position i have levels
//     lcp_{i-1}+1 .. lcp_i. Their pre-order record index follows from an exclusive scan
//     of those counts, and a cell of level L ends at the first position whose lcp is below L;
//  5. summaries. Counts are extents. For whole-number masses (the default deg+1) a cell
//     lighter than 2^24 has the same float mass in every summation order, so its mass and
//     centroid come from exact integer prefix sums over the sorted bodies (fixed-point
//     moments, see Moment); heavier cells are summed in quadrant order. Other masses:
//     bottom-up, children in quadrant order, mass accumulated from 0.0f
//     and centroid (sum m*p)*(1/mass), as the reference's SummarizationKernel
//     (src/RPBHKernels.cu:357-506).
// Nothing waits on another workgroup; every dependency crosses a launch boundary.
#include "engine_internal.h"
#include "attract_device.h"
#include "tree_device.h"

namespace gfa2 {
namespace {

// Reduce bounding-box partials {minx, miny, maxx, maxy} in LDS (every block does it).
__device__ void reduce_bbox(const float4* __restrict__ part, int np, float* root /*[3] LDS*/) {
    __shared__ float4 red[256];
    const int tid = threadIdx.x;
    float4 acc = part[0];
    for (int k = tid; k < np; k += blockDim.x) {
        float4 v = part[k];
        acc.x = fminf(acc.x, v.x);
        acc.y = fminf(acc.y, v.y);
        acc.z = fmaxf(acc.z, v.z);
        acc.w = fmaxf(acc.w, v.w);
    }
    red[tid] = acc;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if (tid < o) {
            float4 v = red[tid + o];
            acc.x = fminf(acc.x, v.x);
            acc.y = fminf(acc.y, v.y);
            acc.z = fmaxf(acc.z, v.z);
            acc.w = fmaxf(acc.w, v.w);
            red[tid] = acc;
        }
        __syncthreads();
    }
    if (tid == 0) {
        float4 t = red[0];
        root[2] = fmaxf(t.z - t.x, t.w - t.y) * 0.5f;   // src/RPBHKernels.cu:140
        root[0] = (t.x + t.z) * 0.5f;                    // :147
        root[1] = (t.y + t.w) * 0.5f;                    // :148
    }
    __syncthreads();
}

// What the displacement leaves for the next iteration, from positions that came from elsewhere: the
// degree-ranked copy, the bounding box's partials (one graph) and, with RESET, also cleared forces
// and the first iteration's state. One launch: at some ten thousand bodies each is little but a
// launch (20k bodies, positions set, then a reset, before one force evaluation: 366 us in all with
// the four launches, six fills and two copies that this takes the place of, 343 with it).
struct NewState {
    float global_speed, speed_efficiency, jitter_tolerance, k_s_max;
    int full_sorts;          // without RESET: the next sorts that are full ones (-1: as they were)
};

template <bool RESET>
__global__ __launch_bounds__(256) void k_new_positions(const float2* __restrict__ pos, const int* __restrict__ rank,
                                                       int n, float2* __restrict__ pos_rank,
                                                       float4* __restrict__ part, DevState* st, NewState init,
                                                       SegState* __restrict__ seg_st, int nseg,
                                                       float2* __restrict__ f, float2* __restrict__ fprev,
                                                       float2* __restrict__ fga) {
    __shared__ float4 red[256];
    const int tid = threadIdx.x;
    float2 p0 = pos[0];
    float4 acc = make_float4(p0.x, p0.y, p0.x, p0.y);
    for (int i = blockIdx.x * 256 + tid; i < n; i += gridDim.x * 256) {
        float2 p = pos[i];
        pos_rank[rank[i]] = p;
        acc.x = fminf(acc.x, p.x);
        acc.y = fminf(acc.y, p.y);
        acc.z = fmaxf(acc.z, p.x);
        acc.w = fmaxf(acc.w, p.y);
        if constexpr (RESET) {
            const float2 z = make_float2(0.0f, 0.0f);
            f[i] = z;
            fprev[i] = z;
            fga[i] = z;
        }
    }
    if constexpr (RESET) {
        for (int q = blockIdx.x * 256 + tid; q < nseg; q += gridDim.x * 256) {
            SegState s{};
            s.global_speed = init.global_speed;
            s.speed_efficiency = init.speed_efficiency;
            s.jitter_tolerance = init.jitter_tolerance;
            s.k_s_max = init.k_s_max;
            seg_st[q] = s;
        }
        static_assert(sizeof(DevState) % 4 == 0, "cleared word by word");
        if (blockIdx.x == 0)
            for (int w = tid; w < (int)(sizeof(DevState) / 4); w += 256) reinterpret_cast<int*>(st)[w] = 0;
    }
    red[tid] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            float4 v = red[tid + o];
            acc.x = fminf(acc.x, v.x);
            acc.y = fminf(acc.y, v.y);
            acc.z = fmaxf(acc.z, v.z);
            acc.w = fmaxf(acc.w, v.w);
            red[tid] = acc;
        }
        __syncthreads();
    }
    if (tid != 0) return;
    if (nseg == 1) part[blockIdx.x] = red[0];
    if (blockIdx.x > 0) return;
    if (nseg == 1) st->nbbox = gridDim.x;
    if constexpr (RESET) {
        st->global_speed = init.global_speed;
        st->speed_efficiency = init.speed_efficiency;
        st->jitter_tolerance = init.jitter_tolerance;
        st->k_s_max = init.k_s_max;
    } else if (init.full_sorts >= 0) {
        st->sort_skip = 0;
        st->full_sorts = init.full_sorts;
    }
}

// Root box + path keys. vals = identity; pm = {x, y, mass} per node, so that k_lcp gathers one
// 16-byte record per sorted body instead of a position and a mass. With dhist (a sort of one
// launch per pass), also the digit counts of all 8 passes, added to the table the previous
// iteration's fix-up cleared (the sort's own histogram launches are then skipped).
struct KeysArgs {
    const float2* pos;
    const float* mass;
    int n;
    const float4* part;
    DevState* st;
    float4* seg_root;
    unsigned long long *k0, *k1;
    unsigned int *v0, *v1;
    float4* pm;
    int first;
    unsigned int* dhist;
    const SegState* seg;
    SegState* seg_cur;
};

__device__ __forceinline__ void keys_block(const KeysArgs& K, int block, int blocks) {
    const float2* __restrict__ pos = K.pos;
    const float* __restrict__ mass = K.mass;
    const float4* __restrict__ part = K.part;
    DevState* st = K.st;
    float4* __restrict__ pm = K.pm;
    unsigned int* __restrict__ dhist = K.dhist;
    const int n = K.n;
    __shared__ float root[3];
    __shared__ unsigned int h[8][256];
    if (dhist)
        for (int p = 0; p < 8; ++p) h[p][threadIdx.x] = 0u;
    // the buffer from which the sort passes that will run (8 less the skipped or unlaunched low
    // ones) end in buffer 0
    const int low = max(st->sort_skip, K.first);
    const bool odd = ((8 - low) & 1) != 0;
    unsigned long long* __restrict__ keys = odd ? K.k1 : K.k0;
    unsigned int* __restrict__ vals = odd ? K.v1 : K.v0;
    reduce_bbox(part, st->nbbox, root);
    const float rootx = root[0], rooty = root[1], radius = root[2];
    if (block == 0 && threadIdx.x == 0) {
        st->rootx = rootx;
        st->rooty = rooty;
        st->radius = radius;
        K.seg_root[0] = make_float4(rootx, rooty, radius, 0.0f);
        *K.seg_cur = K.seg[0];        // for k_advance
    }
    for (int i = block * 256 + threadIdx.x; i < n; i += blocks * 256) {
        const float2 p = pos[i];
        const unsigned long long key = path_key(p, rootx, rooty, radius);
        keys[i] = key;
        vals[i] = (unsigned)i;
        pm[i] = make_float4(p.x, p.y, mass[i], 0.0f);   // one gather per body for k_lcp
        if (dhist)
#pragma unroll
            for (int d = 0; d < 8; ++d)
                if (d >= low) atomicAdd(&h[d][(unsigned)(key >> (8 * d)) & 255u], 1u);
    }
    if (dhist) {
        __syncthreads();
        for (int d = low; d < 8; ++d) {
            const unsigned int c = h[d][threadIdx.x];
            if (c) atomicAdd(&dhist[d * 256 + threadIdx.x], c);
        }
    }
}

__global__ __launch_bounds__(256) void k_keys(const KeysArgs K) { keys_block(K, blockIdx.x, gridDim.x); }

// The keys and the attraction, which both need the positions only, in one launch: on the first
// key_blocks blocks the keys, on one block each the attraction's virtual blocks. Up to some ten
// thousand bodies either is a launch and a few steps in a row, and at any size the one fills the
// chip while the other ends: 92.0 -> 86.2 us an iteration at 10,000 bodies, 138.8 -> 131.0 at 131,000,
// 533 -> 523 at 1M.
template <bool GEN>
__global__ __launch_bounds__(256) void k_keys_attract(const KeysArgs K, int key_blocks, const AttractArgs A,
                                                      const AttractPlan w, const int2* __restrict__ chunks,
                                                      float2* __restrict__ part) {
    __shared__ float2 red[256];
    if ((int)blockIdx.x < key_blocks) keys_block(K, blockIdx.x, key_blocks);
    else attract_block<GEN>(blockIdx.x - key_blocks, w, chunks, part, A, red);
}

// Block-wide exclusive scan of one int per thread (NT threads). Returns the exclusive
// prefix; *total gets the block sum.
template <int NT>
__device__ int block_exclusive_scan(int v, int* total) {
    __shared__ int wsum[NT / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        int s = wsum[w];
        if (w < wave) before += s;
        all += s;
    }
    __syncthreads();
    *total = all;
    return before + inc - v;
}

__device__ __forceinline__ u128 mo_x(const Moment& a) { return ((u128)a.xh << 64) | a.xl; }
__device__ __forceinline__ u128 mo_y(const Moment& a) { return ((u128)a.yh << 64) | a.yl; }

__device__ __forceinline__ Moment mo_make(u128 x, u128 y, unsigned long long m) {
    return Moment{(unsigned long long)x, (unsigned long long)(x >> 64), (unsigned long long)y,
                  (unsigned long long)(y >> 64), m};
}

__device__ __forceinline__ Moment mo_add(const Moment& a, const Moment& b) {
    return mo_make(mo_x(a) + mo_x(b), mo_y(a) + mo_y(b), a.m + b.m);
}

__device__ __forceinline__ Moment mo_sub(const Moment& a, const Moment& b) {
    return mo_make(mo_x(a) - mo_x(b), mo_y(a) - mo_y(b), a.m - b.m);
}

__device__ __forceinline__ Moment mo_shfl_up(const Moment& v, int o) {
    return Moment{__shfl_up(v.xl, o, 64), __shfl_up(v.xh, o, 64), __shfl_up(v.yl, o, 64), __shfl_up(v.yh, o, 64),
                  __shfl_up(v.m, o, 64)};
}

// Block-wide exclusive scan of one Moment per thread (NT threads); *total gets the sum.
template <int NT>
__device__ Moment block_exclusive_scan_mo(const Moment& v, Moment* total) {
    __shared__ Moment ws[NT / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Moment inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const Moment t = mo_shfl_up(inc, o);
        if (lane >= o) inc = mo_add(inc, t);
    }
    if (lane == 63) ws[wave] = inc;
    __syncthreads();
    Moment before{0ull, 0ull, 0ull, 0ull, 0ull}, all{0ull, 0ull, 0ull, 0ull, 0ull};
    for (int w = 0; w < NT / 64; ++w) {
        const Moment s = ws[w];
        if (w < wave) before = mo_add(before, s);
        all = mo_add(all, s);
    }
    __syncthreads();
    *total = all;
    return mo_sub(mo_add(before, inc), v);
}

// Sums over a tile's bodies. They are right for every cell lighter than 2^24, the only ones that
// take them, and for the tiles inside such a cell; a sum over heavier bodies may wrap.
using TileSplit = SplitOf<unsigned long long>;
static_assert(sizeof(TileSplit) == sizeof(Moment));

// lcp per sorted position and the number of cells opened there; block sums (of the
// cell counts and, on the integer-mass path, of body mass sums). Each sorted body's
// {x, y, mass} is gathered here once and written in sorted order (sbody) for the kernels
// that follow.
__global__ __launch_bounds__(kTreeThreads) void k_lcp(const unsigned long long* __restrict__ keys,
                                                      const int* __restrict__ sg, int n,
                                                      signed char* __restrict__ lcp,
                                                      int* __restrict__ blocksum,
                                                      const unsigned int* __restrict__ vals,
                                                      const float4* __restrict__ pm,
                                                      const float4* __restrict__ seg_root,
                                                      Moment* __restrict__ bmass, float4* __restrict__ sbody,
                                                      DevState* __restrict__ st) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {       // for the launches that follow
        st->max_level = 0;
        st->nbig = 0;
    }
    // the tile's keys (with one on each side), graph ids and body ids, read coalesced into
    // LDS; each thread then takes its kTreeItems consecutive positions from there
    __shared__ unsigned long long skey[kTreeTile + 2];
    __shared__ int ssg[kTreeTile + 2];
    __shared__ unsigned int sval[kTreeTile];
    __shared__ int wsum[kTreeThreads / 64];
    __shared__ TileSplit wmass[kTreeThreads / 64];
    const int base = blockIdx.x * kTreeTile;
    for (int t = threadIdx.x; t < kTreeTile + 2; t += kTreeThreads) {
        const int gi = base - 1 + t;
        const bool in = gi >= 0 && gi < n;
        skey[t] = in ? keys[gi] : 0ull;
        if (sg) ssg[t] = in ? sg[gi] : -1;
        if (t < kTreeTile) sval[t] = base + t < n ? vals[base + t] : 0u;
    }
    __syncthreads();
    // over the staged tile (position i at index i - base + 1): whether a graph starts at position i,
    // and the levels shared by positions i and i + 1 (-1 at the end of a graph, except for a graph of
    // one body, whose root, level 0, opens at its only position); the position before the tile is
    // only asked for its lcp when no graph starts at the tile
    auto seg_start_l = [&](int i) { return i == 0 || (sg != nullptr && ssg[i - base] != ssg[i - base + 1]); };
    auto lcp_at_l = [&](int i) -> int {
        if (i < 0) return -1;
        const bool end = i >= n - 1 || (sg != nullptr && ssg[i - base + 1] != ssg[i - base + 2]);
        if (end) return seg_start_l(i) ? 0 : -1;
        return lcp_levels(skey[i - base + 1], skey[i - base + 2]);
    };
    const int i0 = base + threadIdx.x * kTreeItems;
    // all gathers of the thread's items first, outside the per-item branch, so they are in
    // flight together (ids past n are 0, a valid node)
    float4 pp[kTreeItems];
#pragma unroll
    for (int k = 0; k < kTreeItems; ++k) pp[k] = pm[sval[i0 + k - base]];
    int sum = 0;
    TileSplit ms{};
#pragma unroll
    for (int k = 0; k < kTreeItems; ++k) {
        int i = i0 + k;
        if (i < n) {
            const int prev = seg_start_l(i) ? -1 : lcp_at_l(i - 1);
            int l = lcp_at_l(i);
            lcp[i] = (signed char)l;
            sum += max(0, l - prev);
            const float4 bd = make_float4(pp[k].x, pp[k].y, pp[k].z, 0.0f);
            sbody[i] = bd;
            if (bmass) ms = ms + split_of<unsigned long long>(bd, seg_root[sg ? ssg[i - base + 1] : 0]);
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    sum = (int)wave_scan((unsigned int)sum);
    if (bmass) ms = wave_scan(ms);
    if (lane == 63) {
        wsum[wave] = sum;
        if (bmass) wmass[wave] = ms;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kTreeThreads / 64; ++w) wsum[0] += wsum[w];
        blocksum[blockIdx.x] = wsum[0];
        if (bmass) {
            TileSplit all = wmass[0];
            for (int w = 1; w < kTreeThreads / 64; ++w) all = all + wmass[w];
            bmass[blockIdx.x] = mo_make(moment_x(all), moment_y(all), all.m);
        }
    }
}

// Two-level scan of the tile totals, for more tiles than one block scans quickly: per chunk
// of kTileChunk tiles its totals (up), then one block scans the chunk totals (k_scan_blocks,
// which also sets the tree's totals), then every chunk scans its tiles from its offset (down).
// The sums are integers, so the result is the one-level scan's.
__global__ __launch_bounds__(kTileChunk) void k_scan_up(const int* __restrict__ blocksum,
                                                        const Moment* __restrict__ bmass, int nb,
                                                        int* __restrict__ chunk_sum,
                                                        Moment* __restrict__ chunk_mass) {
    const int t = blockIdx.x * kTileChunk + threadIdx.x;
    int total;
    (void)block_exclusive_scan<kTileChunk>(t < nb ? blocksum[t] : 0, &total);
    if (threadIdx.x == 0) chunk_sum[blockIdx.x] = total;
    if (bmass) {
        Moment mt;
        (void)block_exclusive_scan_mo<kTileChunk>(t < nb ? bmass[t] : Moment{0ull, 0ull, 0ull, 0ull, 0ull}, &mt);
        if (threadIdx.x == 0) chunk_mass[blockIdx.x] = mt;
    }
}

__global__ __launch_bounds__(kTileChunk) void k_scan_down(int* __restrict__ blocksum, Moment* __restrict__ bmass,
                                                          int nb, const int* __restrict__ chunk_sum,
                                                          const Moment* __restrict__ chunk_mass) {
    const int t = blockIdx.x * kTileChunk + threadIdx.x;
    int total;
    const int off = block_exclusive_scan<kTileChunk>(t < nb ? blocksum[t] : 0, &total) + chunk_sum[blockIdx.x];
    Moment moff{0ull, 0ull, 0ull, 0ull, 0ull};
    if (bmass) {
        Moment mt;
        moff = mo_add(block_exclusive_scan_mo<kTileChunk>(t < nb ? bmass[t] : Moment{0ull, 0ull, 0ull, 0ull, 0ull}, &mt),
                      chunk_mass[blockIdx.x]);
    }
    if (t < nb) {
        blocksum[t] = off;
        if (bmass) bmass[t] = moff;
    }
}

// Single block: exclusive scan of block sums (in place), cell total, capacity check.
__global__ __launch_bounds__(1024) void k_scan_blocks(int* __restrict__ blocksum, int nb, int n,
                                                      int cap_records, int* __restrict__ rec_end, DevState* st,
                                                      Moment* __restrict__ bmass) {
    __shared__ int wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (nb + 1023) / 1024;
    const int b0 = tid * per;
    // each thread's run of `per` tiles is read kAhead entries at a time with independent loads,
    // then taken in order
    constexpr int kAhead = 8;
    auto valid = [&](int k0, int j) { return k0 + j < per && b0 + k0 + j < nb; };
    if (bmass) {
        Moment loc{0ull, 0ull, 0ull, 0ull, 0ull};
        for (int k0 = 0; k0 < per; k0 += kAhead) {
            Moment c[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) c[j] = valid(k0, j) ? bmass[b0 + k0 + j] : Moment{0ull, 0ull, 0ull, 0ull, 0ull};
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                if (valid(k0, j)) loc = mo_add(loc, c[j]);
        }
        Moment tot;
        Moment run = block_exclusive_scan_mo<1024>(loc, &tot);
        for (int k0 = 0; k0 < per; k0 += kAhead) {
            Moment c[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) c[j] = valid(k0, j) ? bmass[b0 + k0 + j] : Moment{0ull, 0ull, 0ull, 0ull, 0ull};
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                if (valid(k0, j)) {
                    bmass[b0 + k0 + j] = run;
                    run = mo_add(run, c[j]);
                }
        }
    }
    int local = 0;
    for (int k0 = 0; k0 < per; k0 += kAhead) {
        int c[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) c[j] = valid(k0, j) ? blocksum[b0 + k0 + j] : 0;
#pragma unroll
        for (int j = 0; j < kAhead; ++j) local += c[j];
    }
    int inc = local;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < 16; ++w) {
        if (w < wave) before += wsum[w];
        all += wsum[w];
    }
    int run = before + inc - local;
    for (int k0 = 0; k0 < per; k0 += kAhead) {
        int c[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) c[j] = valid(k0, j) ? blocksum[b0 + k0 + j] : 0;
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (valid(k0, j)) {
                blocksum[b0 + k0 + j] = run;
                run += c[j];
            }
    }
    if (tid == 0) {
        st->ncells = all;
        st->nrecords = n + all;
        *rec_end = n + all;
        if (n + all > cap_records) st->err |= kErrTreeOverflow;
    }
}

// The tree's cells in two launches. Positions i and j of a graph lie in one cell of level L if every
// lcp between them is L or more, so a cell that starts at i ends at the first position from i on
// whose lcp is below L, and its 2nd, 3rd and 4th child start behind the first ones of lcp L.
//
// k_tile takes kTreeTile sorted positions: it finds where each cell of the tile ends and where its
// children start from rows of bits in LDS (row L, bit j: lcp(j) < L), and its summary from prefix
// sums in LDS, so a cell inside the tile costs no load from memory. A cell that reaches past
// the tile's end is left to k_cross; such cells contain the tile's last position, so they are nested,
// at most one per level.
// What bounds it: the bytes (a body's record and offset, a cell's record, children and count) at
// 2M bodies, its chain of LDS steps at 50,000. In the place of a pass for the prefix sums over
// bodies (40 bytes written for each, two read per cell), a pass for the cells by searches over
// the keys and one for the child lists: 146 -> 109 us at 2M bodies, 27 -> 21 at 50,000.
constexpr int kTileWords = kTreeTile / 64;
constexpr int kRows = kKeyLevels + 2;
constexpr int kTileCells = 2 * kTreeTile;      // cells per round

struct TileArgs {
    const signed char* lcp;
    const int* sg;
    int n;
    const int* blockoff;        // the tile's first cell, or with fused every tile's cells
    const Moment* bmass;        // the same of the bodies' sums
    int fused;
    int* S;
    const float4* sbody;
    float4* rec;
    int4* kids;
    int* rcount;
    DevState* st;
    const float4* seg_root;
    TileSplit* pm16;            // the sum over the tile's bodies before every 16th position
    int cap_records;
    int* rec_begin;             // each graph's root, then the records' end
    int nseg;
    const int* node_off;
    int* big_rc;
    unsigned char* big_lvl;
    int* kids_part;
    int4* cross;                // per tile up to kCrossMax cells {first position, level, ordinal, graph}
    TileSplit* cross_sum;       // their sums over the bodies of their own tile
    int* ncross;
    signed char* tmin;          // per tile the least lcp
};

// Row L's first bit at position `from` of the tile or later; kTreeTile: none.
__device__ __forceinline__ int next_bit(const unsigned long long (*rows)[kTileWords], int L, int from) {
    if (from >= kTreeTile) return kTreeTile;
    int w = from >> 6;
    unsigned long long v = rows[L][w] & (~0ull << (from & 63));
    while (v == 0ull && ++w < kTileWords) v = rows[L][w];
    return v ? w * 64 + __builtin_ctzll(v) : kTreeTile;
}

// A cell's record: its info word, and on the whole-mass path its summary from its moment d. A cell
// lighter than 2^24 has this exact float mass in any summation order; heavier cells are listed
// and summed in quadrant order later.
__device__ __forceinline__ void write_cell(const TileArgs& A, int rc, int L, unsigned int info, const Moment& d, float4 c) {
    const double M = (double)d.m;
    if (M < 16777216.0) {
        const int sh = moment_shift(c.z);
        A.rec[rc] = make_float4((float)(ldexp(i128_to_double(d.xl, d.xh) / M, -sh) + c.x),
                                (float)(ldexp(i128_to_double(d.yl, d.yh) / M, -sh) + c.y), (float)M,
                                __uint_as_float(info));
        return;
    }
    A.rec[rc].w = __uint_as_float(info);
    const int slot = atomicAdd(&A.st->nbig, 1);
    if (slot < kMaxBig) {
        A.big_rc[slot] = rc;
        A.big_lvl[slot] = (unsigned char)L;
    } else {
        A.st->err |= kErrTreeOverflow;
    }
}

__device__ __forceinline__ unsigned int cell_info(int skip, int L) {
    return ((unsigned int)skip << kInfoLevelBits) | (unsigned int)((L > 0 ? L - 1 : 0) & 31);
}

template <bool MOMENTS>
__global__ __launch_bounds__(kTreeTile) void k_tile(const TileArgs A) {
    __shared__ unsigned long long rows[kRows][kTileWords];
    __shared__ TileSplit pre[MOMENTS ? kTreeTile + 1 : 1];     // relative to the tile's start
    __shared__ TileSplit wsum[kTileWords];
    __shared__ int wopened[kTileWords], wacc[kTileWords];
    __shared__ int first[kTreeTile + 1];                       // cells opened before each position
    __shared__ unsigned char level[kTreeTile];                 // the first opened cell's
    __shared__ unsigned short owner[kTileCells];               // a round's cells' positions
    __shared__ int rmax[8];
    __shared__ int lmax, lmin, ncross, go;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int base = blockIdx.x * kTreeTile, n = A.n, i = base + tid;
    const bool in = i < n;
    const int l = in ? (int)A.lcp[i] : -1;
    int before = in && i > 0 ? (int)A.lcp[i - 1] : -1;
    const float4 bd = in ? A.sbody[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int graph = 0;
    bool ends = !in || i == n - 1;
    if (A.sg) {
        graph = in ? A.sg[i] : 0;
        if (in && i > 0 && A.sg[i - 1] != graph) before = -1;
        if (!ends && A.sg[i + 1] != graph) ends = true;
    }
    const float4 root = A.seg_root[graph];
    int acc = 0;
    if (A.fused)
        for (int t = tid; t < (int)blockIdx.x; t += kTreeTile) acc += A.blockoff[t];
    else if (tid == 0) acc = A.blockoff[blockIdx.x];
    if (tid < 8) rmax[tid] = 0;
    if (tid == 0) {
        lmax = ncross = 0;
        lmin = kMaxLevels;
        go = A.st->err == 0;
    }
    const int opened = in ? max(0, l - before) : 0;
    const int share = ends ? -1 : l;                           // (a graph of one body has lcp 0)
    unsigned long long row = 0ull;
    for (int L = 0; L < kRows; ++L) {
        const unsigned long long word = __builtin_amdgcn_ballot_w64(share < L);
        if (lane == L) row = word;
    }
    if (lane < kRows) rows[lane][wave] = row;
    int run = (int)wave_scan((unsigned int)opened);
    acc = (int)wave_scan((unsigned int)acc);
    TileSplit own{}, p{};
    if (MOMENTS) {
        if (in) own = split_of<unsigned long long>(bd, root);
        p = wave_scan(own);
    }
    if (lane == 63) {
        wopened[wave] = run;
        wacc[wave] = acc;
        if (MOMENTS) wsum[wave] = p;
    }
    __syncthreads();
    // the waves before this one, and all
    const int wl = lane < kTileWords ? lane : 0;
    const unsigned int wo = lane < kTileWords ? (unsigned int)wopened[wl] : 0u;
    const unsigned int wscan = wave_scan(wo);
    const int total = (int)from_lane(wscan, kTileWords - 1);
    const int off = (int)from_lane(wave_scan(lane < kTileWords ? (unsigned int)wacc[wl] : 0u), kTileWords - 1);
    run += (int)from_lane(wscan - wo, wave) - opened;
    if (MOMENTS) {
        const TileSplit w = lane < kTileWords ? wsum[wl] : TileSplit{};
        const TileSplit upto = wave_scan(w);
        p = p - own + from_lane(upto - w, wave);
        pre[tid] = p;
        if (tid == 0) pre[kTreeTile] = from_lane(upto, kTileWords - 1);
        if (tid % 16 == 0 && in) A.pm16[i / 16] = p;
    }
    // records written here: below min(base + tile, n) + off + total (the cells before and in
    // this tile), within capacity whenever the whole tree is
    const bool ok = go != 0 && (!A.fused || min(base + kTreeTile, n) + off + total <= A.cap_records);
    first[tid] = run;
    level[tid] = (unsigned char)(before + 1);
    if (tid == 0) {
        first[kTreeTile] = total;
        if (base + kTreeTile >= n) A.S[n] = off + total;
        if (A.fused && blockIdx.x == gridDim.x - 1) {
            const int all = off + total;
            A.st->ncells = all;
            A.st->nrecords = n + all;
            A.rec_begin[A.nseg] = n + all;
            if (n + all > A.cap_records) A.st->err |= kErrTreeOverflow;
        }
    }
    if (in) {
        A.S[i] = off + run;
        // after its own cells
        if (ok) A.rec[i + off + run + opened] = make_float4(bd.x, bd.y, bd.z, __int_as_float(-1));
    }
    for (int c0 = 0; c0 < total && ok; c0 += kTileCells) {     // uniform
        if (c0 > 0) __syncthreads();                           // the last round's owners
        for (int j = max(0, c0 - run); j < opened && run + j < c0 + kTileCells; ++j)
            owner[run + j - c0] = (unsigned short)tid;
        __syncthreads();
        const int here = min(kTileCells, total - c0);
        for (int c = tid; c < here; c += kTreeTile) {
            const int p = owner[c], L = level[p] + c0 + c - first[p];
            const int ord = off + c0 + c, rc = base + p + ord;
            const int b = next_bit(rows, L, p);                // the cell's last body
            const int g = A.sg ? A.sg[base + p] : 0;
            if (L == 0) A.rec_begin[g] = rc;
            atomicMax(&lmax, L);
            if (b == kTreeTile) {
                const int slot = blockIdx.x * kCrossMax + atomicAdd(&ncross, 1);
                A.cross[slot] = make_int4(base + p, L, ord, g);
                if (MOMENTS) A.cross_sum[slot] = pre[kTreeTile] - pre[p];
                continue;
            }
            int at[3];
            int from = p;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                from = from <= b ? next_bit(rows, L + 1, from) + 1 : kTreeTile + 1;
                at[q] = from <= b ? base + from + off + first[from] : -1;
            }
            A.kids[rc] = make_int4(rc + 1, at[0], at[1], at[2]);
            const unsigned int info = cell_info(base + b + off + first[b + 1] + 1 - rc, L);
            if (MOMENTS) {
                const TileSplit d = pre[b + 1] - pre[p];
                write_cell(A, rc, L, info, mo_make(moment_x(d), moment_y(d), d.m), A.sg ? A.seg_root[g] : root);
            }
            if (!MOMENTS) A.rec[rc].w = __uint_as_float(info);
            A.rcount[rc] = b + 1 - p;
            if (L > 0 && (L & 3) == 0) atomicMax(&rmax[(L >> 2) - 1], b + 1 - p);
        }
    }
    // the tile's least lcp, for k_cross: the first row with a bit
    if (tid < kRows) {
        unsigned long long any = 0ull;
        for (int w = 0; w < kTileWords; ++w) any |= rows[tid][w];
        if (any) atomicMin(&lmin, tid - 1);
    }
    __syncthreads();
    // every block would hit this one word: only blocks above the value seen so far update it
    // (the maximum only grows, so skipping on a stale value is still correct)
    if (tid == 0 && lmax > 0 && lmax > __hip_atomic_load(&A.st->max_level, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(&A.st->max_level, lmax);
    if (tid == 0) {
        A.ncross[blockIdx.x] = ncross;
        A.tmin[blockIdx.x] = (signed char)lmin;
    }
    // per-block maxima, reduced by the speed step (no word shared by the blocks: thousands of
    // device-scope reads or atomics on one line cost more than the kernel itself)
    if (tid < 8) A.kids_part[blockIdx.x * 8 + tid] = rmax[tid];
}

// The cells that reach past their tile, a wave each. Where such a cell ends and its children start is
// found from the tiles' least lcps (1,024 of them per load) and then the 512 lcps of the tiles that
// hold a bound, at most four besides its own: two or three loads in a row for most.
constexpr int kCrossThreads = 1024;   // at most
static_assert(kTreeTile == 64 * 8, "8 lcps per lane");

// Bit b: byte b of v, as a signed number, is below x.
__device__ __forceinline__ unsigned int bytes_below(const unsigned int (&v)[2], int x) {
    unsigned int m = 0u;
#pragma unroll
    for (int b = 0; b < 8; ++b) m |= (unsigned int)((int)(signed char)(v[b >> 2] >> (8 * (b & 3))) < x) << b;
    return m;
}

// Takes the first position out of the lanes' masks of 8 positions each (uniform; -1: none).
__device__ __forceinline__ int take_first(unsigned int& mask, int lane) {
    const unsigned long long some = __builtin_amdgcn_ballot_w64(mask != 0u);
    if (some == 0ull) return -1;
    const int at = __builtin_ctzll(some);
    const int bit = __builtin_ctz((unsigned)__builtin_amdgcn_readlane((int)mask, at));
    if (lane == at) mask &= mask - 1u;
    return at * 8 + bit;
}

template <bool MOMENTS>
__global__ __launch_bounds__(kCrossThreads) void k_cross(const TileArgs A) {
    __shared__ int rmax[8];
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < 8) rmax[tid] = 0;
    __syncthreads();
    const int tile = blockIdx.x, tiles = gridDim.x;
    const int w1 = (tile + 1) & ~15;                           // the first 1,024 tiles looked at
    auto lcps = [&](int t) { return reinterpret_cast<const uint2*>(A.lcp + (size_t)t * kTreeTile)[lane]; };
    auto mins = [&](int w0) {
        const int t0 = w0 + lane * 16;
        return t0 < tiles ? reinterpret_cast<const uint4*>(A.tmin)[t0 / 16] : make_uint4(0u, 0u, 0u, 0u);
    };
    auto below = [](uint2 w, int x) {
        const unsigned int v[2] = {w.x, w.y};
        return bytes_below(v, x);
    };
    const uint2 here = lcps(tile);
    const uint4 next = mins(w1);
    // (a wave's first cell is read along with their number)
    const int c0 = tid >> 6;
    int4 x = A.cross[tile * kCrossMax + c0];
    TileSplit mine{};
    if (MOMENTS) mine = A.cross_sum[tile * kCrossMax + c0];
    const int cells = A.st->err == 0 ? A.ncross[tile] : 0;
    for (int c = c0; c < cells; c += (int)blockDim.x / 64) {
        if (c > c0) {
            x = A.cross[tile * kCrossMax + c];
            if (MOMENTS) mine = A.cross_sum[tile * kCrossMax + c];
        }
        const int i = __builtin_amdgcn_readfirstlane(x.x), L = __builtin_amdgcn_readfirstlane(x.y);
        const int ord = __builtin_amdgcn_readfirstlane(x.z), g = __builtin_amdgcn_readfirstlane(x.w);
        const int rc = i + ord;
        const float4 root = A.seg_root[g];
        int child[3] = {-1, -1, -1}, found = 0;
        auto add_child = [&](int p) {
            if (found == 0) child[0] = p;
            else if (found == 1) child[1] = p;
            else child[2] = p;
            ++found;
        };
        // a root ends where its graph does
        int end = L == 0 ? (A.sg ? A.node_off[g + 1] : A.n) : -1;
        const int last = L == 0 ? (end - 1) / kTreeTile : tiles - 1;
        // its own tile: children only
        {
            unsigned int m = below(here, L + 1);
            const int skip = i - tile * kTreeTile - lane * 8;  // positions of this lane before i
            if (skip > 0) m &= skip >= 8 ? 0u : 0xffu << skip;
            for (int p; found < 3 && (p = take_first(m, lane)) >= 0;) add_child(tile * kTreeTile + p + 1);
        }
        for (int w0 = w1; w0 <= last && (found < 3 || L > 0); w0 += 1024) {
            // the lane's 16 tiles: least lcp below L + 1, below L
            unsigned int mc = 0u, me = 0u;
            const int t0 = w0 + lane * 16;
            if (t0 <= last) {
                const uint4 w = w0 == w1 ? next : mins(w0);
                const unsigned int lo[2] = {w.x, w.y}, hi[2] = {w.z, w.w};
                mc = bytes_below(lo, L + 1) | bytes_below(hi, L + 1) << 8;
                me = bytes_below(lo, L) | bytes_below(hi, L) << 8;
                unsigned int use = 0xffffu;
                if (t0 <= tile) use &= 0xffffu << (tile + 1 - t0);
                if (t0 + 15 > last) use &= 0xffffu >> (t0 + 15 - last);
                mc &= use;
                me &= use;
            }
            bool done = false;
            for (;;) {
                // with all children found only the end is missing
                const unsigned int m = found < 3 ? mc : me;
                const unsigned long long some = __builtin_amdgcn_ballot_w64(m != 0u);
                if (some == 0ull) break;
                const int at = __builtin_ctzll(some);
                const int bit = __builtin_ctz((unsigned)__builtin_amdgcn_readlane((int)m, at));
                if (lane < at) mc = me = 0u;                   // tiles before it hold no bound that is wanted
                else if (lane == at) {
                    mc &= ~1u << bit;
                    me &= ~1u << bit;
                }
                const int t = w0 + at * 16 + bit;
                const uint2 there = lcps(t);
                unsigned int starts = below(there, L + 1);
                int stop = L == 0 ? end - 1 - t * kTreeTile : -1;          // the cell's last body, if here
                if (L > 0) {
                    unsigned int e = below(there, L);
                    stop = take_first(e, lane);
                    if (stop < 0) stop = kTreeTile;
                }
                for (int p; found < 3 && (p = take_first(starts, lane)) >= 0 && p < stop;) add_child(t * kTreeTile + p + 1);
                if (L > 0 && stop < kTreeTile) {
                    end = t * kTreeTile + stop + 1;
                    done = true;
                    break;
                }
                if (L == 0 && found == 3) break;
            }
            if (done) break;
        }
        // lanes 0-2: a child each; lane 3: the end
        const int at = lane == 0 ? child[0] : lane == 1 ? child[1] : lane == 2 ? child[2] : end;
        const int sat = lane < 4 && at >= 0 ? A.S[at] : 0;
        Moment m{0ull, 0ull, 0ull, 0ull, 0ull};
        if (MOMENTS) {
            // lanes 0-15: the bodies of the last tile from the 16th position before the end; lane 16: those before
            // them; lane 17: its own tile's; then the tiles between
            const int from16 = (end - 1) & ~15, t2 = (end - 1) / kTreeTile, j = from16 + lane;
            TileSplit d{};
            if (lane < 16 && j < end) d = split_of<unsigned long long>(A.sbody[j], root);
            if (lane == 16) d = A.pm16[from16 >> 4];
            if (lane == 17) d = mine;
            d = from_lane(wave_scan(d), 63);
            if (!A.fused) {
                m = mo_sub(A.bmass[t2], A.bmass[tile + 1]);
            } else if (t2 > tile + 1) {
                for (int t = tile + 1 + lane; t < t2; t += 64) m = mo_add(m, A.bmass[t]);
#pragma unroll
                for (int o = 1; o < 64; o <<= 1)
                    m = mo_add(m, Moment{__shfl_xor(m.xl, o, 64), __shfl_xor(m.xh, o, 64), __shfl_xor(m.yl, o, 64),
                                         __shfl_xor(m.yh, o, 64), __shfl_xor(m.m, o, 64)});
            }
            m = mo_add(m, mo_make(moment_x(d), moment_y(d), d.m));
        }
        const int rec = lane < 4 && at >= 0 ? at + sat : -1;
        const int4 kids = make_int4(rc + 1, __builtin_amdgcn_readlane(rec, 0), __builtin_amdgcn_readlane(rec, 1),
                                    __builtin_amdgcn_readlane(rec, 2));
        const unsigned int info = cell_info(__builtin_amdgcn_readlane(rec, 3) - rc, L);
        if (lane == 0) {
            A.kids[rc] = kids;
            A.rcount[rc] = end - i;
            if (MOMENTS) write_cell(A, rc, L, info, m, root);
            else A.rec[rc].w = __uint_as_float(info);
            if (L > 0 && (L & 3) == 0) atomicMax(&rmax[(L >> 2) - 1], end - i);
        }
    }
    __syncthreads();
    if (tid < 8) A.kids_part[(gridDim.x + blockIdx.x) * 8 + tid] = rmax[tid];
}

// Summaries of all cells, bottom-up. A block takes kSumBlock records, which lie in preorder, and sums
// the cells that end inside it in LDS, deepest level first. The few that reach past its end contain
// its last record, so they are nested and of different levels: each has a slot of its own (block,
// level). One block then sums the slots of kSumUnits blocks in the same order, with their other
// children read beforehand; what reaches past those has a slot among kSumUnits of such groups, and
// so on to one group. What bounds all are the levels' dependent steps, which here cost a barrier
// each and no launch: 20k bodies with fractional masses 31 us, where a launch per level took 82;
// an iteration of 70k bodies 155 us (per level 199), of 1M 497 (583), of 11.5M 5,142 (5,820).
constexpr int kSumBlock = 4096, kSumThreads = 1024, kSumUnits = 62;
constexpr int kSumLevels = 33;       // slots per block: the root, then a cell's info level + 1
constexpr int kSumOwn = kSumBlock / kSumThreads;
static_assert(kSumUnits * kSumLevels <= 2 * kSumThreads, "two slots per thread of k_sum_spill");

constexpr unsigned int kBodyInfo = 0xffffffffu;

__device__ __forceinline__ int info_level(unsigned int info) { return (int)(info & ((1u << kInfoLevelBits) - 1)); }

// Records to the next one beside this one.
__device__ __forceinline__ int record_hop(unsigned int info) {
    return info == kBodyInfo ? 1 : max((int)(info >> kInfoLevelBits), 1);
}

struct CellSum {
    float m = 0.0f, x = 0.0f, y = 0.0f;
    __device__ __forceinline__ void add(const float4& c) {
        x = fmaf(c.x, c.z, x);
        y = fmaf(c.y, c.z, y);
        m += c.z;
    }
    __device__ __forceinline__ float4 record(float w) const {
        const float inv = 1.0f / m;
        return make_float4(x * inv, y * inv, m, w);
    }
};

// A cell of info level 0 is the root if a child has that level too (the root's own is 0, as its
// children's): first is its first child, end past its last, in R.
__device__ __forceinline__ bool is_root(const float4* R, int first, int end) {
    for (int r = first; r < end;) {
        const unsigned int ci = __float_as_uint(R[r].w);
        if (ci != kBodyInfo && info_level(ci) == 0) return true;
        r += record_hop(ci);
    }
    return false;
}

__global__ __launch_bounds__(kSumThreads) void k_sum_blocks(float4* __restrict__ rec, int* __restrict__ spill,
                                                            const DevState* __restrict__ st) {
    __shared__ float4 R[kSumBlock];
    __shared__ int slot[kSumLevels];
    __shared__ int deepest;
    if (st->err != 0) return;
    const int tid = threadIdx.x, base = blockIdx.x * kSumBlock, total = st->nrecords;
    const int len = min(kSumBlock, total - base);
    if (len <= 0) return;
    if (tid < kSumLevels) slot[tid] = -1;
    if (tid == 0) deepest = -1;
    int level[kSumOwn], end[kSumOwn];            // level -1: no cell, or one that ends in a later block
#pragma unroll
    for (int k = 0; k < kSumOwn; ++k) {
        const int i = tid + k * kSumThreads;
        level[k] = -1;
        end[k] = 0;
        if (i < len) R[i] = rec[base + i];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSumOwn; ++k) {
        const int i = tid + k * kSumThreads;
        if (i >= len) continue;
        const unsigned int info = __float_as_uint(R[i].w);
        if (info == kBodyInfo) continue;
        end[k] = min(base + i + (int)(info >> kInfoLevelBits), total) - base;
        if (end[k] <= len) {
            level[k] = info_level(info);
            continue;
        }
        const bool root = info_level(info) == 0 && is_root(rec, base + i + 1, base + end[k]);
        slot[root ? 0 : info_level(info) + 1] = base + i;
    }
    int most = level[0];
#pragma unroll
    for (int k = 1; k < kSumOwn; ++k) most = max(most, level[k]);
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, 64));
    if ((tid & 63) == 0 && most >= 0) atomicMax(&deepest, most);
    __syncthreads();
    if (tid < kSumLevels) spill[blockIdx.x * kSumLevels + tid] = slot[tid];
    const int from = deepest;
    // round -1 is the root's
    for (int L = from; L >= -1; --L) {
#pragma unroll
        for (int k = 0; k < kSumOwn; ++k) {
            if (level[k] != L || (L == -1 && end[k] >= 0)) continue;
            const int i = tid + k * kSumThreads;
            const int stop = L == -1 ? ~end[k] : end[k];
            if (L == 0 && is_root(R, i + 1, stop)) {
                level[k] = -1;
                end[k] = ~stop;
                continue;
            }
            CellSum s;
            for (int r = i + 1; r < stop;) {
                const float4 c = R[r];
                s.add(c);
                r += record_hop(__float_as_uint(c.w));
            }
            R[i] = s.record(R[i].w);
            rec[base + i] = R[i];
        }
        __syncthreads();
    }
}

// Units of span records; a block takes kSumUnits of them, and the cells that reach past its last
// go to its own slots in up (read by a launch with kSumUnits times the span).
__global__ __launch_bounds__(kSumThreads) void k_sum_spill(float4* __restrict__ rec, const int* __restrict__ spill,
                                                           int span, int* __restrict__ up,
                                                           const DevState* __restrict__ st) {
    __shared__ float4 sum[2 * kSumThreads];
    __shared__ int slot[kSumLevels];
    if (st->err != 0) return;
    const int tid = threadIdx.x, total = st->nrecords;
    const int unit0 = blockIdx.x * kSumUnits;
    const int units = min((int)(((long long)total + span - 1) / span) - unit0, kSumUnits);
    if (units <= 0) return;
    const int slots = units * kSumLevels;
    const int stop = (int)min((long long)(unit0 + units) * span, (long long)total);
    if (tid < kSumLevels) slot[tid] = -1;
    __syncthreads();
    float4 child[2][4], own[2];
    int ref[2][4];               // a child's slot; -1: it is in child; -2: none
    int cell[2];
    bool waits[2] = {false, false};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int q = tid + k * kSumThreads;
        cell[k] = q < slots ? spill[unit0 * kSumLevels + q] : -1;
        if (cell[k] < 0) continue;
        own[k] = rec[cell[k]];
        const int end = min(cell[k] + (int)(__float_as_uint(own[k].w) >> kInfoLevelBits), total);
        if (end > stop) {
            slot[q % kSumLevels] = cell[k];
            continue;
        }
        int r = cell[k] + 1;
        CellSum s;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ref[k][u] = -2;
            if (r >= end) continue;
            child[k][u] = rec[r];
            const unsigned int ci = __float_as_uint(child[k][u].w);
            const int next = r + record_hop(ci);
            ref[k][u] = -1;
            if (ci != kBodyInfo && r / span != (next - 1) / span) {
                ref[k][u] = (r / span - unit0) * kSumLevels + info_level(ci) + 1;
                waits[k] = true;
            }
            s.add(child[k][u]);
            r = next;
        }
        if (waits[k]) continue;          // (such a cell has at most four children)
        while (r < end) {                // bodies at one point
            const float4 c = rec[r];
            s.add(c);
            r += record_hop(__float_as_uint(c.w));
        }
        sum[q] = s.record(own[k].w);
        rec[cell[k]] = sum[q];
    }
    __syncthreads();
    if (up != nullptr && tid < kSumLevels) up[blockIdx.x * kSumLevels + tid] = slot[tid];
    for (int L = kSumLevels - 1; L >= 0; --L) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int q = tid + k * kSumThreads;
            if (!waits[k] || q % kSumLevels != L) continue;
            CellSum s;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (ref[k][u] != -2) s.add(ref[k][u] >= 0 ? sum[ref[k][u]] : child[k][u]);
            sum[q] = s.record(own[k].w);
            rec[cell[k]] = sum[q];
        }
        __syncthreads();
    }
}

// Heavy cells (mass >= 2^24, listed with the cells) of the integer-mass path, in one
// workgroup: sorted by record index in LDS, then summarised deepest level first, children
// in quadrant order (mass from 0.0f, centroid (sum m*p)*(1/mass), as
// src/RPBHKernels.cu:468-494). A heavy child's summary is read from LDS; light children
// and bodies were written by earlier launches.
__global__ __launch_bounds__(256) void k_big(float4* __restrict__ rec, const int* __restrict__ big_rc,
                                             const unsigned char* __restrict__ big_lvl,
                                             const DevState* __restrict__ st) {
    __shared__ int brc[kMaxBig];
    __shared__ int blv[kMaxBig];
    __shared__ float4 res[kMaxBig];
    __shared__ int maxl;
    if (st->err != 0) return;
    const int nb = min(st->nbig, kMaxBig);
    if (nb == 0) return;
    const int tid = threadIdx.x;
    int P = 1;
    while (P < nb) P <<= 1;
    if (tid == 0) maxl = 0;
    for (int t = tid; t < P; t += 256) {
        brc[t] = t < nb ? big_rc[t] : 0x7fffffff;
        blv[t] = t < nb ? (int)big_lvl[t] : -1;
    }
    __syncthreads();
    // bitonic sort by record index
    for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = tid; t < P; t += 256) {
                const int u = t ^ j;
                if (u > t) {
                    const bool up = (t & k) == 0;
                    if ((brc[t] > brc[u]) == up) {
                        const int a = brc[t], b = blv[t];
                        brc[t] = brc[u];
                        blv[t] = blv[u];
                        brc[u] = a;
                        blv[u] = b;
                    }
                }
            }
            __syncthreads();
        }
    for (int t = tid; t < nb; t += 256) atomicMax(&maxl, blv[t]);
    __syncthreads();
    for (int L = maxl; L >= 0; --L) {
        for (int t = tid; t < nb; t += 256) {
            if (blv[t] != L) continue;
            const int rc = brc[t];
            const int end = min(rc + (int)(__float_as_uint(rec[rc].w) >> kInfoLevelBits), st->nrecords);
            float cm = 0.0f, px = 0.0f, py = 0.0f;
            int r = rc + 1;
            while (r < end) {
                float4 c = rec[r];
                const unsigned int ci = __float_as_uint(c.w);
                if (ci != 0xffffffffu) {
                    int lo = 0, hi = nb;   // is r heavy?
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if (brc[mid] <= r) lo = mid;
                        else hi = mid;
                    }
                    if (brc[lo] == r) c = res[lo];
                }
                px = fmaf(c.x, c.z, px);
                py = fmaf(c.y, c.z, py);
                cm += c.z;
                r += ci == 0xffffffffu ? 1 : max((int)(ci >> kInfoLevelBits), 1);
            }
            const float inv = 1.0f / cm;
            res[t] = make_float4(px * inv, py * inv, cm, 0.0f);
        }
        __syncthreads();
    }
    for (int t = tid; t < nb; t += 256) {
        const float4 v = res[t];
        rec[brc[t]].x = v.x;
        rec[brc[t]].y = v.y;
        rec[brc[t]].z = v.z;
    }
}

}  // namespace

int displacement_blocks(const Bufs& b) {
    int cap = b.grid_cap < kPartBlocks ? b.grid_cap : kPartBlocks;
    int g = (b.n + 255) / 256;
    return g < 1 ? 1 : (g > cap ? cap : g);
}

namespace {

template <bool RESET>
void new_positions(const Bufs& b, const NewState& init, hipStream_t s) {
    k_new_positions<RESET><<<displacement_blocks(b), 256, 0, s>>>(b.pos, b.rank, b.n, b.pos_rank, b.bbox_part, b.st,
                                                                 init, b.seg_st, b.nseg, b.f, b.fprev, b.fga);
    if (b.nseg > 1) launch_seg_bbox(b, s);
}

}  // namespace

void launch_new_positions(const Bufs& b, int full_sorts, hipStream_t s) {
    new_positions<false>(b, NewState{0.0f, 0.0f, 0.0f, 0.0f, full_sorts}, s);
}

void launch_reset(const Bufs& b, float global_speed, float speed_efficiency, float jitter_tolerance, float k_s_max,
                  hipStream_t s) {
    new_positions<true>(b, NewState{global_speed, speed_efficiency, jitter_tolerance, k_s_max, -1}, s);
}

namespace {

KeysArgs keys_args(const Bufs& b, int first) {
    return KeysArgs{b.pos, b.mass, b.n, b.bbox_part, b.st, b.seg_root, b.sort.keys[0], b.sort.keys[1], b.sort.vals[0],
                    b.sort.vals[1], b.pm, first, b.sort.hist_in_keys ? b.sort.digit_hist : nullptr, b.seg_st, b.seg_cur};
}

int keys_blocks(const Bufs& b) {
    const int blocks = std::min((b.n + 255) / 256, b.grid_cap);
    // Each block that counts digits adds up to 256 counts per pass to the table: at 131,000 bodies
    // 145.6 us an iteration with 128 blocks, 146.5 with 256, 150.5 with one per 256 bodies; at
    // 262,000 198.2, 196.5, 207.6
    return b.sort.hist_in_keys ? std::min(blocks, std::max(128, (b.n + 1023) / 1024)) : blocks;
}

}  // namespace

void launch_keys(const Bufs& b, int first, hipStream_t s) {
    k_keys<<<keys_blocks(b), 256, 0, s>>>(keys_args(b, first));
}

void launch_keys_attraction(const Bufs& b, const Params& p, int first, hipStream_t s) {
    const AttractPlan w = attract_plan(b);
    const int kb = keys_blocks(b);
    const auto k = p.linlog || b.ew ? k_keys_attract<true> : k_keys_attract<false>;
    k<<<kb + w.total, 256, 0, s>>>(keys_args(b, first), kb, attract_args(b, p), w, b.attr_chunks, b.attr_part);
    launch_attract_heavy(b, p, s);
}

void launch_tree(Bufs& b, hipStream_t s) {
    const int n = b.n;
    const int tiles = (n + kTreeTile - 1) / kTreeTile;
    const int* sg = b.nseg > 1 ? b.sg : nullptr;
    Moment* bm = b.int_mass ? b.bmass : nullptr;
    k_lcp<<<tiles, kTreeThreads, 0, s>>>(b.sort.keys[0], sg, n, b.lcp, b.blocksum, b.sort.vals[0], b.pm,
                                         b.seg_root, bm, b.sbody, b.st);
    // up to kFuseTiles tiles, k_tile sums the tile totals itself
    const bool fused = tiles <= kFuseTiles;
    if (!fused) {
        const int chunks = (tiles + kTileChunk - 1) / kTileChunk;
        Moment* cm = b.int_mass ? b.chunk_mass : nullptr;
        k_scan_up<<<chunks, kTileChunk, 0, s>>>(b.blocksum, bm, tiles, b.chunk_sum, cm);
        k_scan_blocks<<<1, 1024, 0, s>>>(b.chunk_sum, chunks, n, b.cap_records, b.rec_begin + b.nseg, b.st, cm);
        k_scan_down<<<chunks, kTileChunk, 0, s>>>(b.blocksum, bm, tiles, b.chunk_sum, cm);
    }
    const TileArgs T{b.lcp,       sg,      n,       b.blocksum,  bm,        fused ? 1 : 0, b.S,     b.sbody,
                     b.rec,       b.kids,         b.rcount, b.st,
                     b.seg_root,  reinterpret_cast<TileSplit*>(b.pmass),        b.cap_records, b.rec_begin, b.nseg, b.node_off, b.big_rc, b.big_lvl,
                     b.kids_part, b.cross,        reinterpret_cast<TileSplit*>(b.cross_sum), b.ncross, b.tmin};
    // a wave for each of a tile's cells while the tiles fit the chip once (50,000 bodies: 8.4 us with
    // 1,024 threads, 9.5 with 512), fewer where blocks follow one another (2M bodies: 34 us with
    // 256 threads, 39 with 512, 84 with 1,024)
    const int ct = tiles <= 256 ? kCrossThreads : tiles <= 1024 ? 512 : 256;
    if (b.int_mass) {
        k_tile<true><<<tiles, kTreeTile, 0, s>>>(T);
        k_cross<true><<<tiles, ct, 0, s>>>(T);
    } else {
        k_tile<false><<<tiles, kTreeTile, 0, s>>>(T);
        k_cross<false><<<tiles, ct, 0, s>>>(T);
    }
    if (b.int_mass) {
        if (!b.no_big) k_big<<<1, 256, 0, s>>>(b.rec, b.big_rc, b.big_lvl, b.st);
        return;
    }
    int units = (b.cap_records + kSumBlock - 1) / kSumBlock, span = kSumBlock;
    int* spill = b.spill;
    k_sum_blocks<<<units, kSumThreads, 0, s>>>(b.rec, spill, b.st);
    for (;;) {
        const int groups = (units + kSumUnits - 1) / kSumUnits;
        int* up = groups > 1 ? spill + units * kSumLevels : nullptr;
        k_sum_spill<<<groups, kSumThreads, 0, s>>>(b.rec, spill, span, up, b.st);
        if (groups == 1) return;
        spill = up;
        units = groups;
        span *= kSumUnits;           // (units of 2^31 records at most: below 62^4 blocks)
    }
}

}  // namespace gfa2
