// Layout quality: hop distances of sampled node pairs and normalized stress (no counterpart
// in the reference).
//
// Pairs: K sources, T targets each (targets drawn uniformly among the other nodes).
// Hop distances come from a multi-source breadth-first search of up to 1,024 sources at a
// time: every node keeps a row of W 64-bit words, one bit per source, of the sources that have
// reached it and of those that reached it on the last level; a level is one pull over the CSR
// (each node ORs its neighbours' last-level rows; an OR does not depend on its order, so the
// result is deterministic). After each level the pairs whose target bit just appeared get that
// level as their distance. Pairs whose target is never reached keep distance 0 and are left out.
//
// Normalized stress of positions p over the P reachable pairs, with r = |p_a - p_b| / d:
//   alpha = sum r / sum r^2,  NS = (1/P) sum (alpha r - 1)^2 = 1 - (sum r)^2 / (P sum r^2)
// summed in double in one pass (per-block partials, fixed-order final sum).
#include "engine_internal.h"

#include <algorithm>
#include <utility>
#include <vector>

namespace gfa2 {
namespace {

// No source has reached any node; the bits past the nk sources count as reached, so that a row
// is done when its words are all ones.
template <int W>
__global__ __launch_bounds__(256) void k_bfs_init(unsigned long long* __restrict__ seen,
                                                  unsigned long long* __restrict__ front, long long words, int nk) {
    for (long long q = blockIdx.x * 256ll + threadIdx.x; q < words; q += (long long)gridDim.x * 256) {
        const int bits = nk - 64 * (int)(q % W);          // sources of this word
        seen[q] = bits >= 64 ? 0ull : (bits <= 0 ? ~0ull : ~0ull << bits);
        front[q] = 0ull;
    }
}

// The sources are distinct nodes: one thread per source, no word is shared.
template <int W>
__global__ __launch_bounds__(256) void k_bfs_seed(unsigned long long* __restrict__ seen,
                                                  unsigned long long* __restrict__ front,
                                                  const int* __restrict__ src, int k0, int nk) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= nk) return;
    const size_t q = (size_t)src[k0 + k] * W + (k >> 6);
    seen[q] |= 1ull << (k & 63);
    front[q] = 1ull << (k & 63);
}

// One word of the OR of the front rows of entries e, e + stride, ... below e1 (four loads in
// flight).
template <int W>
__device__ __forceinline__ unsigned long long or_rows(const int* __restrict__ col,
                                                      const unsigned long long* __restrict__ front, int e, int e1,
                                                      int stride, int w) {
    unsigned long long acc = 0ull;
    for (; e + 3 * stride < e1; e += 4 * stride) {
        const int j0 = col[e], j1 = col[e + stride], j2 = col[e + 2 * stride], j3 = col[e + 3 * stride];
        const unsigned long long a0 = front[(size_t)j0 * W + w], a1 = front[(size_t)j1 * W + w];
        const unsigned long long a2 = front[(size_t)j2 * W + w], a3 = front[(size_t)j3 * W + w];
        acc |= (a0 | a1) | (a2 | a3);
    }
    for (; e < e1; e += stride) acc |= front[(size_t)col[e] * W + w];
    return acc;
}

// One level over all rows, W lanes per row (one word each, so a neighbour's row is one
// contiguous read). Rows come in the attraction's degree classes: light rows W lanes each,
// medium rows a wave each (64 / W entries at a time), heavy rows a block per chunk of
// kAttrChunk entries ORed into hacc, which k_bfs_heavy turns into the row's result. Lanes whose
// word is complete read nothing. prev: whether the last level reached anything.
//
// Bound by the rows gathered (8 W bytes per CSR entry): 5M entries of an R-MAT graph of 2^18
// ids with W = 16 are 640 MB, read in about 100 us on the levels that gather everything
// (6.4 TB/s, from L2 and MALL), and 1,024 sources take one search of 7 such levels. One word and
// a thread per row left a hub's row of tens of thousands of entries to one thread: 1.12 ms a
// level and 123 levels; the whole set-up with its pairs went from 156 ms to 1.7 ms.
template <int W>
__global__ __launch_bounds__(256) void k_bfs_level(const int* __restrict__ rowptr, const int* __restrict__ col,
                                                   const int* __restrict__ lists, int nlight, int nmedium,
                                                   const int2* __restrict__ chunks, int light_blocks,
                                                   int medium_blocks, const unsigned long long* __restrict__ front,
                                                   unsigned long long* __restrict__ next,
                                                   unsigned long long* __restrict__ seen,
                                                   unsigned long long* __restrict__ hacc,
                                                   const int* __restrict__ prev, int* __restrict__ changed) {
    if (*prev == 0) return;
    constexpr int S = 64 / W;                 // rows (or entries) a wave takes side by side
    const int lane = threadIdx.x & 63, w = lane % W, slot = lane / W;
    const int wave = threadIdx.x >> 6;
    int blk = blockIdx.x;
    if (blk < light_blocks) {
        const int k = (blk * 4 + wave) * S + slot;
        bool any = false;
        if (k < nlight) {
            const int v = lists[k];
            const unsigned long long s = seen[(size_t)v * W + w];
            unsigned long long nw = 0ull;
            if (~s != 0ull) nw = or_rows<W>(col, front, rowptr[v], rowptr[v + 1], 1, w) & ~s;
            next[(size_t)v * W + w] = nw;
            if (nw) seen[(size_t)v * W + w] = s | nw;
            any = nw != 0ull;
        }
        if (__builtin_amdgcn_ballot_w64(any) != 0ull && lane == 0) *changed = 1;
        return;
    }
    blk -= light_blocks;
    if (blk < medium_blocks) {
        const int k = blk * 4 + wave;
        if (k >= nmedium) return;             // uniform per wave
        const int v = lists[nlight + k];
        const unsigned long long s = seen[(size_t)v * W + w];
        unsigned long long acc = 0ull;
        if (~s != 0ull) acc = or_rows<W>(col, front, rowptr[v] + slot, rowptr[v + 1], S, w);
#pragma unroll
        for (int o = 32; o >= W; o >>= 1) acc |= __shfl_xor(acc, o, 64);
        const unsigned long long nw = acc & ~s;
        if (slot == 0) {
            next[(size_t)v * W + w] = nw;
            if (nw) seen[(size_t)v * W + w] = s | nw;
        }
        if (__builtin_amdgcn_ballot_w64(nw != 0ull) != 0ull && lane == 0) *changed = 1;
        return;
    }
    blk -= medium_blocks;
    const int2 ch = chunks[blk];
    const int v = lists[nlight + nmedium + ch.x];
    if (~seen[(size_t)v * W + w] == 0ull) return;      // no barrier below
    const int e1 = min(ch.y + kAttrChunk, rowptr[v + 1]);
    const unsigned long long acc = or_rows<W>(col, front, ch.y + wave * S + slot, e1, 4 * S, w);
    if (acc) atomicOr(&hacc[(size_t)ch.x * W + w], acc);
}

// Heavy rows after a level: the result of the chunks' OR, which is cleared for the next level.
template <int W>
__global__ __launch_bounds__(256) void k_bfs_heavy(const int* __restrict__ heavy, int nheavy,
                                                   unsigned long long* __restrict__ hacc,
                                                   unsigned long long* __restrict__ next,
                                                   unsigned long long* __restrict__ seen,
                                                   const int* __restrict__ prev, int* __restrict__ changed) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= nheavy * W || *prev == 0) return;
    const size_t at = (size_t)heavy[q / W] * W + q % W;
    const unsigned long long s = seen[at], nw = hacc[q] & ~s;
    hacc[q] = 0ull;
    next[at] = nw;
    if (nw) {
        seen[at] = s | nw;
        *changed = 1;
    }
}

// Pairs of sources k0..k0+nk-1 (pair index = source index * T + j).
template <int W>
__global__ __launch_bounds__(256) void k_bfs_pairs(const int* __restrict__ tgt, int T, int k0, int nk,
                                                   const unsigned long long* __restrict__ next, int level,
                                                   int* __restrict__ dist, const int* __restrict__ changed) {
    if (*changed == 0) return;
    // unsigned: a search's pairs are fewer than 2^31, but a grid stride more may not be
    const unsigned int total = (unsigned int)nk * T;
    for (unsigned int q = blockIdx.x * 256u + threadIdx.x; q < total; q += gridDim.x * 256u) {
        const int k = (int)(q / (unsigned int)T);
        const size_t p = (size_t)k0 * T + q;
        if (dist[p] == 0 && ((next[(size_t)tgt[p] * W + (k >> 6)] >> (k & 63)) & 1ull)) dist[p] = level;
    }
}

// Targets of source k: uniform over the other n - 1 nodes, draw number `first` + pair of the
// generator seeded by `seed` (SplitMix64 is a hash of its counter, so every draw stands alone).
__global__ __launch_bounds__(256) void k_draw_targets(const int* __restrict__ src, int T, long long np,
                                                      unsigned long long seed, unsigned long long first, int n,
                                                      int* __restrict__ tgt) {
    for (long long p = blockIdx.x * 256ll + threadIdx.x; p < np; p += (long long)gridDim.x * 256) {
        unsigned long long z = seed + (first + (unsigned long long)p + 1ull) * 0x9E3779B97F4A7C15ull;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        const int u = (int)(z % (unsigned long long)(n - 1));
        tgt[p] = u >= src[p / T] ? u + 1 : u;
    }
}

// Pairs with a distance, one count per block.
__global__ __launch_bounds__(256) void k_count_pairs(const int* __restrict__ dist, long long np,
                                                     int* __restrict__ part) {
    __shared__ int wsum[4];
    int c = 0;
    for (long long p = blockIdx.x * 256ll + threadIdx.x; p < np; p += (long long)gridDim.x * 256) c += dist[p] > 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

__global__ __launch_bounds__(256) void k_stress_partials(const float2* __restrict__ pos, const int* __restrict__ src,
                                                         const int* __restrict__ tgt, const int* __restrict__ dist,
                                                         int T, long long np, double* __restrict__ part) {
    __shared__ double r1[256], r2[256], rc[256];
    double s1 = 0.0, s2 = 0.0, c = 0.0;
    for (long long p = blockIdx.x * 256ll + threadIdx.x; p < np; p += (long long)gridDim.x * 256) {
        const int d = dist[p];
        if (d <= 0) continue;
        const float2 a = pos[src[p / T]], b = pos[tgt[p]];
        const double dx = (double)a.x - b.x, dy = (double)a.y - b.y;
        const double r = sqrt(dx * dx + dy * dy) / d;
        s1 += r;
        s2 += r * r;
        c += 1.0;
    }
    const int t = threadIdx.x;
    r1[t] = s1;
    r2[t] = s2;
    rc[t] = c;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (t < o) {
            r1[t] += r1[t + o];
            r2[t] += r2[t + o];
            rc[t] += rc[t + o];
        }
        __syncthreads();
    }
    if (t == 0) {
        part[3 * blockIdx.x] = r1[0];
        part[3 * blockIdx.x + 1] = r2[0];
        part[3 * blockIdx.x + 2] = rc[0];
    }
}

constexpr int kBfsBatch = 6;       // levels queued between two looks at whether the search has ended
constexpr int kCountBlocks = 256;

int grid_of(long long items, int most) {
    const long long b = (items + 255) / 256;
    return (int)(b < 1 ? 1 : (b > most ? most : b));
}

// Scratch of one search: three rows of W words per node, the heavy rows' accumulators and the
// levels' flags.
struct BfsScratch {
    unsigned long long* words = nullptr;
    int* flags = nullptr;
    ~BfsScratch() {
        if (words) (void)hipFree(words);
        if (flags) (void)hipFree(flags);
    }
};

template <int W>
int bfs_run(const Bufs& b, const int* d_src, int K, const int* d_tgt, int T, int* d_dist, BfsScratch& m,
            hipStream_t s) {
    const int n = b.n;
    const long long words = (long long)n * W;
    unsigned long long *seen = m.words, *cur = seen + words, *nxt = cur + words, *hacc = nxt + words;
    constexpr int S = 64 / W;
    const int light_blocks = (b.nlight + 4 * S - 1) / (4 * S);
    const int medium_blocks = (b.nmedium + 3) / 4;
    const int blocks = light_blocks + medium_blocks + b.nattr_chunks;
    const int* heavy = b.node_lists + b.nlight + b.nmedium;
    if (b.nheavy > 0 && hipMemsetAsync(hacc, 0, sizeof(unsigned long long) * b.nheavy * W, s) != hipSuccess) return -1;
    for (int k0 = 0; k0 < K; k0 += 64 * W) {
        const int nk = K - k0 < 64 * W ? K - k0 : 64 * W;
        k_bfs_init<W><<<grid_of(words, 4096), 256, 0, s>>>(seen, cur, words, nk);
        k_bfs_seed<W><<<grid_of(nk, 1 << 20), 256, 0, s>>>(seen, cur, d_src, k0, nk);
        // flag 0: the last level of the batch before reached something; flag j: level j of this batch did
        int flag[kBfsBatch + 1];
        bool more = true;
        for (int level = 1; more && level <= n;) {
            if (hipMemsetD32Async((hipDeviceptr_t)m.flags, 1, 1, s) != hipSuccess ||
                hipMemsetAsync(m.flags + 1, 0, sizeof(int) * kBfsBatch, s) != hipSuccess)
                return -1;
            for (int j = 1; j <= kBfsBatch; ++j, ++level) {
                k_bfs_level<W><<<blocks, 256, 0, s>>>(b.rowptr, b.col, b.node_lists, b.nlight, b.nmedium,
                                                      b.attr_chunks, light_blocks, medium_blocks, cur, nxt, seen,
                                                      hacc, m.flags + j - 1, m.flags + j);
                if (b.nheavy > 0)
                    k_bfs_heavy<W><<<grid_of((long long)b.nheavy * W, 1 << 20), 256, 0, s>>>(
                        heavy, b.nheavy, hacc, nxt, seen, m.flags + j - 1, m.flags + j);
                k_bfs_pairs<W><<<grid_of((long long)nk * T, 2048), 256, 0, s>>>(d_tgt, T, k0, nk, nxt, level, d_dist,
                                                                               m.flags + j);
                std::swap(cur, nxt);
            }
            if (hipMemcpyAsync(flag, m.flags, sizeof(flag), hipMemcpyDeviceToHost, s) != hipSuccess) return -1;
            if (hipStreamSynchronize(s) != hipSuccess) return -1;
            for (int j = 1; j <= kBfsBatch; ++j) more = more && flag[j] != 0;
        }
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

void stress_draw_targets(const int* d_src, int T, long long np, unsigned long long seed, unsigned long long first, int n,
                         int* d_tgt, hipStream_t s) {
    k_draw_targets<<<grid_of(np, 4096), 256, 0, s>>>(d_src, T, np, seed, first, n, d_tgt);
}

// Words per node: as many as the sources need, up to 16 (1,024 sources: a row of 128 bytes, one
// cache line per CSR entry). Fewer passes read the CSR fewer times and a wider row is gathered
// at a better rate, so the most words that fit are taken: three rows per node within
// kBfsScratch bytes, and half as many whenever the device has no room for them.
int stress_hop_distances(const Bufs& b, const int* d_src, int K, const int* d_tgt, int T, int* d_dist,
                         long long* npairs, hipStream_t s) {
    constexpr long long kBfsScratch = 4ll << 30;
    int W = 1;
    while (W < 16 && 64 * W < K) W *= 2;
    while (W > 1 && 24ll * W * b.n > kBfsScratch) W /= 2;
    BfsScratch m;
    hipError_t e = hipErrorOutOfMemory;
    for (;; W /= 2) {
        e = hipMalloc(&m.words, sizeof(unsigned long long) * W * (3 * (size_t)b.n + (size_t)b.nheavy));
        if (e != hipErrorOutOfMemory || W == 1) break;
        (void)hipGetLastError();               // tried again with fewer words
        m.words = nullptr;
    }
    if (e == hipSuccess) e = hipMalloc(&m.flags, sizeof(int) * std::max(kBfsBatch + 1, kCountBlocks));
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();               // reported here: not again by the next call
        return -2;
    }
    if (e != hipSuccess) return -1;
    if (hipMemsetAsync(d_dist, 0, sizeof(int) * (size_t)K * T, s) != hipSuccess) return -1;
    int rc = 0;
    switch (W) {
        case 1: rc = bfs_run<1>(b, d_src, K, d_tgt, T, d_dist, m, s); break;
        case 2: rc = bfs_run<2>(b, d_src, K, d_tgt, T, d_dist, m, s); break;
        case 4: rc = bfs_run<4>(b, d_src, K, d_tgt, T, d_dist, m, s); break;
        case 8: rc = bfs_run<8>(b, d_src, K, d_tgt, T, d_dist, m, s); break;
        default: rc = bfs_run<16>(b, d_src, K, d_tgt, T, d_dist, m, s); break;
    }
    if (rc == 0 && npairs) {
        int part[kCountBlocks];
        k_count_pairs<<<kCountBlocks, 256, 0, s>>>(d_dist, (long long)K * T, m.flags);
        if (hipGetLastError() != hipSuccess) rc = -1;
        if (rc == 0 && hipMemcpyAsync(part, m.flags, sizeof(part), hipMemcpyDeviceToHost, s) != hipSuccess) rc = -1;
        *npairs = 0;
        if (rc == 0 && hipStreamSynchronize(s) != hipSuccess) rc = -1;
        for (int k = 0; k < kCountBlocks && rc == 0; ++k) *npairs += part[k];
    }
    (void)hipStreamSynchronize(s);             // the scratch is freed on return
    return rc;
}

int stress_reduce(const float2* pos, const int* d_src, const int* d_tgt, const int* d_dist, int T, long long np,
                  double* d_part, int nblocks, double out[3], hipStream_t s) {
    k_stress_partials<<<nblocks, 256, 0, s>>>(pos, d_src, d_tgt, d_dist, T, np, d_part);
    std::vector<double> h((size_t)3 * nblocks);
    if (hipMemcpyAsync(h.data(), d_part, sizeof(double) * 3 * nblocks, hipMemcpyDeviceToHost, s) != hipSuccess)
        return -1;
    if (hipStreamSynchronize(s) != hipSuccess) return -1;
    out[0] = out[1] = out[2] = 0.0;
    for (int k = 0; k < nblocks; ++k) {
        out[0] += h[3 * k];
        out[1] += h[3 * k + 1];
        out[2] += h[3 * k + 2];
    }
    return 0;
}

}  // namespace gfa2
