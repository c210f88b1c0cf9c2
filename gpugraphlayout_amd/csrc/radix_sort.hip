// LSD radix sort of (u64 key, u32 value) pairs for gfx950.
//
// Up to 262,144 pairs: one launch per 8-bit pass ("onesweep"), after one histogram launch for all
// passes.
//   k_sort_hist  digit histograms of every pass at once (order-independent), LDS then global
//                atomics; the table is cleared by k_sort_zero first
//   k_onesweep   per tile (8 pairs per thread): tiles are taken in the order of a global ticket,
//                the tile's digit counts are published, and while they travel the tile ranks its
//                pairs stably (wave64 ballot matching). Then every earlier tile's counts are read,
//                eight at a time, and added: each digit's exclusive prefix, without a chain from
//                tile to tile. A tile only ever waits for tiles with smaller tickets, which started
//                before it and publish their counts before they wait themselves, so the waits end;
//                every wait is also bounded and raises an error flag.
// Larger inputs (or SortBuffers::onesweep = false): three launches per pass (per-tile histograms,
// a scan over tiles per digit, scatter), with every cross-tile dependency through a launch
// boundary.
// Both are stable (hence LSD-correct) and give the same result.
#include "engine_internal.h"

namespace gfa2 {
namespace {

constexpr int kWaves = kSortThreads / 64;

// A pass this iteration's sort skips (see radix_sort_pairs).
__device__ __forceinline__ bool pass_skipped(const DevState* __restrict__ st, int pass) {
    return st != nullptr && pass < st->sort_skip;
}

// The low passes that do not run: those the device skips and those the host did not launch.
__device__ __forceinline__ int passes_below(const DevState* __restrict__ st, int first) {
    return max(st != nullptr ? st->sort_skip : 0, first);
}

// The buffer the first pass that runs reads: buffer 0, or with `lead` (the total number of
// passes, when the keys were written where an odd count of running passes needs them) the one
// that makes the last pass end in buffer 0.
__device__ __forceinline__ int start_buffer(const DevState* __restrict__ st, int first, int lead) {
    return lead ? ((lead - passes_below(st, first)) & 1) : 0;
}

// The buffer a pass reads (it writes the other one): every pass that runs flips it (skipped
// passes move nothing).
__device__ __forceinline__ int pass_src(const DevState* __restrict__ st, int first, int lead, int pass) {
    return (start_buffer(st, first, lead) + pass - passes_below(st, first)) & 1;
}

__global__ __launch_bounds__(kSortThreads) void k_upsweep(const unsigned long long* __restrict__ k0,
                                                          const unsigned long long* __restrict__ k1,
                                                          int n, int shift, unsigned int* __restrict__ hist,
                                                          int tiles, const DevState* __restrict__ st, int first,
                                                          int lead, int pass) {
    if (pass_skipped(st, pass)) return;
    const unsigned long long* __restrict__ keys = pass_src(st, first, lead, pass) ? k1 : k0;
    __shared__ unsigned int h[256];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const int base = blockIdx.x * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        int e = base + r * kSortThreads + tid;
        if (e < n) atomicAdd(&h[(unsigned)(keys[e] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[tid * tiles + blockIdx.x] = h[tid];
}

// One block per digit row: exclusive scan over the tiles, row total into rowtot. The row is
// read in chunks of 256 tiles (one per thread, coalesced), up to kRowChunks chunks requested
// before any is scanned; each chunk is one block scan (shuffles within the waves, then the
// four wave totals) carried into the next.
constexpr int kRowChunks = 16;

__global__ __launch_bounds__(256) void k_rowscan(unsigned int* __restrict__ hist, int tiles,
                                                 unsigned int* __restrict__ rowtot, const DevState* __restrict__ st,
                                                 int pass) {
    if (pass_skipped(st, pass)) return;
    __shared__ unsigned int sh[2][4];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    unsigned int* h = hist + (size_t)blockIdx.x * tiles;
    unsigned int carry = 0u;
    int parity = 0;
    for (int c0 = 0; c0 < tiles; c0 += 256 * kRowChunks) {
        unsigned int v[kRowChunks];
#pragma unroll
        for (int c = 0; c < kRowChunks; ++c) {
            const int t = c0 + c * 256 + tid;
            v[c] = t < tiles ? h[t] : 0u;
        }
#pragma unroll
        for (int c = 0; c < kRowChunks; ++c) {
            if (c0 + c * 256 >= tiles) break;            // uniform
            unsigned int inc = v[c];
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned int t = __shfl_up(inc, o, 64);
                if (lane >= o) inc += t;
            }
            if (lane == 63) sh[parity][wave] = inc;
            __syncthreads();
            unsigned int off = 0u, total = 0u;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const unsigned int x = sh[parity][w];
                if (w < wave) off += x;
                total += x;
            }
            const int t = c0 + c * 256 + tid;
            if (t < tiles) h[t] = carry + off + inc - v[c];
            carry += total;
            parity ^= 1;
        }
    }
    if (tid == 0) rowtot[blockIdx.x] = carry;
}

// Stable ranks within a tile, three block barriers per tile: each wave owns a contiguous
// quarter of the tile (kSortItems rows of 64 pairs), ranks its pairs row by row with
// a wave64 ballot match against its own running digit counts in LDS, then one pass over the
// digits turns the per-wave counts into destinations (wave order is tile order, so the sort
// stays stable).
__device__ __forceinline__ void rank_rows(const unsigned long long (&key)[kSortItems], int wbase, int n, int shift,
                                          unsigned int* __restrict__ wcnt, unsigned int (&rank)[kSortItems]) {
    const int lane = threadIdx.x & 63;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const bool valid = wbase + r * 64 + lane < n;
        const unsigned int d = (unsigned)(key[r] >> shift) & 255u;
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const unsigned long long m = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? m : ~m;
        }
        const unsigned int rr = (unsigned)__popcll(peers & lt);
        // every lane reads the digit's count before its leader writes it (one wave, LDS in order)
        const unsigned int before = valid ? wcnt[d] : 0u;
        rank[r] = before + rr;
        if (valid && rr == 0) wcnt[d] = before + (unsigned)__popcll(peers);
    }
}

// Exclusive scan of one value per thread over the block's 256 threads: shuffle scans within
// the waves, then the four wave totals (one barrier). sh: 4 words of LDS, not reused before
// another barrier.
__device__ __forceinline__ unsigned int block_exscan256(unsigned int v, unsigned int* __restrict__ sh) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    unsigned int inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) sh[wave] = inc;
    __syncthreads();
    unsigned int off = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
        if (w < wave) off += sh[w];
    return off + inc - v;
}

// LDS of the tile step: per-wave digit counts, the staged tile, scan scratch.
struct TileLds {
    unsigned int wcnt[kWaves][256];
    unsigned long long skey[kSortTile];
    unsigned int sval[kSortTile];
    int delta[256];                 // global destination minus tile position, per digit
    unsigned int sh[2][kWaves];
};

// Writes one tile's pairs (held in registers, each wave a contiguous quarter) to their sorted
// places. dglobal: this thread's digit's first destination for the tile. The pairs are ranked
// stably (rank_rows), placed in LDS in digit order, then written out in tile order, so the
// pairs of a digit leave as one run of consecutive addresses.
__device__ __forceinline__ unsigned int scatter_tile(const unsigned long long (&key)[kSortItems],
                                             const unsigned int (&val)[kSortItems], int tile, int n, int shift,
                                             unsigned int dglobal, TileLds& L,
                                             unsigned long long* __restrict__ kout, unsigned int* __restrict__ vout) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wbase = tile * kSortTile + wave * (kSortItems * 64);
    unsigned int rank[kSortItems];
    rank_rows(key, wbase, n, shift, L.wcnt[wave], rank);
    __syncthreads();
    // per digit (one per thread): the tile's count, its start within the tile, each wave's start
    unsigned int c[kWaves], tcount = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        c[w] = L.wcnt[w][tid];
        tcount += c[w];
    }
    const unsigned int tstart = block_exscan256(tcount, L.sh[1]);
    {
        unsigned int run = tstart;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            L.wcnt[w][tid] = run;
            run += c[w];
        }
    }
    L.delta[tid] = (int)dglobal - (int)tstart;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        if (wbase + r * 64 + lane < n) {
            const unsigned int at = L.wcnt[wave][(unsigned)(key[r] >> shift) & 255u] + rank[r];
            L.skey[at] = key[r];
            L.sval[at] = val[r];
        }
    }
    __syncthreads();
    const int count = min(kSortTile, n - tile * kSortTile);
    for (int j = tid; j < count; j += kSortThreads) {
        const unsigned long long k = L.skey[j];
        const unsigned int dst = (unsigned int)(L.delta[(unsigned)(k >> shift) & 255u] + j);
        kout[dst] = k;
        vout[dst] = L.sval[j];
    }
    return tcount;
}

__global__ __launch_bounds__(kSortThreads) void k_scatter(unsigned long long* __restrict__ k0,
                                                          unsigned int* __restrict__ v0,
                                                          unsigned long long* __restrict__ k1,
                                                          unsigned int* __restrict__ v1, int n, int shift,
                                                          const unsigned int* __restrict__ hist, int tiles,
                                                          const unsigned int* __restrict__ rowtot,
                                                          const DevState* __restrict__ st, int first, int lead,
                                                          int pass) {
    if (pass_skipped(st, pass)) return;
    const int src = pass_src(st, first, lead, pass);
    const unsigned long long* __restrict__ kin = src ? k1 : k0;
    const unsigned int* __restrict__ vin = src ? v1 : v0;
    unsigned long long* __restrict__ kout = src ? k0 : k1;
    unsigned int* __restrict__ vout = src ? v0 : v1;
    __shared__ TileLds L;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wbase = blockIdx.x * kSortTile + wave * (kSortItems * 64);
    unsigned long long key[kSortItems];
    unsigned int val[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const int e = wbase + r * 64 + lane;
        key[r] = e < n ? kin[e] : 0ull;
        val[r] = e < n ? vin[e] : 0u;
    }
#pragma unroll
    for (int w = 0; w < kWaves; ++w) L.wcnt[w][tid] = 0;
    // digit starts: exclusive scan of the digit totals, plus this tile's offset within the digit
    const unsigned int dglobal = block_exscan256(rowtot[tid], L.sh[0]) + hist[(size_t)tid * tiles + blockIdx.x];
    scatter_tile(key, val, blockIdx.x, n, shift, dglobal, L, kout, vout);
}

// ---- one block per segment, or four segments per block ---------------------------------------
// Segment g is [node_off[g], node_off[g+1]) of both buffers; its pairs are sorted by the full key,
// stable, into buffer 0. A block of 1,024 threads takes one segment of more than kSegSmall
// pairs, or four smaller ones, a quarter of its threads each (every quarter runs the same passes
// and meets the same barriers). A segment of up to 8 pairs per thread stays in registers and LDS
// from its first pass to its last; a longer one takes its tiles in order in every pass, from one
// buffer to the other, with the running digit starts of all passes counted beforehand. Blocks take
// segments in `order` (largest first), so the longest ones start first. What bounds it is the
// largest segment's chain of tile steps: 192 graphs of 100 to 20,000 bodies 62 us, where blocks of 256
// threads that went through memory in every pass took 104.
constexpr int kSegThreads = 1024;
static_assert(kSegSmall == 256 * kSortItems);

// LDS of a group of T threads.
template <int T>
struct SegLds {
    unsigned int wcnt[T / 64][256];              // per-wave digit counts, then the waves' starts
    int delta[256];                              // destination minus tile position, per digit
    unsigned int sh[4];
    unsigned long long stage[T * kSortItems];
};

// Exclusive scan of one value per thread over the group's first 256 threads (one barrier).
__device__ __forceinline__ unsigned int digit_exscan(unsigned int v, unsigned int* __restrict__ sh, int wave) {
    const int lane = threadIdx.x & 63;
    unsigned int inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63 && wave < 4) sh[wave] = inc;
    __syncthreads();
    unsigned int off = 0u;
#pragma unroll
    for (int w = 0; w < 4; ++w)
        if (w < wave) off += sh[w];
    return off + inc - v;
}

// Ranks a tile of m pairs (each wave a contiguous run): rank[r] becomes the pair's place in the
// tile. Returns the digit's count and start in the tile (the group's first 256 threads). Ends in
// front of a barrier that the caller has to pass before it reads starts another thread may move.
template <int T>
__device__ __forceinline__ unsigned int rank_tile(const unsigned long long (&key)[kSortItems], int m, int shift, int tid,
                                                  SegLds<T>& L, unsigned int (&rank)[kSortItems],
                                                  unsigned int& tstart) {
    const int lane = tid & 63, wave = tid >> 6;
    const int wbase = wave * (kSortItems * 64);
#pragma unroll
    for (int q = 0; q < 4; ++q) L.wcnt[wave][q * 64 + lane] = 0u;      // this wave's own
    __builtin_amdgcn_wave_barrier();
    rank_rows(key, wbase, m, shift, L.wcnt[wave], rank);
    __syncthreads();
    unsigned int count = 0u;
    if (tid < 256)
#pragma unroll
        for (int w = 0; w < T / 64; ++w) count += L.wcnt[w][tid];
    tstart = digit_exscan(count, L.sh, wave);
    if (tid < 256) {
        unsigned int run = tstart;
#pragma unroll
        for (int w = 0; w < T / 64; ++w) {
            const unsigned int c = L.wcnt[w][tid];
            L.wcnt[w][tid] = run;
            run += c;
        }
    }
    return count;
}

// The places themselves, after the barrier.
template <int T>
__device__ __forceinline__ void add_starts(const unsigned long long (&key)[kSortItems], int m, int shift, int tid,
                                           const SegLds<T>& L, unsigned int (&rank)[kSortItems]) {
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
        if (wave * (kSortItems * 64) + r * 64 + lane < m) rank[r] += L.wcnt[wave][(unsigned)(key[r] >> shift) & 255u];
}

// A segment of m <= T * kSortItems pairs.
template <int T>
__device__ __forceinline__ void sort_in_lds(unsigned long long* __restrict__ k, unsigned int* __restrict__ v, int m,
                                            int p0, int tid, SegLds<T>& L) {
    const int base = (tid >> 6) * (kSortItems * 64) + (tid & 63);
    unsigned int* sval = reinterpret_cast<unsigned int*>(L.stage);
    unsigned long long key[kSortItems];
    unsigned int val[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const int e = base + r * 64;
        key[r] = e < m ? k[e] : 0ull;
        val[r] = e < m ? v[e] : 0u;
    }
    for (int p = p0; p < 8; ++p) {
        unsigned int rank[kSortItems], tstart;
        rank_tile<T>(key, m, 8 * p, tid, L, rank, tstart);
        __syncthreads();
        add_starts<T>(key, m, 8 * p, tid, L, rank);
#pragma unroll
        for (int r = 0; r < kSortItems; ++r)
            if (base + r * 64 < m) L.stage[rank[r]] = key[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSortItems; ++r)
            if (base + r * 64 < m) key[r] = L.stage[base + r * 64];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSortItems; ++r)
            if (base + r * 64 < m) sval[rank[r]] = val[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSortItems; ++r)
            if (base + r * 64 < m) val[r] = sval[base + r * 64];
    }
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const int e = base + r * 64;
        if (e >= m) continue;
        k[e] = key[r];
        v[e] = val[r];
    }
}

// A longer segment, by all of the block's threads.
__device__ __forceinline__ void sort_tiles(unsigned long long* __restrict__ k0, unsigned int* __restrict__ v0,
                                           unsigned long long* __restrict__ k1, unsigned int* __restrict__ v1, int m,
                                           int p0, SegLds<kSegThreads>& L, unsigned int* __restrict__ hist) {
    constexpr int kTile = kSegThreads * kSortItems;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    unsigned int* sval = reinterpret_cast<unsigned int*>(L.stage);
    // the digit counts of all passes
    for (int i = tid; i < 8 * 256; i += kSegThreads) hist[i] = 0u;
    __syncthreads();
    for (int e = tid; e < m; e += kSegThreads) {
        const unsigned long long k = k0[e];
        for (int p = p0; p < 8; ++p) atomicAdd(&hist[p * 256 + ((unsigned)(k >> (8 * p)) & 255u)], 1u);
    }
    __syncthreads();
    const int tiles = (m + kTile - 1) / kTile;
    for (int p = p0; p < 8; ++p) {
        const int shift = 8 * p;
        const bool from1 = ((p - p0) & 1) != 0;
        const unsigned long long* kin = from1 ? k1 : k0;
        const unsigned int* vin = from1 ? v1 : v0;
        unsigned long long* kout = from1 ? k0 : k1;
        unsigned int* vout = from1 ? v0 : v1;
        // this thread's digit: its first destination in the segment, advanced tile by tile
        unsigned int dstart = digit_exscan(tid < 256 ? hist[p * 256 + tid] : 0u, L.sh, wave);
        for (int t = 0; t < tiles; ++t) {
            const int here = min(kTile, m - t * kTile);
            const int base = wave * (kSortItems * 64) + lane;
            unsigned long long key[kSortItems];
            unsigned int val[kSortItems], rank[kSortItems], dst[kSortItems], tstart;
#pragma unroll
            for (int r = 0; r < kSortItems; ++r) {
                const int e = base + r * 64;
                key[r] = e < here ? kin[t * kTile + e] : 0ull;
                val[r] = e < here ? vin[t * kTile + e] : 0u;
            }
            // (the barrier inside also ends the previous tile's and the scan's reads)
            const unsigned int count = rank_tile<kSegThreads>(key, here, shift, tid, L, rank, tstart);
            if (tid < 256) L.delta[tid] = (int)dstart - (int)tstart;
            dstart += count;
            __syncthreads();
            add_starts<kSegThreads>(key, here, shift, tid, L, rank);
#pragma unroll
            for (int r = 0; r < kSortItems; ++r)
                if (base + r * 64 < here) L.stage[rank[r]] = key[r];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kSortItems; ++r) {
                const int j = tid + r * kSegThreads;
                if (j >= here) continue;
                const unsigned long long k = L.stage[j];
                dst[r] = (unsigned int)(L.delta[(unsigned)(k >> shift) & 255u] + j);
                kout[dst[r]] = k;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kSortItems; ++r)
                if (base + r * 64 < here) sval[rank[r]] = val[r];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kSortItems; ++r) {
                const int j = tid + r * kSegThreads;
                if (j < here) vout[dst[r]] = sval[j];
            }
        }
        // this pass's writes are read by the next one (one block: workgroup-scope visibility)
        __syncthreads();
    }
    if (((8 - p0) & 1) != 0)
        for (int e = tid; e < m; e += kSegThreads) {
            k0[e] = k1[e];
            v0[e] = v1[e];
        }
}

// A batch of segments of at most T * kSortItems pairs: a block each.
template <int T>
__global__ __launch_bounds__(T) void k_seg_lds(unsigned long long* __restrict__ k0, unsigned int* __restrict__ v0,
                                               const int* __restrict__ node_off, const int* __restrict__ order,
                                               const DevState* __restrict__ st) {
    __shared__ SegLds<T> L;
    const int g = order[blockIdx.x], a = node_off[g];
    sort_in_lds<T>(k0 + a, v0 + a, node_off[g + 1] - a, st ? st->sort_skip : 0, threadIdx.x, L);
}

__global__ __launch_bounds__(kSegThreads) void k_seg_sort(unsigned long long* __restrict__ k0,
                                                          unsigned int* __restrict__ v0,
                                                          unsigned long long* __restrict__ k1,
                                                          unsigned int* __restrict__ v1,
                                                          const int* __restrict__ node_off,
                                                          const int* __restrict__ order, int nseg, int large,
                                                          const DevState* __restrict__ st) {
    union Lds {
        SegLds<kSegThreads> one;
        SegLds<256> four[4];
    };
    __shared__ Lds L;
    __shared__ unsigned int hist[8 * 256];
    // the low passes the previous trees' cells let the sort skip (k_sort_fixup, told the graph
    // of each position, orders what they would have ordered)
    const int p0 = st ? st->sort_skip : 0;
    if ((int)blockIdx.x >= large) {
        const int quarter = threadIdx.x >> 8, q = large + ((int)blockIdx.x - large) * 4 + quarter;
        const int g = q < nseg ? order[q] : 0;
        const int a = node_off[g], m = q < nseg ? node_off[g + 1] - a : 0;
        sort_in_lds<256>(k0 + a, v0 + a, m, p0, threadIdx.x & 255, L.four[quarter]);
        return;
    }
    const int g = order[blockIdx.x], a = node_off[g], m = node_off[g + 1] - a;
    if (m <= kSegThreads * kSortItems) sort_in_lds<kSegThreads>(k0 + a, v0 + a, m, p0, threadIdx.x, L.one);
    else sort_tiles(k0 + a, v0 + a, k1 + a, v1 + a, m, p0, L.one, hist);
}

// ---- onesweep -------------------------------------------------------------------------------
constexpr unsigned int kStatAgg = 1u << 30;      // the tile's digit count is published, with its pass's epoch
constexpr unsigned int kStatCount = (1u << 27) - 1;

// A pass of one launch costs its chain of steps across the chip (ticket, pairs, published counts,
// the other tiles' counts, destinations), not its bytes. Tiles of 256 threads up to 32,768 pairs, where
// they spread over more compute units (20,000 bodies: 99.7 us an iteration, 101.0 with 512
// threads); of 512 up to 262,144, where fewer tiles have to be read (131,000: 145.6, with 256 threads
// 151.1). Beyond, three launches per pass are as fast (262,000: 198.5 us an iteration against 196.5;
// 300,000: 225.7 against 224.8; 2M: 1,118 against 1,159). 1,024 threads were slower
// up to this line. Past it they gain 1% on one stream and lose where a second stream's kernels
// leave such large blocks no room (579,581 bodies, 20M entries, three launches against one: 404.7
// and 400.6 us an iteration alone, 349 and 407 beside the attraction). With a look-back from tile to
// tile the iterations took 104.1 us at 20,000, 121.8 (now 115.0) at 50,000 and 158.2 at 131,000.
constexpr int kSweepSmall = 32768;
constexpr int kSweepMost = 262144;
constexpr int kMaxSpins = 1 << 20;   // per thread and pass: ~1 s at worst, then an error

__global__ void k_sort_zero(unsigned int* __restrict__ digit_hist, int npasses) {
    for (int i = threadIdx.x; i < npasses * 256; i += blockDim.x) digit_hist[i] = 0u;
}

__global__ __launch_bounds__(256) void k_sort_hist(const unsigned long long* __restrict__ k0,
                                                   const unsigned long long* __restrict__ k1, int n, int begin_bit,
                                                   int npasses, unsigned int* __restrict__ digit_hist,
                                                   const DevState* __restrict__ st, int first, int lead) {
    const unsigned long long* __restrict__ keys = start_buffer(st, first, lead) ? k1 : k0;
    __shared__ unsigned int h[8][256];
    for (int p = 0; p < npasses; ++p) h[p][threadIdx.x] = 0u;
    __syncthreads();
    for (int e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
        const unsigned long long k = keys[e];
        for (int p = 0; p < npasses; ++p) atomicAdd(&h[p][(unsigned)(k >> (begin_bit + 8 * p)) & 255u], 1u);
    }
    __syncthreads();
    for (int p = 0; p < npasses; ++p) {
        const unsigned int c = h[p][threadIdx.x];
        if (c) atomicAdd(&digit_hist[p * 256 + threadIdx.x], c);
    }
}

// LDS of a pass of one launch. The tile's keys are staged first, then its values.
template <int T>
struct SweepLds {
    unsigned int wcnt[T / 64][256];              // per-wave digit counts, then the waves' starts
    unsigned int tcount[256];
    unsigned int before[T / 256][256];           // counts of the earlier tiles
    int delta[256];                              // global destination minus tile position, per digit
    unsigned long long stage[T * kSortItems];
    unsigned int sh[2][4];
    int tile;
    unsigned int epoch;
};

template <int T>
__global__ __launch_bounds__(T) void k_onesweep(unsigned long long* __restrict__ k0, unsigned int* __restrict__ v0,
                                                unsigned long long* __restrict__ k1, unsigned int* __restrict__ v1,
                                                int n, int shift, const unsigned int* __restrict__ digit_hist,
                                                unsigned int* __restrict__ status,
                                                unsigned long long* __restrict__ ticket, int tiles,
                                                int* __restrict__ err, const DevState* __restrict__ st, int first,
                                                int lead, int pass) {
    constexpr int kTile = T * kSortItems, kParts = T / 256, kAhead = 8;
    if (pass_skipped(st, pass)) return;   // takes no ticket: the epochs of later passes stay distinct
    const int src = pass_src(st, first, lead, pass);
    const unsigned long long* __restrict__ kin = src ? k1 : k0;
    const unsigned int* __restrict__ vin = src ? v1 : v0;
    unsigned long long* __restrict__ kout = src ? k0 : k1;
    unsigned int* __restrict__ vout = src ? v0 : v1;
    __shared__ SweepLds<T> L;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int digit = tid & 255, part = tid >> 8;
    if (tid == 0) {
        const unsigned long long t = atomicAdd(ticket, 1ull);
        L.tile = (int)(t % (unsigned long long)tiles);
        L.epoch = (unsigned int)((t / (unsigned long long)tiles) & 7ull) << 27;
    }
    for (int i = tid; i < T / 64 * 256; i += T) L.wcnt[0][i] = 0u;
    if (tid < 256) L.tcount[tid] = 0u;
    const unsigned int total = tid < 256 ? digit_hist[tid] : 0u;
    __syncthreads();
    const int tile = L.tile;
    const unsigned int epoch = L.epoch;
    // the tile's pairs, held in registers (each wave a contiguous run), and its digit counts
    const int wbase = tile * kTile + wave * (kSortItems * 64);
    unsigned long long key[kSortItems];
    unsigned int val[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const int e = wbase + r * 64 + lane;
        key[r] = e < n ? kin[e] : 0ull;
        val[r] = e < n ? vin[e] : 0u;
    }
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
        if (wbase + r * 64 + lane < n) atomicAdd(&L.tcount[(unsigned)(key[r] >> shift) & 255u], 1u);
    __syncthreads();
    const unsigned int count = L.tcount[digit];
    if (part == 0)
        __hip_atomic_store(status + (size_t)tile * 256 + digit, kStatAgg | epoch | count, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    // the counts are on their way to the other tiles while this tile ranks its pairs
    unsigned int rank[kSortItems];
    rank_rows(key, wbase, n, shift, L.wcnt[wave], rank);
    unsigned int sum = 0u;
    int spins = 0;                       // bounded over all of a thread's waits
    for (int t0 = part; t0 < tile; t0 += kParts * kAhead) {
        unsigned int v[kAhead];
        bool ready;
        do {
            ready = true;
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int t = t0 + u * kParts;
                v[u] = t < tile ? __hip_atomic_load(status + (size_t)t * 256 + digit, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT)
                                : (kStatAgg | epoch);
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) ready = ready && (v[u] & ~kStatCount) == (kStatAgg | epoch);
        } while (!ready && ++spins < kMaxSpins);
        if (!ready) {                    // (too small a sum keeps every destination in range)
            atomicOr(err, kErrSortWait);
            break;
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) sum += v[u] & kStatCount;
    }
    L.before[part][digit] = sum;
    const unsigned int gstart = digit_exscan(total, L.sh[0], wave);                       // (barrier)
    const unsigned int tstart = digit_exscan(tid < 256 ? count : 0u, L.sh[1], wave);      // (barrier)
    if (tid < 256) {
        unsigned int excl = 0u;
#pragma unroll
        for (int q = 0; q < kParts; ++q) excl += L.before[q][tid];
        L.delta[tid] = (int)(gstart + excl) - (int)tstart;
        unsigned int run = tstart;
#pragma unroll
        for (int w = 0; w < T / 64; ++w) {
            const unsigned int c = L.wcnt[w][tid];
            L.wcnt[w][tid] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
        if (wbase + r * 64 + lane < n) {
            rank[r] += L.wcnt[wave][(unsigned)(key[r] >> shift) & 255u];
            L.stage[rank[r]] = key[r];
        }
    __syncthreads();
    const int here = min(kTile, n - tile * kTile);
    unsigned int dst[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const int j = tid + r * T;
        if (j >= here) continue;
        const unsigned long long k = L.stage[j];
        dst[r] = (unsigned int)(L.delta[(unsigned)(k >> shift) & 255u] + j);
        kout[dst[r]] = k;
    }
    __syncthreads();
    unsigned int* sval = reinterpret_cast<unsigned int*>(L.stage);
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
        if (wbase + r * 64 + lane < n) sval[rank[r]] = val[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const int j = tid + r * T;
        if (j < here) vout[dst[r]] = sval[j];
    }
}

// (key, value) pairs in lexicographic order (values are distinct body ids: a total order).
__device__ __forceinline__ bool pair_less(unsigned long long ka, unsigned int va, unsigned long long kb,
                                          unsigned int vb) {
    return ka < kb || (ka == kb && va < vb);
}

// Heapsort of pairs [0, m) of k/v in place: O(m log m) whatever the input order.
__device__ void heapsort_pairs(unsigned long long* __restrict__ k, unsigned int* __restrict__ v, int m) {
    auto sift = [&](int root, int end) {
        while (2 * root + 1 < end) {
            int c = 2 * root + 1;
            if (c + 1 < end && pair_less(k[c], v[c], k[c + 1], v[c + 1])) ++c;
            if (!pair_less(k[root], v[root], k[c], v[c])) return;
            const unsigned long long tk = k[root];
            const unsigned int tv = v[root];
            k[root] = k[c];
            v[root] = v[c];
            k[c] = tk;
            v[c] = tv;
            root = c;
        }
    };
    for (int r = m / 2 - 1; r >= 0; --r) sift(r, m);
    for (int end = m - 1; end > 0; --end) {
        const unsigned long long tk = k[0];
        const unsigned int tv = v[0];
        k[0] = k[end];
        v[0] = v[end];
        k[end] = tk;
        v[end] = tv;
        sift(0, end);
    }
}

// After a sort that skipped its low passes: the passes that ran left the pairs ordered by
// their top 8 (8 - skip) key bits, in buffer (8 - skip) & 1. Every run of pairs whose keys agree
// in those bits is ordered by (whole key, value), and the result goes to buffer 0 (pairs outside
// runs are copied there when the passes ended in buffer 1). Such runs are the bodies of one cell at
// the sorted depth, few and short when the depth was chosen from the previous tree.
//
// A block takes the runs that start in its kFixTile positions and looks kFixHalo positions past
// them; each pair's place in its run is the number of the run's pairs before it, counted in LDS.
// A run past the window (over kFixHalo pairs) is left to the thread at its first position, which
// heapsorts it in place. Where the result replaces
// its input, a neighbouring block may read positions while their run's own block reorders them;
// it uses only their top bits, which all pairs of a run share.
//
// Bound by the round trips of a few loads: 4.7 us on SBM 50,000 nodes and 16 us on an R-MAT graph of
// 2M nodes, where one thread insertion-sorting each run in global memory took 21.4 and 20.6.
constexpr int kFixThreads = 256;
constexpr int kFixHalo = 64;
constexpr int kFixTile = kFixThreads - kFixHalo;

__global__ __launch_bounds__(kFixThreads) void k_sort_fixup(unsigned long long* __restrict__ k0,
                                                            unsigned int* __restrict__ v0,
                                                            const unsigned long long* k1, const unsigned int* v1,
                                                            int n, const DevState* __restrict__ st, int first,
                                                            int lead, const int* __restrict__ seg,
                                                            unsigned int* __restrict__ clear_hist) {
    __shared__ unsigned long long skey[kFixThreads];
    __shared__ unsigned int sval[kFixThreads];
    __shared__ unsigned long long starts[kFixThreads / 64];
    // the passes are done with the digit table: cleared for the next iteration's k_keys
    if (clear_hist && blockIdx.x == 0)
        for (int i = threadIdx.x; i < 8 * 256; i += kFixThreads) clear_hist[i] = 0u;
    const int skip = passes_below(st, first);
    if (skip == 0) return;                       // all 8 passes ran: sorted, ties by value, in buffer 0
    // the passes that ran ended in buffer 1 (unless the keys started where they end in buffer 0)
    const bool moved = !lead && ((8 - skip) & 1) != 0;
    const unsigned long long* ks = moved ? k1 : k0;
    const unsigned int* vs = moved ? v1 : v0;
    const unsigned long long top = ~0ull << (8 * skip);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // seg (sorted position -> graph, each graph sorted in its own range): runs stop at graphs
    for (int base = blockIdx.x * kFixTile; base < n; base += gridDim.x * kFixTile) {   // uniform
        const int i = base + tid;
        const bool valid = i < n;
        const unsigned long long k = valid ? ks[i] : 0ull;
        const unsigned int v = valid ? vs[i] : 0u;
        const unsigned long long kp = valid && i > 0 ? ks[i - 1] : 0ull;
        const bool start = !valid || i == 0 || ((k ^ kp) & top) != 0ull || (seg && seg[i - 1] != seg[i]);
        __syncthreads();                         // the last tile's reads are done
        skey[tid] = k;
        sval[tid] = v;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(start);
        if (lane == 0) starts[wave] = m;
        __syncthreads();
        // the run [b, e) of this position, within the window
        const unsigned long long upto = (2ull << lane) - 1ull;          // lanes 0 .. lane
        int b = -1, e = kFixThreads;
        {
            unsigned long long q = m & upto;
            for (int w = wave; w >= 0; q = --w >= 0 ? starts[w] : 0ull)
                if (q) {
                    b = 64 * w + 63 - __clzll((long long)q);
                    break;
                }
            q = m & ~upto;
            for (int w = wave; w < kFixThreads / 64; q = ++w < kFixThreads / 64 ? starts[w] : 0ull)
                if (q) {
                    e = 64 * w + __builtin_ctzll(q);
                    break;
                }
        }
        if (!valid || b < 0 || b >= kFixTile) continue;                 // another block's run
        if (e == kFixThreads && base + kFixThreads < n) {
            // the run goes on past the window (or ends with it)
            if (tid != b) continue;
            int j = base + kFixThreads;
            while (j < n && ((ks[j] ^ k) & top) == 0ull && (!seg || seg[j] == seg[i])) ++j;
            if (moved)
                for (int a = i; a < j; ++a) {
                    k0[a] = ks[a];
                    v0[a] = vs[a];
                }
            heapsort_pairs(k0 + i, v0 + i, j - i);
            continue;
        }
        if (e - b == 1) {
            if (moved) {
                k0[i] = k;
                v0[i] = v;
            }
            continue;
        }
        int before = 0;
        for (int q = b; q < e; ++q) before += pair_less(skey[q], sval[q], k, v);
        k0[base + b + before] = k;
        v0[base + b + before] = v;
    }
}

}  // namespace

void launch_sort_fixup(SortBuffers& buf, int n, const DevState* st, hipStream_t s, int first, bool lead,
                       const int* seg, bool clear_hist) {
    if (n < 1) return;
    int blocks = (n + kFixTile - 1) / kFixTile;
    if (blocks > 65535) blocks = 65535;
    k_sort_fixup<<<blocks, kFixThreads, 0, s>>>(buf.keys[0], buf.vals[0], buf.keys[1], buf.vals[1], n, st, first,
                                                lead ? 8 : 0, seg, clear_hist ? buf.digit_hist : nullptr);
}

bool sort_onesweep(const SortBuffers& buf, int n) {
    return buf.onesweep && n <= kSweepMost;
}

void segmented_sort_pairs(SortBuffers& buf, const int* node_off, const int* order, int nseg, int max_seg, int large,
                          hipStream_t s, const DevState* skip) {
    if (nseg <= 0) return;
    // without a long segment, blocks of just the threads it takes, several to a compute unit (4,000
    // graphs of 200 bodies: 242 us an iteration, 253 by quarters; 300 of 2,049: 237, 251)
    if (max_seg <= 256 * kSortItems)
        k_seg_lds<256><<<nseg, 256, 0, s>>>(buf.keys[0], buf.vals[0], node_off, order, skip);
    else if (max_seg <= 512 * kSortItems)
        k_seg_lds<512><<<nseg, 512, 0, s>>>(buf.keys[0], buf.vals[0], node_off, order, skip);
    else
        k_seg_sort<<<large + (nseg - large + 3) / 4, kSegThreads, 0, s>>>(buf.keys[0], buf.vals[0], buf.keys[1],
                                                                         buf.vals[1], node_off, order, nseg, large,
                                                                         skip);
}

void radix_sort_pairs(SortBuffers& buf, int n, int begin_bit, int end_bit, hipStream_t s, const DevState* skip,
                      int first, bool lead_in, bool hist_ready) {
    if (n <= 1) return;
    const int tiles = (n + kSortTile - 1) / kSortTile;
    const int npasses = (end_bit - begin_bit + 7) / 8;
    const int lead = lead_in && skip ? npasses : 0;
    // Every pass picks its buffers on the device (pass_src): with a device skip the passes that
    // run may end in buffer 1, and launch_sort_fixup moves the result to buffer 0.
    unsigned long long *k0 = buf.keys[0], *k1 = buf.keys[1];
    unsigned int *v0 = buf.vals[0], *v1 = buf.vals[1];
    if (sort_onesweep(buf, n)) {
        if (!hist_ready) {
            k_sort_zero<<<1, 256, 0, s>>>(buf.digit_hist, npasses);
            int hb = (n + 255) / 256;
            if (hb > 256) hb = 256;
            k_sort_hist<<<hb, 256, 0, s>>>(k0, k1, n, begin_bit, npasses, buf.digit_hist, skip, first, lead);
        }
        const int threads = n <= kSweepSmall ? 256 : 512;
        const int sweeps = (n + threads * kSortItems - 1) / (threads * kSortItems);
        const auto sweep = threads == 256 ? k_onesweep<256> : k_onesweep<512>;
        for (int p = first; p < npasses; ++p)
            sweep<<<sweeps, threads, 0, s>>>(k0, v0, k1, v1, n, begin_bit + 8 * p, buf.digit_hist + 256 * p,
                                             buf.status, buf.ticket, sweeps, buf.err, skip, first, lead, p);
    } else {
        for (int p = first; p < npasses; ++p) {
            const int shift = begin_bit + 8 * p;
            k_upsweep<<<tiles, kSortThreads, 0, s>>>(k0, k1, n, shift, buf.hist, tiles, skip, first, lead, p);
            k_rowscan<<<256, 256, 0, s>>>(buf.hist, tiles, buf.rowtot, skip, p);
            k_scatter<<<tiles, kSortThreads, 0, s>>>(k0, v0, k1, v1, n, shift, buf.hist, tiles, buf.rowtot, skip, first,
                                                     lead, p);
        }
    }
    if (!skip && ((npasses - first) & 1)) {
        hipMemcpyAsync(k0, k1, sizeof(unsigned long long) * n, hipMemcpyDeviceToDevice, s);
        hipMemcpyAsync(v0, v1, sizeof(unsigned int) * n, hipMemcpyDeviceToDevice, s);
    }
}

}  // namespace gfa2
