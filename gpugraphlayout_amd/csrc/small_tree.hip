// The quadtree of a small graph in one block, for gfx950: path keys, sort, cells, summaries and
// child lists in LDS, with the attraction and gravity in the launch's other blocks.
//
// The kernels of bh_tree.hip and radix_sort.hip spread a graph over the chip and hand every step
// to the next through a launch. On a small graph each of those launches lasts 4-11 us however
// little it does: a chain of loads of what another compute unit has just written, at about a
// microsecond each. Here one block of 1,024 threads keeps keys, order and prefix counts in LDS
// and only the records leave it. The tree is the same, bit for bit: the same keys in the same
// order, the same integer moments, the same arithmetic per cell.
//
// Where the block's time goes at 500 bodies (us of 13.8): keys 2.1, two sort passes 2.8, tied runs
// 0.7, order, prefix counts and bit rows 1.6, records 0.4, moments 2.5, cells 3.4; at 2,048 (22)
// keys 4.8, sort 4.4, cells 6.5. It is bound by its chains: LDS round trips, barriers and FP64.
// Searching the keys for a cell's extent and children took 6.2 us at 500 where the bit rows take 3.4.
//
// What the walk, the speed step and gfa2_get_tree read: rec, kids, rcount, sbody, vals[0] (the
// body order), seg_root, rec_begin, kids_part (one block's worth) and the instance state.
#include "attract_device.h"
#include "engine_internal.h"
#include "tree_device.h"

#include <algorithm>

namespace gfa2 {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kRunCap = 64;          // longest run of tied bodies ordered by counting

using Split = SplitOf<unsigned int>;      // (the launch's rule: under 2^24 in all)

struct SmallArgs {
    const float2* pos;
    const float* mass;
    int n;
    const float4* bbox_part;
    DevState* st;
    float4* seg_root;
    const SegState* seg;
    SegState* seg_cur;
    const unsigned long long* keys;      // when they were formed by a launch of their own
    unsigned int* perm;
    unsigned int* spare;                 // n words (only when the sort is redone)
    float4* sbody;
    float4* rec;
    int4* kids;
    int* rcount;
    int* rec_begin;
    int* kids_part;
    unsigned char* cell_lvl;             // fractional masses only
    Moment* pmass;                       // prefix moments, N > kLdsMoments
    int cap_records;
    int int_mass;
};

constexpr int kLdsMoments = 2048;        // up to this size the prefix moments lie in LDS too

template <int N>
struct SmallLds {
    unsigned long long key[N];
    unsigned short idx[2][N];
    union {
        unsigned int wcnt[kWaves][256];  // sort: per-wave digit counts, then starts
        unsigned short start[kWaves * 512];   // cells: first position of cell c
    };
    int S[N + 1];
    unsigned long long below[kKeyLevels][N / 64];   // bit j of level L: positions j, j + 1 share fewer than L + 1 levels
    unsigned long long some[kKeyLevels];            // bit w: word w of the level has a bit
    union {
        unsigned int dsum[256];
        Split wsum[kWaves];
    };
    Split P[N <= kLdsMoments ? N + 1 : 1];
    float root[4];
    int wtot[kWaves];
    int rmax[8];
    int flag, lmax;
};

// Orders positions 0 .. n-1 by `passes` 8-bit digits of key[] from the top, stably, least
// significant first. Positions and ranks go through idx; the result's buffer is returned.
template <int N>
__device__ int small_sort(SmallLds<N>& L, int n, int rows, int passes) {
    constexpr int R = N / kThreads;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int base = wave * rows * 64;
    int src = 0;
    for (int p = 8 - passes; p < 8; ++p) {
        const int shift = 8 * p;
        for (int q = tid; q < kWaves * 256; q += kThreads) (&L.wcnt[0][0])[q] = 0u;
        __syncthreads();
        unsigned int id[R], rank[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r >= rows) break;                          // uniform
            const int e = base + r * 64 + lane;
            const bool valid = e < n;
            id[r] = p == 8 - passes ? (unsigned)e : (valid ? L.idx[src][e] : 0u);
            const unsigned int d = valid ? (unsigned)(L.key[id[r]] >> shift) & 255u : 0u;
            unsigned long long peers = __builtin_amdgcn_ballot_w64(valid);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const unsigned long long m = __builtin_amdgcn_ballot_w64((d >> b) & 1u);
                peers &= ((d >> b) & 1u) ? m : ~m;
            }
            const unsigned int rr = (unsigned)__popcll(peers & lt);
            // every lane reads the digit's count before its leader writes it (one wave, LDS in order)
            const unsigned int before = L.wcnt[wave][d];
            rank[r] = (before + rr) | (d << 16);
            if (valid && rr == 0) L.wcnt[wave][d] = before + (unsigned)__popcll(peers);
        }
        __syncthreads();
        // digit d, a thread each: the waves' counts become their first destinations
        unsigned int c[kWaves], total = 0u;
        if (tid < 256) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                c[w] = L.wcnt[w][tid];
                total += c[w];
            }
            const unsigned int inc = wave_scan(total);
            if (lane == 63) L.dsum[wave] = inc;
            total = inc - total;
        }
        __syncthreads();
        if (tid < 256) {
            unsigned int run = total;
#pragma unroll
            for (int w = 0; w < 3; ++w)
                if (w < wave) run += L.dsum[w];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                L.wcnt[w][tid] = run;
                run += c[w];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r >= rows) break;
            const int e = base + r * 64 + lane;
            if (e < n) L.idx[src ^ 1][L.wcnt[wave][rank[r] >> 16] + (rank[r] & 0xffffu)] = (unsigned short)id[r];
        }
        src ^= 1;
        __syncthreads();
    }
    return src;
}

// The first position j >= from where positions j and j + 1 share fewer than L levels (1 <= L <= 32;
// the last position always does).
template <int N>
__device__ __forceinline__ int next_below(const SmallLds<N>& L, int level, int from) {
    int w = from >> 6;
    const unsigned long long m = L.below[level - 1][w] >> (from & 63);
    if (m) return from + __builtin_ctzll(m);
    w = __builtin_ctzll(L.some[level - 1] & (~1ull << w));
    return 64 * w + __builtin_ctzll(L.below[level - 1][w]);
}

// The tree of one graph of n <= N bodies, by one block.
template <int N, bool OWN_KEYS>
__device__ void small_tree(const SmallArgs& A, SmallLds<N>& L) {
    constexpr int R = N / kThreads;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = A.n;
    const int rows = (n + kThreads - 1) / kThreads;
    const int base = wave * rows * 64;
    if (tid < 8) L.rmax[tid] = 0;
    if (tid == 0) L.flag = L.lmax = 0;
    const int skip_last = A.st->sort_skip;
    float2 p0[R];                                      // loaded while the root is formed
    if (OWN_KEYS) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int e = base + r * 64 + lane;
            p0[r] = r < rows && e < n ? A.pos[e] : make_float2(0.0f, 0.0f);
        }
    }
    float4 root;
    if (OWN_KEYS) {
        if (wave == 0) {
            float4 b = A.bbox_part[0];
            const int np = A.st->nbbox;
            for (int k = lane; k < np; k += 64) {
                const float4 v = A.bbox_part[k];
                b = make_float4(fminf(b.x, v.x), fminf(b.y, v.y), fmaxf(b.z, v.z), fmaxf(b.w, v.w));
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                b = make_float4(fminf(b.x, __shfl_xor(b.x, o, 64)), fminf(b.y, __shfl_xor(b.y, o, 64)),
                                fmaxf(b.z, __shfl_xor(b.z, o, 64)), fmaxf(b.w, __shfl_xor(b.w, o, 64)));
            if (lane == 0) {
                L.root[2] = fmaxf(b.z - b.x, b.w - b.y) * 0.5f;   // src/RPBHKernels.cu:140-148
                L.root[0] = (b.x + b.z) * 0.5f;
                L.root[1] = (b.y + b.w) * 0.5f;
                A.st->rootx = L.root[0];
                A.st->rooty = L.root[1];
                A.st->radius = L.root[2];
                A.seg_root[0] = make_float4(L.root[0], L.root[1], L.root[2], 0.0f);
                *A.seg_cur = A.seg[0];        // for k_advance
            }
        }
        __syncthreads();
        root = make_float4(L.root[0], L.root[1], L.root[2], 0.0f);
    } else {
        root = A.seg_root[0];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int e = base + r * 64 + lane;
        if (r < rows && e < n) L.key[e] = OWN_KEYS ? path_key(p0[r], root.x, root.y, root.z) : A.keys[e];
    }
    __syncthreads();
    // The passes that leave the previous tree's cells at 16 bodies at most, but no more than four:
    // runs of up to kRunCap tied bodies are ordered below, and a longer one redoes the sort in full.
    int passes = min(max(8 - skip_last, 2), 4);
    int buf = small_sort(L, n, rows, passes);
    unsigned long long k[R];
    unsigned int id[R];
    unsigned long long top = ~0ull << (8 * (8 - passes));
    for (;;) {
        // the keys in sorted order
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int e = base + r * 64 + lane;
            if (r < rows && e < n) {
                const unsigned int at = L.idx[buf][e];
                k[r] = L.key[at];
                id[r] = passes == 8 ? A.spare[at] : at;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int e = base + r * 64 + lane;
            if (r < rows && e < n) {
                L.key[e] = k[r];
                L.idx[buf][e] = (unsigned short)id[r];
            }
        }
        __syncthreads();
        if (passes == 8) break;
        // runs that agree in every sorted bit: a body's place in its run is the number of the run's
        // bodies before it by (whole key, id)
        int to[R];
        bool any = false;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int e = base + r * 64 + lane;
            to[r] = -1;
            if (r < rows && e < n) {
                const unsigned long long t = k[r] & top;
                const bool tied = (e > 0 && (L.key[e - 1] & top) == t) || (e + 1 < n && (L.key[e + 1] & top) == t);
                if (tied) {
                    int b = e, f = e + 1;
                    while (b > 0 && e - b <= kRunCap && (L.key[b - 1] & top) == t) --b;
                    while (f < n && f - e <= kRunCap && (L.key[f] & top) == t) ++f;
                    if (f - b > kRunCap) {
                        L.flag = 1;
                    } else {
                        int before = 0;
                        for (int q = b; q < f; ++q) {
                            const unsigned long long kq = L.key[q];
                            before += kq < k[r] || (kq == k[r] && L.idx[buf][q] < id[r]);
                        }
                        to[r] = b + before;
                        any = true;
                    }
                }
            }
        }
        __syncthreads();
        if (L.flag) {                                  // uniform: redo with every digit
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int e = base + r * 64 + lane;
                if (r < rows && e < n) A.spare[e] = id[r];
            }
            __syncthreads();
            passes = 8;
            buf = small_sort(L, n, rows, 8);
            continue;
        }
        if (any) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (to[r] >= 0) {
                    L.key[to[r]] = k[r];
                    L.idx[buf][to[r]] = (unsigned short)id[r];
                }
        }
        __syncthreads();
        break;
    }
    // Bodies in sorted order, and the cells opened at each position (levels above the one shared
    // with the position before, up to the one shared with the next).
    float4 bd[R];
    int s[R];
    int waves_cells = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int e = base + r * 64 + lane;
        s[r] = 0;
        if (r >= rows || base + r * 64 >= n) continue;  // uniform
        int next = -1;
        if (e < n) {
            const unsigned int v = L.idx[buf][e];
            const float2 p = A.pos[v];
            bd[r] = make_float4(p.x, p.y, A.mass[v], 0.0f);
            A.perm[e] = v;
            const unsigned long long ke = L.key[e];
            const int prev = e == 0 ? -1 : lcp_levels(L.key[e - 1], ke);
            if (e < n - 1) next = lcp_levels(ke, L.key[e + 1]);
            s[r] = max(0, (n == 1 ? 0 : next) - prev);
        }
        // lane l < 32 keeps the row's word of level l + 1
        unsigned long long word = 0ull;
#pragma unroll
        for (int l = 0; l < kKeyLevels; ++l) {
            const unsigned long long m = __builtin_amdgcn_ballot_w64(next <= l);
            if (lane == l) word = m;
        }
        if (lane < kKeyLevels) L.below[lane][wave * rows + r] = word;
    }
    // exclusive prefix of the cells
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (r >= rows) break;
        const int e = base + r * 64 + lane;
        const int inc = (int)wave_scan((unsigned int)s[r]);
        if (e < n) L.S[e] = waves_cells + inc - s[r];
        waves_cells += __builtin_amdgcn_readlane(inc, 63);
    }
    if (lane == 0) L.wtot[wave] = waves_cells;
    __syncthreads();
    for (int l = wave; l < kKeyLevels; l += kWaves) {
        const unsigned long long m = __builtin_amdgcn_ballot_w64(64 * lane < n && L.below[l][lane] != 0ull);
        if (lane == 0) L.some[l] = m;
    }
    const unsigned int tot_cells = lane < kWaves ? (unsigned)L.wtot[lane] : 0u;
    const unsigned int upto_cells = wave_scan(tot_cells);
    const int off = __builtin_amdgcn_readlane((int)(upto_cells - tot_cells), wave);
    const int cells = __builtin_amdgcn_readlane((int)upto_cells, kWaves - 1);
    const bool fits = n + cells <= A.cap_records;
    if (tid == 0) {
        A.st->ncells = cells;
        A.st->nrecords = n + cells;
        A.rec_begin[1] = n + cells;
        A.rec_begin[0] = 0;
        A.st->nbig = 0;
        if (!fits) A.st->err |= kErrTreeOverflow;
        L.S[n] = cells;
    }
    if (!fits) return;                                 // uniform
    constexpr int kStarts = kWaves * 512;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int e = base + r * 64 + lane;
        if (r >= rows || e >= n) continue;
        const int S = L.S[e] + off;
        L.S[e] = S;
        for (int c = S; c < S + s[r] && c < kStarts; ++c) L.start[c] = (unsigned short)e;
        A.sbody[e] = bd[r];
        A.rec[e + S + s[r]] = make_float4(bd[r].x, bd[r].y, bd[r].z, __int_as_float(-1));
    }
    if (A.int_mass) {
        // exclusive prefix of the moments: within the wave row by row, then the waves' totals
        Split ex[R], run{0, 0, 0, 0, 0u};
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r >= rows) break;                      // uniform
            const int e = base + r * 64 + lane;
            const Split own = e < n ? split_of<unsigned int>(bd[r], root) : Split{0, 0, 0, 0, 0u};
            const Split in = wave_scan(own);
            ex[r] = run + (in - own);
            run = run + from_lane(in, 63);
        }
        if (lane == 0) L.wsum[wave] = run;
        __syncthreads();
        const Split tot = lane < kWaves ? L.wsum[lane] : Split{0, 0, 0, 0, 0u};
        const Split upto = wave_scan(tot);
        const Split before = from_lane(upto - tot, wave), all = from_lane(upto, kWaves - 1);
        Split* P = N <= kLdsMoments ? L.P : reinterpret_cast<Split*>(A.pmass);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int e = base + r * 64 + lane;
            if (r < rows && e < n) P[e] = before + ex[r];
        }
        if (tid == 0) P[n] = all;
    }
    __syncthreads();
    // Cells, a thread each. A cell of level lv that starts at i ends at the first position from i
    // that shares fewer than lv levels with the next one; its children part where fewer than
    // lv + 1 are shared. Both come from the levels' bit rows, a few LDS reads whatever the size.
    for (int c = tid; c < cells; c += kThreads) {
        int i;
        if (c < kStarts) {
            i = L.start[c];
        } else {
            int lo = 0, hi = n;                        // S[lo] <= c < S[lo + 1]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (L.S[mid] <= c) lo = mid;
                else hi = mid;
            }
            i = lo;
        }
        const unsigned long long ki = L.key[i];
        const int lv = (i == 0 ? -1 : lcp_levels(L.key[i - 1], ki)) + 1 + (c - L.S[i]);
        const int end = (lv > 0 ? next_below(L, lv, i) : n - 1) + 1;
        const int rc = i + c;
        int kid[4] = {rc + 1, -1, -1, -1};
        int from = i;
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            // (the bodies of a level-32 cell are its children)
            from = lv < kKeyLevels ? next_below(L, lv + 1, from) + 1 : from + 1;
            if (from >= end) break;
            kid[q] = from + L.S[from];
        }
        A.kids[rc] = make_int4(kid[0], kid[1], kid[2], kid[3]);
        const int skip = end + L.S[end] - rc;
        const float info = __uint_as_float(((unsigned)skip << kInfoLevelBits) | (unsigned)((lv > 0 ? lv - 1 : 0) & 31));
        A.rcount[rc] = end - i;
        if (A.int_mass) {
            // lighter than 2^24 in all (the launch's rule): the exact mass in any order
            Split D;
            if (N <= kLdsMoments) {
                D = L.P[end] - L.P[i];
            } else {
                const Split* P = reinterpret_cast<const Split*>(A.pmass);
                D = P[end] - P[i];
            }
            const u128 x = moment_x(D), y = moment_y(D);
            const double M = (double)D.m;
            const int e = -moment_shift(root.z);
            A.rec[rc] = make_float4(
                (float)(ldexp(i128_to_double((unsigned long long)x, (unsigned long long)(x >> 64)) / M, e) + root.x),
                (float)(ldexp(i128_to_double((unsigned long long)y, (unsigned long long)(y >> 64)) / M, e) + root.y),
                (float)M, info);
        } else {
            A.rec[rc].w = info;
            A.cell_lvl[c] = (unsigned char)lv;
        }
        atomicMax(&L.lmax, lv);
        if (lv > 0 && (lv & 3) == 0) atomicMax(&L.rmax[(lv >> 2) - 1], end - i);
    }
    __syncthreads();
    if (tid < 8) A.kids_part[tid] = L.rmax[tid];
    if (tid == 0) A.st->max_level = L.lmax;
    if (!A.int_mass) {
        // bottom-up, children in quadrant order (as k_sum_blocks)
        for (int lv = L.lmax; lv >= 0; --lv) {
            for (int c = tid; c < cells; c += kThreads) {
                if (A.cell_lvl[c] != lv) continue;     // this thread's own write
                int i;
                if (c < kStarts) {
                    i = L.start[c];
                } else {
                    int lo = 0, hi = n;
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if (L.S[mid] <= c) lo = mid;
                        else hi = mid;
                    }
                    i = lo;
                }
                const int rc = i + c;
                const int last = rc + (int)(__float_as_uint(A.rec[rc].w) >> kInfoLevelBits);
                float cm = 0.0f, px = 0.0f, py = 0.0f;
                int r = rc + 1;
                while (r < last) {
                    const float4 v = A.rec[r];
                    const unsigned int ci = __float_as_uint(v.w);
                    px = fmaf(v.x, v.z, px);
                    py = fmaf(v.y, v.z, py);
                    cm += v.z;
                    r += ci == 0xffffffffu ? 1 : max((int)(ci >> kInfoLevelBits), 1);
                }
                const float inv = 1.0f / cm;
                A.rec[rc].x = px * inv;
                A.rec[rc].y = py * inv;
                A.rec[rc].z = cm;
            }
            __syncthreads();
        }
    }
}

// Block 0: the tree. The others: the attraction's light and medium rows, in virtual blocks of 256
// threads (a graph with heavy rows takes the attraction in its own launch, and one block here).
template <int N, bool OWN_KEYS, bool GEN>
__global__ __launch_bounds__(kThreads) void k_small_tree(SmallArgs A, AttractArgs at, int light_blocks,
                                                         int virtual_blocks) {
    __shared__ SmallLds<N> L;
    if (blockIdx.x == 0) {
        if (A.st->err == 0) small_tree<N, OWN_KEYS>(A, L);
        return;
    }
    const int sub = threadIdx.x >> 8, tid = threadIdx.x & 255;
    for (int vb = (blockIdx.x - 1) * 4 + sub; vb < virtual_blocks; vb += (gridDim.x - 1) * 4) {
        if (vb < light_blocks) attract_light<GEN, 0>(vb * 256 + tid, at, nullptr);
        else attract_medium<GEN, 0>((vb - light_blocks) * 4 + (tid >> 6), 1, tid & 63, at, nullptr);
    }
}

template <int N, bool OWN_KEYS>
void launch_size(const SmallArgs& A, const AttractArgs& at, bool gen, int light_blocks, int virtual_blocks,
                 hipStream_t s) {
    const int blocks = 1 + std::min((virtual_blocks + 3) / 4, 255);
    if (gen) k_small_tree<N, OWN_KEYS, true><<<blocks, kThreads, 0, s>>>(A, at, light_blocks, virtual_blocks);
    else k_small_tree<N, OWN_KEYS, false><<<blocks, kThreads, 0, s>>>(A, at, light_blocks, virtual_blocks);
}

}  // namespace

bool small_tree(const Bufs& b) { return b.nseg == 1 && b.n <= kSmallTree && (!b.int_mass || b.no_big); }

void launch_small_tree(const Bufs& b, const Params& p, hipStream_t s) {
    SmallArgs A{};
    A.pos = b.pos;
    A.mass = b.mass;
    A.n = b.n;
    A.bbox_part = b.bbox_part;
    A.st = b.st;
    A.seg_root = b.seg_root;
    A.seg = b.seg_st;
    A.seg_cur = b.seg_cur;
    A.keys = b.sort.keys[0];
    A.perm = b.sort.vals[0];
    A.spare = b.sort.vals[1];
    A.sbody = b.sbody;
    A.rec = b.rec;
    A.kids = b.kids;
    A.rcount = b.rcount;
    A.rec_begin = b.rec_begin;
    A.kids_part = b.kids_part;
    A.cell_lvl = b.cell_lvl;
    A.pmass = b.pmass;
    A.cap_records = b.cap_records;
    A.int_mass = b.int_mass ? 1 : 0;
    const AttractArgs at = attract_args(b, p);
    const bool apart = b.nheavy > 0;
    const int lb = apart ? 0 : (b.nlight + 255) / 256, vb = apart ? 0 : lb + (b.nmedium + 3) / 4;
    if (apart) launch_attraction(b, p, true, s);
    const bool gen = p.linlog || b.ew;
    if (b.n <= kSmallOwnKeys) {
        launch_size<2048, true>(A, at, gen, lb, vb, s);
    } else {
        launch_keys(b, 8, s);                          // into buffer 0
        launch_size<4096, false>(A, at, gen, lb, vb, s);
    }
}

}  // namespace gfa2
