// Rasteriser of a layout on the device: the picture GraphLayout::writeToPNG draws
// (src/RPGraphLayout.cpp:170-207: bounding box fitted to the image, white background,
// black nodes as discs of radius 3 with opacity 10000/V, black edges as lines with opacity
// 100000/E). Each node and each edge (drawn once, from its smaller to its larger id) adds
// to per-pixel hit counters with integer atomics; a pixel's brightness is then
// (1 - a_node)^nodes * (1 - a_edge)^edges, the result of blending that many layers in any
// order. The host layer's CPU rasteriser uses the same pixel walk and the same shading
// arithmetic (powers by repeated squaring, IEEE operations), so both produce the same bytes;
// this file is compiled with -ffp-contract=off, since the *_rn intrinsics alone do not stop
// a multiply and an add from being fused.
//
// gfa2_render counts in LDS: the edges become a list of lines (k_raster_lines), and a block per
// (picture tile, slice of the lines) finds the lines that cross its tile, walks their samples
// there and writes the tile's counts to a copy of the tile of its own (k_raster_tiles), so that
// no counter is shared; k_shade adds the copies. A tile gets slices in proportion to the samples
// a part of the lines put there (k_raster_cost, k_raster_plan): in a finished layout one tile of
// fifty can hold a sixth of them. Where tiles do not pay (tiles_pay, kFewSamples) or their scratch
// is out of proportion or not to be had, and in gfa2_render_noalloc, which has no memory for a list
// or copies, every sample is added to one counter per pixel with device atomics (k_raster_pixels;
// k_raster_nodes, k_raster_edges).
#include "engine_internal.h"
#include "../../include/gfa2.h"

#include <algorithm>
#include <mutex>

// Fixed scratch of gfa2_render_noalloc (one copy per device, loaded with the code object and
// held until the process ends): the node and edge hit counters, 2 x kNoAllocMaxPixels words,
// then the picture, kNoAllocMaxPixels bytes; 9 MiB in all. Host code never passes this name
// to a kernel or a copy: it uses the device address hipGetSymbolAddress gives for it.
namespace gfa2 {
constexpr long long kNoAllocMaxPixels = 1ll << 20;
constexpr size_t kScratchWords = (size_t)(2 * kNoAllocMaxPixels + kNoAllocMaxPixels / 4);
}  // namespace gfa2
static __device__ __align__(256) unsigned int scratch[gfa2::kScratchWords];

namespace gfa2 {
namespace {

constexpr int kScratchMaxDevices = 64;
std::mutex g_scratch_mu;                               // also serialises the calls of one process
unsigned int* g_scratch[kScratchMaxDevices] = {};      // device address of `scratch`, per device

__global__ __launch_bounds__(256) void k_fill_zero(unsigned int* __restrict__ p, long long n) {
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (long long)gridDim.x * 256) p[i] = 0u;
}

struct Frame {
    float x0, y0, sx, sy;
    int w, h;
};

__device__ __forceinline__ void hit(unsigned int* __restrict__ cnt, const Frame& f, int x, int y) {
    if (x < 0 || y < 0 || x >= f.w || y >= f.h) return;
    atomicAdd(&cnt[(size_t)(f.h - 1 - y) * f.w + x], 1u);   // y up
}

__device__ __forceinline__ float to_px(float v, float v0, float s) { return __fmul_rn(__fsub_rn(v, v0), s); }

__global__ __launch_bounds__(256) void k_minmax(const float2* __restrict__ pos, int n, float4* __restrict__ part) {
    __shared__ float4 red[256];
    float4 m = make_float4(3.402823466e38f, -3.402823466e38f, 3.402823466e38f, -3.402823466e38f);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const float2 p = pos[i];
        m.x = fminf(m.x, p.x);
        m.y = fmaxf(m.y, p.x);
        m.z = fminf(m.z, p.y);
        m.w = fmaxf(m.w, p.y);
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            const float4 a = red[threadIdx.x], b = red[threadIdx.x + o];
            red[threadIdx.x] = make_float4(fminf(a.x, b.x), fmaxf(a.y, b.y), fminf(a.z, b.z), fmaxf(a.w, b.w));
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(64) void k_minmax_final(const float4* __restrict__ part, int nb,
                                                     float4* __restrict__ out) {
    float4 m = part[0];
    for (int b = threadIdx.x; b < nb; b += 64) {
        const float4 a = part[b];
        m = make_float4(fminf(m.x, a.x), fmaxf(m.y, a.y), fminf(m.z, a.z), fmaxf(m.w, a.w));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        m = make_float4(fminf(m.x, __shfl_xor(m.x, o, 64)), fmaxf(m.y, __shfl_xor(m.y, o, 64)),
                        fminf(m.z, __shfl_xor(m.z, o, 64)), fmaxf(m.w, __shfl_xor(m.w, o, 64)));
    if (threadIdx.x == 0) *out = m;
}

// A disc of radius 3 around the rounded node centre.
__device__ __forceinline__ void node_hits(float2 p, const Frame& f, unsigned int* __restrict__ cnt) {
    const int cx = (int)lroundf(to_px(p.x, f.x0, f.sx)), cy = (int)lroundf(to_px(p.y, f.y0, f.sy));
    for (int dy = -3; dy <= 3; ++dy)
        for (int dx = -3; dx <= 3; ++dx)
            if (dx * dx + dy * dy <= 9) hit(cnt, f, cx + dx, cy + dy);
}

__global__ __launch_bounds__(256) void k_raster_nodes(const float2* __restrict__ pos, int n, Frame f,
                                                      unsigned int* __restrict__ cnt) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) node_hits(pos[i], f, cnt);
}

// One thread per CSR entry (i, j) with i < j: the line from node i to node j, sampled at
// ceil(max(|dx|, |dy|)) + 1 evenly spaced points (positions formed in double), each rounded
// to the nearest pixel.
__global__ __launch_bounds__(256) void k_raster_edges(const float2* __restrict__ pos, const int* __restrict__ rowptr,
                                                      const int* __restrict__ col, int n, long long nnz, Frame f,
                                                      unsigned int* __restrict__ cnt) {
    for (long long e = blockIdx.x * 256ll + threadIdx.x; e < nnz; e += (long long)gridDim.x * 256) {
        const int j = col[e];
        int lo = 0, hi = n;              // row: rowptr[lo] <= e < rowptr[lo + 1]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if ((long long)rowptr[mid] <= e) lo = mid;
            else hi = mid;
        }
        const int i = lo;
        if (!(i < j)) continue;
        const float2 a = pos[i], b = pos[j];
        const float x0 = to_px(a.x, f.x0, f.sx), y0 = to_px(a.y, f.y0, f.sy);
        const float x1 = to_px(b.x, f.x0, f.sx), y1 = to_px(b.y, f.y0, f.sy);
        const float ddx = __fsub_rn(x1, x0), ddy = __fsub_rn(y1, y0);
        const float len = fmaxf(fabsf(ddx), fabsf(ddy));
        const int steps = (int)ceilf(len);
        if (steps == 0) {
            hit(cnt, f, (int)lroundf(x0), (int)lroundf(y0));
            continue;
        }
        // sample positions in double (IEEE-exact divide on both processors), then float
        for (int k = 0; k <= steps; ++k) {
            const double t = __ddiv_rn((double)k, (double)steps);
            const float sx = (float)__dadd_rn((double)x0, __dmul_rn(t, (double)ddx));
            const float sy = (float)__dadd_rn((double)y0, __dmul_rn(t, (double)ddy));
            hit(cnt, f, (int)lroundf(sx), (int)lroundf(sy));
        }
    }
}

// ---- counting in picture tiles ----------------------------------------------------------------

constexpr int kTileW = 256, kTileH = 128;         // 257-word rows: a vertical line's samples fall in different banks
constexpr int kTileThreads = 1024;
constexpr int kTilePixels = kTileW * kTileH;
constexpr int kQueueGo = 32;                      // a wave walks its tile's lines once it has found this many
constexpr int kSpareSlices = 1024;                // slices beyond the first of each tile: four per compute unit
constexpr int kSliceSamples = 16384;              // least samples for a slice beyond a tile's first: 15 us, as long
                                                  // as its block takes to clear and write its copy
// Small pictures of so few lines that they hold no more samples than this are counted by atomics
// without a list (the tiles' launches take 40 us and more: mesh of 10,000 nodes at 256 x 128 20 us,
// by tiles 56; 500 nodes and 1,491 random lines 82 and 70).
constexpr long long kFewSamples = 6ll << 20;
constexpr int kFewPixels = 256;
// Least tests of lines and nodes against tiles (0.2 ms) for which the device may choose atomics after
// all (tiles_pay); below, that form's launch and the totals it needs are left out (40 us of a picture
// of 71,000 nodes and 1M lines at 1,250 x 1,250; a mesh of 90,000 nodes there takes 120 us for 90).
constexpr long long kManyTests = 100'000'000;
// Scratch up to which tiles are used whatever the picture's shape; beyond, up to four times what
// the atomics take (a picture of one column has 128 KB of counters for 128 pixels).
constexpr size_t kTileMemory = 1ull << 30;
constexpr long long kListEntries = 4ll << 20;     // CSR entries whose lines are listed at a time (64 MB at most)
constexpr int kLineThreads = 256, kLineItems = 16;
// Lines with an end this far out (in pixels) are drawn sample by sample (k_raster_lines): below it
// a sample's float rounding stays under half a pixel, and steps under 2^24 (quotient below).
constexpr float kFarOut = 4194304.0f;

// k / steps correctly rounded, from the correctly rounded y = 1 / steps. q is within two units of
// the quotient, so r = k - steps q is exact (steps is an integer below 2^24), and q + r y errs from
// the quotient by under 2^-100 of it before its own rounding; a quotient of integers below 2^24
// that is no double lies at least 2^-78 of itself from the midpoint of two doubles.
__device__ __forceinline__ double quotient(double k, double steps, double y) {
    const double q = __dmul_rn(k, y);
    return __fma_rn(__fma_rn(-steps, q, k), y, q);
}

// The samples [k0, k1] of a line that may fall in the pixels [x0, x1) x [y0, y1): pad is two
// pixels and what a sample's rounding can add, and the ends are widened by a sample.
__device__ __forceinline__ bool clip_line(const float4 l, int steps, float x0, float x1, float y0, float y1,
                                          float pad, int* k0, int* k1) {
    if (fmaxf(l.x, l.z) < x0 - pad || fminf(l.x, l.z) > x1 + pad || fmaxf(l.y, l.w) < y0 - pad ||
        fminf(l.y, l.w) > y1 + pad)
        return false;
    double t0 = 0.0, t1 = 1.0;
    const double dx = (double)l.z - l.x, dy = (double)l.w - l.y;
    if (fabs(dx) > 1e-3) {
        const double a = ((double)x0 - pad - l.x) / dx, b = ((double)x1 + pad - l.x) / dx;
        t0 = fmax(t0, fmin(a, b));
        t1 = fmin(t1, fmax(a, b));
    }
    if (fabs(dy) > 1e-3) {
        const double a = ((double)y0 - pad - l.y) / dy, b = ((double)y1 + pad - l.y) / dy;
        t0 = fmax(t0, fmin(a, b));
        t1 = fmin(t1, fmax(a, b));
    }
    if (!(t0 <= t1)) return false;
    *k0 = max(0, (int)floor(t0 * steps) - 1);
    *k1 = min(steps, (int)ceil(t1 * steps) + 1);
    return true;
}

// Orders this wave's LDS writes before its later LDS reads by other lanes.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int line_steps(const float4 l) {
    return (int)ceilf(fmaxf(fabsf(__fsub_rn(l.z, l.x)), fabsf(__fsub_rn(l.w, l.y))));
}

// What a list holds.
struct ListTotals {
    unsigned long long samples;
    unsigned int lines, longest;       // the longest in samples
};

// The lines of CSR entries [e0, e1) with i < j, in no order (counts do not depend on it), as
// {x0, y0, x1, y1} in pixels; the far-out ones are drawn here, into far. totals: the list's samples
// are wanted too.
__global__ __launch_bounds__(kLineThreads) void k_raster_lines(const float2* __restrict__ pos,
                                                               const int* __restrict__ rowptr,
                                                               const int* __restrict__ col, int n, long long e0,
                                                               long long e1, Frame f, float4* __restrict__ lines,
                                                               ListTotals* __restrict__ list,
                                                               unsigned int* __restrict__ far, int totals) {
    __shared__ unsigned int wsum[kLineThreads / 64], wlong[kLineThreads / 64];
    __shared__ unsigned long long wsamples[kLineThreads / 64];
    __shared__ unsigned int base;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long long first = e0 + ((long long)blockIdx.x * kLineThreads + tid) * kLineItems;
    const long long last = first + kLineItems < e1 ? first + kLineItems : e1;
    float4 mine[kLineItems];
    unsigned int take = 0u;                         // bit q: mine[q] is a line
    unsigned long long samples = 0ull;
    unsigned int longest = 0u;
    if (first < last) {
        int lo = 0, hi = n;                         // row: rowptr[lo] <= first < rowptr[lo + 1]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if ((long long)rowptr[mid] <= first) lo = mid;
            else hi = mid;
        }
        int i = lo;
        long long end = rowptr[i + 1];
#pragma unroll
        for (int q = 0; q < kLineItems; ++q) {
            const long long e = first + q;
            if (e < last) {
                while (end <= e) end = rowptr[++i + 1];
                const int j = col[e];
                if (i < j) {
                    const float2 a = pos[i], b = pos[j];
                    mine[q] = make_float4(to_px(a.x, f.x0, f.sx), to_px(a.y, f.y0, f.sy), to_px(b.x, f.x0, f.sx),
                                          to_px(b.y, f.y0, f.sy));
                    take |= 1u << q;
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kLineItems; ++q) {
        if (!((take >> q) & 1u)) continue;
        const float4 l = mine[q];
        const float out = fmaxf(fmaxf(fabsf(l.x), fabsf(l.y)), fmaxf(fabsf(l.z), fabsf(l.w)));
        const bool nan = l.x != l.x || l.y != l.y || l.z != l.z || l.w != l.w;
        if (out < kFarOut && !nan) {
            if (totals) {
                const unsigned int k = (unsigned int)line_steps(l) + 1u;
                samples += k;
                longest = max(longest, k);
            }
            continue;
        }
        take &= ~(1u << q);
        const float ddx = __fsub_rn(l.z, l.x), ddy = __fsub_rn(l.w, l.y);
        const float len = fmaxf(fabsf(ddx), fabsf(ddy));
        if (!(len < 2147483648.0f) && len == len) continue;   // more samples than can be counted
        const int steps = (int)ceilf(len);
        if (steps == 0) {
            hit(far, f, (int)lroundf(l.x), (int)lroundf(l.y));
            continue;
        }
        int k0 = 0, k1 = steps;
        // up to 2^30 a sample's float rounding is under 2^-23 of the farthest end (further out, a
        // pixel's number may wrap: every sample is looked at)
        if (out < 1073741824.0f && !nan &&
            !clip_line(l, steps, 0.0f, (float)f.w, 0.0f, (float)f.h, 2.0f + 2.4e-7f * out, &k0, &k1))
            continue;
        for (long long k = k0; k <= k1; ++k) {
            const double t = __ddiv_rn((double)k, (double)steps);
            const float sx = (float)__dadd_rn((double)l.x, __dmul_rn(t, (double)ddx));
            const float sy = (float)__dadd_rn((double)l.y, __dmul_rn(t, (double)ddy));
            hit(far, f, (int)lroundf(sx), (int)lroundf(sy));
        }
    }
    if (totals) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            samples += __shfl_xor(samples, o, 64);
            longest = max(longest, (unsigned int)__shfl_xor((int)longest, o, 64));
        }
        if (lane == 0) {
            wsamples[wave] = samples;
            wlong[wave] = longest;
        }
    }
    // the block's lines get one run of the list
    const unsigned int c = (unsigned int)__popc(take);
    unsigned int inc = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    unsigned int before = 0u, total = 0u;
#pragma unroll
    for (int w = 0; w < kLineThreads / 64; ++w) {
        if (w < wave) before += wsum[w];
        total += wsum[w];
    }
    if (tid == 0) {
        base = 0u;
        if (total) {
            base = atomicAdd(&list->lines, total);
            static_assert(kLineThreads / 64 == 4, "four waves");
            if (totals) {
                atomicAdd(&list->samples, wsamples[0] + wsamples[1] + wsamples[2] + wsamples[3]);
                atomicMax(&list->longest, max(max(wlong[0], wlong[1]), max(wlong[2], wlong[3])));
            }
        }
    }
    __syncthreads();
    unsigned int at = base + before + inc - c;
#pragma unroll
    for (int q = 0; q < kLineItems; ++q)
        if ((take >> q) & 1u) lines[at++] = mine[q];
}

// lroundf (half away from zero) of a value below 2^22 in magnitude: the float steps are exact.
__device__ __forceinline__ int round_px(float v) {
    const float t = truncf(v);
    return (int)(t + (fabsf(__fsub_rn(v, t)) >= 0.5f ? copysignf(1.0f, v) : 0.0f));
}

// A tile of the picture: columns [c0, c0 + cw), rows [r0, r0 + rh); y is up, so these rows are
// y = ylo + rh - 1 down to ylo.
struct Tile {
    int c0, r0, cw, rh, ylo;
};

__device__ __forceinline__ Tile tile_of(int t, int tiles_x, const Frame& f) {
    Tile a;
    a.c0 = (t % tiles_x) * kTileW;
    a.r0 = (t / tiles_x) * kTileH;
    a.cw = min(kTileW, f.w - a.c0);
    a.rh = min(kTileH, f.h - a.r0);
    a.ylo = f.h - a.r0 - a.rh;
    return a;
}

__device__ __forceinline__ bool clip_to_tile(const float4 l, const Tile& a, int* k0, int* k1) {
    return clip_line(l, line_steps(l), (float)a.c0, (float)(a.c0 + a.cw), (float)a.ylo, (float)(a.ylo + a.rh), 2.0f, k0,
                     k1);
}

__device__ __forceinline__ bool node_in_tile(float2 p, const Frame& f, const Tile& a, int* cx, int* cy) {
    *cx = (int)lroundf(to_px(p.x, f.x0, f.sx));
    *cy = (int)lroundf(to_px(p.y, f.y0, f.sy));
    return *cx >= a.c0 - 3 && *cx <= a.c0 + a.cw + 2 && *cy >= a.ylo - 3 && *cy <= a.ylo + a.rh + 2;
}

// Whether the lines and nodes are counted in tiles or by a device atomic per sample (k_raster_pixels),
// from the first list's totals: the least times of both forms, in ns, as fitted to pictures of 64 x 64
// to 8,000 x 8,000. Tiles pay for long lines (100,000 nodes, 1M lines at 1,250 x 1,250: 1.9 ms, 22.4
// with atomics); every line is tested against every tile, so atomics do for many lines of a few
// pixels, where their hits spread over the picture (a mesh of 1M nodes and 2M lines: 0.26 and
// 0.71 ms at 1,250 x 1,250, 0.57 and 3.1 at 4,000 x 4,000, but 0.75 and 0.40 at 500 x 500, 130 hits a
// pixel). A wave of atomics takes as long as its longest line, hence lines times the longest.
__device__ __forceinline__ bool tiles_pay(const ListTotals& l, int n, int tiles, const Frame& f) {
    const float samples = (float)l.samples, lines = (float)l.lines, nodes = (float)n;
    if (samples + 29.0f * nodes > 32.0f * (float)f.w * (float)f.h) return true;
    const float plain = 50e3f + 0.04f * lines * (float)l.longest + 0.15f * nodes;
    const float tiled = 60e3f + 0.002f * (float)tiles * (lines + nodes) + 0.3f * nodes + 0.004f * samples;
    return tiled < plain;
}

// Work of tile t (lines, t < tiles; nodes, t - tiles) in samples, from every kCostStride-th line
// or node: its samples, 8 per line or node that crosses it, and a quarter per one looked at.
constexpr int kCostStride = 16;

__global__ __launch_bounds__(256) void k_raster_cost(const float4* __restrict__ lines,
                                                     const ListTotals* __restrict__ list,
                                                     const float2* __restrict__ pos, int n, Frame f, int tiles,
                                                     int tiles_x, unsigned long long* __restrict__ cost,
                                                     unsigned int* __restrict__ copies, int either) {
    __shared__ unsigned long long wsum[4];
    const int t = blockIdx.x;
    if (either && !tiles_pay(*list, n, tiles, f)) {
        // the nodes' counters of k_raster_pixels
        const long long npix = (long long)f.w * f.h, step = (long long)gridDim.x * gridDim.y * 256;
        for (long long p = ((long long)blockIdx.y * gridDim.x + t) * 256 + threadIdx.x; p < npix; p += step) copies[p] = 0u;
        return;
    }
    const bool nodes = t >= tiles;
    const Tile a = tile_of(nodes ? t - tiles : t, tiles_x, f);
    const unsigned int total = nodes ? (unsigned int)n : list->lines;
    unsigned long long c = 0ull;
    for (unsigned int i = (blockIdx.y * 256u + threadIdx.x) * kCostStride; i < total; i += gridDim.y * 256u * kCostStride) {
        int k0, k1;
        if (nodes) c += node_in_tile(pos[i], f, a, &k0, &k1) ? 4u * (29 + 8) : 0u;
        else if (clip_to_tile(lines[i], a, &k0, &k1)) c += 4u * (unsigned int)(k1 - k0 + 1 + 8);
        c += 1u;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&cost[t], wsum[0] + wsum[1] + wsum[2] + wsum[3]);
}

// first[t]: the first copy of tile t's slices; every tile gets one slice and a share of the spare
// ones by its cost; no copies at all where tiles do not pay. One block.
__global__ __launch_bounds__(1024) void k_raster_plan(const unsigned long long* __restrict__ cost, int count,
                                                      int spare, const ListTotals* __restrict__ list, int n, Frame f,
                                                      int* __restrict__ first, int either) {
    __shared__ unsigned long long wcost[16];
    __shared__ int wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (either && !tiles_pay(*list, n, count / 2, f)) {
        for (int t = tid; t <= count; t += 1024) first[t] = 0;
        return;
    }
    unsigned long long c = 0ull;
    for (int t = tid; t < count; t += 1024) c += cost[t];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if (lane == 0) wcost[wave] = c;
    __syncthreads();
    unsigned long long total = 1ull;
    for (int w = 0; w < 16; ++w) total += wcost[w];
    // (costs are quarters of samples, of every kCostStride-th line)
    spare = (int)min((unsigned long long)spare, total * (kCostStride / 4) / kSliceSamples);
    int carry = 0;
    for (int t0 = 0; t0 < count; t0 += 1024) {
        const int t = t0 + tid;
        const int s = t < count ? 1 + (int)((double)cost[t] / (double)total * spare) : 0;
        int inc = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(inc, o, 64);
            if (lane >= o) inc += u;
        }
        if (lane == 63) wsum[wave] = inc;
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) before += wsum[w];
            all += wsum[w];
        }
        if (t < count) first[t] = carry + before + inc - s;
        carry += all;
        __syncthreads();
    }
    if (tid == 0) first[count] = carry;
}

// One block per copy: its tile (lines or nodes) and slice, counted in LDS and written to the
// copy, copies[block][pixel of the tile] (added to for the lines beyond the first list).
//
// Bound by vector instructions (issued in 80 % of the time a compute unit has a block): about 45 per
// sample, 10 of them FP64, with 16 lanes per line, and half as much again to find the lines. With one device atomic per sample the 1M edges of an R-MAT layout (275M samples, 1250 x
// 1250) took 11.9 ms, 23 samples/ns; with equal slices per tile 1.94 ms, with slices by cost and
// block-wide batches 1.31 ms, as here 1.02 ms, 270 samples/ns.
__global__ __launch_bounds__(kTileThreads) void k_raster_tiles(const float4* __restrict__ lines,
                                                               const ListTotals* __restrict__ list,
                                                               const float2* __restrict__ pos, int n, Frame f,
                                                               int tiles, int tiles_x, const int* __restrict__ first,
                                                               unsigned int* __restrict__ copies, int more) {
    __shared__ unsigned int cnt[kTileH * (kTileW + 1)];
    __shared__ int3 queues[kTileThreads / 64][kQueueGo + 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int count_all = 2 * tiles, me = blockIdx.x;
    if (me >= first[count_all]) return;              // uniform
    int lo = 0, hi = count_all;                      // first[lo] <= me < first[lo + 1]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (first[mid] <= me) lo = mid;
        else hi = mid;
    }
    const bool nodes = lo >= tiles;
    if (nodes && more) return;                       // the nodes went with the first list
    const int slice = me - first[lo], slices = first[lo + 1] - first[lo];
    const Tile a = tile_of(nodes ? lo - tiles : lo, tiles_x, f);
    for (int q = tid; q < kTileH * (kTileW + 1); q += kTileThreads) cnt[q] = 0u;
    __syncthreads();
    // a pixel counts if it lies in the tile
    auto count = [&](int x, int y) {
        const int cx = x - a.c0, cy = y - a.ylo;
        if ((unsigned)cx < (unsigned)a.cw && (unsigned)cy < (unsigned)a.rh) {
            const int row = a.rh - 1 - cy;
            atomicAdd(&cnt[(row << 8) + row + cx], 1u);
        }
    };
    static_assert(kTileW == 256, "a row of the counters is 257 words");
    const unsigned int total = nodes ? (unsigned int)n : list->lines;
    const unsigned int i0 = (unsigned int)((unsigned long long)total * slice / slices);
    const unsigned int i1 = (unsigned int)((unsigned long long)total * (slice + 1) / slices);
    // nodes: a wave per disc of radius 3 around the rounded centre
    const int dx = lane % 7 - 3, dy = lane / 7 - 3;
    const bool disc = lane < 49 && dx * dx + dy * dy <= 9;
    // Each wave looks at 64 lines (or nodes) at a time, the next ones loaded meanwhile, and keeps
    // those that cross the tile in a queue of its own: no barrier until the block is done.
    int3* queue = queues[wave];
    int have = 0;                                    // uniform
    float4 next = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto load = [&](unsigned int id) {
        if (id < i1) {
            if (nodes) {
                const float2 p = pos[id];
                next = make_float4(p.x, p.y, 0.0f, 0.0f);
            } else {
                next = lines[id];
            }
        }
    };
    load(i0 + tid);
    for (unsigned int at = i0 + 64 * wave; at < i1; at += kTileThreads) {  // uniform per wave
        const float4 l = next;
        const unsigned int id = at + lane;
        load(id + kTileThreads);
        int k0 = 0, k1 = 0;
        bool in = false;
        if (id < i1) in = nodes ? node_in_tile(make_float2(l.x, l.y), f, a, &k0, &k1) : clip_to_tile(l, a, &k0, &k1);
        const unsigned long long m = __builtin_amdgcn_ballot_w64(in);
        if (in)
            queue[have + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                nodes ? make_int3(k0, k1, 0) : make_int3((int)id, k0, k1);
        have += __popcll(m);
        if (have < kQueueGo && at + kTileThreads < i1) continue;
        wave_lds_sync();
        if (nodes) {
            for (int q = 0; q < have; ++q)
                if (disc) count(queue[q].x + dx, queue[q].y + dy);
        } else {
            // 16 lanes per line
            for (int q = lane >> 4; q < have; q += 4) {
                const int3 it = queue[q];
                const float4 g = lines[(unsigned int)it.x];
                const int steps = line_steps(g);
                if (steps == 0) {
                    if ((lane & 15) == 0) count(round_px(g.x), round_px(g.y));
                    continue;
                }
                const double ddx = (double)__fsub_rn(g.z, g.x), ddy = (double)__fsub_rn(g.w, g.y);
                const double lx = (double)g.x, ly = (double)g.y;
                const double n_steps = (double)steps, y = __ddiv_rn(1.0, n_steps);
                for (int k = it.y + (lane & 15); k <= it.z; k += 16) {
                    const double t = quotient((double)k, n_steps, y);
                    const float sx = (float)__dadd_rn(lx, __dmul_rn(t, ddx));
                    const float sy = (float)__dadd_rn(ly, __dmul_rn(t, ddy));
                    count(round_px(sx), round_px(sy));
                }
            }
        }
        have = 0;
        wave_lds_sync();
    }
    __syncthreads();
    unsigned int* out = copies + (size_t)me * kTilePixels;
    for (int q = tid; q < a.rh * kTileW; q += kTileThreads) {
        const unsigned int v = cnt[q / kTileW * (kTileW + 1) + q % kTileW];
        out[q] = more ? out[q] + v : v;
    }
}

// The same without tiles: a device atomic per sample, a thread per line and per node (cn: the
// nodes' counters, far: the lines').
__global__ __launch_bounds__(256) void k_raster_pixels(const float4* __restrict__ lines,
                                                       const ListTotals* __restrict__ list,
                                                       const float2* __restrict__ pos, int n, Frame f, int tiles,
                                                       const int* __restrict__ first, unsigned int* __restrict__ cn,
                                                       unsigned int* __restrict__ far, int more) {
    if (first[2 * tiles] != 0) return;
    const unsigned int nodes = more ? 0u : (unsigned int)n, total = list->lines + nodes;
    for (unsigned int q = blockIdx.x * 256u + threadIdx.x; q < total; q += gridDim.x * 256u) {
        if (q < nodes) {
            node_hits(pos[q], f, cn);
            continue;
        }
        const float4 l = lines[q - nodes];
        const int steps = line_steps(l);
        if (steps == 0) {
            hit(far, f, round_px(l.x), round_px(l.y));
            continue;
        }
        const double ddx = (double)__fsub_rn(l.z, l.x), ddy = (double)__fsub_rn(l.w, l.y);
        const double n_steps = (double)steps, y = __ddiv_rn(1.0, n_steps);
        for (int k = 0; k <= steps; ++k) {
            const double t = quotient((double)k, n_steps, y);
            const float sx = (float)__dadd_rn((double)l.x, __dmul_rn(t, ddx));
            const float sy = (float)__dadd_rn((double)l.y, __dmul_rn(t, ddy));
            hit(far, f, round_px(sx), round_px(sy));
        }
    }
}

__device__ __forceinline__ float powi(float b, unsigned int k) {
    float r = 1.0f;
    while (k) {
        if (k & 1u) r = __fmul_rn(r, b);
        b = __fmul_rn(b, b);
        k >>= 1;
    }
    return r;
}

__device__ __forceinline__ unsigned char brightness(float keep_n, unsigned int nodes, float keep_e,
                                                    unsigned int edges) {
    const float keep = __fmul_rn(powi(keep_n, nodes), powi(keep_e, edges));
    return (unsigned char)lroundf(__fmul_rn(255.0f, keep));
}

__global__ __launch_bounds__(256) void k_shade(const unsigned int* __restrict__ cn, const unsigned int* __restrict__ ce,
                                               long long npix, float keep_n, float keep_e,
                                               unsigned char* __restrict__ out) {
    for (long long p = blockIdx.x * 256ll + threadIdx.x; p < npix; p += (long long)gridDim.x * 256)
        out[p] = brightness(keep_n, cn[p], keep_e, ce[p]);
}

// The same from the tiles' copies and the far-out lines' counters (from k_raster_pixels' counters,
// the nodes' in place of the copies, if it counted); a block per row of a tile.
__global__ __launch_bounds__(kTileW) void k_shade_tiles(const unsigned int* __restrict__ copies,
                                                        const int* __restrict__ first, int tiles, int tiles_x,
                                                        const unsigned int* __restrict__ far, Frame f, float keep_n,
                                                        float keep_e, unsigned char* __restrict__ out) {
    const int t = blockIdx.x / kTileH, row = blockIdx.x % kTileH;
    const Tile a = tile_of(t, tiles_x, f);
    if (row >= a.rh || (int)threadIdx.x >= a.cw) return;
    const size_t p = (size_t)(a.r0 + row) * f.w + a.c0 + threadIdx.x;
    const unsigned int* c = copies + (size_t)row * kTileW + threadIdx.x;
    unsigned int edges = far[p], nodes = first[2 * tiles] == 0 ? copies[p] : 0u;
    const int e1 = first[t + 1], n1 = first[tiles + t + 1];
#pragma unroll 8
    for (int k = first[t]; k < e1; ++k) edges += c[(size_t)k * kTilePixels];
    for (int k = first[tiles + t]; k < n1; ++k) nodes += c[(size_t)k * kTilePixels];
    out[p] = brightness(keep_n, nodes, keep_e, edges);
}

// The picture by a device atomic per sample: cnt holds 2 npix cleared counters, the nodes' first.
void count_pixels(const Bufs& b, const Frame& f, unsigned int* cnt, unsigned char* img, const gfa2_raster* r,
                  hipStream_t s) {
    const long long npix = (long long)f.w * f.h;
    k_raster_nodes<<<(b.n + 255) / 256, 256, 0, s>>>(b.pos, b.n, f, cnt);
    long long eb = (b.nnz + 255) / 256;
    if (eb > 8192) eb = 8192;
    if (eb > 0) k_raster_edges<<<(int)eb, 256, 0, s>>>(b.pos, b.rowptr, b.col, b.n, b.nnz, f, cnt + npix);
    long long pb = (npix + 255) / 256;
    if (pb > 8192) pb = 8192;
    k_shade<<<(int)pb, 256, 0, s>>>(cnt, cnt + npix, npix, 1.0f - r->node_alpha, 1.0f - r->edge_alpha, img);
}

}  // namespace
}  // namespace gfa2

using namespace gfa2;

extern "C" {

int gfa2_get_bbox(gfa2_handle h, float* out) {
    const Bufs* b = nullptr;
    int device = 0;
    hipStream_t s = nullptr;
    if (!h || !out) return GFA2_ERR_INVALID_ARG;
    if (!engine_graph(h, &b, &device, &s)) return GFA2_ERR_NO_GRAPH;
    if (hipSetDevice(device) != hipSuccess) return GFA2_ERR_HIP;
    const int nb = 256;
    EngineScratch scratch(h);
    float4* part = static_cast<float4*>(scratch.get(sizeof(float4) * (nb + 1)));
    if (!part) return GFA2_ERR_OOM;
    k_minmax<<<nb, 256, 0, s>>>(b->pos, b->n, part);
    k_minmax_final<<<1, 64, 0, s>>>(part, nb, part + nb);
    float4 m;
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(&m, part + nb, sizeof(float4), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return GFA2_ERR_HIP;
    out[0] = m.x;
    out[1] = m.y;
    out[2] = m.z;
    out[3] = m.w;
    return GFA2_OK;
}

int gfa2_render(gfa2_handle h, const gfa2_raster* r, uint8_t* gray) {
    const Bufs* b = nullptr;
    int device = 0;
    hipStream_t s = nullptr;
    if (!h || !r || !gray || r->width <= 0 || r->height <= 0) return GFA2_ERR_INVALID_ARG;
    if (!engine_graph(h, &b, &device, &s)) return GFA2_ERR_NO_GRAPH;
    if (b->nseg > 1) return GFA2_ERR_UNSUPPORTED;
    if (hipSetDevice(device) != hipSuccess) return GFA2_ERR_HIP;
    const long long npix = (long long)r->width * r->height;
    const Frame f{r->x0, r->y0, r->sx, r->sy, r->width, r->height};
    const long long across = ((long long)f.w + kTileW - 1) / kTileW, down = ((long long)f.h + kTileH - 1) / kTileH;
    const long long most_samples = (b->nnz / 2) * std::max(f.w, f.h);
    const int spare = (int)std::min<long long>(kSpareSlices, (most_samples + 29ll * b->n) / kSliceSamples);
    const long long copies_ll = 2 * across * down + spare;
    const long long lists = std::max<long long>(1, (b->nnz + kListEntries - 1) / kListEntries);
    const size_t list_len = (size_t)std::min<long long>(b->nnz, kListEntries);
    // the scratch: line list, its totals, tile costs, far-out lines' counters, plan, copies, picture
    size_t size = 0;
    auto place = [&](size_t bytes) {
        const size_t at = size;
        size += (bytes + 255) & ~(size_t)255;
        return at;
    };
    const size_t two_tiles = 2 * (size_t)(across * down);
    const size_t at_lines = place(sizeof(float4) * list_len), at_list = place(sizeof(ListTotals));
    const size_t at_cost = place(sizeof(unsigned long long) * two_tiles);
    const size_t at_far = place(sizeof(unsigned int) * (size_t)npix);
    const size_t at_first = place(sizeof(int) * (two_tiles + 1));
    const size_t at_copies = place(sizeof(unsigned int) * kTilePixels * (size_t)copies_ll), at_img = place((size_t)npix);
    const size_t plain = 9 * (size_t)npix + 1024;
    const bool few = most_samples <= std::min(kFewSamples, 512 * npix) && std::max(f.w, f.h) <= kFewPixels;
    const bool either = across * down * (b->nnz / 2 + b->n) > kManyTests;
    EngineScratch scratch(h);
    char* mem = nullptr;
    if (!few && (size <= kTileMemory || size / 4 <= plain)) mem = static_cast<char*>(scratch.get(size));
    unsigned char* img = nullptr;
    hipError_t e = hipSuccess;
    if (!mem) {
        mem = static_cast<char*>(scratch.get(plain));
        if (!mem) return GFA2_ERR_OOM;
        unsigned int* cnt = reinterpret_cast<unsigned int*>(mem);
        img = reinterpret_cast<unsigned char*>(cnt + 2 * npix);
        e = hipMemsetAsync(cnt, 0, sizeof(unsigned int) * 2 * (size_t)npix, s);
        if (e == hipSuccess) {
            count_pixels(*b, f, cnt, img, r, s);
            e = hipGetLastError();
        }
    } else {
        const int tiles_x = (int)across, tiles = (int)(across * down), copies = (int)copies_ll;
        float4* lines = reinterpret_cast<float4*>(mem + at_lines);
        ListTotals* list = reinterpret_cast<ListTotals*>(mem + at_list);
        unsigned long long* cost = reinterpret_cast<unsigned long long*>(mem + at_cost);
        unsigned int* far = reinterpret_cast<unsigned int*>(mem + at_far);
        int* first = reinterpret_cast<int*>(mem + at_first);
        unsigned int* copy = reinterpret_cast<unsigned int*>(mem + at_copies);
        img = reinterpret_cast<unsigned char*>(mem + at_img);
        e = hipMemsetAsync(list, 0, at_first - at_list, s);      // totals, costs and counters
        for (long long q = 0; q < lists && e == hipSuccess; ++q) {
            const long long e0 = q * kListEntries, e1 = std::min<long long>(b->nnz, e0 + kListEntries);
            if (q > 0) e = hipMemsetAsync(list, 0, sizeof(ListTotals), s);
            constexpr long long kPer = kLineThreads * kLineItems;
            if (e1 > e0)
                k_raster_lines<<<(int)((e1 - e0 + kPer - 1) / kPer), kLineThreads, 0, s>>>(b->pos, b->rowptr, b->col, b->n,
                                                                                         e0, e1, f, lines, list, far,
                                                                                         either && q == 0);
            const long long most = std::max<long long>(b->n, (long long)list_len);
            if (q == 0) {
                // the plan of the first list serves the others
                const int per_tile = (int)std::min<long long>(most / (256 * kCostStride) + 1, 8);
                k_raster_cost<<<dim3(2 * tiles, per_tile), 256, 0, s>>>(lines, list, b->pos, b->n, f, tiles, tiles_x, cost,
                                                                        copy, either);
                k_raster_plan<<<1, 1024, 0, s>>>(cost, 2 * tiles, spare, list, b->n, f, first, either);
            }
            k_raster_tiles<<<copies, kTileThreads, 0, s>>>(lines, list, b->pos, b->n, f, tiles, tiles_x, first, copy, q > 0);
            if (either)
                k_raster_pixels<<<(int)std::min<long long>(most / 256 + 1, 2048), 256, 0, s>>>(lines, list, b->pos, b->n, f,
                                                                                           tiles, first, copy, far, q > 0);
        }
        if (e == hipSuccess) {
            k_shade_tiles<<<tiles * kTileH, kTileW, 0, s>>>(copy, first, tiles, tiles_x, far, f, 1.0f - r->node_alpha,
                                                            1.0f - r->edge_alpha, img);
            e = hipGetLastError();
        }
    }
    if (e == hipSuccess) e = hipMemcpyAsync(gray, img, (size_t)npix, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    return e == hipSuccess ? GFA2_OK : GFA2_ERR_HIP;
}

int gfa2_render_noalloc(gfa2_handle h, const gfa2_raster* r, uint8_t* gray) {
    const Bufs* b = nullptr;
    int device = 0;
    hipStream_t s = nullptr;
    if (!h || !r || !gray || r->width <= 0 || r->height <= 0) return GFA2_ERR_INVALID_ARG;
    const long long npix = (long long)r->width * r->height;
    if (npix > kNoAllocMaxPixels) return GFA2_ERR_SCRATCH_LIMIT;
    if (!engine_graph(h, &b, &device, &s)) return GFA2_ERR_NO_GRAPH;
    if (b->nseg > 1) return GFA2_ERR_UNSUPPORTED;
    if (device < 0 || device >= kScratchMaxDevices) return GFA2_ERR_UNSUPPORTED;
    if (hipSetDevice(device) != hipSuccess) return GFA2_ERR_HIP;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[device]) {
        // once per device, with that device current: this device's copy of the array
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return GFA2_ERR_HIP;
        g_scratch[device] = static_cast<unsigned int*>(p);
    }
    unsigned int* cnt = g_scratch[device];                       // node counters [0, npix), edges [npix, 2 npix)
    unsigned char* img = reinterpret_cast<unsigned char*>(cnt + 2 * kNoAllocMaxPixels);
    const Frame f{r->x0, r->y0, r->sx, r->sy, r->width, r->height};
    // the counters keep the previous call's hits: cleared by a kernel (no memset node)
    long long zb = (2 * npix + 255) / 256;
    if (zb > 8192) zb = 8192;
    k_fill_zero<<<(int)zb, 256, 0, s>>>(cnt, 2 * npix);
    count_pixels(*b, f, cnt, img, r, s);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(gray, img, (size_t)npix, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    return e == hipSuccess ? GFA2_OK : GFA2_ERR_HIP;
}

}  // extern "C"
