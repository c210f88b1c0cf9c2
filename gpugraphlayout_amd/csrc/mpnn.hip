// Learned initial layout: a small message-passing network whose output positions
// ForceAtlas2 then refines (no counterpart in the reference).
//
// Network (fixed shape): inputs X [V x 16] (9 features, zero padded), hidden 64, output 2.
//   A0 = mean_agg(X)                     mean over CSR neighbours (0 for isolated nodes)
//   H1 = relu(X W1s + A0 W1n + b1)       [V x 64]
//   A1 = mean_agg(H1)
//   H2 = relu(H1 W2s + A1 W2n + b2)      [V x 64]
//   Y  = H2 Wo + bo                      [V x 2]
// Weights are stored in BF16 (round to nearest even from FP32 master copies kept for
// Adam); every product accumulates in FP32. Gradients are taken with respect to the
// BF16-rounded weights and applied to the masters.
//
// Features: column 0 = log(deg+1); columns 1..8 = seeded standard normal fields smoothed by
// `steps` rounds of z <- (z + mean_agg(z)) / 2; every column then standardised (zero mean,
// unit variance over the nodes).
//
// Loss (invariant to translation and rotation/reflection of the target; the target is
// centred and scaled to unit RMS radius): over a symmetric set P of ordered pairs - each
// node's CSR neighbours plus the nodes (i +/- o_k) mod V for R seeded offsets o_k -
//   L = (1/|P|) sum_{(i,j) in P} (|y_i - y_j| - |t_i - t_j|)^2
// Because P is symmetric, dL/dy_i = (4/|P|) sum_{j in P(i)} (|y_ij| - |t_ij|) (y_i-y_j)/|y_ij|
// is a per-node gather: no atomics anywhere, so training is deterministic.
//
// Every reduction over nodes (weight gradients, column statistics, loss) writes per-block
// partials that a second kernel sums in a fixed order.
//
// Dense products run on the FP32 matrix instructions (v_mfma_f32_16x16x4_f32: 16 x 16 results, 4
// inner terms, FP32 throughout), which do twice the FP32 work per cycle of a vector FMA. A lane
// of the instruction holds A[i = lane % 16][k = lane / 16], B[k = lane / 16][j = lane % 16] and
// four results C[i = 4 (lane / 16) + r][j = lane % 16]; which inner index a (step, lane / 16)
// slot stands for is free as long as A and B agree.
#include "engine_internal.h"
#include "mpnn_internal.h"

#include <vector>

namespace gfa2 {
namespace {

__device__ __forceinline__ float bf16_to_f32(unsigned short b) { return __uint_as_float((unsigned int)b << 16); }

__device__ __forceinline__ unsigned short f32_to_bf16(float f) {
    unsigned int u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)(u >> 16);   // inf / nan
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// ---- features -----------------------------------------------------------------------------

// Z [V x 8]: standard normal by Box-Muller from two 24-bit uniforms of mix64(seed, i*8+f).
__global__ __launch_bounds__(256) void k_normal_fields(int n, unsigned long long seed, float* __restrict__ Z) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n * 8) return;
    const unsigned long long r = mix64(seed ^ mix64((unsigned long long)t));
    const float u1 = ((float)(r >> 40) + 0.5f) * (1.0f / 16777216.0f);
    const float u2 = (float)((r >> 16) & 0xffffffull) * (1.0f / 16777216.0f);
    Z[t] = sqrtf(-2.0f * logf(u1)) * cosf(6.2831853071795864f * u2);
}

// The features are column 0 log(deg + 1) and columns 1 to 8 Z, each with its mean taken away and
// divided by its deviation, and zeros. They are written once, normalised: a pass over Z for the
// columns' sums (each row's entries and offsets are all that it reads), a block that adds the
// passes' partials, a pass that writes X. All three are bound by memory (R-MAT 2^20, 580k nodes:
// with the raw features written, read and rewritten and the partials added by one thread per
// column 144 us, now 28).
constexpr int kStat = 9;             // columns that are not padding
constexpr int kStatBlocks = 448;     // partials of 2 kStat doubles each
static_assert(kStatBlocks * 2 * kStat <= kPartDoubles);

__device__ __forceinline__ float degree_feature(const int* __restrict__ rowptr, int i) {
    return logf((float)(rowptr[i + 1] - rowptr[i]) + 1.0f);
}

__device__ __forceinline__ double wave_sum(double v, int low) {
    for (int o = low; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Per-block sums and sums of squares of the columns. Two lanes per row, a half of Z each; the even
// one takes the degree too.
__global__ __launch_bounds__(256) void k_colstats(const int* __restrict__ rowptr, const float* __restrict__ Z, int n,
                                                  double* __restrict__ part) {
    __shared__ double sums[4][2 * kStat];
    const int half = threadIdx.x & 1;
    double a[5] = {}, b[5] = {};        // the degree, four columns of Z
    for (long long i = (long long)blockIdx.x * 128 + threadIdx.x / 2; i < n; i += (long long)gridDim.x * 128) {
        const float4 z = *reinterpret_cast<const float4*>(Z + i * 8 + 4 * half);
        const float x[5] = {half ? 0.0f : degree_feature(rowptr, (int)i), z.x, z.y, z.z, z.w};
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            const double v = x[c];
            a[c] += v;
            b[c] += v * v;
        }
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        const double A = wave_sum(a[c], 2), B = wave_sum(b[c], 2);
        const int f = c == 0 ? 0 : 4 * half + c;
        if (lane < 2 && (c > 0 || half == 0)) {
            sums[wave][2 * f] = A;
            sums[wave][2 * f + 1] = B;
        }
    }
    __syncthreads();
    if (threadIdx.x < 2 * kStat)
        part[blockIdx.x * 2 * kStat + threadIdx.x] = sums[0][threadIdx.x] + sums[1][threadIdx.x] +
                                                     sums[2][threadIdx.x] + sums[3][threadIdx.x];
}

// A wave per column.
__global__ __launch_bounds__(64 * kStat) void k_colnorm_finish(const double* __restrict__ part, int nb, int n,
                                                               float* __restrict__ mu_sd) {
    const int f = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double A = 0.0, B = 0.0;
#pragma unroll 4
    for (int b = lane; b < nb; b += 64) {
        A += part[b * 2 * kStat + 2 * f];
        B += part[b * 2 * kStat + 2 * f + 1];
    }
    A = wave_sum(A, 1);
    B = wave_sum(B, 1);
    if (lane > 0) return;
    const double mu = A / n;
    const double var = B / n - mu * mu;
    mu_sd[2 * f] = (float)mu;
    mu_sd[2 * f + 1] = var > 1e-12 ? (float)(1.0 / sqrt(var)) : 0.0f;
}

// Four lanes per row, four columns of X each.
__global__ __launch_bounds__(256) void k_features(const int* __restrict__ rowptr, const float* __restrict__ Z, int n,
                                                  const float* __restrict__ mu_sd, float* __restrict__ X) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long i = t / 4;
    if (i >= n) return;
    const int q = (int)(t % 4);
    float x[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int f = 4 * q + c;
        x[c] = 0.0f;
        if (f < kStat) x[c] = ((f == 0 ? degree_feature(rowptr, (int)i) : Z[i * 8 + f - 1]) - mu_sd[2 * f]) * mu_sd[2 * f + 1];
    }
    *reinterpret_cast<float4*>(X + i * kIn + 4 * q) = make_float4(x[0], x[1], x[2], x[3]);
}

// ---- neighbour aggregation -----------------------------------------------------------------

// out[i][:] = epilogue(sum over CSR neighbours j of in[j][:]), F features per node (8, 16 or 64):
//   kAggMean       out = sum / deg(i) (0 for an isolated node)     forward mean
//   kAggSmooth     out = (in[i] + sum / deg(i)) / 2                 feature smoothing
//   kAggBack       out = H[i] > 0 ? P[i] + sum : 0                  backward of the mean and relu
//                  (in[j] already divided by deg(j))
// Light rows (at most kAggLight entries): kAggSlots slots of F / 4 lanes per row, which read a
// float4 each of every entry of the slot; medium rows (listed): a wave per row with 256 / F slots;
// heavy rows (over kAggHeavy entries, the hubs of a skewed graph, which would otherwise leave one
// wave looping over 10^5 entries): a block per chunk of kAggChunk entries, whose four waves sum a
// quarter each into a partial, added by k_agg_heavy. A slot has the loads of four or eight entries
// under way at once, and the slots are added in a fixed tree, so results are deterministic.
// What bounds it are the lines that the L2s miss, which come at the 4 to 5 TB/s of a plain copy
// (R-MAT 2^20, 20M entries: F = 64 asks for 40M lines of 128 bytes; halves or quarters of the
// features to different dies gave nothing, 681 and 862 us). There with 4-byte loads, one row after
// another per group and 512-entry chunks in a launch of their own: F = 8 325 -> 167 us, F = 16
// 414 -> 208, F = 64 889 -> 622.
enum AggMode { kAggMean = 0, kAggSmooth = 1, kAggBack = 2 };

// Slots per light row, and entries under way at once per slot of a medium row (4 in a light one).
template <int F>
constexpr int kAggSlots = F == 64 ? 1 : 4;
template <int F>
constexpr int kAggAhead = F == 64 ? 8 : 4;

struct AggArgs {
    const int* rowptr;
    const int* col;
    int n;
    const int* medium;          // rows of more than kAggLight entries up to kAggHeavy
    int nmedium;
    const int* heavy;
    const int2* chunks;         // {index into heavy, first entry}
    int nchunks;
    const float* in;
    const float* P;
    const float* H;
    float* out;
    float* part;                // [4 nchunks][F]
};

__device__ __forceinline__ float4 add4(float4 a, float4 b) {
    return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

template <int MODE>
__device__ __forceinline__ float agg_finish(float s, int deg, float in, float P, float H) {
    if (MODE == kAggBack) return H > 0.0f ? P + s : 0.0f;
    const float m = deg > 0 ? s / (float)deg : 0.0f;
    return MODE == kAggSmooth ? 0.5f * (in + m) : m;
}

// Row i's result from its sum, features at4 to at4 + 3 of the float array.
template <int MODE>
__device__ __forceinline__ void agg_store(const AggArgs& A, float4 s, int deg, size_t at) {
    const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 v = z, P = z, H = z;
    if (MODE == kAggSmooth) v = *reinterpret_cast<const float4*>(A.in + at);
    if (MODE == kAggBack) {
        P = *reinterpret_cast<const float4*>(A.P + at);
        H = *reinterpret_cast<const float4*>(A.H + at);
    }
    *reinterpret_cast<float4*>(A.out + at) =
        make_float4(agg_finish<MODE>(s.x, deg, v.x, P.x, H.x), agg_finish<MODE>(s.y, deg, v.y, P.y, H.y),
                    agg_finish<MODE>(s.z, deg, v.z, P.z, H.z), agg_finish<MODE>(s.w, deg, v.w, P.w, H.w));
}

// The sum of entries slot, slot + S, slot + 2 S, ... of len, for this lane's four features.
template <int F, int S, int U>
__device__ __forceinline__ float4 agg_slot(const int* __restrict__ col, int len, int slot, const float* __restrict__ in) {
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int e = slot; e < len; e += U * S) {
        int j[U];
#pragma unroll
        for (int u = 0; u < U; ++u) j[u] = e + u * S < len ? col[e + u * S] : 0;
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const float4*>(in + (size_t)j[u] * F);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (e + u * S < len) s = add4(s, v[u]);
    }
    return s;
}

// The sum over the slots of a group: lanes that differ by low, 2 low, ... up to high / 2.
__device__ __forceinline__ float4 agg_fold(float4 s, int low, int high) {
    for (int o = low; o < high; o <<= 1)
        s = add4(s, make_float4(__shfl_xor(s.x, o, 64), __shfl_xor(s.y, o, 64), __shfl_xor(s.z, o, 64),
                                __shfl_xor(s.w, o, 64)));
    return s;
}

// Virtual blocks: the chunks, then light and medium blocks in turns.
template <int F, int MODE>
__global__ __launch_bounds__(256) void k_agg(const AggArgs A, int light_blocks, int medium_blocks) {
    constexpr int L = F / 4, G = L * kAggSlots<F>;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int f = 4 * (lane % L);                // this lane's first feature
    const float* in = A.in + f;
    const unsigned int vb = blockIdx.x;
    if (vb < (unsigned int)A.nchunks) {
        const int2 ch = A.chunks[vb];
        const int len = min(kAggChunk, A.rowptr[A.heavy[ch.x] + 1] - ch.y);
        const int first = wave * (kAggChunk / 4);
        float4 s = agg_slot<F, 64 / L, kAggAhead<F>>(A.col + ch.y + first, min(kAggChunk / 4, len - first), lane / L, in);
        s = agg_fold(s, L, 64);
        if (lane < L) *reinterpret_cast<float4*>(A.part + ((size_t)vb * 4 + wave) * F + f) = s;
        return;
    }
    const unsigned int i = vb - A.nchunks, t = light_blocks + medium_blocks;
    const int m0 = (int)((unsigned long long)i * medium_blocks / t);       // medium blocks before i
    if ((int)((i + 1ull) * medium_blocks / t) > m0) {
        const int k = m0 * 4 + wave;
        if (k >= A.nmedium) return;
        const int v = A.medium[k], e0 = A.rowptr[v], len = A.rowptr[v + 1] - e0;
        const float4 s = agg_fold(agg_slot<F, 64 / L, kAggAhead<F>>(A.col + e0, len, lane / L, in), L, 64);
        if (lane < L) agg_store<MODE>(A, s, len, (size_t)v * F + f);
    } else {
        const long long v = (long long)(i - m0) * (256 / G) + threadIdx.x / G;
        if (v >= A.n) return;
        const int e0 = A.rowptr[v], len = A.rowptr[v + 1] - e0;
        if (len > kAggLight) return;
        const float4 s = agg_fold(agg_slot<F, kAggSlots<F>, 4>(A.col + e0, len, lane % G / L, in), L, G);
        if (lane % G < L) agg_store<MODE>(A, s, len, (size_t)v * F + f);
    }
}

// A wave per heavy row: its partials, 256 / F at a time.
template <int F, int MODE>
__global__ __launch_bounds__(256) void k_agg_heavy(const AggArgs A, const int* __restrict__ heavy_c0, int nheavy) {
    constexpr int L = F / 4, S = 64 / L;
    const int lane = threadIdx.x & 63, h = blockIdx.x * 4 + (threadIdx.x >> 6), f = 4 * (lane % L);
    if (h >= nheavy) return;
    const int v = A.heavy[h], c0 = 4 * heavy_c0[h], c1 = 4 * heavy_c0[h + 1];
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 4
    for (int c = c0 + lane / L; c < c1; c += S) s = add4(s, *reinterpret_cast<const float4*>(A.part + (size_t)c * F + f));
    s = agg_fold(s, L, 64);
    if (lane < L) agg_store<MODE>(A, s, A.rowptr[v + 1] - A.rowptr[v], (size_t)v * F + f);
}

using f32x4 = __attribute__((ext_vector_type(4))) float;

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The weights are read from LDS for every tile: held in registers across tiles (the compiler's own
// choice, 242 of them) they leave one wave per SIMD.
__device__ __forceinline__ void keep_in_lds() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ float at4(const float4& v, int m) { return m == 0 ? v.x : m == 1 ? v.y : m == 2 ? v.z : v.w; }

// H[i][o] = relu(b[o] + sum_k (A[i][k] Ws[k][o] + B[i][k] Wn[k][o])) and, with HEAD, Y = H Wo + bo
// as well (H is then written only if asked for: inference needs none of it). A wave takes 16 nodes
// and all 64 outputs: four result tiles with i = output and j = node, so that a lane ends up with 4
// consecutive outputs of one node and node data goes from memory straight into the instruction's
// operand (four inner indices per 16-byte load, slot (m, lane / 16) standing for 4 (lane / 16) + m).
// The weights, FP32 from BF16, lie in LDS in operand order.
//
// Bound by memory for K = 16 (580,000 nodes read 74 MB and write 148: 50 us, 4.4 TB/s, as the
// vector kernel before) and by the matrix instructions for K = 64 (9.5 GFLOP and 302 MB in 106 us;
// register-tiled vector FMAs took 194 us and a head launch 33 more).
template <int K, bool HEAD>
__global__ __launch_bounds__(256) void k_dense(const float* __restrict__ A, const float* __restrict__ B, int n,
                                               const unsigned short* __restrict__ Ws,
                                               const unsigned short* __restrict__ Wn,
                                               const unsigned short* __restrict__ bias, float* __restrict__ H,
                                               const unsigned short* __restrict__ Wo,
                                               const unsigned short* __restrict__ bo, float2* __restrict__ Y) {
    constexpr int S = K / 16;                                 // 16-index steps per input
    __shared__ float4 w[4][2 * S][64];                        // [output tile][step][lane]
    __shared__ float2 wo[kHid];
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int tiles = (n + 15) / 16, stride = gridDim.x * 4;
    float4 nx[2 * S];                                         // the next tile's inputs, loaded meanwhile
    auto load = [&](int tile) {
        const size_t row = (size_t)min(tile * 16 + j, n - 1) * K;
#pragma unroll
        for (int q = 0; q < S; ++q) {
            nx[q] = *reinterpret_cast<const float4*>(A + row + 16 * q + 4 * g);
            nx[S + q] = *reinterpret_cast<const float4*>(B + row + 16 * q + 4 * g);
        }
    };
    const int tile0 = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile0 < tiles) load(tile0);
#pragma unroll
    for (int q0 = 0; q0 < 2 * K * (kHid / 4); q0 += 256) {
        const int q = q0 + threadIdx.x;
        const int k = q >> 4, o = 4 * (q & 15);               // inner index, first of four outputs
        const ushort4 u = *reinterpret_cast<const ushort4*>((k < K ? Ws + k * kHid : Wn + (k - K) * kHid) + o);
        float* at = reinterpret_cast<float*>(&w[o >> 4][k >> 4][16 * ((k >> 2) & 3) + (o & 15)]) + (k & 3);
        at[0] = bf16_to_f32(u.x);
        at[4] = bf16_to_f32(u.y);
        at[8] = bf16_to_f32(u.z);
        at[12] = bf16_to_f32(u.w);
    }
    if (HEAD && threadIdx.x < kHid)
        wo[threadIdx.x] = make_float2(bf16_to_f32(Wo[2 * threadIdx.x]), bf16_to_f32(Wo[2 * threadIdx.x + 1]));
    __syncthreads();
    f32x4 b0[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) b0[t][r] = bf16_to_f32(bias[16 * t + 4 * g + r]);
    const float y0 = HEAD ? bf16_to_f32(bo[0]) : 0.0f, y1 = HEAD ? bf16_to_f32(bo[1]) : 0.0f;
    for (int tile = tile0; tile < tiles; tile += stride) {
        const int i = tile * 16 + j;
        float4 x[2 * S];
#pragma unroll
        for (int q = 0; q < 2 * S; ++q) x[q] = nx[q];
        if (tile + stride < tiles) load(tile + stride);
        keep_in_lds();
        f32x4 acc[4] = {b0[0], b0[1], b0[2], b0[3]};
#pragma unroll
        for (int q = 0; q < 2 * S; ++q) {
            float4 u[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) u[t] = w[t][q][lane];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[t] = mfma(at4(u[t], m), at4(x[q], m), acc[t]);
        }
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[t][r] = fmaxf(acc[t][r], 0.0f);
                if (HEAD) {
                    const float2 u = wo[16 * t + 4 * g + r];
                    s0 = fmaf(acc[t][r], u.x, s0);
                    s1 = fmaf(acc[t][r], u.y, s1);
                }
            }
            if (i < n && H)
                *reinterpret_cast<float4*>(H + (size_t)i * kHid + 16 * t + 4 * g) =
                    make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
        }
        if (HEAD) {
            // the node's four lanes hold a quarter of the outputs each
            s0 += __shfl_xor(s0, 16, 64);
            s1 += __shfl_xor(s1, 16, 64);
            s0 += __shfl_xor(s0, 32, 64);
            s1 += __shfl_xor(s1, 32, 64);
            if (g == 0 && i < n) Y[i] = make_float2(s0 + y0, s1 + y1);
        }
    }
}

// ---- loss ----------------------------------------------------------------------------------

// Per node: loss terms over P(i) and dY[i]; per-block loss partials. Eight lanes per node take
// its pairs in turn and add up in a fixed tree.
__global__ __launch_bounds__(256) void k_loss(const int* __restrict__ rowptr, const int* __restrict__ col, int n,
                                              const float2* __restrict__ Y, const float2* __restrict__ T,
                                              const int* __restrict__ offs, int R, double inv_pairs,
                                              float2* __restrict__ dY, double* __restrict__ part) {
    __shared__ double red[256];
    const int lane8 = threadIdx.x & 7;
    const float c = (float)(4.0 * inv_pairs);
    double l = 0.0;
    for (long long i0 = blockIdx.x * 32ll; i0 < n; i0 += gridDim.x * 32ll) {
        const long long ii = i0 + (threadIdx.x >> 3);
        float gx = 0.0f, gy = 0.0f;
        if (ii < n) {
            const int i = (int)ii;
            const float2 y = Y[i], t = T[i];
            const int e0 = rowptr[i], deg = rowptr[i + 1] - e0;
            const int cnt = deg + 2 * R;
#pragma unroll 2
            for (int q = lane8; q < cnt; q += 8) {
                int j;
                if (q < deg) j = col[e0 + q];
                else {
                    // offsets are below n
                    const int k = q - deg;
                    const int o = (k & 1) ? n - offs[k >> 1] : offs[k >> 1];
                    j = i < n - o ? i + o : i - (n - o);
                }
                const float2 yj = Y[j], tj = T[j];
                const float dx = y.x - yj.x, dy = y.y - yj.y;
                const float ex = t.x - tj.x, ey = t.y - tj.y;
                const float d = sqrtf(dx * dx + dy * dy) + 1e-12f;
                const float r = d - sqrtf(ex * ex + ey * ey);
                l += (double)r * r;
                const float s = r / d;
                gx = fmaf(s, dx, gx);
                gy = fmaf(s, dy, gy);
            }
        }
#pragma unroll
        for (int o = 4; o > 0; o >>= 1) {
            gx += __shfl_xor(gx, o, 64);
            gy += __shfl_xor(gy, o, 64);
        }
        if (lane8 == 0 && ii < n) dY[ii] = make_float2(c * gx, c * gy);
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0] * inv_pairs;
}

// ---- backward ------------------------------------------------------------------------------

// dZ2[i][o] = H2[i][o] > 0 ? sum_c dY[i][c] Wo[o][c] : 0, formed wherever it is needed.
__device__ __forceinline__ float d_z2(float h, float2 dy, float2 wo) {
    return h > 0.0f ? fmaf(dy.x, wo.x, dy.y * wo.y) : 0.0f;
}

// P[i][k] = sum_o dZ2[i][o] W2s[k][o], Q[i][k] = sum_o dZ2[i][o] W2n[k][o] / deg(i): both input
// gradients of the second layer in one pass over H2 and dY, laid out as k_dense (four result
// tiles each, i = input, j = node).
//
// Bound by memory (H2 read, P and Q written): one wave per node with shuffled inputs took 124 us
// for each of the two products on 50,000 nodes, after a launch that wrote dZ2; both take 19 us here.
__global__ __launch_bounds__(256) void k_back(const float2* __restrict__ dY, const float* __restrict__ H2, int n,
                                              const int* __restrict__ rowptr, const unsigned short* __restrict__ Wo,
                                              const unsigned short* __restrict__ W2s,
                                              const unsigned short* __restrict__ W2n, float* __restrict__ P,
                                              float* __restrict__ Q) {
    __shared__ float4 w[8][4][64];                            // [P's tiles, Q's tiles][step][lane]
    __shared__ float2 wo[kHid];
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int tiles = (n + 15) / 16, stride = gridDim.x * 4;
    float4 nx[4];                                             // the next tile's inputs, loaded meanwhile
    float2 ndy = make_float2(0.0f, 0.0f);
    int ndeg = 0;
    auto load = [&](int tile) {
        const int ic = min(tile * 16 + j, n - 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) nx[q] = *reinterpret_cast<const float4*>(H2 + (size_t)ic * kHid + 16 * q + 4 * g);
        ndy = dY[ic];
        ndeg = rowptr[ic + 1] - rowptr[ic];
    };
    const int tile0 = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile0 < tiles) load(tile0);
#pragma unroll
    for (int q0 = 0; q0 < 2 * kHid * (kHid / 4); q0 += 256) {
        const int q = q0 + threadIdx.x;
        const int k = (q >> 4) & 63, o = 4 * (q & 15), n2 = q >> 10;      // row, first of four inner indices, matrix
        const ushort4 u = *reinterpret_cast<const ushort4*>((n2 ? W2n : W2s) + k * kHid + o);
        w[4 * n2 + (k >> 4)][o >> 4][16 * ((o >> 2) & 3) + (k & 15)] =
            make_float4(bf16_to_f32(u.x), bf16_to_f32(u.y), bf16_to_f32(u.z), bf16_to_f32(u.w));
    }
    if (threadIdx.x < kHid)
        wo[threadIdx.x] = make_float2(bf16_to_f32(Wo[2 * threadIdx.x]), bf16_to_f32(Wo[2 * threadIdx.x + 1]));
    __syncthreads();
    for (int tile = tile0; tile < tiles; tile += stride) {
        const int i = tile * 16 + j;
        float4 x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = nx[q];
        const float2 dy = ndy;
        const int deg = ndeg;
        if (tile + stride < tiles) load(tile + stride);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float2* u = wo + 16 * q + 4 * g;
            x[q] = make_float4(d_z2(x[q].x, dy, u[0]), d_z2(x[q].y, dy, u[1]), d_z2(x[q].z, dy, u[2]),
                               d_z2(x[q].w, dy, u[3]));
        }
        keep_in_lds();
        f32x4 acc[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float4 u[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) u[t] = w[t][q][lane];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int t = 0; t < 8; ++t) acc[t] = mfma(at4(u[t], m), at4(x[q], m), acc[t]);
        }
        if (i >= n) continue;
        const float inv = deg > 0 ? 1.0f / (float)deg : 0.0f;     // no neighbour reads Q of an isolated node
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const size_t at = (size_t)i * kHid + 16 * t + 4 * g;
            *reinterpret_cast<float4*>(P + at) = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
            *reinterpret_cast<float4*>(Q + at) =
                make_float4(acc[4 + t][0] * inv, acc[4 + t][1] * inv, acc[4 + t][2] * inv, acc[4 + t][3] * inv);
        }
    }
}

// Weight gradients: products over the nodes (the inner index; a lane's slot lane / 16 is the node
// within a step of four). Blocks take runs of 64 nodes in turn; a run is summed in FP32 and added
// to FP64 sums kept in registers, which become the block's partial at the end. Partials are laid
// out as the parameters are, so that k_sum_grad writes the gradient itself.
//
// A partial per run of 64 nodes (782 of them at 50,000 nodes, each of 4,160 values) summed by one
// thread per value took 185 us per matrix, 925 of the gradient's 1,530 us on 50,000 nodes, and the
// products 130; here both layers' products take 31 us and the sum 7. A run's loads are issued
// together: left to the compiler they were waited for step by step (35 and 37 us).
constexpr int kRun = 64;

// Layer 1: W1s (16 rows, from X), W1n (16 rows, from A0), b1. Each wave has 16 of the outputs.
__global__ __launch_bounds__(256) void k_wgrad1(const float* __restrict__ X, const float* __restrict__ A0,
                                                const float* __restrict__ dZ1, int n, double* __restrict__ part) {
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4, b = threadIdx.x >> 6;
    double sum[2][4] = {}, bias = 0.0;
    for (long long i0 = (long long)blockIdx.x * kRun; i0 < n; i0 += (long long)gridDim.x * kRun) {
        f32x4 acc[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
        float bs = 0.0f;
        // the run's loads together, then its products
        float x[kRun / 4], a0[kRun / 4], z[kRun / 4];
#pragma unroll
        for (int st = 0; st < kRun / 4; ++st) {
            const size_t r = (size_t)min(i0 + 4 * st + g, (long long)n - 1);
            x[st] = X[r * kIn + j];
            a0[st] = A0[r * kIn + j];
            z[st] = dZ1[r * kHid + 16 * b + j];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int st = 0; st < kRun / 4; ++st) {
            const float zi = i0 + 4 * st + g < n ? z[st] : 0.0f;
            acc[0] = mfma(x[st], zi, acc[0]);
            acc[1] = mfma(a0[st], zi, acc[1]);
            bs += zi;
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[a][r] += (double)acc[a][r];
        bias += (double)bs;
    }
    double* out = part + (size_t)blockIdx.x * kGrad1;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(16 * a + 4 * g + r) * kHid + 16 * b + j] = sum[a][r];
    bias += __shfl_xor(bias, 16, 64);
    bias += __shfl_xor(bias, 32, 64);
    if (g == 0) out[2 * kIn * kHid + 16 * b + j] = bias;
}

// Layer 2 and head: W2s (64 rows, from H1), W2n (64 rows, from A1), b2, Wo, bo. Each wave has 32
// of the rows, and one of the small sums.
__global__ __launch_bounds__(256) void k_wgrad2(const float* __restrict__ H1, const float* __restrict__ A1,
                                                const float* __restrict__ H2, const float2* __restrict__ dY, int n,
                                                const unsigned short* __restrict__ Wo, double* __restrict__ part) {
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float* src = wave < 2 ? H1 : A1;
    const int c0 = 32 * (wave & 1);
    float2 wo[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
        wo[b] = make_float2(bf16_to_f32(Wo[2 * (16 * b + j)]), bf16_to_f32(Wo[2 * (16 * b + j) + 1]));
    double sum[2][4][4] = {}, small[8] = {};
    for (long long i0 = (long long)blockIdx.x * kRun; i0 < n; i0 += (long long)gridDim.x * kRun) {
        f32x4 acc[2][4];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0, 0, 0, 0};
        float sm[8] = {};
        constexpr int kPart = 8;                         // steps whose loads go together
        for (int s0 = 0; s0 < kRun / 4; s0 += kPart) {
            float2 dy[kPart];
            float x0[kPart], x1[kPart], h[kPart][4];
#pragma unroll
            for (int st = 0; st < kPart; ++st) {
                const size_t r = (size_t)min(i0 + 4 * (s0 + st) + g, (long long)n - 1);
                dy[st] = dY[r];
                x0[st] = src[r * kHid + c0 + j];
                x1[st] = src[r * kHid + c0 + 16 + j];
#pragma unroll
                for (int b = 0; b < 4; ++b) h[st][b] = H2[r * kHid + 16 * b + j];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < kPart; ++st) {
                const float2 d = i0 + 4 * (s0 + st) + g < n ? dy[st] : make_float2(0.0f, 0.0f);
                float z[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    z[b] = d_z2(h[st][b], d, wo[b]);       // 0 past the last node
                    acc[0][b] = mfma(x0[st], z[b], acc[0][b]);
                    acc[1][b] = mfma(x1[st], z[b], acc[1][b]);
                }
                if (wave == 0) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) sm[b] += z[b];
                } else if (wave == 1) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        sm[2 * b] = fmaf(h[st][b], d.x, sm[2 * b]);
                        sm[2 * b + 1] = fmaf(h[st][b], d.y, sm[2 * b + 1]);
                    }
                } else if (wave == 2) {
                    sm[0] += d.x;
                    sm[1] += d.y;
                }
            }
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[a][b][r] += (double)acc[a][b][r];
#pragma unroll
        for (int q = 0; q < 8; ++q) small[q] += (double)sm[q];
    }
    double* out = part + (size_t)blockIdx.x * kGrad2;
    const int row0 = 32 * wave;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(row0 + 16 * a + 4 * g + r) * kHid + 16 * b + j] = sum[a][b][r];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        small[q] += __shfl_xor(small[q], 16, 64);
        small[q] += __shfl_xor(small[q], 32, 64);
    }
    if (g != 0) return;
    double* b2 = out + 2 * kHid * kHid;
    if (wave == 0) {
#pragma unroll
        for (int b = 0; b < 4; ++b) b2[16 * b + j] = small[b];
    } else if (wave == 1) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            b2[kHid + 2 * (16 * b + j)] = small[2 * b];
            b2[kHid + 2 * (16 * b + j) + 1] = small[2 * b + 1];
        }
    } else if (wave == 2 && j == 0) {
        b2[kHid + 2 * kHid] = small[0];
        b2[kHid + 2 * kHid + 1] = small[1];
    }
}

// grad[p] = the sum of parameter p's partials, in FP64 and a fixed order: 64 parameters per block,
// four runs of the partials each.
__global__ __launch_bounds__(256) void k_sum_grad(const double* __restrict__ part1, const double* __restrict__ part2,
                                                  int nb, float* __restrict__ grad) {
    __shared__ double red[4][64];
    const int p = blockIdx.x * 64 + (threadIdx.x & 63), run = threadIdx.x >> 6;
    double s = 0.0;
    if (p < kParams) {
        const double* src = p < kGrad1 ? part1 + p : part2 + (p - kGrad1);
        const size_t len = p < kGrad1 ? kGrad1 : kGrad2;
        const int b1 = nb * (run + 1) / 4;
#pragma unroll 8
        for (int b = nb * run / 4; b < b1; ++b) s += src[b * len];
    }
    red[run][threadIdx.x & 63] = s;
    __syncthreads();
    if (run == 0 && p < kParams)
        grad[p] = (float)(((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x]);
}

// Adam on the FP32 masters, then the BF16 copies.
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, unsigned short* __restrict__ wb, int len, float lr,
                                              float b1, float b2, float c1, float c2, float eps) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= len) return;
    const float gt = g[t];
    const float mt = b1 * m[t] + (1.0f - b1) * gt;
    const float vt = b2 * v[t] + (1.0f - b2) * gt * gt;
    m[t] = mt;
    v[t] = vt;
    const float wt = w[t] - lr * (mt / c1) / (sqrtf(vt / c2) + eps);
    w[t] = wt;
    wb[t] = f32_to_bf16(wt);
}

__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ w, int len, unsigned short* __restrict__ wb) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < len) wb[t] = f32_to_bf16(w[t]);
}

// Output scaled to the layout size: xy = s * (Y - mean Y) / rms, with mean / rms from
// per-block partials summed in a fixed order.
__global__ __launch_bounds__(256) void k_ystats(const float* __restrict__ Y, int n, double* __restrict__ part) {
    __shared__ double a[256], b[256], c[256];
    double sx = 0.0, sy = 0.0, sq = 0.0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const double x = Y[2 * i], y = Y[2 * i + 1];
        sx += x;
        sy += y;
        sq += x * x + y * y;
    }
    a[threadIdx.x] = sx;
    b[threadIdx.x] = sy;
    c[threadIdx.x] = sq;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            a[threadIdx.x] += a[threadIdx.x + o];
            b[threadIdx.x] += b[threadIdx.x + o];
            c[threadIdx.x] += c[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x] = a[0];
        part[3 * blockIdx.x + 1] = b[0];
        part[3 * blockIdx.x + 2] = c[0];
    }
}

__global__ __launch_bounds__(256) void k_place(const float* __restrict__ Y, int n, const double* __restrict__ part,
                                               int nb, float scale, float2* __restrict__ xy) {
    __shared__ float coef[3];
    if (threadIdx.x < 64) {
        double sx = 0.0, sy = 0.0, sq = 0.0;
        for (int b = threadIdx.x; b < nb; b += 64) {
            sx += part[3 * b];
            sy += part[3 * b + 1];
            sq += part[3 * b + 2];
        }
        sx = wave_sum(sx, 1);
        sy = wave_sum(sy, 1);
        sq = wave_sum(sq, 1);
        const double mx = sx / n, my = sy / n;
        const double var = sq / n - mx * mx - my * my;
        if (threadIdx.x == 0) {
            coef[0] = (float)mx;
            coef[1] = (float)my;
            coef[2] = var > 0 ? (float)(scale / sqrt(var)) : scale;
        }
    }
    __syncthreads();
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        xy[i] = make_float2((Y[2 * i] - coef[0]) * coef[2], (Y[2 * i + 1] - coef[1]) * coef[2]);
}

int blocks_for(long long work) {
    long long b = (work + 255) / 256;
    return (int)(b < 1 ? 1 : b);
}

// Waves of 16 nodes; at most the four blocks per compute unit that the weights' LDS lets run at a
// time (each stages the weights once).
int dense_blocks(int n) {
    const int b = (n + 63) / 64;
    return b < 1024 ? b : 1024;
}

template <int F, int MODE>
void aggregate(const MpnnGraph& g, const float* in, float* out, hipStream_t st, const float* P = nullptr,
               const float* H = nullptr) {
    const AggArgs A{g.rowptr, g.col, g.n, g.medium, g.nmedium, g.heavy_row, g.chunks, g.nchunks, in, P, H, out, g.part};
    const int light = (int)(((long long)g.n * (F / 4 * kAggSlots<F>) + 255) / 256), medium = (g.nmedium + 3) / 4;
    k_agg<F, MODE><<<light + medium + g.nchunks, 256, 0, st>>>(A, light, medium);
    if (g.nheavy > 0) k_agg_heavy<F, MODE><<<(g.nheavy + 3) / 4, 256, 0, st>>>(A, g.heavy_c0, g.nheavy);
}

}  // namespace

void mpnn_agg_plan(const int* rowptr, int n, std::vector<int>& medium, std::vector<int>& heavy_row,
                   std::vector<int>& heavy_c0, std::vector<int2>& chunks) {
    medium.clear();
    heavy_row.clear();
    heavy_c0.assign(1, 0);
    chunks.clear();
    for (int i = 0; i < n; ++i) {
        const int e0 = rowptr[i], len = rowptr[i + 1] - e0;
        if (len <= kAggLight) continue;
        if (len <= kAggHeavy) {
            medium.push_back(i);
            continue;
        }
        for (int e = 0; e < len; e += kAggChunk) chunks.push_back(make_int2((int)heavy_row.size(), e0 + e));
        heavy_row.push_back(i);
        heavy_c0.push_back((int)chunks.size());
    }
}

void mpnn_features(const MpnnGraph& g, unsigned long long seed, int steps, MpnnScratch& s, hipStream_t st) {
    const int n = g.n;
    k_normal_fields<<<blocks_for((long long)n * 8), 256, 0, st>>>(n, seed, s.z0);
    float* a = s.z0;
    float* b = s.z1;
    for (int k = 0; k < steps; ++k) {
        aggregate<8, kAggSmooth>(g, a, b, st);
        float* t = a;
        a = b;
        b = t;
    }
    const int nb = (n + 127) / 128 < kStatBlocks ? (n + 127) / 128 : kStatBlocks;
    k_colstats<<<nb, 256, 0, st>>>(g.rowptr, a, n, s.dpart);
    k_colnorm_finish<<<1, 64 * kStat, 0, st>>>(s.dpart, nb, n, s.musd);
    k_features<<<blocks_for((long long)n * 4), 256, 0, st>>>(g.rowptr, a, n, s.musd, g.X);
    aggregate<kIn, kAggMean>(g, g.X, g.A0, st);
}

void mpnn_forward(const MpnnGraph& g, const MpnnWeights& w, MpnnScratch& s, bool keep, hipStream_t st) {
    const int n = g.n;
    const int db = dense_blocks(n);
    k_dense<kIn, false><<<db, 256, 0, st>>>(g.X, g.A0, n, w.bf + kOffW1s, w.bf + kOffW1n, w.bf + kOffB1, s.H1, nullptr,
                                            nullptr, nullptr);
    aggregate<kHid, kAggMean>(g, s.H1, s.A1, st);
    k_dense<kHid, true><<<db, 256, 0, st>>>(s.H1, s.A1, n, w.bf + kOffW2s, w.bf + kOffW2n, w.bf + kOffB2,
                                            keep ? s.H2 : nullptr, w.bf + kOffWo, w.bf + kOffBo,
                                            reinterpret_cast<float2*>(s.Y));
}

int mpnn_loss_backward(const MpnnGraph& g, const MpnnWeights& w, MpnnScratch& s, const int* d_offs, int R,
                       double* loss, hipStream_t st) {
    const int n = g.n;
    const long long pairs = (long long)g.nnz + 2ll * R * n;
    const double inv = 1.0 / (double)pairs;
    const int lb = (n + 31) / 32 < kLossBlocks ? (n + 31) / 32 : kLossBlocks;
    float2* dY = reinterpret_cast<float2*>(s.dY);
    k_loss<<<lb, 256, 0, st>>>(g.rowptr, g.col, n, reinterpret_cast<const float2*>(s.Y),
                               reinterpret_cast<const float2*>(g.T), d_offs, R, inv, dY, s.dpart);
    // layer 2 and head
    const int runs = (n + kRun - 1) / kRun, nb = runs < kGradBlocks ? runs : kGradBlocks;
    k_wgrad2<<<nb, 256, 0, st>>>(s.H1, s.A1, s.H2, dY, n, w.bf + kOffWo, s.part2);
    // dZ1 = (dZ2 W2s^T + agg^T(dZ2 W2n^T)) masked by H1 > 0
    k_back<<<dense_blocks(n), 256, 0, st>>>(dY, s.H2, n, g.rowptr, w.bf + kOffWo, w.bf + kOffW2s, w.bf + kOffW2n, s.P,
                                            s.Q);
    aggregate<kHid, kAggBack>(g, s.Q, s.dZ1, st, s.P, s.H1);
    // layer 1
    k_wgrad1<<<nb, 256, 0, st>>>(g.X, g.A0, s.dZ1, n, s.part1);
    k_sum_grad<<<(kParams + 63) / 64, 256, 0, st>>>(s.part1, s.part2, nb, w.grad);
    if (loss) {
        std::vector<double> h((size_t)lb);
        if (hipMemcpyAsync(h.data(), s.dpart, sizeof(double) * lb, hipMemcpyDeviceToHost, st) != hipSuccess) return -1;
        if (hipStreamSynchronize(st) != hipSuccess) return -1;
        double L = 0.0;
        for (double v : h) L += v;
        *loss = L;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

void mpnn_adam(MpnnWeights& w, float lr, int step, hipStream_t st) {
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    k_adam<<<blocks_for(kParams), 256, 0, st>>>(w.master, w.grad, w.m, w.v, w.bf, kParams, lr, b1, b2, c1, c2, 1e-8f);
}

void mpnn_sync_bf16(MpnnWeights& w, hipStream_t st) { k_to_bf16<<<blocks_for(kParams), 256, 0, st>>>(w.master, kParams, w.bf); }

void mpnn_place(const MpnnGraph& g, MpnnScratch& s, float scale, float2* xy, hipStream_t st) {
    const int nb = 128;
    k_ystats<<<nb, 256, 0, st>>>(s.Y, g.n, s.dpart);
    k_place<<<blocks_for(g.n) < 1024 ? blocks_for(g.n) : 1024, 256, 0, st>>>(s.Y, g.n, s.dpart, nb, scale, xy);
}

}  // namespace gfa2
