// Shapes, parameter layout and buffers of the learned-initialisation network.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

namespace gfa2 {

constexpr int kIn = 16;      // input features (9 used, zero padded)
constexpr int kHid = 64;     // hidden width
// Parameter layout (FP32 masters and BF16 copies share it): W[k][o] row-major.
constexpr int kOffW1s = 0;
constexpr int kOffW1n = kOffW1s + kIn * kHid;
constexpr int kOffB1 = kOffW1n + kIn * kHid;
constexpr int kOffW2s = kOffB1 + kHid;
constexpr int kOffW2n = kOffW2s + kHid * kHid;
constexpr int kOffB2 = kOffW2n + kHid * kHid;
constexpr int kOffWo = kOffB2 + kHid;
constexpr int kOffBo = kOffWo + kHid * 2;
constexpr int kParams = kOffBo + 2;

// Gradient partials: layer 1 (W1s, W1n, b1) and layer 2 with the head (W2s, W2n, b2, Wo, bo).
constexpr int kGrad1 = kOffW2s;
constexpr int kGrad2 = kParams - kOffW2s;
constexpr int kGradBlocks = 256;
constexpr int kLossBlocks = 2048;
constexpr int kPartDoubles = 8192;

// Rows of up to kAggLight entries are aggregated by a few lanes each, up to kAggHeavy by a wave
// each, longer ones in chunks of kAggChunk entries, a block each.
constexpr int kAggLight = 32;
constexpr int kAggHeavy = 2048;
constexpr int kAggChunk = 4096;

struct MpnnGraph {
    int n = 0;
    long long nnz = 0;
    int* rowptr = nullptr;
    int* col = nullptr;
    int nmedium = 0;            // rows of more than kAggLight entries up to kAggHeavy
    int nheavy = 0;             // longer ones
    int nchunks = 0;
    int* medium = nullptr;      // [nmedium]
    int* heavy_row = nullptr;   // [nheavy]
    int* heavy_c0 = nullptr;    // [nheavy + 1] first chunk of each heavy row
    int2* chunks = nullptr;     // [nchunks] {index into heavy_row, first entry}
    float* part = nullptr;      // [4 nchunks x kHid] partial sums, one per quarter of a chunk
    float* X = nullptr;     // [n x kIn] features
    float* A0 = nullptr;    // [n x kIn] mean_agg(X)
    float* T = nullptr;     // [n x 2] normalised target, or null
    float target_scale = 0.0f;
};

struct MpnnWeights {
    float* master = nullptr;
    unsigned short* bf = nullptr;
    float* grad = nullptr;
    float* m = nullptr;
    float* v = nullptr;
};

struct MpnnScratch {
    int cap = 0;            // nodes the buffers hold
    float *z0 = nullptr, *z1 = nullptr;
    double* dpart = nullptr;    // kPartDoubles: column statistics, loss partials
    float* musd = nullptr;      // 2 * kIn
    float *H1 = nullptr, *A1 = nullptr, *H2 = nullptr, *Y = nullptr, *dY = nullptr;
    float *P = nullptr, *Q = nullptr, *dZ1 = nullptr;
    double *part1 = nullptr, *part2 = nullptr;  // kGradBlocks x kGrad1 and kGrad2: weight-gradient partials
};

// Host side: the medium and heavy rows and the chunk list of a CSR given by its row offsets.
void mpnn_agg_plan(const int* rowptr, int n, std::vector<int>& medium, std::vector<int>& heavy_row,
                   std::vector<int>& heavy_c0, std::vector<int2>& chunks);
void mpnn_features(const MpnnGraph& g, unsigned long long seed, int steps, MpnnScratch& s, hipStream_t st);
// keep: H2 is written too (the backward pass reads it).
void mpnn_forward(const MpnnGraph& g, const MpnnWeights& w, MpnnScratch& s, bool keep, hipStream_t st);
int mpnn_loss_backward(const MpnnGraph& g, const MpnnWeights& w, MpnnScratch& s, const int* d_offs, int R,
                       double* loss, hipStream_t st);
void mpnn_adam(MpnnWeights& w, float lr, int step, hipStream_t st);
void mpnn_sync_bf16(MpnnWeights& w, hipStream_t st);
void mpnn_place(const MpnnGraph& g, MpnnScratch& s, float scale, float2* xy, hipStream_t st);

}  // namespace gfa2
