// C ABI of the learned initialiser (include/gfa2.h, gfa2_mpnn_*).
#include "engine_internal.h"
#include "mpnn_internal.h"
#include "../../include/gfa2.h"

#include <algorithm>
#include <cmath>
#include <new>
#include <type_traits>
#include <utility>
#include <vector>

using namespace gfa2;

static_assert(kAggLight == kAttrLight && kAggHeavy == kAttrHeavy && kAggChunk == kAttrChunk,
              "the engine's lists of rows are used as they are");

namespace {
struct GraphBlock {
    char* p = nullptr;
    size_t bytes = 0;
};
// A released graph's memory is kept for the next graph of the handle up to this size. Allocating and
// freeing the 160 MB of an R-MAT 2^20 graph (20M entries) in nine pieces, with its row lists built
// here from offsets read back, took 1.8 of the 3.5 ms of its learned start.
constexpr size_t kSpareKeep = 256u << 20;
}  // namespace

struct gfa2_mpnn {
    int device = 0;
    hipStream_t stream = nullptr;
    MpnnWeights w;
    MpnnScratch s;
    std::vector<MpnnGraph> graphs;
    std::vector<void*> allocs;          // weights and scratch
    std::vector<GraphBlock> blocks;     // each graph's device memory
    GraphBlock spare;                   // a released graph's, for the next one
    int adam_step = 0;
    int* offs = nullptr;                // training offsets, steps x R
    long long offs_cap = 0;
};

namespace {

int st_of(hipError_t e) {
    if (e == hipSuccess) return GFA2_OK;
    if (e != hipErrorOutOfMemory) return GFA2_ERR_HIP;
    (void)hipGetLastError();            // reported here: not again by the next call
    return GFA2_ERR_OOM;
}

#define MP_TRY(expr)                           \
    do {                                       \
        hipError_t _e = (expr);                \
        if (_e != hipSuccess) return st_of(_e); \
    } while (0)

template <typename T>
int mp_alloc(std::vector<void*>& list, T** p, size_t count) {
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, sizeof(T) * (count ? count : 1));
    if (e != hipSuccess) return st_of(e);
    list.push_back(q);
    *p = static_cast<T*>(q);
    return GFA2_OK;
}

struct SplitMix {
    uint64_t x;
    uint64_t next() {
        uint64_t z = (x += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    double uniform() { return (double)(next() >> 11) * (1.0 / 9007199254740992.0); }
};

void drop_spare(gfa2_mpnn* m) {
    if (m->spare.p) (void)hipFree(m->spare.p);
    m->spare = GraphBlock{};
}

void free_scratch(MpnnScratch& s) {
    for (float** p : {&s.z0, &s.z1, &s.H1, &s.A1, &s.H2, &s.Y, &s.dY, &s.P, &s.Q, &s.dZ1}) {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
    }
    s.cap = 0;
}

// Scratch for n nodes, before every use of it (it grows and never shrinks, but is gone after a
// growth that found no memory, so that the next graph finds all of the memory there is).
int ensure_scratch(gfa2_mpnn* m, int n) {
    MpnnScratch& s = m->s;
    if (n <= s.cap) return GFA2_OK;
    drop_spare(m);
    free_scratch(s);
    hipError_t e = hipSuccess;
    auto take = [&](float*& p, size_t width) {
        if (e == hipSuccess) e = hipMalloc(&p, sizeof(float) * (size_t)n * width);
        if (e != hipSuccess) p = nullptr;
    };
    take(s.z0, 8);
    take(s.z1, 8);
    take(s.H1, kHid);
    take(s.A1, kHid);
    take(s.H2, kHid);
    take(s.Y, 2);
    take(s.dY, 2);
    take(s.P, kHid);
    take(s.Q, kHid);
    take(s.dZ1, kHid);
    if (e == hipSuccess) s.cap = n;
    else free_scratch(s);
    return st_of(e);
}

// Room for the training offsets.
int ensure_offsets(gfa2_mpnn* m, long long count) {
    if (count <= m->offs_cap) return GFA2_OK;
    if (m->offs) (void)hipFree(m->offs);
    m->offs = nullptr;
    m->offs_cap = 0;
    const hipError_t e = hipMalloc(&m->offs, sizeof(int) * (size_t)count);
    if (e == hipSuccess) m->offs_cap = count;
    else m->offs = nullptr;
    return st_of(e);
}

// The block's work is done. The larger of it and the spare one is kept.
void give_back(gfa2_mpnn* m, GraphBlock& b) {
    if (b.bytes <= kSpareKeep && b.bytes > m->spare.bytes) std::swap(b, m->spare);
    if (b.p) (void)hipFree(b.p);
    b = GraphBlock{};
}

// The spare block if it is large enough and at least half of it is used.
int take_block(gfa2_mpnn* m, size_t bytes, GraphBlock& b) {
    if (m->spare.bytes >= bytes && m->spare.bytes / 2 <= bytes) {
        std::swap(b, m->spare);
        return GFA2_OK;
    }
    drop_spare(m);
    void* p = nullptr;
    const hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) return st_of(e);
    b.p = static_cast<char*>(p);
    b.bytes = bytes;
    return GFA2_OK;
}

// One block for all of a graph's arrays (n, nnz, nmedium, nheavy and nchunks are set).
int lay_out(gfa2_mpnn* m, MpnnGraph& g, bool target, GraphBlock& b) {
    size_t at = 0;
    auto place = [&](auto*& p, size_t count) {
        p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(b.p ? b.p + at : nullptr);
        at += (sizeof(*p) * count + 255) / 256 * 256;
    };
    auto all = [&]() {
        const size_t n = (size_t)g.n;
        at = 0;
        place(g.rowptr, n + 1);
        place(g.col, (size_t)g.nnz);
        place(g.medium, (size_t)g.nmedium + g.nheavy);
        g.heavy_row = g.medium ? g.medium + g.nmedium : nullptr;
        place(g.heavy_c0, (size_t)g.nheavy + 1);
        place(g.chunks, (size_t)g.nchunks);
        place(g.part, (size_t)g.nchunks * 4 * kHid);
        place(g.X, n * kIn);
        place(g.A0, n * kIn);
        if (target) place(g.T, n * 2);
    };
    all();
    const int st = take_block(m, at, b);
    if (st == GFA2_OK) all();
    return st;
}

// A new graph's block: given back unless the graph is kept.
struct NewBlock {
    gfa2_mpnn* m;
    GraphBlock b;
    explicit NewBlock(gfa2_mpnn* m_) : m(m_) {}
    ~NewBlock() {
        if (!b.p) return;
        (void)hipStreamSynchronize(m->stream);
        give_back(m, b);
    }
    int keep(const MpnnGraph& g) {
        m->graphs.push_back(g);
        m->blocks.push_back(b);
        b = GraphBlock{};
        return (int)m->graphs.size() - 1;
    }
};

int check_graph(const gfa2_mpnn* m, int id) {
    if (!m || id < 0 || id >= (int)m->graphs.size() || m->graphs[id].n == 0) return GFA2_ERR_INVALID_ARG;
    return GFA2_OK;
}

}  // namespace

extern "C" {

int32_t gfa2_mpnn_num_params(void) { return kParams; }

int gfa2_mpnn_create(int device, uint64_t seed, gfa2_mpnn_t* out) {
    if (!out) return GFA2_ERR_INVALID_ARG;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return GFA2_ERR_NO_DEVICE;
    if (device < 0 || device >= count) return GFA2_ERR_INVALID_ARG;
    MP_TRY(hipSetDevice(device));
    gfa2_mpnn* m = new (std::nothrow) gfa2_mpnn();
    if (!m) return GFA2_ERR_OOM;
    m->device = device;
    int st = GFA2_OK;
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess ||
        (st = mp_alloc(m->allocs, &m->w.master, kParams)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->w.bf, kParams)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->w.grad, kParams)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->w.m, kParams)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->w.v, kParams)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->s.dpart, kPartDoubles)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->s.musd, 2 * kIn)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->s.part1, (size_t)kGradBlocks * kGrad1)) != GFA2_OK ||
        (st = mp_alloc(m->allocs, &m->s.part2, (size_t)kGradBlocks * kGrad2)) != GFA2_OK) {
        gfa2_mpnn_destroy(m);
        return st != GFA2_OK ? st : GFA2_ERR_HIP;
    }
    // Glorot-uniform weights (fan_in + fan_out of each matrix), zero biases.
    std::vector<float> w(kParams, 0.0f);
    SplitMix rng{seed};
    auto fill = [&](int off, int fan_in, int fan_out, int rows_used) {
        const double a = std::sqrt(6.0 / (fan_in + fan_out));
        for (int k = 0; k < rows_used; ++k)
            for (int o = 0; o < fan_out; ++o) w[off + k * fan_out + o] = (float)((2.0 * rng.uniform() - 1.0) * a);
    };
    fill(kOffW1s, 9, kHid, 9);
    fill(kOffW1n, 9, kHid, 9);
    fill(kOffW2s, kHid, kHid, kHid);
    fill(kOffW2n, kHid, kHid, kHid);
    fill(kOffWo, kHid, 2, kHid);
    st = gfa2_mpnn_set_params(m, w.data());
    if (st != GFA2_OK) {
        gfa2_mpnn_destroy(m);
        return st;
    }
    *out = m;
    return GFA2_OK;
}

int gfa2_mpnn_set_params(gfa2_mpnn_t m, const float* params) {
    if (!m || !params) return GFA2_ERR_INVALID_ARG;
    MP_TRY(hipSetDevice(m->device));
    MP_TRY(hipMemcpyAsync(m->w.master, params, sizeof(float) * kParams, hipMemcpyHostToDevice, m->stream));
    MP_TRY(hipMemsetAsync(m->w.m, 0, sizeof(float) * kParams, m->stream));
    MP_TRY(hipMemsetAsync(m->w.v, 0, sizeof(float) * kParams, m->stream));
    mpnn_sync_bf16(m->w, m->stream);
    MP_TRY(hipStreamSynchronize(m->stream));
    m->adam_step = 0;
    return GFA2_OK;
}

int gfa2_mpnn_get_params(gfa2_mpnn_t m, float* params) {
    if (!m || !params) return GFA2_ERR_INVALID_ARG;
    MP_TRY(hipSetDevice(m->device));
    MP_TRY(hipMemcpyAsync(params, m->w.master, sizeof(float) * kParams, hipMemcpyDeviceToHost, m->stream));
    MP_TRY(hipStreamSynchronize(m->stream));
    return GFA2_OK;
}

int gfa2_mpnn_add_graph(gfa2_mpnn_t m, int32_t n, const int64_t* rowptr, const int32_t* col, const float* target_xy,
                        uint64_t feature_seed, int32_t smoothing_steps, int32_t* graph_id) {
    if (!m || !rowptr || n < 1 || smoothing_steps < 0) return GFA2_ERR_INVALID_ARG;
    const int64_t nnz = rowptr[n];
    if (rowptr[0] != 0 || nnz < 0 || nnz >= (int64_t)1 << 31 || (nnz > 0 && !col)) return GFA2_ERR_INVALID_GRAPH;
    std::vector<int> rp((size_t)n + 1);
    for (int v = 0; v <= n; ++v) {
        if (v < n && (rowptr[v + 1] < rowptr[v])) return GFA2_ERR_INVALID_GRAPH;
        rp[v] = (int)rowptr[v];
    }
    for (int64_t e = 0; e < nnz; ++e)
        if (col[e] < 0 || col[e] >= n) return GFA2_ERR_INVALID_GRAPH;
    MP_TRY(hipSetDevice(m->device));
    int st = ensure_scratch(m, n);
    if (st != GFA2_OK) return st;
    MpnnGraph g;
    g.n = n;
    g.nnz = nnz;
    std::vector<int> medium, heavy_row, heavy_c0;
    std::vector<int2> chunks;
    mpnn_agg_plan(rp.data(), n, medium, heavy_row, heavy_c0, chunks);
    g.nmedium = (int)medium.size();
    g.nheavy = (int)heavy_row.size();
    g.nchunks = (int)chunks.size();
    medium.insert(medium.end(), heavy_row.begin(), heavy_row.end());
    std::vector<float> t;               // the target, copied by the stream
    NewBlock mine(m);                   // drains the stream before the vectors go
    if ((st = lay_out(m, g, target_xy != nullptr, mine.b)) != GFA2_OK) return st;
    auto upload = [&](void* to, const void* from, size_t bytes) {
        return bytes ? hipMemcpyAsync(to, from, bytes, hipMemcpyHostToDevice, m->stream) : hipSuccess;
    };
    MP_TRY(upload(g.rowptr, rp.data(), sizeof(int) * ((size_t)n + 1)));
    MP_TRY(upload(g.col, col, sizeof(int) * (size_t)nnz));
    MP_TRY(upload(g.medium, medium.data(), sizeof(int) * medium.size()));
    MP_TRY(upload(g.heavy_c0, heavy_c0.data(), sizeof(int) * heavy_c0.size()));
    MP_TRY(upload(g.chunks, chunks.data(), sizeof(int2) * chunks.size()));
    if (target_xy) {
        // centre and scale to unit RMS radius
        double cx = 0.0, cy = 0.0;
        for (int i = 0; i < n; ++i) {
            cx += target_xy[2 * i];
            cy += target_xy[2 * i + 1];
        }
        cx /= n;
        cy /= n;
        double r2 = 0.0;
        for (int i = 0; i < n; ++i) {
            const double dx = target_xy[2 * i] - cx, dy = target_xy[2 * i + 1] - cy;
            r2 += dx * dx + dy * dy;
        }
        const double rms = std::sqrt(r2 / n);
        t.resize((size_t)2 * n);
        for (int i = 0; i < n; ++i) {
            t[2 * i] = (float)((target_xy[2 * i] - cx) / (rms > 0 ? rms : 1.0));
            t[2 * i + 1] = (float)((target_xy[2 * i + 1] - cy) / (rms > 0 ? rms : 1.0));
        }
        g.target_scale = (float)rms;
        MP_TRY(hipMemcpyAsync(g.T, t.data(), sizeof(float) * 2 * n, hipMemcpyHostToDevice, m->stream));
    }
    mpnn_features(g, feature_seed, smoothing_steps, m->s, m->stream);
    MP_TRY(hipGetLastError());
    MP_TRY(hipStreamSynchronize(m->stream));
    const int id = mine.keep(g);
    if (graph_id) *graph_id = id;
    return GFA2_OK;
}

int gfa2_mpnn_add_engine_graph(gfa2_mpnn_t m, gfa2_handle h, uint64_t feature_seed, int32_t smoothing_steps,
                               int32_t* graph_id) {
    if (!m || !h || smoothing_steps < 0) return GFA2_ERR_INVALID_ARG;
    EngineView v;
    if (!engine_view(h, &v)) return GFA2_ERR_NO_GRAPH;
    if (v.nseg > 1) return GFA2_ERR_UNSUPPORTED;
    if (v.device != m->device) return GFA2_ERR_INVALID_ARG;
    MP_TRY(hipSetDevice(m->device));
    const int n = v.n;
    int st = ensure_scratch(m, n);
    if (st != GFA2_OK) return st;
    MpnnGraph g;
    g.n = n;
    g.nnz = v.nnz;
    g.nmedium = v.nmedium;
    g.nheavy = v.nheavy;
    g.nchunks = v.nchunks;
    NewBlock mine(m);
    if ((st = lay_out(m, g, false, mine.b)) != GFA2_OK) return st;
    // the engine's CSR was validated when it was set; it and the engine's lists of rows, which are
    // those of the aggregation, are copied device to device after the engine's queued work
    MP_TRY(hipStreamSynchronize(v.stream));
    auto copy = [&](void* to, const void* from, size_t bytes) {
        return bytes ? hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToDevice, m->stream) : hipSuccess;
    };
    MP_TRY(copy(g.rowptr, v.rowptr, sizeof(int) * ((size_t)n + 1)));
    MP_TRY(copy(g.col, v.col, sizeof(int) * (size_t)g.nnz));
    MP_TRY(copy(g.medium, v.medium, sizeof(int) * ((size_t)g.nmedium + g.nheavy)));
    if (g.nheavy > 0) {
        MP_TRY(copy(g.heavy_c0, v.chunk0, sizeof(int) * ((size_t)g.nheavy + 1)));
        MP_TRY(copy(g.chunks, v.chunks, sizeof(int2) * (size_t)g.nchunks));
    }
    mpnn_features(g, feature_seed, smoothing_steps, m->s, m->stream);
    MP_TRY(hipGetLastError());
    MP_TRY(hipStreamSynchronize(m->stream));
    const int id = mine.keep(g);
    if (graph_id) *graph_id = id;
    return GFA2_OK;
}

int gfa2_mpnn_release_graph(gfa2_mpnn_t m, int32_t graph_id) {
    int st = check_graph(m, graph_id);
    if (st != GFA2_OK) return st;
    MP_TRY(hipSetDevice(m->device));
    MP_TRY(hipStreamSynchronize(m->stream));
    give_back(m, m->blocks[graph_id]);
    m->graphs[graph_id] = MpnnGraph{};     // n = 0, no target: skipped by training, rejected by id
    return GFA2_OK;
}

int gfa2_mpnn_features(gfa2_mpnn_t m, int32_t graph_id, float* X) {
    int st = check_graph(m, graph_id);
    if (st != GFA2_OK || !X) return st != GFA2_OK ? st : GFA2_ERR_INVALID_ARG;
    const MpnnGraph& g = m->graphs[graph_id];
    MP_TRY(hipSetDevice(m->device));
    MP_TRY(hipMemcpy(X, g.X, sizeof(float) * (size_t)g.n * kIn, hipMemcpyDeviceToHost));
    return GFA2_OK;
}

int gfa2_mpnn_loss_grad(gfa2_mpnn_t m, int32_t graph_id, const int32_t* offsets, int32_t R, double* loss, float* grad) {
    int st = check_graph(m, graph_id);
    if (st != GFA2_OK) return st;
    const MpnnGraph& g = m->graphs[graph_id];
    if (!g.T || R < 0 || (R > 0 && !offsets)) return GFA2_ERR_INVALID_ARG;
    for (int k = 0; k < R; ++k)
        if (offsets[k] < 1 || offsets[k] >= g.n) return GFA2_ERR_INVALID_ARG;
    MP_TRY(hipSetDevice(m->device));
    if ((st = ensure_scratch(m, g.n)) != GFA2_OK || (st = ensure_offsets(m, R)) != GFA2_OK) return st;
    if (R) MP_TRY(hipMemcpyAsync(m->offs, offsets, sizeof(int) * R, hipMemcpyHostToDevice, m->stream));
    mpnn_forward(g, m->w, m->s, true, m->stream);
    if (mpnn_loss_backward(g, m->w, m->s, m->offs, R, loss, m->stream) != 0) return GFA2_ERR_HIP;
    if (grad) {
        MP_TRY(hipMemcpyAsync(grad, m->w.grad, sizeof(float) * kParams, hipMemcpyDeviceToHost, m->stream));
        MP_TRY(hipStreamSynchronize(m->stream));
    }
    return GFA2_OK;
}

int gfa2_mpnn_train(gfa2_mpnn_t m, int32_t steps, float lr, int32_t R, uint64_t seed, double* last_loss) {
    if (!m || steps < 0 || R < 0) return GFA2_ERR_INVALID_ARG;
    std::vector<int> ids;
    for (size_t k = 0; k < m->graphs.size(); ++k)
        if (m->graphs[k].T) ids.push_back((int)k);
    if (ids.empty()) return GFA2_ERR_NO_GRAPH;
    MP_TRY(hipSetDevice(m->device));
    // all steps' offsets drawn up front (seeded) and uploaded once
    SplitMix rng{seed};
    std::vector<int> offs((size_t)steps * (R > 0 ? R : 1), 1);
    for (int s = 0; s < steps; ++s) {
        const int n = m->graphs[ids[s % ids.size()]].n;
        for (int k = 0; k < R; ++k) offs[(size_t)s * R + k] = n > 1 ? 1 + (int)(rng.next() % (uint64_t)(n - 1)) : 1;
    }
    int most = 0;
    for (int k : ids) most = std::max(most, m->graphs[k].n);
    int st = ensure_scratch(m, most);
    if (st != GFA2_OK || (st = ensure_offsets(m, (long long)offs.size())) != GFA2_OK) return st;
    MP_TRY(hipMemcpyAsync(m->offs, offs.data(), sizeof(int) * offs.size(), hipMemcpyHostToDevice, m->stream));
    for (int s = 0; s < steps; ++s) {
        const MpnnGraph& g = m->graphs[ids[s % ids.size()]];
        mpnn_forward(g, m->w, m->s, true, m->stream);
        double* lp = (s == steps - 1) ? last_loss : nullptr;
        if (mpnn_loss_backward(g, m->w, m->s, m->offs + (size_t)s * R, R, lp, m->stream) != 0) return GFA2_ERR_HIP;
        mpnn_adam(m->w, lr, ++m->adam_step, m->stream);
    }
    MP_TRY(hipGetLastError());
    MP_TRY(hipStreamSynchronize(m->stream));
    return GFA2_OK;
}

float gfa2_mpnn_target_scale(gfa2_mpnn_t m) {
    if (!m) return 0.0f;
    double s = 0.0;
    int c = 0;
    for (const MpnnGraph& g : m->graphs)
        if (g.T) {
            s += g.target_scale;
            ++c;
        }
    return c ? (float)(s / c) : 0.0f;
}

int gfa2_mpnn_infer(gfa2_mpnn_t m, int32_t graph_id, float scale, float* xy) {
    int st = check_graph(m, graph_id);
    if (st != GFA2_OK || !xy) return st != GFA2_OK ? st : GFA2_ERR_INVALID_ARG;
    const MpnnGraph& g = m->graphs[graph_id];
    MP_TRY(hipSetDevice(m->device));
    if ((st = ensure_scratch(m, g.n)) != GFA2_OK) return st;
    mpnn_forward(g, m->w, m->s, false, m->stream);
    mpnn_place(g, m->s, scale, reinterpret_cast<float2*>(m->s.dY), m->stream);
    MP_TRY(hipMemcpyAsync(xy, m->s.dY, sizeof(float) * 2 * g.n, hipMemcpyDeviceToHost, m->stream));
    MP_TRY(hipStreamSynchronize(m->stream));
    return GFA2_OK;
}

int gfa2_mpnn_infer_to_engine(gfa2_mpnn_t m, int32_t graph_id, float scale, gfa2_handle h) {
    int st = check_graph(m, graph_id);
    if (st != GFA2_OK) return st;
    EngineView v;
    if (!engine_view(h, &v)) return GFA2_ERR_NO_GRAPH;
    const MpnnGraph& g = m->graphs[graph_id];
    if (v.n != g.n || v.device != m->device) return GFA2_ERR_INVALID_ARG;
    MP_TRY(hipSetDevice(m->device));
    if ((st = ensure_scratch(m, g.n)) != GFA2_OK) return st;
    MP_TRY(hipStreamSynchronize(v.stream));
    mpnn_forward(g, m->w, m->s, false, m->stream);
    mpnn_place(g, m->s, scale, v.pos, m->stream);
    MP_TRY(hipGetLastError());
    MP_TRY(hipStreamSynchronize(m->stream));
    return engine_positions_written(h);
}

int gfa2_mpnn_destroy(gfa2_mpnn_t m) {
    if (!m) return GFA2_ERR_INVALID_ARG;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    for (const GraphBlock& b : m->blocks)
        if (b.p) (void)hipFree(b.p);
    drop_spare(m);
    for (void* p : m->allocs) (void)hipFree(p);
    free_scratch(m->s);
    if (m->offs) (void)hipFree(m->offs);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return GFA2_OK;
}

}  // extern "C"
