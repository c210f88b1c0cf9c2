// The engine behind include/gfa2.h: one handle = one layout instance with its own HIP
// stream, device buffers and device-resident FA2 state (the reference keeps that state
// in __device__ globals, src/RPFA2Kernels.cu:28-33 and src/RPBHKernels.cu:53-62, which
// allows one instance per process).
#include "engine_internal.h"
#include "../../include/gfa2.h"

#include <algorithm>
#include <cstdio>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <vector>

using namespace gfa2;

namespace {

const char* const kGroupNames[] = {"attraction", "keys", "sort", "tree", "walk", "combine", "speed", "displacement"};
constexpr int kGroups = 8;
// Timing events recorded per iteration, and the pair of events that brackets each group. The
// attraction's pair is recorded on the stream it runs on (the second stream when it runs beside
// the walk); "combine" is the wait for that stream plus k_combine (empty on one stream).
// Events 0 and 11 bracket the whole iteration.
constexpr int kEvents = 12;
constexpr int kSpan[kGroups][2] = {{1, 2}, {3, 4}, {4, 5}, {5, 6}, {7, 8}, {8, 9}, {9, 10}, {10, 11}};
constexpr int kWalkGroup = 4;

}  // namespace

struct gfa2_engine {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t side = nullptr;         // the attraction's stream (default priority, like `stream`)
    hipEvent_t fork = nullptr;          // stream -> side: the iteration's inputs are in place
    hipEvent_t join = nullptr;          // side -> stream: the attraction + gravity is written
    gfa2_params user{};
    Params p{};
    Bufs b{};
    bool has_graph = false;
    bool has_pos = false;
    long long edges = 0;
    bool capture_rep = false;
    float2* rep_buf = nullptr;          // repulsion of the last captured iteration (kept when capture stops)
    float* ew_buf = nullptr;            // w^delta per CSR entry, once weights were given
    std::vector<void*> allocs;
    // timing
    int timing = 0;                     // 0, GFA2_TIMING_GROUPS or GFA2_TIMING_WALK
    std::vector<hipEvent_t> events;     // pool, kEvents per pending iteration
    int pending = 0;                    // iterations with recorded, unread events
    double acc_ms[kGroups] = {0};
    long long timed_iters = 0;
    // graph capture
    bool use_graph = false;
    bool graph_valid = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    // layout-quality pairs (gfa2_stress_setup)
    int stress_K = 0, stress_T = 0;
    int* stress_src = nullptr;
    int* stress_tgt = nullptr;
    int* stress_dist = nullptr;
    double* stress_part = nullptr;
    float2* stress_pos = nullptr;
    // graphs of a batch (one for a single graph)
    std::vector<int> node_off_host;
    int groups_cap = 0;
    // the lowest path-key sort pass launched: one below the lowest the device ran when the host
    // last read its state (a full sort after new positions or parameters)
    int sort_first = 0;
    // workspace of calls that need scratch (EngineScratch)
    std::mutex scratch_mu;
    void* scratch = nullptr;
    size_t scratch_bytes = 0;
    // launch shapes (autotuned per graph-size bucket)
    int cus = 256;
    LaunchConfig tune{256, 8, 0, 0};
};

namespace {

// Process-wide autotuning results: graph-size bucket floor(log2 V) -> launch shapes.
std::mutex g_tune_mu;
std::map<int, LaunchConfig> g_tune_table;

int size_bucket(int n) {
    int b = 0;
    while ((2ll << b) <= n) ++b;
    return b;
}

// Parameter checks shared by gfa2_create and gfa2_set_params.
int validate_params(const gfa2_params& p) {
    if (p.prevent_overlap) return GFA2_ERR_UNSUPPORTED;
    if (p.group_size != 32 && p.group_size != 64) return GFA2_ERR_INVALID_ARG;
    if (!(p.theta > 0.0f) || !(p.epssq >= 0.0f)) return GFA2_ERR_INVALID_ARG;
    if (!std::isfinite(p.edge_weight_influence)) return GFA2_ERR_INVALID_ARG;
    return GFA2_OK;
}

void apply_tune(gfa2_engine* h) {
    h->p.walk_bt = h->tune.walk_bt;
    h->b.grid_cap = h->tune.blocks_per_cu * h->cus;
    h->b.attr_grid = h->tune.attraction_bpc * h->cus;
}

}  // namespace

namespace {

int hip_status(hipError_t e) {
    if (e == hipSuccess) return GFA2_OK;
    if (e != hipErrorOutOfMemory) return GFA2_ERR_HIP;
    (void)hipGetLastError();            // reported here: not again by the next call
    return GFA2_ERR_OOM;
}

#define GFA2_TRY(expr)                       \
    do {                                     \
        hipError_t _e = (expr);              \
        if (_e != hipSuccess) return hip_status(_e); \
    } while (0)

template <typename T>
int dalloc(gfa2_engine* h, T** ptr, size_t count) {
    void* p = nullptr;
    size_t bytes = sizeof(T) * (count ? count : 1);
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) return hip_status(e);
    h->allocs.push_back(p);
    *ptr = static_cast<T*>(p);
    return GFA2_OK;
}

void free_all(gfa2_engine* h) {
    if (h->gexec) { hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { hipGraphDestroy(h->graph); h->graph = nullptr; }
    h->graph_valid = false;
    for (void* p : h->allocs) hipFree(p);
    h->allocs.clear();
    if (h->scratch) hipFree(h->scratch);
    h->scratch = nullptr;
    h->scratch_bytes = 0;
    h->b = Bufs{};
    h->rep_buf = nullptr;
    h->ew_buf = nullptr;
    h->has_graph = false;
    h->has_pos = false;
    h->stress_K = h->stress_T = 0;
    h->stress_src = h->stress_tgt = h->stress_dist = nullptr;
    h->stress_part = nullptr;
    h->stress_pos = nullptr;
}

// splitmix64: the engine's own seeded generator for pair sampling.
struct SplitMix {
    uint64_t x;
    uint64_t next() {
        uint64_t z = (x += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    uint64_t below(uint64_t r) { return next() % r; }
};

constexpr int kStressBlocks = 512;

// Whether the launch shape says where the attraction runs: not where it is part of a small graph's
// one launch, nor beside all pairs.
bool attraction_placed(const gfa2_engine* h) { return !h->p.exact && !small_tree(h->b); }

void enqueue_iteration(gfa2_engine* h, hipEvent_t* ev) {
    hipStream_t s = h->stream;
    Bufs& b = h->b;
    // with GFA2_TIMING_WALK only the walk's pair is recorded (each mark costs a little)
    auto mark = [&](int i, hipStream_t on) {
        if (ev && (h->timing != GFA2_TIMING_WALK || i == kSpan[kWalkGroup][0] || i == kSpan[kWalkGroup][1]))
            hipEventRecord(ev[i], on);
    };
    // Gravity + attraction reads only the positions, which nothing in the iteration writes
    // before the displacement, and writes only F_ga, which only the walk's epilogue reads. So it
    // can run on a second stream: beside the walk (mode 1: the walk is launched split and
    // k_combine forms F afterwards, as the fused epilogue would), or beside keys, sort and tree
    // (mode 2: joined before the walk).
    // A small graph's tree is one launch that carries the attraction along, in every mode.
    const bool small = !h->p.exact && small_tree(b);
    const int mode = attraction_placed(h) ? h->tune.attraction_stream : 0;
    auto attraction_on_side = [&]() {
        hipEventRecord(h->fork, s);
        hipStreamWaitEvent(h->side, h->fork, 0);
        mark(1, h->side);
        launch_attraction(b, h->p, false, h->side);
        mark(2, h->side);
        hipEventRecord(h->join, h->side);
    };
    mark(0, s);
    // one launch with the keys, unless it has a grid or blocks of its own or their times are asked
    // for one by one
    const bool apart = ev && h->timing != GFA2_TIMING_WALK;
    const bool keyed = mode == 0 && !h->p.exact && !small && !apart && b.attr_grid == 0 && !attract_wide(b);
    if (mode == 0) {
        mark(1, s);
        if (!small && !keyed) launch_attraction(b, h->p, true, s);
        mark(2, s);
    } else if (mode == 2) {
        attraction_on_side();
    }
    mark(3, s);
    if (!h->p.exact && !small) {
        if (b.nseg > 1) {
            if (!advance_seg(b)) launch_seg_bbox(b, s);
            if (keyed) launch_seg_keys_attraction(b, h->p, s);
            else launch_seg_keys(b, s);
        } else {
            if (keyed) launch_keys_attraction(b, h->p, h->sort_first, s);
            else launch_keys(b, h->sort_first, s);
        }
    }
    mark(4, s);
    if (!h->p.exact && !small) {
        if (b.nseg > 1 && b.max_seg <= kSegSortMax) {
            // every graph fits one block's sort: by (graph, key) in one launch, the low passes
            // skipped as for one graph; the result is in buffer 0 and runs stop at graphs
            segmented_sort_pairs(b.sort, b.node_off, b.seg_order, b.nseg, b.max_seg, b.large_segs, s, b.st);
            launch_sort_fixup(b.sort, b.n, b.st, s, 0, true, b.seg_of);
        } else {
            // the previous tree's depth bounds the key bits the order needs (skipped low passes
            // are made up for by the fix-up, so the order is the full sort's whatever the depth)
            // a single graph's keys start where the passes that run end in buffer 0
            const bool lead = b.nseg == 1;
            radix_sort_pairs(b.sort, b.n, 0, 64, s, b.st, h->sort_first, lead, b.sort.hist_in_keys);
            launch_sort_fixup(b.sort, b.n, b.st, s, h->sort_first, lead, nullptr, b.sort.hist_in_keys);
            if (b.nseg > 1) launch_seg_graph_sort(b, s);
        }
    }
    mark(5, s);
    if (small) launch_small_tree(b, h->p, s);
    else if (!h->p.exact) launch_tree(b, s);
    mark(6, s);
    if (mode == 1) attraction_on_side();
    if (mode == 2) hipStreamWaitEvent(s, h->join, 0);
    mark(7, s);
    if (h->p.exact) launch_exact(b, h->p, s);
    else launch_walk(b, h->p, mode == 1, s);
    mark(8, s);
    if (mode == 1) {
        hipStreamWaitEvent(s, h->join, 0);
        launch_combine(b, h->p, s);
    }
    mark(9, s);
    launch_speed(b, s);
    mark(10, s);
    launch_displacement(b, s);
    mark(11, s);
}

// Reads back the events of completed timed iterations.
int drain_timing(gfa2_engine* h) {
    if (h->pending == 0) return GFA2_OK;
    GFA2_TRY(hipStreamSynchronize(h->stream));
    for (int it = 0; it < h->pending; ++it) {
        hipEvent_t* ev = &h->events[(size_t)it * kEvents];
        for (int g = 0; g < kGroups; ++g) {
            if (h->timing == GFA2_TIMING_WALK && g != kWalkGroup) continue;
            float ms = 0.0f;
            GFA2_TRY(hipEventElapsedTime(&ms, ev[kSpan[g][0]], ev[kSpan[g][1]]));
            h->acc_ms[g] += ms;
        }
    }
    h->timed_iters += h->pending;
    h->pending = 0;
    return GFA2_OK;
}

int reset_state(gfa2_engine* h) {
    launch_reset(h->b, h->user.global_speed, h->user.speed_efficiency, h->user.jitter_tolerance, h->user.k_s_max,
                 h->stream);
    GFA2_TRY(hipGetLastError());
    GFA2_TRY(hipStreamSynchronize(h->stream));
    return GFA2_OK;
}

int build_groups(gfa2_engine* h);

// New positions or parameters: the previous tree's depth says nothing about the next one, so
// the next path-key sort sorts every key bit.
void invalidate_graph(gfa2_engine* h) {
    h->graph_valid = false;
    if (h->gexec) { (void)hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
}

// The passes the host launches follow the device's choice, as last read, with one pass to
// spare (fewer passes than the device asks for only lengthen the fix-up's runs; the order is
// the same). A change of launches needs a new captured graph.
void set_sort_first(gfa2_engine* h, int first) {
    if (first == h->sort_first) return;
    h->sort_first = first;
    invalidate_graph(h);
}

// New positions: the next sort is a full one, and so are those of the following
// kFullSortsAfterNew iterations. The first steps from a fresh layout move bodies the most, so a
// tree would underestimate the next one's tied runs (at R-MAT 2^24 from a random start, the
// second iteration's runs took the fix-up 31 ms).
constexpr int kFullSortsAfterNew = 3;

// The positions on the device are new ones.
void positions_changed(gfa2_engine* h) {
    set_sort_first(h, 0);
    launch_new_positions(h->b, kFullSortsAfterNew, h->stream);
}

hipError_t full_sort_next(gfa2_engine* h) {
    set_sort_first(h, 0);
    hipError_t e = hipMemsetAsync(&h->b.st->sort_skip, 0, sizeof(int), h->stream);
    if (e == hipSuccess) e = hipMemsetD32Async((hipDeviceptr_t)&h->b.st->full_sorts, kFullSortsAfterNew, 1, h->stream);
    return e;
}

// The ABI status of the device error word (tree overflow first: it is the one a caller can
// act on, with a larger cell_factor).
int device_error(int err) {
    if (err & kErrTreeOverflow) return GFA2_ERR_TREE_OVERFLOW;
    if (err & kErrSortWait) return GFA2_ERR_DEVICE_WAIT;
    return GFA2_OK;
}

// Copies DevState back (waits for the stream).
int read_state(gfa2_engine* h, DevState* st) {
    GFA2_TRY(hipMemcpyAsync(st, h->b.st, sizeof(DevState), hipMemcpyDeviceToHost, h->stream));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    // (a small graph's sort is inside its tree's launch)
    if (!small_tree(h->b)) set_sort_first(h, std::max(0, std::min(st->sort_skip, 7) - 1));
    return GFA2_OK;
}

}  // namespace

extern "C" {

void gfa2_default_params(gfa2_params* p) {
    if (!p) return;
    p->use_barneshut = 1;
    p->strong_gravity = 0;
    p->gravity = 1.0f;
    p->scale = 1.0f;
    p->theta = 1.0f;
    p->epssq = (float)(0.05 * 0.05);
    p->jitter_tolerance = 1.0f;
    p->k_s_max = 10.0f;
    p->global_speed = 1.0f;
    p->speed_efficiency = 1.0f;
    p->group_size = 32;
    p->cell_factor = 0;
    p->linlog = 0;
    p->edge_weight_influence = 0.0f;   // src/RPForceAtlas2.cpp:49
    p->prevent_overlap = 0;
}

int gfa2_device_info(int device, int32_t* cus, int32_t* wave, int64_t* mem_bytes) {
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return GFA2_ERR_NO_DEVICE;
    if (device < 0 || device >= count) return GFA2_ERR_INVALID_ARG;
    hipDeviceProp_t prop;
    GFA2_TRY(hipGetDeviceProperties(&prop, device));
    if (cus) *cus = prop.multiProcessorCount;
    if (wave) *wave = prop.warpSize;
    if (mem_bytes) *mem_bytes = (int64_t)prop.totalGlobalMem;
    return GFA2_OK;
}

int gfa2_create(const gfa2_params* params, int device, gfa2_handle* out) {
    if (!out) return GFA2_ERR_INVALID_ARG;
    *out = nullptr;
    gfa2_params prm;
    if (params) prm = *params;
    else gfa2_default_params(&prm);
    const int valid = validate_params(prm);
    if (valid != GFA2_OK) return valid;
    if (prm.cell_factor < 0) return GFA2_ERR_INVALID_ARG;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return GFA2_ERR_NO_DEVICE;
    if (device < 0 || device >= count) return GFA2_ERR_INVALID_ARG;
    hipDeviceProp_t prop;
    GFA2_TRY(hipGetDeviceProperties(&prop, device));
    // The kernels are written for 64-lane wavefronts (the reference likewise refuses any
    // warp size but its own, src/RPGPUForceAtlas2.cu:90-95).
    if (prop.warpSize != 64) return GFA2_ERR_UNSUPPORTED;
    GFA2_TRY(hipSetDevice(device));
    gfa2_engine* h = new (std::nothrow) gfa2_engine();
    if (!h) return GFA2_ERR_OOM;
    h->device = device;
    h->user = prm;
    h->p.strong_gravity = prm.strong_gravity;
    h->p.k_g = prm.gravity;
    h->p.k_r = prm.scale;
    h->p.itolsq = 1.0f / (prm.theta * prm.theta);
    h->p.epssq = prm.epssq;
    h->p.group = prm.group_size;
    h->p.exact = prm.use_barneshut ? 0 : 1;
    h->p.linlog = prm.linlog ? 1 : 0;
    h->cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    hipError_t e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&h->side, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&h->fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&h->join, hipEventDisableTiming);
    if (e != hipSuccess) {
        if (h->fork) (void)hipEventDestroy(h->fork);
        if (h->side) (void)hipStreamDestroy(h->side);
        if (h->stream) (void)hipStreamDestroy(h->stream);
        delete h;
        return hip_status(e);
    }
    *out = h;
    return GFA2_OK;
}

int gfa2_set_params(gfa2_handle h, const gfa2_params* prm) {
    if (!h || !prm) return GFA2_ERR_INVALID_ARG;
    const int valid = validate_params(*prm);
    if (valid != GFA2_OK) return valid;
    const bool new_delta = prm->edge_weight_influence != h->user.edge_weight_influence;
    const int keep_factor = h->user.cell_factor;
    h->user = *prm;
    h->user.cell_factor = keep_factor;   // capacity is fixed by set_graph
    h->p.strong_gravity = prm->strong_gravity;
    h->p.k_g = prm->gravity;
    h->p.k_r = prm->scale;
    h->p.itolsq = 1.0f / (prm->theta * prm->theta);
    h->p.epssq = prm->epssq;
    h->p.exact = prm->use_barneshut ? 0 : 1;
    h->p.linlog = prm->linlog ? 1 : 0;
    const bool regroup = h->p.group != prm->group_size;
    h->p.group = prm->group_size;
    if (regroup && h->has_graph) {
        const int rc = build_groups(h);
        if (rc != GFA2_OK) return rc;
    }
    if (h->has_graph) {
        GFA2_TRY(hipSetDevice(h->device));
        GFA2_TRY(full_sort_next(h));
    }
    if (new_delta && h->b.ew) {
        GFA2_TRY(hipSetDevice(h->device));
        launch_edge_weights(h->b, prm->edge_weight_influence, h->stream);
        GFA2_TRY(hipGetLastError());
        GFA2_TRY(hipStreamSynchronize(h->stream));
    }
    h->graph_valid = false;
    if (h->gexec) { (void)hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
    return GFA2_OK;
}

}  // extern "C"

namespace {

// Walk groups: per graph, runs of G sorted positions starting at the graph's first.
int build_groups(gfa2_engine* h) {
    Bufs& b = h->b;
    const int G = h->p.group;
    std::vector<int2> groups;
    std::vector<int> first((size_t)b.nseg + 1);
    for (int g = 0; g < b.nseg; ++g) {
        first[g] = (int)groups.size();
        for (int k = h->node_off_host[g]; k < h->node_off_host[g + 1]; k += G) groups.push_back(make_int2(k, g));
    }
    first[b.nseg] = (int)groups.size();
    if ((int)groups.size() > h->groups_cap) return GFA2_ERR_INVALID_ARG;
    b.ngroups = (int)groups.size();
    GFA2_TRY(hipMemcpyAsync(b.groups, groups.data(), sizeof(int2) * groups.size(), hipMemcpyHostToDevice, h->stream));
    GFA2_TRY(hipMemcpyAsync(b.grp_first, first.data(), sizeof(int) * first.size(), hipMemcpyHostToDevice, h->stream));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    return GFA2_OK;
}

// Validates a symmetric CSR whose edges stay inside their graph, allocates every buffer and
// uploads the graph. node_off: nseg+1 node offsets (nseg = 1 for a single graph).
int set_graph_impl(gfa2_engine* h, int32_t n, const int64_t* rowptr, const int32_t* col, const float* mass,
                   int nseg, const int32_t* node_off) {
    // bodies and cells share the 27-bit record index space: up to 2^26 bodies
    if (n < 1 || n > (1 << 26) || nseg < 1 || nseg > n) return GFA2_ERR_INVALID_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    if (rowptr[0] != 0) return GFA2_ERR_INVALID_GRAPH;
    if (node_off[0] != 0 || node_off[nseg] != n) return GFA2_ERR_INVALID_GRAPH;
    for (int g = 0; g < nseg; ++g)
        if (node_off[g + 1] <= node_off[g]) return GFA2_ERR_INVALID_GRAPH;
    const int64_t nnz = rowptr[n];
    if (nnz < 0 || nnz >= (int64_t)1 << 31 || (nnz > 0 && !col)) return GFA2_ERR_INVALID_GRAPH;
    std::vector<int> rp32((size_t)n + 1);
    std::vector<int> lists;
    lists.reserve(n);
    std::vector<int> medium, heavy, seg_of;
    std::vector<float> m((size_t)n);
    if (nseg > 1) seg_of.resize(n);
    int g = 0;
    for (int v = 0; v < n; ++v) {
        while (v >= node_off[g + 1]) ++g;
        if (nseg > 1) seg_of[v] = g;
        const int64_t a = rowptr[v], e1 = rowptr[v + 1];
        if (e1 < a || e1 > nnz) return GFA2_ERR_INVALID_GRAPH;
        for (int64_t e = a; e < e1; ++e)
            if (col[e] < node_off[g] || col[e] >= node_off[g + 1] || col[e] == v) return GFA2_ERR_INVALID_GRAPH;
        rp32[v] = (int)a;
        const int64_t deg = e1 - a;
        if (deg <= kAttrLight) lists.push_back(v);
        else if (deg <= kAttrHeavy) medium.push_back(v);
        else heavy.push_back(v);
        m[v] = mass ? mass[v] : (float)(deg + 1.0);
    }
    rp32[n] = (int)nnz;
    const int nlight = (int)lists.size();
    lists.insert(lists.end(), medium.begin(), medium.end());
    lists.insert(lists.end(), heavy.begin(), heavy.end());
    std::vector<int2> attr_chunks;
    std::vector<int> attr_c0(1, 0);
    for (size_t q = 0; q < heavy.size(); ++q) {
        for (int e = rp32[heavy[q]]; e < (int)rowptr[heavy[q] + 1]; e += kAttrChunk) attr_chunks.push_back(make_int2((int)q, e));
        attr_c0.push_back((int)attr_chunks.size());
    }

    free_all(h);
    const int factor = h->user.cell_factor > 0 ? h->user.cell_factor : 3;
    long long cap = (long long)n + (long long)factor * n + 1024;
    if (cap > kMaxRecords) cap = kMaxRecords;
    if ((long long)n * 3 / 2 + 2 > cap) return GFA2_ERR_UNSUPPORTED;
    Bufs& b = h->b;
    b.n = n;
    b.nnz = nnz;
    b.cap_records = (int)cap;
    b.nseg = nseg;
    b.seg_bits = 0;
    while ((1 << b.seg_bits) < nseg) ++b.seg_bits;
    h->node_off_host.assign(node_off, node_off + nseg + 1);
    int groups_cap = 0;
    for (int q = 0; q < nseg; ++q) groups_cap += (node_off[q + 1] - node_off[q] + 31) / 32;
    h->groups_cap = groups_cap;
    const int sort_tiles = (n + kSortTile - 1) / kSortTile;
    const int tree_tiles = (n + kTreeTile - 1) / kTreeTile;
    int st = GFA2_OK;
#define GFA2_ALLOC(ptr, cnt) \
    if ((st = dalloc(h, &(ptr), (cnt))) != GFA2_OK) { free_all(h); return st; }
    GFA2_ALLOC(b.pos, n);
    GFA2_ALLOC(b.mass, n);
    GFA2_ALLOC(b.rowptr, (size_t)n + 1);
    GFA2_ALLOC(b.col, (size_t)nnz);
    GFA2_ALLOC(b.node_lists, n);
    GFA2_ALLOC(b.attr_chunks, attr_chunks.size());
    GFA2_ALLOC(b.attr_c0, attr_c0.size());
    GFA2_ALLOC(b.attr_part, attr_chunks.size());
    GFA2_ALLOC(b.rank, n);
    GFA2_ALLOC(b.col_rank, (size_t)nnz);
    GFA2_ALLOC(b.pos_rank, n);
    GFA2_ALLOC(b.fga, n);
    GFA2_ALLOC(b.f, n);
    GFA2_ALLOC(b.fprev, n);
    GFA2_ALLOC(b.sort.keys[0], n);
    GFA2_ALLOC(b.sort.keys[1], n);
    GFA2_ALLOC(b.sort.vals[0], n);
    GFA2_ALLOC(b.sort.vals[1], n);
    GFA2_ALLOC(b.sort.hist, (size_t)256 * sort_tiles);
    GFA2_ALLOC(b.sort.rowtot, 256);
    GFA2_ALLOC(b.sort.digit_hist, 8 * 256);
    // one graph sorted with one launch per pass: k_keys counts the digits into a table that
    // starts clear and that every iteration's fix-up clears again
    b.sort.hist_in_keys = nseg == 1 && sort_onesweep(b.sort, n);
    GFA2_TRY(hipMemsetAsync(b.sort.digit_hist, 0, sizeof(unsigned int) * 8 * 256, h->stream));
    GFA2_ALLOC(b.sort.status, (size_t)256 * sort_tiles);
    GFA2_ALLOC(b.sort.ticket, 1);
    // no tile has published counts, ticket 0
    GFA2_TRY(hipMemsetAsync(b.sort.status, 0, sizeof(unsigned int) * 256 * (size_t)sort_tiles, h->stream));
    GFA2_TRY(hipMemsetAsync(b.sort.ticket, 0, sizeof(unsigned long long), h->stream));
    GFA2_ALLOC(b.rec, (size_t)cap);
    GFA2_ALLOC(b.kids, (size_t)cap);
    GFA2_ALLOC(b.sbody, n);
    GFA2_ALLOC(b.pm, n);
    GFA2_ALLOC(b.rcount, (size_t)cap);
    GFA2_ALLOC(b.bbox_part, kPartBlocks);
    GFA2_ALLOC(b.st, 1);
    // a sort wait that runs out raises the instance's error word, so every later kernel of the
    // iteration skips and gfa2_sync reports it (cleared by reset_state)
    b.sort.err = &b.st->err;
    GFA2_ALLOC(b.node_off, (size_t)nseg + 1);
    GFA2_ALLOC(b.seg_root, nseg);
    GFA2_ALLOC(b.rec_begin, (size_t)nseg + 1);
    GFA2_ALLOC(b.groups, groups_cap);
    GFA2_ALLOC(b.grp_first, (size_t)nseg + 1);
    GFA2_ALLOC(b.seg_st, nseg);
    GFA2_ALLOC(b.seg_cur, 1);
    GFA2_ALLOC(b.grp_part, groups_cap);
    if (nseg > 1) {
        int* so = nullptr;
        GFA2_ALLOC(so, n);
        b.seg_of = so;
        GFA2_ALLOC(b.sg, n);
        GFA2_ALLOC(b.pkey, n);
        GFA2_TRY(hipMemcpyAsync(so, seg_of.data(), sizeof(int) * n, hipMemcpyHostToDevice, h->stream));
        // a graph's sorted positions are its own node range, so sorted position -> graph is
        // the node -> graph table (the global sort path rewrites it each iteration)
        GFA2_TRY(hipMemcpyAsync(b.sg, seg_of.data(), sizeof(int) * n, hipMemcpyHostToDevice, h->stream));
        // graphs by decreasing node count, for the per-graph sort
        std::vector<int> order((size_t)nseg);
        for (int g = 0; g < nseg; ++g) order[g] = g;
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
            return node_off[x + 1] - node_off[x] > node_off[y + 1] - node_off[y];
        });
        b.max_seg = node_off[order[0] + 1] - node_off[order[0]];
        b.large_segs = 0;
        for (int q : order) b.large_segs += node_off[q + 1] - node_off[q] > kSegSmall;
        GFA2_ALLOC(b.seg_order, nseg);
        GFA2_TRY(hipMemcpyAsync(b.seg_order, order.data(), sizeof(int) * nseg, hipMemcpyHostToDevice, h->stream));
        GFA2_TRY(hipStreamSynchronize(h->stream));   // order goes out of scope
    }
    h->rep_buf = nullptr;
    if (h->capture_rep) {
        GFA2_ALLOC(h->rep_buf, n);
        b.rep = h->rep_buf;
    }
    {
        double total = 0.0;
        bool whole = true;
        for (int v = 0; v < n && whole; ++v) {
            whole = m[v] >= 0.0f && m[v] < 16777216.0f && m[v] == std::floor(m[v]);
            total += m[v];
        }
        b.int_mass = whole && total < 16777216.0 * 62.0;
        // no cell (a part of one graph) can reach 2^24
        b.no_big = total < 16777216.0;
    }
    if (small_tree(b)) {
        b.kids_blocks = 1;
        b.sort.hist_in_keys = false;
        if (b.int_mass) {
            GFA2_ALLOC(b.pmass, (size_t)n + 1);
        } else {
            GFA2_ALLOC(b.cell_lvl, (size_t)(cap - n));
        }
    } else {
        b.kids_blocks = 2 * tree_tiles;
        GFA2_ALLOC(b.lcp, (size_t)tree_tiles * kTreeTile);      // read by whole tiles
        GFA2_ALLOC(b.blocksum, tree_tiles);
        GFA2_ALLOC(b.chunk_sum, (tree_tiles + kTileChunk - 1) / kTileChunk);
        GFA2_ALLOC(b.S, (size_t)n + 1);
        // the tables of the crossing cells
        const size_t slots = ((size_t)tree_tiles * kCrossMax + 1) / 2 * 2, groups = ((size_t)tree_tiles + 15) / 16 * 16;
        char* tables = nullptr;
        GFA2_ALLOC(tables, slots * (sizeof(int4) + sizeof(Moment)) + groups * (sizeof(int) + 1));
        b.cross = reinterpret_cast<int4*>(tables);
        b.cross_sum = reinterpret_cast<Moment*>(b.cross + slots);
        b.ncross = reinterpret_cast<int*>(b.cross_sum + slots);
        b.tmin = reinterpret_cast<signed char*>(b.ncross + groups);
        if (b.int_mass) {
            GFA2_ALLOC(b.pmass, (size_t)n / 16 + 1);
            GFA2_ALLOC(b.bmass, tree_tiles);
            GFA2_ALLOC(b.chunk_mass, (tree_tiles + kTileChunk - 1) / kTileChunk);
            GFA2_ALLOC(b.big_rc, kMaxBig);
            GFA2_ALLOC(b.big_lvl, kMaxBig);
        } else {
            GFA2_ALLOC(b.spill, 66 * ((size_t)cap / 4096 + 8));   // (33 slots per block, fewer in all for the groups)
        }
    }
    GFA2_ALLOC(b.kids_part, (size_t)b.kids_blocks * 8);
#undef GFA2_ALLOC
    b.cus = h->cus;
    b.nlight = nlight;
    b.nmedium = (int)medium.size();
    b.nheavy = (int)heavy.size();
    GFA2_TRY(hipMemcpyAsync(b.rowptr, rp32.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, h->stream));
    if (nnz > 0)
        GFA2_TRY(hipMemcpyAsync(b.col, col, sizeof(int) * nnz, hipMemcpyHostToDevice, h->stream));
    GFA2_TRY(hipMemcpyAsync(b.mass, m.data(), sizeof(float) * n, hipMemcpyHostToDevice, h->stream));
    GFA2_TRY(hipMemcpyAsync(b.node_lists, lists.data(), sizeof(int) * n, hipMemcpyHostToDevice, h->stream));
    b.nattr_chunks = (int)attr_chunks.size();
    if (!attr_chunks.empty())
        GFA2_TRY(hipMemcpyAsync(b.attr_chunks, attr_chunks.data(), sizeof(int2) * attr_chunks.size(), hipMemcpyHostToDevice,
                                h->stream));
    GFA2_TRY(hipMemcpyAsync(b.attr_c0, attr_c0.data(), sizeof(int) * attr_c0.size(), hipMemcpyHostToDevice, h->stream));
    {
        // rank = position in the order of decreasing degree (ties by id), by counting sort
        int maxdeg = 0;
        for (int v = 0; v < n; ++v) maxdeg = std::max(maxdeg, rp32[v + 1] - rp32[v]);
        std::vector<int> start((size_t)maxdeg + 2, 0);
        for (int v = 0; v < n; ++v) ++start[(size_t)(maxdeg - (rp32[v + 1] - rp32[v])) + 1];
        for (int d = 0; d <= maxdeg; ++d) start[(size_t)d + 1] += start[(size_t)d];
        long long hub_entries = 0;
        for (int d = 0; d <= maxdeg && start[(size_t)d] < kWideHubs; ++d)
            hub_entries += (long long)(maxdeg - d) * (std::min(start[(size_t)d + 1], kWideHubs) - start[(size_t)d]);
        b.hub_entries = hub_entries;
        std::vector<int> rank((size_t)n);
        for (int v = 0; v < n; ++v) rank[v] = start[(size_t)(maxdeg - (rp32[v + 1] - rp32[v]))]++;
        GFA2_TRY(hipMemcpyAsync(b.rank, rank.data(), sizeof(int) * n, hipMemcpyHostToDevice, h->stream));
        launch_col_rank(b, h->stream);
        GFA2_TRY(hipStreamSynchronize(h->stream));   // rank goes out of scope
    }
    GFA2_TRY(hipMemcpyAsync(b.node_off, node_off, sizeof(int) * (nseg + 1), hipMemcpyHostToDevice, h->stream));
    GFA2_TRY(hipMemsetAsync(b.pos, 0, sizeof(float2) * n, h->stream));
    GFA2_TRY(hipMemsetAsync(b.kids_part, 0, sizeof(int) * 8 * (size_t)b.kids_blocks, h->stream));
    GFA2_TRY(hipMemsetAsync(b.rec_begin, 0, sizeof(int) * (nseg + 1), h->stream));
    h->edges = nnz / 2;
    h->has_graph = true;
    h->has_pos = false;
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        auto it = g_tune_table.find(size_bucket(n));
        if (it != g_tune_table.end()) h->tune = it->second;
    }
    apply_tune(h);
    st = build_groups(h);
    if (st != GFA2_OK) return st;
    return reset_state(h);
}

}  // namespace

extern "C" {

int gfa2_set_graph(gfa2_handle h, int32_t n, const int64_t* rowptr, const int32_t* col, const float* mass) {
    if (!h || !rowptr) return GFA2_ERR_INVALID_ARG;
    const int32_t off[2] = {0, n};
    return set_graph_impl(h, n, rowptr, col, mass, 1, off);
}

int gfa2_set_graph_batch(gfa2_handle h, int32_t ngraphs, const int32_t* node_off, const int64_t* rowptr,
                         const int32_t* col, const float* mass) {
    if (!h || !rowptr || !node_off || ngraphs < 1) return GFA2_ERR_INVALID_ARG;
    return set_graph_impl(h, node_off[ngraphs], rowptr, col, mass, ngraphs, node_off);
}

int gfa2_get_batch_stats(gfa2_handle h, int32_t cap, float* speed, float* efficiency, double* swing,
                         double* traction, int64_t* interactions) {
    if (!h || cap < 0) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    const int ns = h->b.nseg < cap ? h->b.nseg : cap;
    std::vector<SegState> seg((size_t)h->b.nseg);
    GFA2_TRY(hipMemcpyAsync(seg.data(), h->b.seg_st, sizeof(SegState) * h->b.nseg, hipMemcpyDeviceToHost, h->stream));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    for (int g = 0; g < ns; ++g) {
        if (speed) speed[g] = seg[g].global_speed;
        if (efficiency) efficiency[g] = seg[g].speed_efficiency;
        if (swing) swing[g] = seg[g].swing;
        if (traction) traction[g] = seg[g].traction;
        if (interactions) interactions[g] = (int64_t)seg[g].interactions;
    }
    return GFA2_OK;
}

int gfa2_set_graph_coo(gfa2_handle h, int32_t n, int64_t m, const int32_t* src, const int32_t* dst,
                       const float* mass) {
    if (!h || n < 1 || m < 0 || (m > 0 && (!src || !dst))) return n < 1 ? GFA2_ERR_INVALID_GRAPH : GFA2_ERR_INVALID_ARG;
    std::vector<int64_t> rowptr((size_t)n + 1, 0);
    for (int64_t e = 0; e < m; ++e) {
        if (src[e] < 0 || src[e] >= n || dst[e] < 0 || dst[e] >= n || src[e] == dst[e]) return GFA2_ERR_INVALID_GRAPH;
        rowptr[src[e] + 1]++;
        rowptr[dst[e] + 1]++;
    }
    for (int v = 0; v < n; ++v) rowptr[v + 1] += rowptr[v];
    std::vector<int64_t> cur(rowptr.begin(), rowptr.end() - 1);
    std::vector<int32_t> col((size_t)(2 * m));
    for (int64_t e = 0; e < m; ++e) {
        col[cur[src[e]]++] = dst[e];
        col[cur[dst[e]]++] = src[e];
    }
    return gfa2_set_graph(h, n, rowptr.data(), col.data(), mass);
}

int gfa2_set_positions(gfa2_handle h, const float* xy) {
    if (!h || !xy) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    GFA2_TRY(hipMemcpyAsync(h->b.pos, xy, sizeof(float2) * h->b.n, hipMemcpyHostToDevice, h->stream));
    positions_changed(h);
    GFA2_TRY(hipGetLastError());
    GFA2_TRY(hipStreamSynchronize(h->stream));
    h->has_pos = true;
    return GFA2_OK;
}

int gfa2_get_positions(gfa2_handle h, float* xy) {
    if (!h || !xy) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    GFA2_TRY(hipMemcpyAsync(xy, h->b.pos, sizeof(float2) * h->b.n, hipMemcpyDeviceToHost, h->stream));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    return GFA2_OK;
}

int gfa2_reset(gfa2_handle h) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    return reset_state(h);
}

int gfa2_step(gfa2_handle h, int32_t iters) {
    if (!h || iters < 0) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    if (!h->has_pos) return GFA2_ERR_INVALID_ARG;
    GFA2_TRY(hipSetDevice(h->device));
    if (h->timing) {
        // events are recycled: at most kTimedBatch iterations are pending between reads
        constexpr int kTimedBatch = 1024;
        int left = iters;
        while (left > 0) {
            if (h->pending >= kTimedBatch) {
                const int rc = drain_timing(h);
                if (rc != GFA2_OK) return rc;
            }
            const int now = std::min(left, kTimedBatch - h->pending);
            const size_t need = (size_t)(h->pending + now) * kEvents;
            while (h->events.size() < need) {
                // timing only: no system-scope fence (its cache writeback would slow the
                // kernels between the marks); the stream order and the kernels' own fences
                // are what orders the work
                hipEvent_t e;
                GFA2_TRY(hipEventCreateWithFlags(&e, hipEventDisableSystemFence));
                h->events.push_back(e);
            }
            for (int i = 0; i < now; ++i) {
                enqueue_iteration(h, &h->events[(size_t)(h->pending) * kEvents]);
                h->pending++;
            }
            left -= now;
        }
        GFA2_TRY(hipGetLastError());
        return GFA2_OK;
    }
    if (h->use_graph) {
        if (!h->graph_valid) {
            GFA2_TRY(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
            enqueue_iteration(h, nullptr);
            hipError_t e = hipStreamEndCapture(h->stream, &h->graph);
            if (e != hipSuccess) return hip_status(e);
            GFA2_TRY(hipGraphInstantiate(&h->gexec, h->graph, nullptr, nullptr, 0));
            h->graph_valid = true;
        }
        for (int i = 0; i < iters; ++i) GFA2_TRY(hipGraphLaunch(h->gexec, h->stream));
        return GFA2_OK;
    }
    for (int i = 0; i < iters; ++i) enqueue_iteration(h, nullptr);
    GFA2_TRY(hipGetLastError());
    return GFA2_OK;
}

int gfa2_sync(gfa2_handle h) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_OK;
    GFA2_TRY(hipSetDevice(h->device));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    int rc = drain_timing(h);
    if (rc != GFA2_OK) return rc;
    DevState st;
    rc = read_state(h, &st);
    if (rc != GFA2_OK) return rc;
    return device_error(st.err);
}

int gfa2_get_forces(gfa2_handle h, int32_t kind, float* xy) {
    if (!h || !xy) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    const float2* src = nullptr;
    if (kind == GFA2_FORCE_TOTAL) src = h->b.f;
    else if (kind == GFA2_FORCE_REPULSION) src = h->rep_buf;
    else if (kind == GFA2_FORCE_ATTRACTION_GRAVITY) src = h->b.fga;
    else return GFA2_ERR_INVALID_ARG;
    if (!src) return GFA2_ERR_INVALID_ARG;
    GFA2_TRY(hipMemcpyAsync(xy, src, sizeof(float2) * h->b.n, hipMemcpyDeviceToHost, h->stream));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    return GFA2_OK;
}

int gfa2_set_capture(gfa2_handle h, int32_t on) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    h->capture_rep = on != 0;
    if (h->has_graph && h->capture_rep && !h->rep_buf) {
        GFA2_TRY(hipSetDevice(h->device));
        int st = dalloc(h, &h->rep_buf, h->b.n);
        if (st != GFA2_OK) return st;
        GFA2_TRY(hipMemsetAsync(h->rep_buf, 0, sizeof(float2) * h->b.n, h->stream));
    }
    // the walk writes the repulsion only while capture is on; the last capture stays readable
    if (h->has_graph) h->b.rep = h->capture_rep ? h->rep_buf : nullptr;
    h->graph_valid = false;
    if (h->gexec) { hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { hipGraphDestroy(h->graph); h->graph = nullptr; }
    return GFA2_OK;
}

int gfa2_get_tree(gfa2_handle h, int32_t cap, int32_t* ncells, int32_t* level, int32_t* count, float* mass,
                  float* xy, int32_t* perm) {
    if (!h || cap < 0) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    DevState st;
    int rc = read_state(h, &st);
    if (rc != GFA2_OK) return rc;
    rc = device_error(st.err);
    if (rc != GFA2_OK) return rc;
    const int nrec = st.nrecords;
    std::vector<float4> rec((size_t)std::max(nrec, 1));
    std::vector<int> rcount((size_t)std::max(nrec, 1));
    if (nrec > 0) {
        GFA2_TRY(hipMemcpyAsync(rec.data(), h->b.rec, sizeof(float4) * nrec, hipMemcpyDeviceToHost, h->stream));
        GFA2_TRY(hipMemcpyAsync(rcount.data(), h->b.rcount, sizeof(int) * nrec, hipMemcpyDeviceToHost, h->stream));
    }
    if (perm)
        GFA2_TRY(hipMemcpyAsync(perm, h->b.sort.vals[0], sizeof(int) * h->b.n, hipMemcpyDeviceToHost, h->stream));
    // each graph's root record (a cell stores level - 1, and a root level 0 as 0 too)
    std::vector<int> root((size_t)h->b.nseg + 1, 0);
    GFA2_TRY(hipMemcpyAsync(root.data(), h->b.rec_begin, sizeof(int) * root.size(), hipMemcpyDeviceToHost, h->stream));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    int c = 0;
    size_t g = 0;
    for (int r = 0; r < nrec; ++r) {
        int info;
        memcpy(&info, &rec[r].w, sizeof(int));
        if (info == -1) continue;
        while (g + 1 < root.size() && root[g] < r) ++g;
        if (c < cap) {
            if (level) level[c] = (g < root.size() && root[g] == r) ? 0 : (info & 31) + 1;
            if (count) count[c] = rcount[r];
            if (mass) mass[c] = rec[r].z;
            if (xy) { xy[2 * c] = rec[r].x; xy[2 * c + 1] = rec[r].y; }
        }
        ++c;
    }
    if (ncells) *ncells = c;
    return GFA2_OK;
}

int gfa2_get_stats(gfa2_handle h, gfa2_stats* s) {
    if (!h || !s) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    DevState st;
    int rc = read_state(h, &st);
    if (rc != GFA2_OK) return rc;
    s->iteration = st.iteration;
    s->nodes = h->b.n;
    s->edges = h->edges;
    s->global_speed = st.global_speed;
    s->speed_efficiency = st.speed_efficiency;
    s->swing = st.swing;
    s->traction = st.traction;
    s->interactions = (int64_t)st.interactions;
    {
        // the running totals are kept per graph
        std::vector<SegState> seg((size_t)h->b.nseg);
        GFA2_TRY(hipMemcpyAsync(seg.data(), h->b.seg_st, sizeof(SegState) * seg.size(), hipMemcpyDeviceToHost,
                                h->stream));
        GFA2_TRY(hipStreamSynchronize(h->stream));
        unsigned long long total = 0;
        for (const SegState& q : seg) total += q.interactions_total;
        s->interactions_total = (int64_t)total;
    }
    s->cells = st.ncells;
    s->max_level = st.max_level;
    s->root_x = st.rootx;
    s->root_y = st.rooty;
    s->radius = st.radius;
    s->error_flags = st.err;
    return GFA2_OK;
}

int gfa2_set_timing(gfa2_handle h, int32_t on) {
    if (!h || on < 0 || on > GFA2_TIMING_WALK) return GFA2_ERR_INVALID_ARG;
    if (h->pending) {
        int rc = drain_timing(h);
        if (rc != GFA2_OK) return rc;
    }
    h->timing = on;
    for (double& a : h->acc_ms) a = 0.0;
    h->timed_iters = 0;
    return GFA2_OK;
}

int gfa2_get_timing(gfa2_handle h, int32_t cap, int32_t* count, const char** names, double* ms) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    int rc = drain_timing(h);
    if (rc != GFA2_OK) return rc;
    // the groups the last timed iterations measured
    int k = 0;
    for (int g = 0; g < kGroups; ++g) {
        if (h->timing == GFA2_TIMING_WALK && g != kWalkGroup) continue;
        if (k < cap) {
            if (names) names[k] = kGroupNames[g];
            if (ms) ms[k] = h->timed_iters ? h->acc_ms[g] / (double)h->timed_iters : 0.0;
        }
        ++k;
    }
    if (count) *count = k < cap ? k : cap;
    return GFA2_OK;
}

int gfa2_set_graph_capture(gfa2_handle h, int32_t on) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    h->use_graph = on != 0;
    h->graph_valid = false;
    if (h->gexec) { hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { hipGraphDestroy(h->graph); h->graph = nullptr; }
    return GFA2_OK;
}

int gfa2_set_edge_weights(gfa2_handle h, int64_t count, const float* w) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    Bufs& b = h->b;
    GFA2_TRY(hipSetDevice(h->device));
    if (!w) {
        b.ew = nullptr;                  // buffers stay allocated until the next graph
    } else {
        if (count != b.nnz) return GFA2_ERR_INVALID_ARG;
        for (int64_t e = 0; e < count; ++e)
            if (!(w[e] > 0.0f) || !std::isfinite(w[e])) return GFA2_ERR_INVALID_ARG;
        if (!b.ew_raw) {
            int st = dalloc(h, &b.ew_raw, (size_t)b.nnz);
            if (st == GFA2_OK) st = dalloc(h, &h->ew_buf, (size_t)b.nnz);
            if (st != GFA2_OK) return st;
        }
        GFA2_TRY(hipMemcpyAsync(b.ew_raw, w, sizeof(float) * (size_t)count, hipMemcpyHostToDevice, h->stream));
        b.ew = h->ew_buf;
        launch_edge_weights(b, h->user.edge_weight_influence, h->stream);
        GFA2_TRY(hipGetLastError());
        GFA2_TRY(hipStreamSynchronize(h->stream));
    }
    h->graph_valid = false;
    if (h->gexec) { (void)hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
    return GFA2_OK;
}

int gfa2_set_graph_coo_weighted(gfa2_handle h, int32_t n, int64_t m, const int32_t* src, const int32_t* dst,
                                const float* weight, const float* mass) {
    if (!h || n < 1 || m < 0 || (m > 0 && (!src || !dst || !weight)))
        return n < 1 ? GFA2_ERR_INVALID_GRAPH : GFA2_ERR_INVALID_ARG;
    std::vector<int64_t> rowptr((size_t)n + 1, 0);
    for (int64_t e = 0; e < m; ++e) {
        if (src[e] < 0 || src[e] >= n || dst[e] < 0 || dst[e] >= n || src[e] == dst[e]) return GFA2_ERR_INVALID_GRAPH;
        rowptr[src[e] + 1]++;
        rowptr[dst[e] + 1]++;
    }
    for (int v = 0; v < n; ++v) rowptr[v + 1] += rowptr[v];
    std::vector<int64_t> cur(rowptr.begin(), rowptr.end() - 1);
    std::vector<int32_t> col((size_t)(2 * m));
    std::vector<float> w((size_t)(2 * m));
    for (int64_t e = 0; e < m; ++e) {
        w[cur[src[e]]] = weight[e];
        col[cur[src[e]]++] = dst[e];
        w[cur[dst[e]]] = weight[e];
        col[cur[dst[e]]++] = src[e];
    }
    int st = gfa2_set_graph(h, n, rowptr.data(), col.data(), mass);
    if (st != GFA2_OK) return st;
    return gfa2_set_edge_weights(h, 2 * m, w.data());
}

int gfa2_exact_repulsion(gfa2_handle h, int32_t fp64, double* xy) {
    if (!h || !xy) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph || !h->has_pos) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    int rc = drain_timing(h);
    if (rc != GFA2_OK) return rc;
    double2* out = nullptr;
    GFA2_TRY(hipMalloc(&out, sizeof(double2) * (size_t)h->b.n));
    launch_exact_only(h->b, h->p, fp64 != 0, out, h->stream);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpyAsync(xy, out, sizeof(double2) * (size_t)h->b.n, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    (void)hipFree(out);
    return e == hipSuccess ? GFA2_OK : hip_status(e);
}

int gfa2_get_launch_config(gfa2_handle h, gfa2_launch_config* c) {
    if (!h || !c) return GFA2_ERR_INVALID_ARG;
    c->walk_block = h->tune.walk_bt;
    c->blocks_per_cu = h->tune.blocks_per_cu;
    c->attraction_stream = h->tune.attraction_stream;
    c->attraction_blocks_per_cu = h->tune.attraction_bpc;
    c->ms_per_iteration = 0.0;
    return GFA2_OK;
}

int gfa2_set_launch_config(gfa2_handle h, const gfa2_launch_config* c) {
    if (!h || !c) return GFA2_ERR_INVALID_ARG;
    const int bt = c->walk_block;
    if ((bt != 64 && bt != 128 && bt != 256 && bt != 512) || c->blocks_per_cu < 1 || c->blocks_per_cu > 64 ||
        c->attraction_stream < 0 || c->attraction_stream > 2 || c->attraction_blocks_per_cu < 0 ||
        c->attraction_blocks_per_cu > 64)
        return GFA2_ERR_INVALID_ARG;
    h->tune = LaunchConfig{bt, c->blocks_per_cu, c->attraction_stream, c->attraction_blocks_per_cu};
    apply_tune(h);
    h->graph_valid = false;
    if (h->gexec) { (void)hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
    return GFA2_OK;
}

int gfa2_tuned_config(int32_t nodes, gfa2_launch_config* c) {
    if (!c || nodes < 1) return GFA2_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(g_tune_mu);
    auto it = g_tune_table.find(size_bucket(nodes));
    if (it == g_tune_table.end()) return GFA2_ERR_NO_GRAPH;
    c->walk_block = it->second.walk_bt;
    c->blocks_per_cu = it->second.blocks_per_cu;
    c->attraction_stream = it->second.attraction_stream;
    c->attraction_blocks_per_cu = it->second.attraction_bpc;
    c->ms_per_iteration = 0.0;
    return GFA2_OK;
}

// Times every candidate launch shape over `iters` real iterations (HIP events on the
// handle's stream), keeps the fastest, and restores the layout state so the caller's
// trajectory is the one it would have been without tuning (no candidate changes a result
// bit, so only the advanced iterations need undoing).
int gfa2_autotune(gfa2_handle h, int32_t iters, gfa2_launch_config* best) {
    if (!h || iters < 1) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph || !h->has_pos) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    int rc = drain_timing(h);
    if (rc != GFA2_OK) return rc;
    Bufs& b = h->b;
    const size_t n = (size_t)b.n;
    // snapshot
    float2 *spos = nullptr, *sfp = nullptr, *sf = nullptr, *sfga = nullptr;
    DevState* sst = nullptr;
    SegState* sseg = nullptr;
    auto free_snapshot = [&]() {
        for (void* p : {(void*)spos, (void*)sfp, (void*)sf, (void*)sfga, (void*)sst, (void*)sseg})
            if (p) (void)hipFree(p);
    };
    {
        hipError_t ea = hipMalloc(&spos, sizeof(float2) * n);
        if (ea == hipSuccess) ea = hipMalloc(&sfp, sizeof(float2) * n);
        if (ea == hipSuccess) ea = hipMalloc(&sf, sizeof(float2) * n);
        if (ea == hipSuccess) ea = hipMalloc(&sfga, sizeof(float2) * n);
        if (ea == hipSuccess) ea = hipMalloc(&sst, sizeof(DevState));
        if (ea == hipSuccess) ea = hipMalloc(&sseg, sizeof(SegState) * b.nseg);
        if (ea != hipSuccess) {
            free_snapshot();
            return hip_status(ea);
        }
    }
    auto copy_all = [&](bool save) -> hipError_t {
        hipError_t e = hipSuccess;
        auto cp = [&](void* dst, const void* src, size_t bytes) {
            if (e == hipSuccess) e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, h->stream);
        };
        if (save) {
            cp(spos, b.pos, sizeof(float2) * n);
            cp(sfp, b.fprev, sizeof(float2) * n);
            cp(sf, b.f, sizeof(float2) * n);
            cp(sfga, b.fga, sizeof(float2) * n);
            cp(sst, b.st, sizeof(DevState));
            cp(sseg, b.seg_st, sizeof(SegState) * b.nseg);
        } else {
            cp(b.pos, spos, sizeof(float2) * n);
            cp(b.fprev, sfp, sizeof(float2) * n);
            cp(b.f, sf, sizeof(float2) * n);
            cp(b.fga, sfga, sizeof(float2) * n);
            cp(b.st, sst, sizeof(DevState));
            cp(b.seg_st, sseg, sizeof(SegState) * b.nseg);
            launch_new_positions(b, -1, h->stream);
        }
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        return e;
    };
    hipError_t e = copy_all(true);
    hipEvent_t t0 = nullptr, t1 = nullptr;
    if (e == hipSuccess) e = hipEventCreateWithFlags(&t0, hipEventDisableSystemFence);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&t1, hipEventDisableSystemFence);
    const LaunchConfig keep = h->tune;
    LaunchConfig win = keep;
    float win_ms = 1e30f;
    std::vector<std::pair<float, LaunchConfig>> timed;
    // Times one candidate over `reps` iterations after one untimed one, then restores the state.
    auto time_one = [&](LaunchConfig cand, int reps) -> float {
        if (e != hipSuccess) return 1e30f;
        h->tune = cand;
        apply_tune(h);
        enqueue_iteration(h, nullptr);   // warm
        e = hipEventRecord(t0, h->stream);
        for (int i = 0; i < reps && e == hipSuccess; ++i) enqueue_iteration(h, nullptr);
        if (e == hipSuccess) e = hipEventRecord(t1, h->stream);
        if (e == hipSuccess) e = hipEventSynchronize(t1);
        float ms = 0.0f;
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, t0, t1);
        if (e == hipSuccess) e = copy_all(false);
        return e == hipSuccess ? ms : 1e30f;
    };
    auto trial = [&](LaunchConfig cand) {
        const float ms = time_one(cand, iters);
        timed.push_back({ms, cand});
        if (ms < win_ms) {
            win_ms = ms;
            win = cand;
        }
    };
    // Stage 1: the walk's block size (the walk dominates); stage 2: the grid of the
    // grid-stride kernels, then where the attraction runs (and with how many blocks when it runs
    // beside keys, sort and tree), each with the winner so far.
    const int bts[] = {64, 128, 256, 512};
    const int bpcs[] = {1, 2, 4, 8};
    for (int bt : bts) trial(LaunchConfig{bt, keep.blocks_per_cu, keep.attraction_stream, keep.attraction_bpc});
    const LaunchConfig shape = win;
    for (int bpc : bpcs)
        if (bpc != shape.blocks_per_cu)
            trial(LaunchConfig{shape.walk_bt, bpc, shape.attraction_stream, shape.attraction_bpc});
    const LaunchConfig shape2 = win;
    const int modes[][2] = {{0, 0}, {1, 0}, {2, 0}, {2, 2}, {2, 3}, {2, 4}};
    if (attraction_placed(h))
        for (const auto& m : modes)
            if (m[0] != shape2.attraction_stream || m[1] != shape2.attraction_bpc)
                trial(LaunchConfig{shape2.walk_bt, shape2.blocks_per_cu, m[0], m[1]});
    // Stage 3: the three fastest shapes again, three rounds each over twice the iterations,
    // interleaved so that a drift of the clock or the layout affects them alike.
    std::stable_sort(timed.begin(), timed.end(),
                     [](const std::pair<float, LaunchConfig>& a, const std::pair<float, LaunchConfig>& b) {
                         return a.first < b.first;
                     });
    const size_t finalists = std::min<size_t>(3, timed.size());
    if (finalists > 1 && e == hipSuccess) {
        std::vector<float> total(finalists, 0.0f);
        for (int round = 0; round < 3; ++round)
            for (size_t k = 0; k < finalists; ++k) total[k] += time_one(timed[k].second, 2 * iters);
        size_t bestk = 0;
        for (size_t k = 1; k < finalists; ++k)
            if (total[k] < total[bestk]) bestk = k;
        win = timed[bestk].second;
        win_ms = total[bestk] / 6.0f;
    }
    if (t0) (void)hipEventDestroy(t0);
    if (t1) (void)hipEventDestroy(t1);
    free_snapshot();
    if (e != hipSuccess) {
        h->tune = keep;
        apply_tune(h);
        return hip_status(e);
    }
    h->tune = win;
    apply_tune(h);
    h->graph_valid = false;
    if (h->gexec) { (void)hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        LaunchConfig& entry = g_tune_table[size_bucket(b.n)];
        LaunchConfig found = win;
        if (!attraction_placed(h)) {
            // what others of these nodes measured, or the default
            found.attraction_stream = entry.attraction_stream;
            found.attraction_bpc = entry.attraction_bpc;
        }
        entry = found;
    }
    if (best) {
        best->walk_block = win.walk_bt;
        best->blocks_per_cu = win.blocks_per_cu;
        best->attraction_stream = win.attraction_stream;
        best->attraction_blocks_per_cu = win.attraction_bpc;
        best->ms_per_iteration = win_ms / iters;
    }
    return GFA2_OK;
}

int gfa2_stress_setup(gfa2_handle h, int32_t nsources, int32_t targets_per_source, uint64_t seed, int64_t* npairs) {
    if (!h || nsources < 1 || targets_per_source < 1) return GFA2_ERR_INVALID_ARG;
    if (!h->has_graph) return GFA2_ERR_NO_GRAPH;
    const int n = h->b.n;
    if (n < 2) return GFA2_ERR_INVALID_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    GFA2_TRY(hipStreamSynchronize(h->stream));
    const int K = nsources < n ? nsources : n;
    const int T = targets_per_source;
    if ((long long)K * T >= (1ll << 31)) return GFA2_ERR_INVALID_ARG;
    // sources: the first K entries of a seeded Fisher-Yates shuffle; targets: uniform over
    // the other n-1 nodes, with replacement
    SplitMix rng{seed};
    std::vector<int> perm(n);
    for (int i = 0; i < n; ++i) perm[i] = i;
    for (int i = 0; i < K; ++i) {
        const int j = i + (int)rng.below((uint64_t)(n - i));
        std::swap(perm[i], perm[j]);
    }
    std::vector<int> src(perm.begin(), perm.begin() + K);
    int st = GFA2_OK;
    if (!h->stress_part) {
        if ((st = dalloc(h, &h->stress_part, 3 * kStressBlocks)) != GFA2_OK) return st;
        if ((st = dalloc(h, &h->stress_pos, n)) != GFA2_OK) return st;
    }
    if (K * T > h->stress_K * h->stress_T) {
        if ((st = dalloc(h, &h->stress_tgt, (size_t)K * T)) != GFA2_OK) return st;
        if ((st = dalloc(h, &h->stress_dist, (size_t)K * T)) != GFA2_OK) return st;
    }
    if (K > h->stress_K && (st = dalloc(h, &h->stress_src, K)) != GFA2_OK) return st;
    h->stress_K = K;
    h->stress_T = T;
    GFA2_TRY(hipMemcpyAsync(h->stress_src, src.data(), sizeof(int) * K, hipMemcpyHostToDevice, h->stream));
    // the targets take the generator's draws after the K of the shuffle
    stress_draw_targets(h->stress_src, T, (long long)K * T, seed, (unsigned long long)K, n, h->stress_tgt, h->stream);
    long long reached = 0;
    const int rc = stress_hop_distances(h->b, h->stress_src, K, h->stress_tgt, T, h->stress_dist,
                                        npairs ? &reached : nullptr, h->stream);
    if (rc != 0) return rc == -2 ? GFA2_ERR_OOM : GFA2_ERR_HIP;
    if (npairs) *npairs = reached;
    return GFA2_OK;
}

int gfa2_stress_pairs(gfa2_handle h, int64_t cap, int32_t* a, int32_t* b, int32_t* d) {
    if (!h || cap < 0) return GFA2_ERR_INVALID_ARG;
    if (!h->stress_K) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    const int64_t np = (int64_t)h->stress_K * h->stress_T;
    const int64_t c = np < cap ? np : cap;
    std::vector<int> src(h->stress_K);
    GFA2_TRY(hipMemcpy(src.data(), h->stress_src, sizeof(int) * h->stress_K, hipMemcpyDeviceToHost));
    if (b) GFA2_TRY(hipMemcpy(b, h->stress_tgt, sizeof(int) * c, hipMemcpyDeviceToHost));
    if (d) GFA2_TRY(hipMemcpy(d, h->stress_dist, sizeof(int) * c, hipMemcpyDeviceToHost));
    if (a)
        for (int64_t k = 0, p = 0; p < c; ++k) {
            const int64_t end = std::min<int64_t>(p + h->stress_T, c);
            for (; p < end; ++p) a[p] = src[(size_t)k];
        }
    return GFA2_OK;
}

int gfa2_normalized_stress(gfa2_handle h, const float* xy, double* ns, double* alpha) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    if (!h->stress_K) return GFA2_ERR_NO_GRAPH;
    GFA2_TRY(hipSetDevice(h->device));
    const float2* pos = h->b.pos;
    if (xy) {
        GFA2_TRY(hipMemcpyAsync(h->stress_pos, xy, sizeof(float2) * h->b.n, hipMemcpyHostToDevice, h->stream));
        pos = h->stress_pos;
    }
    double s[3];
    if (stress_reduce(pos, h->stress_src, h->stress_tgt, h->stress_dist, h->stress_T,
                      (long long)h->stress_K * h->stress_T, h->stress_part, kStressBlocks, s, h->stream) != 0)
        return GFA2_ERR_HIP;
    const double P = s[2];
    if (ns) *ns = (P > 0 && s[1] > 0) ? 1.0 - s[0] * s[0] / (P * s[1]) : 0.0;
    if (alpha) *alpha = s[1] > 0 ? s[0] / s[1] : 0.0;
    return GFA2_OK;
}

}  // extern "C"

namespace gfa2 {

bool engine_graph(gfa2_engine* h, const Bufs** b, int* device, hipStream_t* stream) {
    if (!h || !h->has_graph || !h->has_pos) return false;
    *b = &h->b;
    *device = h->device;
    *stream = h->stream;
    return true;
}

EngineScratch::EngineScratch(gfa2_engine* engine) : h(engine) { h->scratch_mu.lock(); }

EngineScratch::~EngineScratch() {
    if (own) (void)hipFree(own);
    h->scratch_mu.unlock();
}

void* EngineScratch::get(size_t bytes) {
    if (bytes <= h->scratch_bytes) return h->scratch;
    if (bytes > kScratchKeep) {
        if (hipMalloc(&own, bytes) != hipSuccess) {
            (void)hipGetLastError();
            own = nullptr;
        }
        return own;
    }
    if (h->scratch) (void)hipFree(h->scratch);      // waits for the device
    h->scratch = nullptr;
    h->scratch_bytes = 0;
    if (hipMalloc(&h->scratch, bytes) != hipSuccess) {
        (void)hipGetLastError();
        h->scratch = nullptr;
        return nullptr;
    }
    h->scratch_bytes = bytes;
    return h->scratch;
}

bool engine_view(gfa2_engine* h, EngineView* v) {
    if (!h || !h->has_graph) return false;
    v->n = h->b.n;
    v->device = h->device;
    v->pos = h->b.pos;
    v->stream = h->stream;
    v->rowptr = h->b.rowptr;
    v->col = h->b.col;
    v->nnz = h->b.nnz;
    v->nseg = h->b.nseg;
    v->medium = h->b.node_lists + h->b.nlight;
    v->nmedium = h->b.nmedium;
    v->nheavy = h->b.nheavy;
    v->chunk0 = h->b.attr_c0;
    v->chunks = h->b.attr_chunks;
    v->nchunks = h->b.nattr_chunks;
    return true;
}

int engine_positions_written(gfa2_engine* h) {
    h->has_pos = true;
    positions_changed(h);
    GFA2_TRY(hipGetLastError());
    GFA2_TRY(hipStreamSynchronize(h->stream));
    return GFA2_OK;
}

}  // namespace gfa2

extern "C" {

int gfa2_destroy(gfa2_handle h) {
    if (!h) return GFA2_ERR_INVALID_ARG;
    hipSetDevice(h->device);
    if (h->stream) hipStreamSynchronize(h->stream);
    free_all(h);
    for (hipEvent_t e : h->events) hipEventDestroy(e);
    if (h->fork) hipEventDestroy(h->fork);
    if (h->join) hipEventDestroy(h->join);
    if (h->side) hipStreamDestroy(h->side);
    if (h->stream) hipStreamDestroy(h->stream);
    delete h;
    return GFA2_OK;
}

const char* gfa2_strerror(int code) {
    switch (code) {
        case GFA2_OK: return "ok";
        case GFA2_ERR_NO_DEVICE: return "no HIP device found";
        case GFA2_ERR_OOM: return "out of device memory";
        case GFA2_ERR_INVALID_ARG: return "invalid argument";
        case GFA2_ERR_INVALID_GRAPH: return "invalid graph (empty, malformed CSR, self-loop or id out of range)";
        case GFA2_ERR_TREE_OVERFLOW: return "quadtree cell capacity exceeded";
        case GFA2_ERR_HIP: return "HIP runtime error";
        case GFA2_ERR_NO_GRAPH: return "no graph loaded";
        case GFA2_ERR_UNSUPPORTED: return "unsupported configuration";
        case GFA2_ERR_DEVICE_WAIT: return "a bounded device wait ran out (the iteration was skipped)";
        case GFA2_ERR_SCRATCH_LIMIT: return "request exceeds the fixed scratch of the allocation-free entry point";
        default: return "unknown error";
    }
}

}  // extern "C"
