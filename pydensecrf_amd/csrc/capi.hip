// Host orchestration and the extern "C" boundary (include/dcrf_hip.h).
//
// A dcrf_model mirrors the reference's DenseCRF (pydensecrf/densecrf/src/densecrf.cpp):
// it owns the unary, the list of pairwise terms (each a lattice + normaliser + label
// compatibility, pairwise.cpp:116-122 / labelcompatibility.cpp) and runs mean-field
// inference.  Construction touches no device; the first call that needs the GPU
// creates the model's stream on the current HIP device.  No C++ exception crosses the
// boundary: every entry point returns a status and records a message.
#include "dcrf_internal.h"

#include <sys/mman.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <limits>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <numeric>
#include <thread>

using namespace dcrf;

namespace dcrf {
namespace {
thread_local std::string g_last_error;
}
void set_error(int code, const std::string& msg) {
    (void)code;
    g_last_error = msg;
}
}  // namespace dcrf

namespace {

constexpr int kDefaultChunk = 32;

struct TermLayout {
    DevBuf<int2> nbr;    // [(d+1)][V] global rows
    // multi-step blur passes: steps per pass, table offsets (ints) per pass, tables
    // forward / reverse
    std::vector<int> pass_steps, pass_off;
    DevBuf<int> passF, passT;
    DevBuf<int> vtx;     // [N][d+1] global rows
    DevBuf<float> swF;   // slice weights, forward
    DevBuf<float> swT;   // slice weights, transpose (unused when symmetric)
};

// Kernel classes timed by dcrf_enable_timing.
enum { KC_SPLAT = 0, KC_COMBINE = 1, KC_BLUR = 2, KC_MEANFIELD = 3, KC_COUNT = 4 };

struct PendingTiming {
    hipEvent_t start, stop;
    int cls;
    double bytes;
};

}  // namespace

namespace dcrf {

// ---------------------------------------------------------------- host transfers
// Large copies between pageable host memory (the caller's arrays) and the device go
// through one page-locked staging area per process (hipHostMalloc, grown on demand,
// shared by all models under a lock, kept until dcrf_release_cached_memory) in chunks:
// the DMA engine moves some chunks while host threads copy others in or out, where the
// runtime would stage pageable memory through one host thread.
constexpr size_t kStageMax = (size_t)256 << 20;  // larger copies: windows of this size
constexpr int kCopyThreads = 8;

struct HostStage {
    std::mutex mu;
    char* p = nullptr;
    size_t cap = 0;
};
HostStage& host_stage() {
    static HostStage* h = new HostStage;  // never destroyed: no runtime call at process exit
    return *h;
}

// Threads for a host copy of n bytes: about one per 2 MiB, at most kCopyThreads and the
// hardware threads.
int copy_threads(size_t n) {
    const size_t hw = std::max(1u, std::thread::hardware_concurrency());
    return (int)std::max<size_t>(1, std::min({(size_t)kCopyThreads, hw, n >> 21}));
}

// Chunk t of n bytes split T ways, 4 KiB aligned: [off(t), off(t + 1)).
inline size_t chunk_off(size_t n, int T, int t) { return t >= T ? n : (n / T * t) & ~(size_t)4095; }

// Chunks of one staged window of n bytes uploaded by T threads: about 2 MiB each, at
// least one and at most 8 per thread (thread t takes chunks t, t + T, ...).  The host copy
// made before the window's first DMA is then one small chunk rather than a thread's whole
// share.
inline int window_chunks(size_t n, int T) { return (int)std::clamp<size_t>(n >> 21, (size_t)T, (size_t)8 * T); }

// work(t) for t < T: t = 0 on this thread, the others on threads of their own where the
// system starts them (else here as well).  work must not throw.
template <typename F>
void run_parallel(int T, const F& work) {
    std::vector<std::thread> th;
    int t = 1;
    try {
        for (; t < T; t++) th.emplace_back(work, t);
    } catch (...) {
    }
    work(0);
    for (int u = t; u < T; u++) work(u);
    for (auto& x : th) x.join();
}

// dst = src (host memory, n bytes) with copy_threads(n) threads.
void host_copy(void* dst, const void* src, size_t n) {
    const int T = copy_threads(n);
    run_parallel(T, [&](int t) {
        const size_t a = chunk_off(n, T, t), b = chunk_off(n, T, t + 1);
        std::memcpy((char*)dst + a, (const char*)src + a, b - a);
    });
}

// rows rows of cols floats from src (row stride ss) to dst (row stride ds), rows shared
// out among copy_threads threads (row t, t + T, ...).
void copy_rows(float* dst, size_t ds, const float* src, size_t ss, int rows, size_t cols) {
    const int T = std::min(copy_threads((size_t)rows * cols * sizeof(float)), std::max(rows, 1));
    run_parallel(T, [&](int t) {
        for (int r = t; r < rows; r += T) std::memcpy(dst + r * ds, src + r * ss, sizeof(float) * cols);
    });
}

// The staging area of at least n bytes, or null where the runtime cannot give that much
// page-locked memory (the caller then copies without staging).
char* stage_reserve(HostStage& H, size_t n) {
    if (n > H.cap) {
        if (H.p) DCRF_HIP_CHECK(hipHostFree(H.p));
        H.p = nullptr;
        H.cap = 0;
        if (hipHostMalloc((void**)&H.p, n, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();  // clear the failure: the copy goes unstaged
            H.p = nullptr;
            return nullptr;
        }
        H.cap = n;
    }
    return H.p;
}

// Page-locked buffers that hold a unary between dcrf_set_unary and its upload.  At most
// kPinnedMax bytes exist at a time, in use or kept for the next model (until
// dcrf_release_cached_memory); a request beyond that, or one that the runtime refuses,
// gets none and the caller uses pageable memory.  Nothing is allocated before the process
// has used a device: setting a unary alone does not initialise one.
constexpr size_t kPinnedMax = (size_t)512 << 20;
constexpr size_t kPinnedMin = (size_t)1 << 20;  // smaller unaries: pageable, the copies cost less than the events
std::atomic<bool> g_device_used{false};

struct PinnedPool {
    std::mutex mu;
    std::multimap<size_t, void*> free;
    size_t total = 0;  // bytes allocated: in use and free
};
PinnedPool& pinned_pool() {
    static PinnedPool* p = new PinnedPool;  // never destroyed: no runtime call at process exit
    return *p;
}

// Frees the buffers not in use; returns their bytes.  The caller holds the lock.
size_t release_pinned(PinnedPool& P) {
    size_t b = 0;
    for (auto& f : P.free) {
        (void)hipHostFree(f.second);
        b += f.first;
    }
    P.free.clear();
    P.total -= b;
    return b;
}
size_t release_pinned() {
    PinnedPool& P = pinned_pool();
    std::lock_guard<std::mutex> lk(P.mu);
    return release_pinned(P);
}

// A buffer taken from the pool.
struct PinnedBuf {
    char* p = nullptr;
    size_t cap = 0;
    PinnedBuf() = default;
    PinnedBuf(const PinnedBuf&) = delete;
    PinnedBuf& operator=(const PinnedBuf&) = delete;
    ~PinnedBuf() { give(); }
    void give() {
        if (!p) return;
        PinnedPool& P = pinned_pool();
        std::lock_guard<std::mutex> lk(P.mu);
        P.free.emplace(cap, p);
        p = nullptr;
        cap = 0;
    }
    // At least n bytes in p, or false.
    bool take(size_t n) {
        if (p && cap >= n && cap <= 4 * n) return true;
        give();
        if (!g_device_used || n < kPinnedMin || n > kPinnedMax) return false;
        PinnedPool& P = pinned_pool();
        std::lock_guard<std::mutex> lk(P.mu);
        auto it = P.free.lower_bound(n);
        if (it == P.free.end() || it->first > 4 * n) {
            const size_t size = (n + ((size_t)2 << 20) - 1) & ~(((size_t)2 << 20) - 1);
            if (P.total + size > kPinnedMax) release_pinned(P);
            if (P.total + size > kPinnedMax) return false;
            // (a stream capture that another part of the program has open is not touched)
            hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
            (void)hipThreadExchangeStreamCaptureMode(&mode);
            void* q = nullptr;
            const hipError_t e = hipHostMalloc(&q, size, hipHostMallocPortable);
            (void)hipThreadExchangeStreamCaptureMode(&mode);
            if (e != hipSuccess) {
                (void)hipGetLastError();  // clear the failure
                return false;
            }
            P.total += size;
            it = P.free.emplace(size, q);
        }
        p = static_cast<char*>(it->second);
        cap = it->first;
        P.free.erase(it);
        return true;
    }
};

// The stream of the current device that uploads unaries beside the models' own work.
hipStream_t upload_stream() {
    static std::mutex* mu = new std::mutex;
    static std::map<int, hipStream_t>* streams = new std::map<int, hipStream_t>;
    int dev = 0;
    DCRF_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(*mu);
    auto it = streams->find(dev);
    if (it == streams->end()) {
        hipStream_t s = nullptr;
        DCRF_HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        it = streams->emplace(dev, s).first;
    }
    return it->second;
}

// Events of one staged copy, destroyed on every exit.
struct ChunkEvents {
    std::vector<hipEvent_t> ev;
    explicit ChunkEvents(int T) : ev(T, nullptr) {
        for (auto& e : ev) DCRF_HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    ~ChunkEvents() {
        for (auto e : ev)
            if (e) (void)hipEventDestroy(e);
    }
};

void copy_to_host_window(char* stage, void* dst, const void* src, size_t n, hipStream_t s);
void copy_to_device_window(char* stage, void* dst, const void* src, size_t n, hipStream_t s);

// dst (host) = src (device), n bytes, after the work queued on s; returns when done.
// Copies above kStageMax go through the staging area one window at a time.
void copy_to_host(void* dst, const void* src, size_t n, hipStream_t s) {
    if (n < kStagedMin) {
        DCRF_HIP_CHECK(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s));
        DCRF_HIP_CHECK(hipStreamSynchronize(s));
        return;
    }
    HostStage& H = host_stage();
    std::lock_guard<std::mutex> lk(H.mu);
    char* stage = stage_reserve(H, std::min(n, kStageMax));
    if (!stage) {
        DCRF_HIP_CHECK(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s));
        DCRF_HIP_CHECK(hipStreamSynchronize(s));
        return;
    }
    for (size_t o = 0; o < n; o += kStageMax)
        copy_to_host_window(stage, (char*)dst + o, (const char*)src + o, std::min(kStageMax, n - o), s);
}

// dst (device) = src (host), n bytes, queued on s; returns when the copy is done.
void copy_to_device(void* dst, const void* src, size_t n, hipStream_t s) {
    if (n < kStagedMin) {
        DCRF_HIP_CHECK(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, s));
        DCRF_HIP_CHECK(hipStreamSynchronize(s));
        return;
    }
    HostStage& H = host_stage();
    std::lock_guard<std::mutex> lk(H.mu);
    char* stage = stage_reserve(H, std::min(n, kStageMax));
    if (!stage) {
        DCRF_HIP_CHECK(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, s));
        DCRF_HIP_CHECK(hipStreamSynchronize(s));
        return;
    }
    for (size_t o = 0; o < n; o += kStageMax)
        copy_to_device_window(stage, (char*)dst + o, (const char*)src + o, std::min(kStageMax, n - o), s);
}

// One window (n <= the staging area's size) of copy_to_host: every chunk's DMA is
// queued at once, in order; while the device works the threads touch the pages the copy
// will fill (their contents kept), then each chunk is copied out by all of them as soon
// as its event fires.  Chunks of 8 MiB, or a quarter of less: each costs a launch and an
// event, and the host copy left after the last one is a thread's share of it.  (In chunks
// of 2 MiB, one thread each and the pages not touched before, 66 MB into fresh memory
// took 2.2 ms behind 1.5 ms of iterations; now 1.55.)
void copy_to_host_window(char* stage, void* dst, const void* src, size_t n, hipStream_t s) {
    const int T = copy_threads(n), C = (int)std::max<size_t>({n >> 23, std::min<size_t>(n >> 21, 4), 1});
    ChunkEvents E(C);
    for (int c = 0; c < C; c++) {  // all chunks queued before any thread starts
        const size_t a = chunk_off(n, C, c), b = chunk_off(n, C, c + 1);
        DCRF_HIP_CHECK(hipMemcpyAsync(stage + a, (const char*)src + a, b - a, hipMemcpyDeviceToHost, s));
        DCRF_HIP_CHECK(hipEventRecord(E.ev[c], s));
    }
    std::vector<hipError_t> err(T, hipSuccess);
    run_parallel(T, [&](int t) {  // each chunk leaves the staging area as soon as it arrived
        for (int pass = 0; pass < 2; pass++)
            for (int c = 0; c < C; c++) {
                const size_t a = chunk_off(n, C, c), m = chunk_off(n, C, c + 1) - a;
                const size_t x = a + chunk_off(m, T, t), y = a + chunk_off(m, T, t + 1);
                if (pass == 0) {  // while the device works: the pages the copy will fill
                    for (size_t o = x; o < y; o += 4096) {
                        volatile char* q = (volatile char*)dst + o;
                        *q = *q;
                    }
                    continue;
                }
                err[t] = hipEventSynchronize(E.ev[c]);
                if (err[t] != hipSuccess) return;
                std::memcpy((char*)dst + x, stage + x, y - x);
            }
    });
    for (hipError_t e : err) DCRF_HIP_CHECK(e);
}

// One window of copy_to_device: each thread stages its chunks in turn and queues each
// chunk's DMA as soon as it is staged; returns when the window's copies are done (the
// staging area is free again).
void copy_to_device_window(char* stage, void* dst, const void* src, size_t n, hipStream_t s) {
    const int T = copy_threads(n), C = window_chunks(n, T);
    std::vector<hipError_t> err(C, hipSuccess);
    run_parallel(T, [&](int t) {
        for (int c = t; c < C; c += T) {
            const size_t a = chunk_off(n, C, c), b = chunk_off(n, C, c + 1);
            std::memcpy(stage + a, (const char*)src + a, b - a);
            err[c] = hipMemcpyAsync((char*)dst + a, stage + a, b - a, hipMemcpyHostToDevice, s);
            if (err[c] != hipSuccess) return;
        }
    });
    const hipError_t sync = hipStreamSynchronize(s);  // the staging area is free again
    for (hipError_t e : err) DCRF_HIP_CHECK(e);
    DCRF_HIP_CHECK(sync);
}

// Frees the staging area; returns its bytes.
size_t release_host_stage() {
    HostStage& H = host_stage();
    std::lock_guard<std::mutex> lk(H.mu);
    const size_t b = H.cap;
    if (H.p) DCRF_HIP_CHECK(hipHostFree(H.p));
    H.p = nullptr;
    H.cap = 0;
    return b;
}

}  // namespace dcrf

// Host floats left uninitialised when allocated (a copy fills them).  Blocks of 4 MiB
// and more are 2 MiB aligned and advised for transparent huge pages: a 66 MB unary then
// faults in ~33 pages on its first copy instead of ~16,000.
struct HostFloats {
    struct Free {
        void operator()(float* q) const { std::free(q); }
    };
    std::unique_ptr<float, Free> p;
    size_t n = 0;
    void resize(size_t count) {
        if (count == n) return;
        p.reset();
        n = 0;
        if (!count) return;
        const size_t bytes = sizeof(float) * count;
        void* q = nullptr;
        if (bytes >= ((size_t)4 << 20)) {
            if (posix_memalign(&q, (size_t)2 << 20, bytes) != 0) q = nullptr;
            if (q) (void)madvise(q, bytes, MADV_HUGEPAGE);  // advice only
        } else {
            q = std::malloc(bytes);
        }
        if (!q) throw std::bad_alloc();
        p.reset(static_cast<float*>(q));
        n = count;
    }
    float* data() { return p.get(); }
    const float* data() const { return p.get(); }
    size_t size() const { return n; }
};

struct dcrf_model {
    Geometry geo;
    GeometryDev geod;
    int L = 0;
    bool dev_ready = false;
    hipStream_t stream = nullptr;
    HostFloats unary_host;  // (L, N) row-major as given, unless unary_pin holds it
    // a single instance's unary on its way to the device: set, and (unary_ev) being copied
    // to `stage` by the device's upload stream
    PinnedBuf unary_pin;
    hipEvent_t unary_ev = nullptr;
    bool unary_uploading = false;
    std::vector<char> unary_unset;  // per instance: its columns of unary_host hold no data yet
    bool has_unary = false, unary_dirty = false;
    DevBuf<float> unary;  // [N][L]
    // LogisticUnaryEnergy (U = L f): parameters L [L][F] row-major, features [N][F]
    bool logistic = false;
    int lF = 0;
    std::vector<float> lL;
    DevBuf<float> lL_dev, lf, lfFN;  // features [N][F] and as given [F][N]
    std::vector<float> ugrad_param;  // its parameter gradient from the last dcrf_gradient
    std::vector<std::unique_ptr<Term>> terms;
    DevBuf<float> Q, work, tmp1, tmp2, stage;
    DevBuf<float> Qp;  // inference iterate with the vertex-row stride (see run_inference)
    int ldv = 0;       // row stride (floats) of the vertex rows and Qp: padded_labels(L), or L
    float hash_load = 0.5f;
    int splat_chunk = 0;  // 0: default
    int tile_side = 0;  // 0: default_tile_side(L)
    TileMap tiles;
    bool tiles_ready = false;

    // global filter layout
    bool layout_valid = false;
    int V_total = 0, rows0 = 0, E_total = 0, max_d = 0;
    size_t noalloc_rows = 0;  // the rows that the allocation-free inference's limit counts
    std::vector<int> order, vbase;
    std::vector<int> prefixV;
    DevBuf<float> vals[2];
    SegLists seg;                      // splat segments and recombination items
    DevBuf<int> g_tile_seg, g_tile_e;  // first segment / entry of each tile
    bool tiled = false;                // splat through LDS tiles (else the global form)
    size_t lds_cap = 0;                // LDS bytes one workgroup may allocate
    TiledSplat tsplat{};
    DevBuf<int2> g_entF, g_entT;  // splat entries (pixel, weight bits), forward / transposed
    // opt-in: Q between inference iterations in 8 x 8 pixel blocks (2-D single images),
    // read by the splat through entries holding block positions
    bool qblocks = false, qblocks_ready = false;
    // opt-in: blur passes of fewer than blur_small_v vertices with blur_r labels per lane
    int blur_r = 0, blur_small_v = 0;
    DevBuf<int2> g_entB;
    DevBuf<float> Qb;
    bool fused = false;           // inference through k_meanfield_fused
    DevBuf<int2> g_slc;           // its per-pixel slice pairs of every term
    DevBuf<int2> g_slcT;          // the same with the transposed filter's slice weights (adjoint;
    bool slcT_valid = false;      // built on first use when they differ from the forward's)
    bool runs = false;            // ... or through k_meanfield_runs (rows staged per pixel run)
    int mf_mode = 0;              // dcrf_set_meanfield_kernel: 0 auto (fused), 1 generic, 2 fused, 3 runs
    bool pairs = true;            // blur up to three steps per pass (dcrf_set_blur_pairs)
    int blur_steps = 2;           // most steps per multi-step pass, 2 or 3 (dcrf_set_blur_steps)
    int n_passes = 0;             // launches per filter with multi-step passes
    std::vector<int> prefixP;     // vertices of the terms with more than p passes
    int run_rows = 16;            // pixel rows of a run rectangle
    RunSlice rslice;
    int rows_lds = 0;
    bool all_symmetric = true;
    std::vector<std::unique_ptr<TermLayout>> tl;

    // term weights (device, [T]); null unless set
    DevBuf<float> kw;
    bool kw_set = false;
    // training checkpoints: Q_0..Q_n and the raw messages K~_k Q_t
    int train_n = -1;
    const float* train_kw = nullptr;
    DevBuf<float> qcache, mcache, bbuf, partial;
    DevBuf<double> rmid;  // first-stage sums of launch_sum_rows
    DevBuf<double> gacc, gacc2;
    // objective on the device: ground truth, Hamming's class weights, partial sums
    DevBuf<int16_t> gt_dev;
    DevBuf<float> obj_w;
    DevBuf<double> obj_partial;
    // kernel-parameter gradient: the filter plans (built on first use for the lattices of
    // generation lat_gen, which every lattice change advances), 4 [N][L] work slabs per
    // term of a plan ([a | c], x, lbl), 2 [N][d] feature gradients (one-thread-per-point
    // form), per-block partials and the accumulated gradient of all terms
    std::vector<std::unique_ptr<KgPlan>> kgplans;
    int lat_gen = 0;
    DevBuf<float> kgbuf, kgdf;
    DevBuf<int16_t> labels;  // dcrf_map / dcrf_current_map
    DevBuf<double> kpartial, kacc;

    // captured inference (dcrf_capture_inference)
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    bool graph_valid = false;

    // timing
    bool timing = false;
    long long kc_launches[KC_COUNT] = {};
    double kc_ms[KC_COUNT] = {}, kc_bytes[KC_COUNT] = {};
    std::vector<PendingTiming> pending;
    std::vector<hipEvent_t> free_events;

    ~dcrf_model() {
        for (auto& p : pending) {
            (void)hipEventDestroy(p.start);
            (void)hipEventDestroy(p.stop);
        }
        for (auto e : free_events) (void)hipEventDestroy(e);
        drop_graph();
        if (unary_uploading) (void)hipEventSynchronize(unary_ev);
        if (unary_ev) (void)hipEventDestroy(unary_ev);
        if (stream) (void)hipStreamDestroy(stream);
    }

    // what a captured graph reads: the model's own unary buffer (nullptr: the caller's
    // unary, or none) and the term-weight buffer (nullptr: no weights)
    bool graph_own_unary = false;
    const float* graph_unary = nullptr;
    const float* graph_kw = nullptr;

    void drop_graph() {
        if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
        if (graph) (void)hipGraphDestroy(graph);
        graph_exec = nullptr;
        graph = nullptr;
        graph_valid = false;
    }

    int N() const { return geo.N_total(); }
    int chunk() const { return splat_chunk > 0 ? splat_chunk : kDefaultChunk; }
};

namespace {

template <typename F>
int guard(F&& f) {
    try {
        f();
        set_error(DCRF_OK, "");
        return DCRF_OK;
    } catch (const Error& e) {
        set_error(e.code, e.msg);
        return e.code;
    } catch (const std::bad_alloc&) {
        set_error(DCRF_ERR_MEMORY, "host allocation failed");
        return DCRF_ERR_MEMORY;
    } catch (const std::exception& e) {
        set_error(DCRF_ERR_DEVICE, e.what());
        return DCRF_ERR_DEVICE;
    }
}

void require(bool cond, const std::string& msg, int code = DCRF_ERR_VALUE) {
    if (!cond) throw Error{code, msg};
}

hipEvent_t take_event(dcrf_model& m) {
    if (!m.free_events.empty()) {
        hipEvent_t e = m.free_events.back();
        m.free_events.pop_back();
        return e;
    }
    hipEvent_t e;
    DCRF_HIP_CHECK(hipEventCreate(&e));
    return e;
}

void collect_timing(dcrf_model& m) {
    for (auto& p : m.pending) {
        DCRF_HIP_CHECK(hipEventSynchronize(p.stop));
        float ms = 0.f;
        DCRF_HIP_CHECK(hipEventElapsedTime(&ms, p.start, p.stop));
        m.kc_ms[p.cls] += ms;
        m.kc_bytes[p.cls] += p.bytes;
        m.kc_launches[p.cls]++;
        m.free_events.push_back(p.start);
        m.free_events.push_back(p.stop);
    }
    m.pending.clear();
}

// Brackets one launch with events when timing is on.
struct Timed {
    dcrf_model& m;
    hipStream_t s;
    int cls;
    double bytes;
    hipEvent_t e0 = nullptr;
    Timed(dcrf_model& m_, hipStream_t s_, int cls_, double bytes_) : m(m_), s(s_), cls(cls_), bytes(bytes_) {
        if (m.timing) {
            e0 = take_event(m);
            DCRF_HIP_CHECK(hipEventRecord(e0, s));
        }
    }
    void done() {
        if (!e0) return;
        hipEvent_t e1 = take_event(m);
        DCRF_HIP_CHECK(hipEventRecord(e1, s));
        m.pending.push_back(PendingTiming{e0, e1, cls, bytes});
        e0 = nullptr;
    }
};

void ensure_device(dcrf_model& m) {
    if (m.dev_ready) return;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
        throw Error{DCRF_ERR_DEVICE, "no HIP device is available"};
    DCRF_HIP_CHECK(hipStreamCreateWithFlags(&m.stream, hipStreamNonBlocking));
    int dev = 0, lds = 0;
    DCRF_HIP_CHECK(hipGetDevice(&dev));
    DCRF_HIP_CHECK(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    m.lds_cap = (size_t)std::max(lds, 0);
    const Geometry& g = m.geo;
    m.geod.pix_base.reserve(g.pix_base.size());
    m.geod.pad_base.reserve(g.pad_base.size());
    m.geod.W.reserve(g.n_inst);
    DCRF_HIP_CHECK(hipMemcpy(m.geod.pix_base.get(), g.pix_base.data(), sizeof(int) * g.pix_base.size(),
                             hipMemcpyHostToDevice));
    DCRF_HIP_CHECK(hipMemcpy(m.geod.pad_base.get(), g.pad_base.data(), sizeof(int) * g.pad_base.size(),
                             hipMemcpyHostToDevice));
    std::vector<int> W = g.is2d ? g.W : std::vector<int>(g.n_inst, 1);
    DCRF_HIP_CHECK(hipMemcpy(m.geod.W.get(), W.data(), sizeof(int) * g.n_inst, hipMemcpyHostToDevice));
    m.dev_ready = true;
    g_device_used = true;
}

// Waits for the unary's copy in flight, if any; the page-locked buffer is free after.
void finish_unary_upload(dcrf_model& m) {
    if (!m.unary_uploading) return;
    DCRF_HIP_CHECK(hipEventSynchronize(m.unary_ev));
    m.unary_uploading = false;
}

// Starts the copy of a unary that waits in page-locked memory, so that it runs beside the
// lattice builds (one copy of 66 MB takes 1.2 ms, the two builds at 1024x768 about as
// long).
void start_unary_upload(dcrf_model& m) {
    if (!m.unary_pin.p || m.unary_uploading) return;
    const size_t n = (size_t)m.N() * m.L;
    m.stage.reserve(n);
    if (!m.unary_ev) DCRF_HIP_CHECK(hipEventCreateWithFlags(&m.unary_ev, hipEventDisableTiming));
    hipStream_t s = upload_stream();
    DCRF_HIP_CHECK(hipMemcpyAsync(m.stage.get(), m.unary_pin.p, sizeof(float) * n, hipMemcpyHostToDevice, s));
    const hipError_t e = hipEventRecord(m.unary_ev, s);
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    DCRF_HIP_CHECK(e);
    m.unary_uploading = true;
}

// dst = src on the device (large lists through the staging area; then the copy is
// complete on return, else it is queued on s).
template <typename T>
void upload(DevBuf<T>& dst, const std::vector<T>& src, hipStream_t s) {
    dst.reserve(src.size());
    if (src.empty()) return;
    const size_t bytes = sizeof(T) * src.size();
    if (bytes >= kStagedMin)
        copy_to_device(dst.get(), src.data(), bytes, s);
    else
        DCRF_HIP_CHECK(hipMemcpyAsync(dst.get(), src.data(), bytes, hipMemcpyHostToDevice, s));
}

void ensure_unary(dcrf_model& m) {
    if (!m.has_unary || !m.unary_dirty) return;
    const size_t n = (size_t)m.N() * m.L;
    if (m.logistic) {
        // LogisticUnaryEnergy::get (unary.cpp:50-52) on the matrix cores
        m.unary.reserve(n);
        upload(m.lL_dev, m.lL, m.stream);
        launch_logistic_unary(m.lfFN.get(), m.lL_dev.get(), m.N(), m.lF, m.L, m.unary.get(), m.stream);
        DCRF_HIP_CHECK(hipStreamSynchronize(m.stream));
        m.unary_dirty = false;
        return;
    }
    if (m.unary_pin.p) {
        m.unary.reserve(n);
        start_unary_upload(m);
        DCRF_HIP_CHECK(hipStreamWaitEvent(m.stream, m.unary_ev, 0));
        launch_transpose(m.stage.get(), m.unary.get(), m.L, m.N(), m.stream);
        DCRF_HIP_CHECK(hipStreamSynchronize(m.stream));
        m.unary_uploading = false;
        m.unary_pin.give();
        m.unary_dirty = false;
        return;
    }
    m.stage.reserve(n);
    m.unary.reserve(n);
    for (int i = 0; i < (int)m.unary_unset.size(); i++)
        if (m.unary_unset[i]) {  // an instance never given a unary: zeros, as the first set left them
            const int b = m.geo.pix_base[i], Ni = m.geo.N[i];
            for (int l = 0; l < m.L; l++) std::fill_n(m.unary_host.data() + (size_t)l * m.N() + b, Ni, 0.f);
            m.unary_unset[i] = 0;
        }
    copy_to_device(m.stage.get(), m.unary_host.data(), sizeof(float) * n, m.stream);
    launch_transpose(m.stage.get(), m.unary.get(), m.L, m.N(), m.stream);
    DCRF_HIP_CHECK(hipStreamSynchronize(m.stream));
    m.unary_dirty = false;
}

inline bool pre_norm(int ntype, bool transpose) {
    return ntype == DCRF_NORMALIZE_SYMMETRIC || (ntype == DCRF_NORMALIZE_BEFORE && !transpose) ||
           (ntype == DCRF_NORMALIZE_AFTER && transpose);
}
inline bool post_norm(int ntype, bool transpose) {
    return ntype == DCRF_NORMALIZE_SYMMETRIC || (ntype == DCRF_NORMALIZE_BEFORE && transpose) ||
           (ntype == DCRF_NORMALIZE_AFTER && !transpose);
}
// Alpha of the slice (permutohedral.cpp:571): 1 / (1 + 2^-d) in float.
inline float slice_alpha(int d) { return 1.0f / (1.0f + std::pow(2.0f, (float)-d)); }

TileGeom tile_geom(const dcrf_model& m) {
    return TileGeom{m.tiles.base_dev.get(), m.geod.pix_base.get(), m.geo.is2d ? m.geod.W.get() : nullptr,
                    m.geo.n_inst, m.geo.is2d ? 1 : 0, m.tiles.side};
}

// Multi-step blur schedule: a lattice runs its d+1 steps in ceil((d+1)/K) passes of at
// most K steps, spread as evenly as possible (longer passes first); the number of passes
// falls with d, so in the global filter pass p covers a prefix of the vertex space.
// K = 2 by default: passes of three steps (27 rows per vertex) for every lattice
// measured slower at 1024x768x21 (49 us against 28 us of blur per iteration), as the
// 27 gathers per vertex of the large Gaussian lattice cost more than the launch saved.
constexpr int kMaxPassSteps = 2;
std::vector<int> pass_schedule(int steps, int K = kMaxPassSteps) {
    const int n = (steps + K - 1) / K;
    std::vector<int> out(n, steps / n);
    for (int i = 0; i < steps % n; i++) out[i]++;
    return out;
}

// Most steps per pass of every term (dcrf_set_blur_steps: 2, the default, or 3).  Each
// pass is one launch over the terms that still have passes, and a short launch costs
// ~5 us whatever its work (a pass over the 36 k vertices of the 1024x768 bilateral
// lattice alone: 5.1-5.5 us), but three-step passes for that lattice only (3 + 3 beside
// the Gaussian lattice's 2 + 1: two launches instead of three) measured 2 x 25.8 us of
// blur per iteration against 3 x 12.9 us: its 27-row trees, folded one 9-row subtree
// after another, make each launch's tail three memory round trips long.
std::vector<int> pass_step_limits(const dcrf_model& m) {
    return std::vector<int>(m.terms.size(), m.blur_steps);
}

// Pass tables of one lattice (forward axes 0..d, reverse d..0) over its neighbour rows
// nbr [(d+1)][V] (global rows from vbase, zero row zero_row), passes of at most K steps.
void build_pass_tables(const int2* nbr, int V, int d, int vbase, int zero_row, std::vector<int>& steps,
                       std::vector<int>& off, DevBuf<int>& fwd, DevBuf<int>& rev, int K,
                       std::vector<PassTableJob>& jobs) {
    steps = pass_schedule(d + 1, K);
    off.assign(1, 0);
    for (int q : steps) off.push_back(off.back() + V * (q == 1 ? 3 : q == 2 ? 9 : 27));
    fwd.reserve(off.back());
    rev.reserve(off.back());
    int first = 0;
    for (size_t p = 0; p < steps.size(); p++) {
        const int q = steps[p];
        PassTableJob f{nbr, fwd.get() + off[p], V, vbase, zero_row, q, {}};
        PassTableJob r{nbr, rev.get() + off[p], V, vbase, zero_row, q, {}};
        for (int j = 0; j < q; j++) {
            f.axes[j] = first + j;
            r.axes[j] = d - first - j;
        }
        jobs.push_back(f);
        jobs.push_back(r);
        first += q;
    }
}

// The counting of the segment lists for rows of Lr floats (padding included): in-wave runs
// where a segment's lanes fit a wave (and runs is set), recombination in one launch.
void plan_segments(const RunSet& rs, int Lr, bool runs, SegPlan& P, hipStream_t s) {
    const LaunchShape sh = shape_for(Lr);
    count_segments(rs, sh.wave && runs ? splat_shape(Lr).per : 0, sh.wave ? sh.per : 0, false, P, s);
}

// The same for the filters of the kernel-parameter gradient: every vertex's segments in one
// sequence, whatever the row length and the other terms (the normalisers' sums have that
// order too, splat_ones).  The
// parameter gradient amplifies the last bits of its vertex rows and of the normalisers a
// hundred times (two orders of summation differ by 1e-5 of the result at 512x512x21), so
// these sums keep one order; it costs 11 us a recombination there against in-wave runs
// and whole waves for the long ones.
void plan_sequential(const RunSet& rs, SegPlan& P, hipStream_t s) { count_segments(rs, 0, 0, true, P, s); }

// Splat of rows of Lr floats (stride Lr) over a list, and its recombination.
void splat_lists(const SegLists& l, const int2* ent, const float* in, size_t rows_in, int Lr, float* vals,
                 hipStream_t s) {
    launch_splat(l.ch.get(), l.nch, ent, in, rows_in, Lr, vals, Lr, Lr, s);
}
void combine_lists(const SegLists& l, int Lr, float* vals, hipStream_t s) {
    if (l.waves)
        launch_combine_waves(l.cb.get(), l.ncb, vals, Lr, Lr, s);
    else
        launch_combine(l.cb.get(), l.ncb, vals, Lr, Lr, s);
    launch_combine(l.cb2.get(), l.ncb2, vals, Lr, Lr, s);
}

// ---------------------------------------------------------------- kernel-parameter gradient
// The blur passes of one layout (x: the x chains, else the forward and reverse chains
// of the paired inputs) from the splat rows src through the ping-pong pair buf: pass p
// runs the chains of the parts with more than p passes over rows [0, vp[p]).  Part i's
// result is in buf[(passes - 1) & 1].
void kg_blur(const KgPlan& P, bool x, const float* src, float* const buf[2], int Lc, hipStream_t s) {
    const float* in = src;
    for (int p = 0; p < P.passes; p++) {
        PassTable pt{};
        pt.nterms = 0;
        for (size_t i = 0; i < P.parts.size() && P.parts[i].passes > p; i++) {
            const KgPart& part = P.parts[i];
            const int q = part.steps[p];
            const int* tab = P.tab.get();
            const std::vector<int>& off = P.tab_off[p];
            if (x) {
                pt.t[pt.nterms++] = PassTerm{part.X, part.V, tab + off[3 * i + 2], q};
            } else {
                pt.t[pt.nterms++] = PassTerm{part.F, part.V, tab + off[3 * i], q};
                pt.t[pt.nterms++] = PassTerm{part.R, part.V, tab + off[3 * i + 1], q};
            }
        }
        pt.zero_row = x ? P.Z1 : P.Z2;
        launch_blur_pass(in, buf[p & 1], 0, x ? P.vp1[p] : P.vp2[p], Lc, Lc, pt, s);
        in = buf[p & 1];
    }
}

// Fill plan P for the model terms `terms` (at most DCRF_MAX_TERMS / 2; P's device
// buffers are reused where they are large enough): the layouts of KgPlan, the merged
// segment and entry lists (those of the paired rows mapped from the x layout's on the
// device), the pass tables
// of every chain, and per term the slice weights and the all-ones input splatted and
// blurred in reverse order (one value per vertex, through the plan's own launches: the
// same segments, sums and pass order as a filter of that term alone).
void build_kg_plan(dcrf_model& m, std::vector<int> terms, KgPlan& P) {
    hipStream_t s = m.stream;
    const int N = m.N();
    const size_t L = m.L;
    auto steps_of = [&](int k) { return pass_schedule(m.terms[k]->lat.d + 1, kMaxPassSteps); };
    std::stable_sort(terms.begin(), terms.end(),
                     [&](int a, int b) { return steps_of(a).size() > steps_of(b).size(); });
    std::vector<KgPart> old = std::move(P.parts);
    P.parts.clear();
    P.passes = 0;
    int row = 0, xrow = 0;
    size_t E = 0;
    for (size_t i = 0; i < terms.size(); i++) {
        const int k = terms[i];
        const TermLattice& lat = m.terms[k]->lat;
        KgPart part;
        if (i < old.size()) part.sw = std::move(old[i].sw);
        part.term = k;
        part.V = lat.V;
        part.steps = steps_of(k);
        part.passes = (int)part.steps.size();
        part.F = row;
        part.R = row + lat.V;
        part.X = xrow;
        row += 2 * lat.V;
        xrow += lat.V;
        E += (size_t)N * (lat.d + 1);
        P.passes = std::max(P.passes, part.passes);
        P.parts.push_back(std::move(part));
    }
    P.Z2 = row;
    P.Z1 = xrow;
    // merged segment lists in the x layout's rows (the terms' vertices one after another):
    // one for x, one for [a | c] and the all-ones input, whose rows are then moved to the
    // paired layout
    RunSet rs;
    {
        std::vector<const TermLattice*> lats;
        std::vector<int> xbase;
        for (const KgPart& part : P.parts) {
            lats.push_back(&m.terms[part.term]->lat);
            xbase.push_back(part.X);
        }
        build_run_set(lats, xbase, m.tiles.n_tiles(), m.chunk(), rs, s);
    }
    SegPlan sp;
    plan_sequential(rs, sp, s);
    P.ent.reserve(E);
    for (size_t i = 0; i < P.parts.size(); i++) {
        const TermLattice& lat = m.terms[P.parts[i].term]->lat;
        const int d1 = lat.d + 1;
        launch_entry_gather(lat.csr_e.get(), N * d1, d1, lat.bary.get(), nullptr, 0, lat.tile_ptr.get(),
                            rs.gebase.get(), rs.NT, rs.T, (int)i, nullptr, P.ent.get(), s, (int)i * N);
    }
    KgRowMap rm{};
    rm.n = (int)P.parts.size();
    rm.Z2 = P.Z2;
    rm.Z1 = P.Z1;
    for (size_t i = 0; i < P.parts.size(); i++) {
        rm.F[i] = P.parts[i].F;
        rm.X[i] = P.parts[i].X;
    }
    DCRF_HIP_CHECK(hipStreamSynchronize(s));  // the counts
    emit_segments(rs, sp, P.Z1 + 1, P.l1, s);
    emit_segments(rs, sp, P.Z1 + 1, P.l2, s);
    launch_kg_relayout(P.l2.ch.get(), P.l2.nch, P.l2.cb.get(), P.l2.ncb, rm, s);
    P.l2.rows += P.Z2 - P.Z1;
    // pass tables: pass p of term i expands the axes of its p-th pass; the forward chain
    // reads rows from F, the reverse chain from F in its first pass (the splat rows) and
    // from R after, the x chain from X
    size_t tab_total = 0;
    for (const KgPart& part : P.parts)
        for (int q : part.steps) tab_total += (size_t)3 * part.V * (q == 1 ? 3 : 9);
    P.tab.reserve(std::max<size_t>(tab_total, 1));
    P.tab_off.assign(P.passes, std::vector<int>(3 * P.parts.size(), -1));
    P.vp2.assign(P.passes, 0);
    P.vp1.assign(P.passes, 0);
    size_t toff = 0;
    std::vector<PassTableJob> jobs;
    std::vector<std::array<DevBuf<int2>, 3>> nbrs(P.parts.size());  // until the tables are built
    for (size_t i = 0; i < P.parts.size(); i++) {
        KgPart& part = P.parts[i];
        const TermLattice& lat = m.terms[part.term]->lat;
        const int V = lat.V, d = lat.d, d1 = d + 1;
        DevBuf<int2>&nF = nbrs[i][0], &nR = nbrs[i][1], &nX = nbrs[i][2];  // the neighbour rows in each chain's numbering
        nF.reserve((size_t)d1 * V);
        nR.reserve((size_t)d1 * V);
        nX.reserve((size_t)d1 * V);
        launch_remap_nbr(lat.nbr.get(), nF.get(), d1 * V, part.F, P.Z2, s);
        launch_remap_nbr(lat.nbr.get(), nR.get(), d1 * V, part.R, P.Z2, s);
        launch_remap_nbr(lat.nbr.get(), nX.get(), d1 * V, part.X, P.Z1, s);
        int first = 0;
        for (int p = 0; p < part.passes; p++) {
            const int q = part.steps[p];
            int fa[3], ta[3];
            for (int j = 0; j < q; j++) {
                fa[j] = first + j;
                ta[j] = d - first - j;
            }
            const size_t n = (size_t)V * (q == 1 ? 3 : 9);
            std::vector<int>& off = P.tab_off[p];
            off[3 * i] = (int)toff;
            auto table = [&](const int2* nbr, int base, int zero_row, const int* axes) {
                PassTableJob t{nbr, P.tab.get() + toff, V, base, zero_row, q, {}};
                std::copy(axes, axes + q, t.axes);
                jobs.push_back(t);
            };
            table(nF.get(), part.F, P.Z2, fa);
            toff += n;
            off[3 * i + 1] = (int)toff;
            if (p == 0)
                table(nF.get(), part.F, P.Z2, ta);
            else
                table(nR.get(), part.R, P.Z2, ta);
            toff += n;
            off[3 * i + 2] = (int)toff;
            table(nX.get(), part.X, P.Z1, fa);
            toff += n;
            P.vp2[p] = part.R + V;  // the parts are in decreasing pass count
            P.vp1[p] = part.X + V;
            first += q;
        }
        DevBuf<int> gv;
        gv.reserve((size_t)N * d1);
        part.sw.reserve((size_t)N * d1);
        launch_slice_weights(lat.vtx.get(), lat.bary.get(), nullptr, 0, slice_alpha(d), N, d1, 0, gv.get(),
                             part.sw.get(), nullptr, 0, 0, s);
    }
    launch_pass_tables(jobs, s);
    // vertex rows: the zero rows stay zero (splats write vertex and partial rows, the
    // blur passes rows below the zero row)
    auto zeroed = [&](DevBuf<float>& b, size_t n) {
        b.reserve(n);
        launch_fill(b.get(), 0.f, n, s);
    };
    zeroed(P.S2, (size_t)P.l2.rows * 2 * L);
    zeroed(P.X2[0], (size_t)(P.Z2 + 1) * 2 * L);
    zeroed(P.X2[1], (size_t)(P.Z2 + 1) * 2 * L);
    zeroed(P.S1, (size_t)P.l1.rows * L);
    zeroed(P.B1, (size_t)(P.Z1 + 1) * L);
    // the all-ones input of every term (stacked, one value per pixel) through the plan's
    // splat and both chains; the reverse rows are the terms' K^T 1
    zeroed(P.ones[0], (size_t)P.l2.rows);
    zeroed(P.ones[1], (size_t)P.Z2 + 1);
    zeroed(P.ones[2], (size_t)P.Z2 + 1);
    DevBuf<float> in1;
    in1.reserve((size_t)P.parts.size() * N);
    launch_fill(in1.get(), 1.f, (size_t)P.parts.size() * N, s);
    splat_lists(P.l2, P.ent.get(), in1.get(), P.parts.size() * (size_t)N, 1, P.ones[0].get(), s);
    combine_lists(P.l2, 1, P.ones[0].get(), s);
    float* const obuf[2] = {P.ones[1].get(), P.ones[2].get()};
    kg_blur(P, false, P.ones[0].get(), obuf, 1, s);
    for (KgPart& part : P.parts) part.ones_rev = obuf[(part.passes - 1) & 1] + part.R;
    P.gen = m.lat_gen;
    DCRF_HIP_CHECK(hipStreamSynchronize(s));  // the uploads from host lists are complete
}

// The plans of the terms with kernel parameters, rebuilt (in place) when a lattice
// changed.  A plan takes at most DCRF_MAX_TERMS / 2 terms (a pass launch holds two chains
// per term), and its stacked input rows, entries and vertex rows stay within int.
void ensure_kg_plans(dcrf_model& m) {
    if (!m.kgplans.empty() && m.kgplans.front()->gen == m.lat_gen) return;
    const long long N = m.N(), lim = std::numeric_limits<int>::max();
    std::vector<std::vector<int>> groups;
    std::vector<int> g;
    long long e = 0, rows = 0;
    for (int k = 0; k < (int)m.terms.size(); k++) {
        const Term& t = *m.terms[k];
        if (!t.num_kparams()) continue;
        // (sequential lists: at most one partial row per segment, no second level)
        const long long ek = N * (t.lat.d + 1), rk = 2LL * t.lat.V + ek / std::max(1, m.chunk()) + t.lat.n_runs;
        if (!g.empty() && ((int)g.size() == DCRF_MAX_TERMS / 2 || e + ek > lim || rows + rk + 1 > lim ||
                           (long long)(g.size() + 1) * N > lim)) {
            groups.push_back(g);
            g.clear();
            e = rows = 0;
        }
        g.push_back(k);
        e += ek;
        rows += rk;
    }
    if (!g.empty()) groups.push_back(g);
    m.kgplans.resize(groups.size());
    for (size_t i = 0; i < groups.size(); i++) {
        if (!m.kgplans[i]) m.kgplans[i] = std::make_unique<KgPlan>();
        build_kg_plan(m, groups[i], *m.kgplans[i]);
    }
}

// acc_k += kernelGradient(b, Q_t) for every term k of plan P (pairwise.cpp:202-207,
// 152-163, 88-114): fg = -G(x, 1) + G(a, c) with a, c and x per the normalisation type.
// One pass forms the terms' inputs a and c from C (w Q_t) and b; the [a | c] of all the
// plan's terms are splatted together and blurred in both orders: the forward rows give
// K a (G(a, c), direction 0) and K c, the reverse rows K^T a and K^T c (G(a, c),
// direction 1).  x (from the slices K^T a and K c in one pass per term) needs one more
// splat and forward blur, and G(x, 1)'s direction 1 is the term's reverse-blurred ones.
// The four slicing gradients and the parameter products then run in one pass per term
// (its partial rows at partial + k * pstride, summed after the last iteration) where the
// lane-group kernel covers the shape, else per direction with a reduction into acc.
void kernel_grad_group(dcrf_model& m, const KgPlan& P, const float* b, const float* Qt, const float* kw,
                       const std::vector<int>& koff, size_t pstride, hipStream_t s) {
    const int N = m.N(), L = m.L, L2 = 2 * L;
    const size_t NL = (size_t)N * L;
    const int T = (int)P.parts.size();
    float* pk = m.kgbuf.get();            // [T][N][2L]
    float* xb = pk + (size_t)2 * T * NL;  // [T][N][L]
    float* lbl = xb + (size_t)T * NL;     // [T][N][L]
    bool any_x = false;
    SliceTable pst{};
    KgInputs in{};
    pst.nterms = T;
    for (int i = 0; i < T; i++) {
        const int k = P.parts[i].term;
        const Term& t = *m.terms[k];
        any_x = any_x || t.ntype != DCRF_NO_NORMALIZATION;
        pst.t[i] = SliceTerm{nullptr, nullptr, nullptr, 1, t.ckind, t.d_compat.get(), kw ? kw + k : nullptr, nullptr, L};
        in.norm[i] = t.norm.get();
        in.ntype[i] = t.ntype;
        // x reads fa and lbl, but for AFTER
        const bool need_fa = t.ntype != DCRF_NO_NORMALIZATION && t.ntype != DCRF_NORMALIZE_AFTER;
        in.lbl[i] = need_fa ? lbl + (size_t)i * NL : nullptr;
    }
    launch_kg_prepare(Qt, b, m.ldv, in, N, L, pst, pk, s);
    splat_lists(P.l2, P.ent.get(), pk, (size_t)T * N, L2, P.S2.get(), s);
    combine_lists(P.l2, L2, P.S2.get(), s);
    float* const pbuf[2] = {P.X2[0].get(), P.X2[1].get()};
    kg_blur(P, false, P.S2.get(), pbuf, L2, s);
    float* const xbuf[2] = {P.B1.get(), P.S1.get()};  // pass 0 reads the splat rows S1
    auto fwd_of = [&](int i) { return pbuf[(P.parts[i].passes - 1) & 1] + (size_t)P.parts[i].F * L2; };
    auto rev_of = [&](int i) { return pbuf[(P.parts[i].passes - 1) & 1] + (size_t)P.parts[i].R * L2; };
    if (any_x) {
        for (int i = 0; i < T; i++) {
            const Term& t = *m.terms[P.parts[i].term];
            float* x = xb + (size_t)i * NL;
            if (t.ntype == DCRF_NO_NORMALIZATION) {  // splatted with the others, never read
                launch_fill(x, 0.f, NL, s);
                continue;
            }
            const bool need_fa = t.ntype != DCRF_NORMALIZE_AFTER, need_fb = t.ntype != DCRF_NORMALIZE_BEFORE;
            SliceTable st{};
            st.nterms = 2;
            const int* vtx = t.lat.vtx.get();
            const float* sw = P.parts[i].sw.get();
            const int d1 = t.lat.d + 1;
            st.t[0] = SliceTerm{vtx, sw, need_fa ? rev_of(i) : nullptr, d1, -1, nullptr, nullptr, nullptr, L2};  // K^T a
            st.t[1] = SliceTerm{vtx, sw, need_fb ? fwd_of(i) + L : nullptr, d1, -1, nullptr, nullptr, nullptr, L2};  // K c
            launch_kg_x(b, m.ldv, lbl + (size_t)i * NL, t.norm.get(), N, L, st, t.ntype, x, s);
        }
        splat_lists(P.l1, P.ent.get(), xb, (size_t)T * N, L, P.S1.get(), s);
        combine_lists(P.l1, L, P.S1.get(), s);
        kg_blur(P, true, P.S1.get(), xbuf, L, s);
    }
    for (int i = 0; i < T; i++) {
        const KgPart& part = P.parts[i];
        const int k = part.term;
        const Term& t = *m.terms[k];
        const int d = t.lat.d;
        const bool has_x = t.ntype != DCRF_NO_NORMALIZATION;
        const float* fwd = fwd_of(i);
        const float* rev = rev_of(i);
        const float* xr = has_x ? xbuf[(part.passes - 1) & 1] + (size_t)part.X * L : nullptr;
        const float* pki = pk + (size_t)i * 2 * NL;
        const float* x = xb + (size_t)i * NL;
        const int* vtx = t.lat.vtx.get();
        const int* rank = t.lat.rank.get();
        const bool full = t.ktype == DCRF_FULL_KERNEL;
        double* partial = m.kpartial.get() + (size_t)k * pstride;
        if (kg_grad_fused(L, d)) {
            launch_kg_grad(vtx, rank, fwd, rev, pki, xr, part.ones_rev, x, t.feat0.get(), m.geod.pix_base.get(),
                           m.geod.pad_base.get(), m.geo.n_inst, N, L, d, full, partial, s);
            continue;
        }
        // more labels than a wave's lanes hold, or d > 6: one thread per point and direction
        float* dfr = m.kgdf.get();
        float* dfg = dfr + (size_t)N * d;
        if (has_x) {
            launch_slice_grad(xr, L, 1, vtx, rank, nullptr, 0, N, L, d, 0, dfr, s);
            launch_slice_grad(part.ones_rev, 1, 0, vtx, rank, x, L, N, L, d, 1, dfr, s);
        }
        launch_slice_grad(fwd, L2, 1, vtx, rank, pki + L, L2, N, L, d, 0, dfg, s);
        launch_slice_grad(rev + L, L2, 1, vtx, rank, pki, L2, N, L, d, 1, dfg, s);
        launch_kparam_reduce(has_x ? dfr : nullptr, dfg, t.feat0.get(), m.geod.pix_base.get(), m.geod.pad_base.get(),
                             m.geo.n_inst, N, d, full, partial, m.kacc.get() + koff[k], s);
    }
}

int num_kernel_params(const dcrf_model& m) {
    int n = 0;
    for (const auto& t : m.terms) n += t->num_kparams();
    return n;
}

void add_term(dcrf_model& m, int d, int ckind, const float* compat, int ktype, int ntype,
              const std::function<void(float*)>& make_features) {
    require((int)m.terms.size() < DCRF_MAX_TERMS, "at most " + std::to_string(DCRF_MAX_TERMS) + " pairwise terms");
    require(d >= 1 && d <= DCRF_MAX_DIM, "feature dimension must be between 1 and " + std::to_string(DCRF_MAX_DIM));
    require(ckind >= DCRF_COMPAT_POTTS && ckind <= DCRF_COMPAT_MATRIX, "unknown label compatibility kind");
    require(ktype >= DCRF_CONST_KERNEL && ktype <= DCRF_FULL_KERNEL, "unknown kernel type");
    require(ntype >= DCRF_NO_NORMALIZATION && ntype <= DCRF_NORMALIZE_SYMMETRIC, "unknown normalization type");
    require(compat != nullptr, "compatibility parameters missing");
    ensure_device(m);
    auto t = std::make_unique<Term>();
    t->ktype = ktype;
    t->ntype = ntype;
    t->ckind = ckind;
    const int L = m.L;
    if (ckind == DCRF_COMPAT_POTTS) {
        t->compat.assign(compat, compat + 1);
    } else if (ckind == DCRF_COMPAT_DIAGONAL) {
        t->compat.assign(compat, compat + L);
    } else {
        // MatrixCompatibility stores 0.5*(m + m^T) (labelcompatibility.cpp:79)
        t->compat.resize((size_t)L * L);
        for (int a = 0; a < L; a++)
            for (int b = 0; b < L; b++) {
                const float s = compat[a * L + b] + compat[b * L + a];
                t->compat[(size_t)a * L + b] = 0.5f * s;
            }
    }
    try {
        start_unary_upload(m);
    } catch (const Error&) {  // no memory for it yet: the first inference uploads
    }
    t->d_compat.reserve(t->compat.size());
    DCRF_HIP_CHECK(hipMemcpy(t->d_compat.get(), t->compat.data(), sizeof(float) * t->compat.size(),
                             hipMemcpyHostToDevice));
    DevBuf<float> feat;
    feat.reserve((size_t)m.geo.npad_total() * d);
    make_features(feat.get());
    if (!m.tiles_ready) {
        make_tile_map(m.geo, m.tile_side ? m.tile_side : default_tile_side(m.L), m.tiles);
        m.tiles_ready = true;
    }
    build_lattice(m.geo, m.geod, m.tiles, feat.get(), d, t->lat, m.hash_load, m.stream);
    if (t->lat.overflow)
        throw Error{DCRF_ERR_OVERFLOW,
                    "a lattice coordinate exceeds the int16 range of the lattice keys; scale the features down"};
    // (the normaliser is computed with the layout)
    // DenseKernel keeps f_ and starts from unit scales / the identity (pairwise.cpp:116-122)
    t->feat0 = std::move(feat);
    t->kparams.assign(ktype == DCRF_FULL_KERNEL ? (size_t)d * d : (size_t)d, 0.0f);
    for (int j = 0; j < d; j++) t->kparams[ktype == DCRF_FULL_KERNEL ? j * d + j : j] = 1.0f;
    m.terms.push_back(std::move(t));
    m.layout_valid = false;
    m.lat_gen++;
    m.kw_set = false;  // term weights are per term: set them again after adding terms
    m.train_n = -1;
}

SliceTable slice_table(const dcrf_model& m, bool transpose, const float* kw = nullptr, float* mout = nullptr);

// The vertex buffer holding term k's filtered rows after the global filter: one buffer
// switch per blur step, or per multi-step pass.
int result_parity(const dcrf_model& m, int k) {
    return (m.pairs ? (int)m.tl[k]->pass_steps.size() : m.terms[k]->lat.d + 1) & 1;
}

// Launches per filter with multi-step passes (after the terms' pass tables exist).
int blur_launches(const dcrf_model& m) {
    int P = 0;
    for (const auto& tl : m.tl) P = std::max(P, (int)tl->pass_steps.size());
    return P;
}

BlurTable blur_table(const dcrf_model& m);

// All blur passes over rows of Lv floats, between the buffers v0 (the splat rows) and v1:
// afterwards term k's rows are in the one of result_parity(m, k).
void blur_rows(dcrf_model& m, float* v0, float* v1, int Lv, bool transpose, hipStream_t s) {
    float* const v[2] = {v0, v1};
    const int L = m.L;
    if (m.pairs) {
        // up to three blur steps per pass; terms in layout order, pass p covers the
        // terms with more than p passes (a prefix of the vertex space)
        for (int p = 0; p < m.n_passes; p++) {
            PassTable pt{};
            pt.nterms = (int)m.order.size();
            pt.zero_row = m.V_total;  // zero in both vertex buffers
            double bytes = 0.0;
            for (int i = 0; i < pt.nterms; i++) {
                const int k = m.order[i];
                const TermLattice& lat = m.terms[k]->lat;
                const TermLayout& lay = *m.tl[k];
                const bool on = (int)lay.pass_steps.size() > p;
                const int steps = on ? lay.pass_steps[p] : 1;
                pt.t[i] = PassTerm{m.vbase[k], lat.V,
                                   on ? (transpose ? lay.passT.get() : lay.passF.get()) + lay.pass_off[p] : nullptr,
                                   steps};
                if (on) bytes += (double)lat.V * steps * (2.0 * L * 4 + 8);
            }
            Timed t(m, s, KC_BLUR, bytes);
            const int pr = m.blur_r > 0 && (m.blur_small_v <= 0 || m.prefixP[p] < m.blur_small_v) ? m.blur_r : 0;
            launch_blur_pass(v[p & 1], v[(p + 1) & 1], 0, m.prefixP[p], Lv, Lv, pt, s, pr);
            t.done();
        }
        return;
    }
    const BlurTable bt = blur_table(m);
    for (int step = 0; step <= m.max_d; step++) {
        Timed t(m, s, KC_BLUR, (double)m.prefixV[step] * (2.0 * L * 4 + 8));
        launch_blur(v[step & 1], v[(step + 1) & 1], 0, m.prefixV[step], Lv, Lv, bt, step,
                    transpose ? 1 : 0, s);
        t.done();
    }
}

// norm = N / sum(norm) per instance, in float (pairwise.cpp:46-53).
void mean_norms(const dcrf_model& m, float* norm, hipStream_t s) {
    const int N = m.N();
    std::vector<float> h(N);
    DCRF_HIP_CHECK(hipMemcpyAsync(h.data(), norm, sizeof(float) * N, hipMemcpyDeviceToHost, s));
    DCRF_HIP_CHECK(hipStreamSynchronize(s));
    for (int i = 0; i < m.geo.n_inst; i++) {
        const int b = m.geo.pix_base[i], e = m.geo.pix_base[i + 1];
        float mean = 0.f;
        for (int p = b; p < e; p++) mean += h[p];
        mean = (float)(e - b) / mean;
        for (int p = b; p < e; p++) h[p] = mean;
    }
    DCRF_HIP_CHECK(hipMemcpyAsync(norm, h.data(), sizeof(float) * N, hipMemcpyHostToDevice, s));
    DCRF_HIP_CHECK(hipStreamSynchronize(s));
}

NormTerm norm_term(const Term& t, const float* vals, int vbase, float* norm) {
    const TermLattice& lat = t.lat;
    return NormTerm{lat.vtx.get(), lat.bary.get(), vals, norm, slice_alpha(lat.d), lat.d + 1, vbase, t.ntype};
}

// The normalisers of all terms: norm = K 1 (pairwise.cpp:44), then the normalisation of
// :46-61.  One filter of the all-ones input over every term's lattice, one float a row,
// through the layout's run set and pass tables.
//   A new small model is a chain of short launches (64x48: 94 with the two lattice builds),
// so their number counts.  The sums need an order of their own (see plan_sequential), but
// no segment list and no entries (splat_ones); with those, and a slice per term, a new
// model took 127.  First inference of a new model, 10 iterations: 64x48x21 606 -> 444 us,
// 320x213x21 740 -> 580, 1024x768x21 2090 -> 1870.
void compute_norms(dcrf_model& m, const std::vector<const TermLattice*>& lats, const RunSet& rs, const SegPlan& sp,
                   hipStream_t s) {
    struct Untimed {  // these launches are no part of the timed classes
        dcrf_model& m;
        bool was;
        explicit Untimed(dcrf_model& m_) : m(m_), was(m_.timing) { m.timing = false; }
        ~Untimed() { m.timing = was; }
    } untimed(m);
    const int V = m.V_total;
    DevBuf<float> v0, v1;
    v0.reserve((size_t)V + 1);
    v1.reserve((size_t)V + 1);
    splat_ones(lats, rs, sp, v0.get(), v1.get(), s);
    blur_rows(m, v0.get(), v1.get(), 1, false, s);
    NormTerms nt{};
    for (int k : m.order) {
        Term& t = *m.terms[k];
        t.norm.reserve(m.N());
        nt.t[nt.T++] = norm_term(t, result_parity(m, k) ? v1.get() : v0.get(), m.vbase[k], t.norm.get());
    }
    launch_norms(nt, m.N(), s);
    for (int k : m.order)
        if (m.terms[k]->ntype == DCRF_NO_NORMALIZATION) mean_norms(m, m.terms[k]->norm.get(), s);
}

// One term's normaliser without a layout (dcrf_get_lattice): the same sums.
void term_norm(const dcrf_model& m, const Term& t, DevBuf<float>& norm) {
    const TermLattice& lat = t.lat;
    const int V = lat.V, d1 = lat.d + 1;
    hipStream_t s = m.stream;
    RunSet rs;
    SegPlan sp;
    build_run_set({&lat}, {0}, lat.n_tiles, m.chunk(), rs, s);
    count_segments(rs, 0, 0, true, sp, s);
    DevBuf<float> v[2];
    for (DevBuf<float>& b : v) b.reserve((size_t)V + 1);
    splat_ones({&lat}, rs, sp, v[0].get(), v[1].get(), s);
    DevBuf<int2> nbr;
    nbr.reserve((size_t)d1 * V);
    launch_remap_nbr(lat.nbr.get(), nbr.get(), d1 * V, 0, V, s);
    BlurTable bt{};
    bt.nterms = 1;
    bt.t[0] = BlurTerm{0, V, lat.d, nbr.get()};
    for (int step = 0; step < d1; step++)
        launch_blur(v[step & 1].get(), v[(step + 1) & 1].get(), 0, V, 1, 1, bt, step, 0, s);
    norm.reserve(m.N());
    NormTerms nt{};
    nt.T = 1;
    nt.t[0] = norm_term(t, v[d1 & 1].get(), 0, norm.get());
    launch_norms(nt, m.N(), s);
    if (t.ntype == DCRF_NO_NORMALIZATION) mean_norms(m, norm.get(), s);
    DCRF_HIP_CHECK(hipStreamSynchronize(s));
}

// The limit of the allocation-free inference counts the rows of a layout without padding
// labels and with one lane group per segment, whatever the splat's form: the quad form has
// more partial rows, padded rows of fewer lanes have fewer, and neither moves the line
// between the models that the call takes and those it refuses.
constexpr size_t kNoAllocRowBytes = (size_t)64 << 20;
size_t noalloc_rows(const dcrf_model& m, const RunSet& rs, const SegPlan& sp, hipStream_t s) {
    const LaunchShape sh = shape_for(m.L);
    const int per = sh.wave ? sh.per : 0;
    const size_t rows = (size_t)m.rows0 + m.V_total + 1;
    if (m.tiled || !rs.T || (sp.per == per && sp.perc == per)) return rows;
    // no layout has more partial and second-level rows than twice the segments
    const size_t most = 2 * ((size_t)m.V_total + 1) + 2 * (size_t)sp.host[1].partial;
    if (most * m.L * sizeof(float) <= kNoAllocRowBytes) return rows;
    SegPlan p;
    count_segments(rs, per, per, false, p, s);
    DCRF_HIP_CHECK(hipStreamSynchronize(s));
    return 2 * ((size_t)m.V_total + 1) + p.host[0].partial + (per ? 0 : p.host[0].pieces);
}

// Sets the stride of the gathered rows.  A training forward's Q_t were stored with the
// stride of its time and a later backward reads them with the present one: they move along.
void set_row_stride(dcrf_model& m, int ldv, hipStream_t s) {
    if (ldv != m.ldv && m.train_n > 0) {
        const int N = m.N(), L = m.L, n = m.train_n;
        DevBuf<float> q;  // (layout: forward_train)
        q.reserve((size_t)N * ((size_t)n * ldv + L));
        // (the caller's stream wrote them)
        DCRF_HIP_CHECK(hipDeviceSynchronize());
        for (int t = 0; t <= n; t++)
            launch_restride_rows(m.qcache.get() + (size_t)t * N * m.ldv, t < n ? m.ldv : L,
                                 q.get() + (size_t)t * N * ldv, t < n ? ldv : L, N, L, s);
        m.qcache = std::move(q);
    }
    m.ldv = ldv;
}

void build_layout(dcrf_model& m);

void ensure_layout(dcrf_model& m) {
    if (m.layout_valid) return;
    try {
        build_layout(m);
    } catch (...) {
        m.train_n = -1;  // (a backward reads the layout)
        throw;
    }
}

void build_layout(dcrf_model& m) {
    m.drop_graph();
    m.qblocks_ready = false;
    hipStream_t s = m.stream;
    const int T = (int)m.terms.size();
    const int N = m.N(), L = m.L;
    // terms in layout order: more blur passes first (then higher d), so that the terms
    // of pass p are a prefix of the vertex space
    const std::vector<int> step_limit = pass_step_limits(m);
    std::vector<int> npass(T);
    for (int k = 0; k < T; k++) npass[k] = (int)pass_schedule(m.terms[k]->lat.d + 1, step_limit[k]).size();
    m.order.resize(T);
    std::iota(m.order.begin(), m.order.end(), 0);
    std::stable_sort(m.order.begin(), m.order.end(), [&](int a, int b) {
        if (npass[a] != npass[b]) return npass[a] > npass[b];
        return m.terms[a]->lat.d > m.terms[b]->lat.d;
    });
    m.vbase.assign(T, 0);
    int V = 0, E = 0;
    m.max_d = -1;
    m.all_symmetric = true;
    for (int k : m.order) {
        const TermLattice& lat = m.terms[k]->lat;
        m.vbase[k] = V;
        V += lat.V;
        E += N * (lat.d + 1);
        m.max_d = std::max(m.max_d, lat.d);
        if (m.terms[k]->ntype != DCRF_NORMALIZE_SYMMETRIC && m.terms[k]->ntype != DCRF_NO_NORMALIZATION)
            m.all_symmetric = false;
    }
    m.V_total = V;
    m.E_total = E;
    // Segments and entries, tile by tile, the terms in layout order inside a tile
    // (segments.hip).  In-wave runs: a vertex's segments that sit side by side in one wave
    // are added inside the wave (k_splat folds each such run into its first lane group),
    // which at 1024x768x21 cuts the partial rows from 188 k to 72 k and the vertices with
    // more than 16 of them from 2,581 to 52.  The runs are part of the summation order, so
    // every (tile, term) group starts a wave: an instance of a batch then gets the bits of
    // the same image alone.  Vertices with more than 16 partial rows are recombined by a
    // whole wave (their rows in pieces summed side by side), in block-mode shapes in two
    // levels.  Block-mode shapes and the tiled splat have no in-wave runs.
    const int NT = m.tiles.n_tiles();
    RunSet rs;
    std::vector<const TermLattice*> lats;
    {
        std::vector<int> vb;
        for (int k : m.order) {
            lats.push_back(&m.terms[k]->lat);
            vb.push_back(m.vbase[k]);
        }
        build_run_set(lats, vb, NT, m.chunk(), rs, s);
    }
    // the LDS-tiled splat (a tile side set by the caller) if the largest tile's entries and
    // segments fit
    const TileGeom tg = tile_geom(m);
    int e_max = 0, s_max = 0;
    m.tiled = false;
    SegPlan sp;
    if (m.tile_side && T) {
        count_segments(rs, 0, 0, false, sp, s);
        std::vector<int> gs(rs.G + 1), ge(rs.G + 1), ts(NT + 1), te(NT + 1);
        copy_to_host(gs.data(), sp.gseg.get(), sizeof(int) * gs.size(), s);
        copy_to_host(ge.data(), rs.gebase.get(), sizeof(int) * ge.size(), s);
        for (int t = 0; t <= NT; t++) {
            ts[t] = gs[(size_t)t * T];
            te[t] = ge[(size_t)t * T];
        }
        for (int t = 0; t < NT; t++) {
            e_max = std::max(e_max, te[t + 1] - te[t]);
            s_max = std::max(s_max, ts[t + 1] - ts[t]);
        }
        s_max += sp.host[0].empty;  // the empty segments go with the last tile
        m.tiled = tiled_splat_lds(L, tg.side, e_max, s_max, m.lds_cap) > 0;
        if (m.tiled) {
            ts[NT] += sp.host[0].empty;
            upload(m.g_tile_seg, ts, s);
            upload(m.g_tile_e, te, s);
            DCRF_HIP_CHECK(hipStreamSynchronize(s));  // (the lists above are on this frame)
        }
    }
    // (the LDS-tiled splat stages unpadded rows)
    set_row_stride(m, m.tiled ? L : padded_labels(L), s);
    // a valid layout has the iterate's buffer: run_inference may allocate nothing
    if (m.ldv != L) m.Qp.reserve((size_t)N * m.ldv);
    if (T) plan_segments(rs, m.ldv, !m.tiled, sp, s);
    m.tl.clear();
    m.tl.resize(T);
    std::vector<PassTableJob> jobs;
    for (int k : m.order) {  // what the normalisers' filter needs
        const TermLattice& lat = m.terms[k]->lat;
        const int d1 = lat.d + 1;
        auto lay = std::make_unique<TermLayout>();
        lay->nbr.reserve((size_t)d1 * lat.V);
        launch_remap_nbr(lat.nbr.get(), lay->nbr.get(), d1 * lat.V, m.vbase[k], V, s);
        if (m.pairs)  // forward passes walk axes 0..d, the transpose's d..0 (permutohedral.cpp:556)
            build_pass_tables(lay->nbr.get(), lat.V, lat.d, m.vbase[k], V, lay->pass_steps, lay->pass_off,
                              lay->passF, lay->passT, step_limit[k], jobs);
        m.tl[k] = std::move(lay);
    }
    launch_pass_tables(jobs, s);
    m.n_passes = m.pairs ? blur_launches(m) : 0;
    m.prefixP.assign(m.n_passes, 0);
    for (int p = 0; p < m.n_passes; p++)
        for (int k = 0; k < T; k++)
            if ((int)m.tl[k]->pass_steps.size() > p) m.prefixP[p] += m.terms[k]->lat.V;
    m.prefixV.assign(std::max(m.max_d + 1, 0), 0);
    for (int st = 0; st <= m.max_d; st++)
        for (int k = 0; k < T; k++)
            if (m.terms[k]->lat.d >= st) m.prefixV[st] += m.terms[k]->lat.V;
    m.g_entF.reserve(E);
    if (!m.all_symmetric) m.g_entT.reserve(E);
    DCRF_HIP_CHECK(hipStreamSynchronize(s));  // the counts
    m.rows0 = V + 1;
    if (T) {
        emit_segments(rs, sp, V + 1, m.seg, s);
        m.rows0 = m.seg.rows;
        compute_norms(m, lats, rs, sp, s);
    }
    m.noalloc_rows = noalloc_rows(m, rs, sp, s);
    m.tsplat = TiledSplat{m.seg.ch.get(), m.g_tile_seg.get(), m.g_tile_e.get(), NT, tg, e_max, s_max};

    m.vals[0].reserve((size_t)m.rows0 * m.ldv);
    m.vals[1].reserve((size_t)(V + 1) * m.ldv);
    launch_fill(m.vals[0].get(), 0.f, (size_t)m.rows0 * m.ldv, s);
    launch_fill(m.vals[1].get(), 0.f, (size_t)(V + 1) * m.ldv, s);
    // interleaved slice pairs for the fused mean-field kernel, in term order
    m.runs = false;
    m.slcT_valid = false;
    m.fused = m.mf_mode != 1 &&
              fused_meanfield_ok(L, T, T > 0 ? m.terms[0]->lat.d + 1 : 0, T > 1 ? m.terms[1]->lat.d + 1 : 0);
    int ds = 0;
    std::vector<int> slc_off(T);
    for (int k = 0; k < T; k++) {
        slc_off[k] = ds;
        ds += m.terms[k]->lat.d + 1;
    }
    if (m.fused) m.g_slc.reserve((size_t)N * ds);
    for (int i = 0; i < T; i++) {
        const int k = m.order[i];
        Term& t = *m.terms[k];
        const TermLattice& lat = t.lat;
        TermLayout& lay = *m.tl[k];
        const int d1 = lat.d + 1, Ek = N * d1;
        const TileGeom* local = m.tiled ? &tg : nullptr;
        launch_entry_gather(lat.csr_e.get(), Ek, d1, lat.bary.get(), t.norm.get(), pre_norm(t.ntype, false),
                            lat.tile_ptr.get(), rs.gebase.get(), NT, T, i, local, m.g_entF.get(), s);
        if (!m.all_symmetric)
            launch_entry_gather(lat.csr_e.get(), Ek, d1, lat.bary.get(), t.norm.get(), pre_norm(t.ntype, true),
                                lat.tile_ptr.get(), rs.gebase.get(), NT, T, i, local, m.g_entT.get(), s);
        lay.vtx.reserve(Ek);
        lay.swF.reserve(Ek);
        const float alpha = slice_alpha(lat.d);
        launch_slice_weights(lat.vtx.get(), lat.bary.get(), t.norm.get(), post_norm(t.ntype, false), alpha, N, d1,
                             m.vbase[k], lay.vtx.get(), lay.swF.get(), m.fused ? m.g_slc.get() : nullptr, ds,
                             slc_off[k], s);
        if (!m.all_symmetric) {
            lay.swT.reserve(Ek);
            launch_slice_weights(lat.vtx.get(), lat.bary.get(), t.norm.get(), post_norm(t.ntype, true), alpha, N, d1,
                                 m.vbase[k], lay.vtx.get(), lay.swT.get(), nullptr, 0, 0, s);
        }
    }
    if (m.fused) {
        // pixel runs (on request): entry j reads vals[result_parity] of its term
        if (m.mf_mode == 3 && m.V_total < (1 << 30)) {
            unsigned par = 0;
            int j = 0;
            for (int k = 0; k < T; k++) {
                const int d1 = m.terms[k]->lat.d + 1;
                for (int q = 0; q < d1; q++, j++)
                    if (result_parity(m, k)) par |= 1u << j;
            }
            // rectangles two waves of pixels wide (18 at 21 labels), at most run_rows
            // high and at most 24 KiB of slice pairs
            const int TW = 2 * shape_for(L).per;
            const int TH = std::max(1, std::min(m.run_rows, (24 * 1024) / (TW * ds * 8)));
            build_run_slice(m.geo, m.geod, m.g_slc.get(), ds, par, TW, TH, m.rslice, s);
            m.rows_lds = (m.rslice.u_max * m.ldv + 1) & ~1;
            SliceTable probe = slice_table(m, false);
            const int cwf = assign_compat_lds(probe, L);
            const size_t lds = meanfield_runs_lds(L, ds, m.rslice.P, m.rows_lds, cwf);
            m.runs = m.mf_mode == 3 && lds <= 64 * 1024 && lds <= m.lds_cap;
        }
    }
    DCRF_HIP_CHECK(hipStreamSynchronize(s));
    m.layout_valid = true;
}

BlurTable blur_table(const dcrf_model& m) {
    BlurTable bt{};
    bt.nterms = (int)m.order.size();
    for (int i = 0; i < bt.nterms; i++) {
        const int k = m.order[i];
        bt.t[i] = BlurTerm{m.vbase[k], m.terms[k]->lat.V, m.terms[k]->lat.d, m.tl[k]->nbr.get()};
    }
    return bt;
}

// kw: device [T] term weights or null; mout: device [T][N][L] raw-message output or null.
SliceTable slice_table(const dcrf_model& m, bool transpose, const float* kw, float* mout) {
    SliceTable st{};
    st.nterms = (int)m.terms.size();
    st.rows = (size_t)m.V_total + 1;  // the slices read vertex rows (and the zero row)
    const size_t NL = (size_t)m.N() * m.L;
    for (int k = 0; k < st.nterms; k++) {
        const Term& t = *m.terms[k];
        const TermLayout& lay = *m.tl[k];
        const float* sw = (transpose && !m.all_symmetric) ? lay.swT.get() : lay.swF.get();
        st.t[k] = SliceTerm{lay.vtx.get(), sw, m.vals[result_parity(m, k)].get(), t.lat.d + 1, t.ckind,
                            t.d_compat.get(), kw ? kw + k : nullptr, mout ? mout + (size_t)k * NL : nullptr, m.ldv};
    }
    return st;
}

int compat_raw_len(int ckind, int L) {
    return ckind == DCRF_COMPAT_POTTS ? 1 : (ckind == DCRF_COMPAT_DIAGONAL ? L : L * L);
}
int compat_packed_len(int ckind, int L) {
    return ckind == DCRF_COMPAT_MATRIX ? L * (L + 1) / 2 : compat_raw_len(ckind, L);
}
int stat_len(int ckind, int L) { return ckind == DCRF_COMPAT_MATRIX ? L * L : L; }

// Splat, combine and blur every term's lattice: afterwards term k's filtered rows are
// in vals[result_parity(m, d_k)].  `transpose` selects the transposed filter (reverse blur
// order and the transpose's normaliser placement, pairwise.cpp:63-80).
// Algorithmic bytes of the splat (input rows once; per term the (pixel, weight) pairs,
// the normaliser and the vertex rows written) and of the per-pixel update (unary read,
// Q written; per term the slice pairs, the normaliser and the vertex rows read).  With
// the blur steps' V (2 L 4 + 8) they add up to dcrf_iteration_bytes.
double splat_bytes(const dcrf_model& m) {
    const double N = m.N(), L = m.L;
    double b = N * L * 4.0;
    for (const auto& t : m.terms) b += N * (t->lat.d + 1) * 8.0 + N * 4.0 + (double)t->lat.V * L * 4.0;
    return b;
}
double meanfield_bytes(const dcrf_model& m) { return splat_bytes(m) + m.N() * (double)m.L * 4.0; }

// Rows of the splat's input: the pixels, or the 8 x 8 block positions of entries ent_in.
size_t in_rows(const dcrf_model& m, const int2* ent_in) {
    return ent_in ? q_block_rows(m.geo.W[0], m.geo.H[0]) : (size_t)m.N();
}

// in: the [N] input rows with row stride m.ldv (floats).
void run_filter(dcrf_model& m, const float* in, bool transpose, hipStream_t s, const int2* ent_in = nullptr) {
    const int L = m.L, Lv = m.ldv;  // the filter works on whole rows, padding labels included
    const int2* ent = ent_in ? ent_in : ((transpose && !m.all_symmetric) ? m.g_entT.get() : m.g_entF.get());
    {
        Timed t(m, s, KC_SPLAT, splat_bytes(m));
        if (m.tiled)
            launch_splat_tiled(m.tsplat, ent, in, m.vals[0].get(), m.ldv, L, m.lds_cap, s);  // ldv == L
        else
            splat_lists(m.seg, ent, in, in_rows(m, ent_in), Lv, m.vals[0].get(), s);
        t.done();
    }
    if (m.seg.ncb) {
        Timed t(m, s, KC_COMBINE, 0.0);
        combine_lists(m.seg, Lv, m.vals[0].get(), s);
        t.done();
    }
    blur_rows(m, m.vals[0].get(), m.vals[1].get(), Lv, transpose, s);
}

void prepare(dcrf_model& m) {
    ensure_device(m);
    ensure_unary(m);
    ensure_layout(m);
    const size_t n = (size_t)m.N() * m.L;
    m.Q.reserve(n);
    if (m.qblocks && !m.qblocks_ready && m.fused && !m.runs && !m.tiled && m.geo.is2d &&
        m.geo.n_inst == 1) {
        m.g_entB.reserve(m.E_total);
        launch_entry_block(m.g_entF.get(), (size_t)m.E_total, m.geo.W[0], m.g_entB.get(), m.stream);
        m.Qb.reserve(q_block_rows(m.geo.W[0], m.geo.H[0]) * m.ldv);
        DCRF_HIP_CHECK(hipStreamSynchronize(m.stream));
        m.qblocks_ready = true;
    }
}

// Splat input rows from rows in the caller's layout ([N][L]): themselves, or m.Qp with the
// padding labels added.
const float* splat_rows(dcrf_model& m, const float* Q, hipStream_t s) {
    if (m.ldv == m.L) return Q;
    launch_restride_rows(Q, m.L, m.Qp.get(), m.ldv, m.N(), m.L, s);
    return m.Qp.get();
}

// Q between the iterations has rows of ldv floats: where those are padded it stays in m.Qp
// and only the last update writes the caller's Q.
void run_inference(dcrf_model& m, int n_iter, const float* U, float* Q, hipStream_t s) {
    const int L = m.L, N = m.N(), Lv = m.ldv;
    float* Qi = Lv != L && n_iter > 0 ? m.Qp.get() : Q;
    launch_softmax_neg(U, Qi, Qi == Q ? L : Lv, N, L, Lv, s);
    const SliceTable st = slice_table(m, false, m.kw_set ? m.kw.get() : nullptr);
    // Q in 8 x 8 blocks between iterations: the first splat reads Q_0 in pixel order, the
    // later ones m.Qb through the block-position entries; the last update writes Q
    const bool blk = m.qblocks_ready && n_iter > 1 && m.fused && !m.runs && !m.tiled;
    for (int it = 0; it < n_iter; it++) {
        const bool last = it + 1 == n_iter;
        if (blk) {
            run_filter(m, it > 0 ? m.Qb.get() : Qi, false, s, it > 0 ? m.g_entB.get() : nullptr);
            Timed t(m, s, KC_MEANFIELD, meanfield_bytes(m));
            launch_meanfield_fused(U, last ? Q : m.Qb.get(), last ? L : Lv, N, L, Lv, st, m.g_slc.get(), s,
                                   last ? 0 : m.geo.W[0]);
            t.done();
            continue;
        }
        run_filter(m, Qi, false, s);
        float* Qo = last ? Q : Qi;
        const int ldo = last ? L : Lv;
        Timed t(m, s, KC_MEANFIELD, meanfield_bytes(m));
        if (m.runs)
            launch_meanfield_runs(U, Qo, ldo, N, L, Lv, st,
                                  RunSliceDev{m.rslice.P, m.rslice.n_runs, m.rows_lds, m.rslice.base.get(),
                                              m.rslice.rows.get(), m.rslice.pix_base.get(), m.rslice.rpix.get(),
                                              m.rslice.loc.get(), m.vals[0].get(), m.vals[1].get()},
                                  s);
        else if (m.fused)
            launch_meanfield_fused(U, Qo, ldo, N, L, Lv, st, m.g_slc.get(), s);
        else
            launch_meanfield(U, Qo, ldo, N, L, Lv, st, nullptr, nullptr, s);
        t.done();
    }
}

int matrix_terms(const dcrf_model& m) {
    int nm = 0;
    for (const auto& t : m.terms) nm += t->ckind == DCRF_COMPAT_MATRIX;
    return nm;
}

// Forward pass that keeps Q_0..Q_n and the Matrix terms' raw messages for the adjoint.
void forward_train(dcrf_model& m, int n_iter, const float* U, const float* compat_raw, const float* kw,
                   hipStream_t s) {
    const int N = m.N(), L = m.L, T = (int)m.terms.size();
    const int Lv = m.ldv;
    const size_t NL = (size_t)N * L, NLv = (size_t)N * Lv;  // Q_t (t < n): rows of ldv floats; Q_n: of L
    m.train_n = -1;  // until the store is complete: a failed allocation below has lost the old one
    if (compat_raw) {
        size_t off = 0;
        for (auto& t : m.terms) {
            launch_set_compat(compat_raw + off, t->ckind, L, t->d_compat.get(), s);
            off += compat_raw_len(t->ckind, L);
        }
    }
    m.qcache.reserve((size_t)n_iter * NLv + NL);
    // raw messages of the Matrix terms only (their statistic is a full L x L product
    // taken after the adjoint loop); the others' statistic comes from the adjoint kernels
    const int nm = matrix_terms(m);
    m.mcache.reserve(std::max<size_t>((size_t)n_iter * nm * NL, 1));
    launch_softmax_neg(U, m.qcache.get(), n_iter ? Lv : L, N, L, Lv, s);
    for (int it = 0; it < n_iter; it++) {
        const float* Qt = m.qcache.get() + (size_t)it * NLv;
        float* Qn = m.qcache.get() + (size_t)(it + 1) * NLv;
        const int ldn = it + 1 < n_iter ? Lv : L;
        run_filter(m, Qt, false, s);
        SliceTable st = slice_table(m, false, kw);
        for (int k = 0, j = 0; k < T; k++)
            if (m.terms[k]->ckind == DCRF_COMPAT_MATRIX)
                st.t[k].mout = m.mcache.get() + ((size_t)it * nm + j++) * NL;
        if (m.fused)  // same arithmetic as k_meanfield, gathers of all entries up front
            launch_meanfield_fused(U, Qn, ldn, N, L, Lv, st, m.g_slc.get(), s);
        else
            launch_meanfield(U, Qn, ldn, N, L, Lv, st, nullptr, nullptr, s);
    }
    m.train_n = n_iter;
    m.train_kw = kw;
}

// Adjoint of forward_train.  dQ: dL/dQ_n.  Outputs dU (always), per-term statistics in
// m.gacc, and optionally raw compatibility / term-weight gradients on the device.
// kernel: also accumulate the kernel-parameter gradient of every term into m.kacc.
// The interleaved slice pairs of the adjoint's fused kernel: the forward's when every
// term's transposed slice weights equal its forward ones (SYMMETRIC / NO_NORMALIZATION),
// else pairs with the transposed weights, built once per layout.
const int2* adjoint_pairs(dcrf_model& m, hipStream_t s) {
    if (m.all_symmetric) return m.g_slc.get();
    if (!m.slcT_valid) {
        const int T = (int)m.terms.size(), N = m.N();
        int ds = 0;
        for (int k = 0; k < T; k++) ds += m.terms[k]->lat.d + 1;
        m.g_slcT.reserve((size_t)N * ds);
        int off = 0;
        for (int k = 0; k < T; k++) {
            const int d1 = m.terms[k]->lat.d + 1;
            launch_interleave_slice(m.tl[k]->vtx.get(), m.tl[k]->swT.get(), N, d1, ds, off, m.g_slcT.get(), s);
            off += d1;
        }
        m.slcT_valid = true;
    }
    return m.g_slcT.get();
}

void backward(dcrf_model& m, const float* dQ, float* dU, float* dcompat, float* dkw, hipStream_t s,
              bool kernel = false) {
    if (m.train_n < 0) throw Error{DCRF_ERR_STATE, "backward needs a preceding training forward"};
    const int N = m.N(), L = m.L, Lv = m.ldv, T = (int)m.terms.size(), n = m.train_n;
    const size_t NL = (size_t)N * L, NLv = (size_t)N * Lv;
    // b_t, the adjoint entering reverse iteration t - 1, in slot t (t = n .. 0).  The
    // Matrix terms' statistic reads every b_t after the loop, so with such a term every
    // slot stays; otherwise a ring of the slots that dU still needs and the step's own.
    const int nm = matrix_terms(m);
    const int ring = nm ? n + 1 : std::min(n + 1, UnarySum::kPending + 1);
    m.bbuf.reserve((size_t)ring * NLv);
    auto bslot = [&](int t) { return m.bbuf.get() + (size_t)(t % ring) * NLv; };
    const float* Qc = m.qcache.get();
    launch_sn_first(Qc + (size_t)n * NLv, dQ, bslot(n), n ? nullptr : dU, N, L, Lv, s);
    int first_pending = n;  // slots first_pending .. it + 1 are not in dU yet
    std::vector<size_t> goff(T + 1, 0);
    for (int k = 0; k < T; k++) goff[k + 1] = goff[k] + stat_len(m.terms[k]->ckind, L);
    m.gacc.reserve(std::max<size_t>(goff[T], 1));
    launch_fill_double(m.gacc.get(), goff[T], s);
    // the other terms' statistic rows: term j (in term order among them), iteration it
    // at partial + (j * n + it) * nblk * L, one row of L sums per adjoint block
    const int nd = T - nm;
    const size_t nblk = (size_t)adjoint_blocks(N, Lv);
    size_t pf = std::max<size_t>((size_t)nd * n * nblk * L, 1);
    if (nm) pf = std::max(pf, grad_partial_floats(N, L, n));
    m.partial.reserve(pf);
    m.rmid.reserve(rows_mid_doubles(nm ? L * L : L));
    std::vector<int> koff(T + 1, 0);
    for (int k = 0; k < T; k++) koff[k + 1] = koff[k] + m.terms[k]->num_kparams();
    kernel = kernel && koff[T] > 0;
    size_t pstride = 0;  // per term: its partial rows in kpartial
    if (kernel) {
        ensure_kg_plans(m);
        int dmax = 1, dslow = 0;  // dslow: largest d of a term without the one-pass gradient
        for (auto& t : m.terms) {
            dmax = std::max(dmax, t->lat.d);
            if (t->num_kparams() && !kg_grad_fused(L, t->lat.d)) dslow = std::max(dslow, t->lat.d);
        }
        size_t tmax = 1;
        for (const auto& P : m.kgplans) tmax = std::max(tmax, P->parts.size());
        m.kgbuf.reserve(4 * tmax * NL);
        if (dslow) m.kgdf.reserve((size_t)2 * N * dslow);
        pstride = kparam_partial_doubles(dmax);
        m.kpartial.reserve(pstride * T);
        m.kacc.reserve(koff[T]);
        launch_fill_double(m.kacc.get(), koff[T], s);
        for (int k = 0; k < T; k++)  // the one-pass kernel adds every iteration to its rows
            if (m.terms[k]->num_kparams() && kg_grad_fused(L, m.terms[k]->lat.d))
                launch_fill_double(m.kpartial.get() + (size_t)k * pstride,
                                   (size_t)kg_grad_blocks(N, L) * m.terms[k]->num_kparams(), s);
    }
    for (int it = n - 1; it >= 0; it--) {
        float* b = bslot(it + 1);
        if (kernel) {
            // DenseCRF::gradient takes the kernel gradient with b before its update
            // (densecrf.cpp:280-284)
            for (const auto& P : m.kgplans)
                kernel_grad_group(m, *P, b, Qc + (size_t)it * NLv, m.train_kw, koff, pstride, s);
        }
        run_filter(m, b, true, s);
        SliceTable st = slice_table(m, true, m.train_kw);
        for (int k = 0, j = 0; k < T; k++)
            if (m.terms[k]->ckind != DCRF_COMPAT_MATRIX) {
                st.t[k].gstat = m.partial.get() + ((size_t)j * n + it) * nblk * L;
                st.t[k].gslot = j++;
                st.nstat = j;
            }
        UnarySum us{};
        us.n = first_pending - it;
        if (us.n == UnarySum::kPending || it == 0) {
            us.mode = first_pending == n ? UnarySum::START : UnarySum::ADD;
            for (int i = 0; i < us.n; i++) us.prev[i] = bslot(first_pending - i);
            first_pending = it - 1;
        }
        if (m.fused)
            launch_adjoint_fused(Qc + (size_t)it * NLv, bslot(it), dU, us, N, L, Lv, st, adjoint_pairs(m, s), s);
        else
            launch_adjoint(Qc + (size_t)it * NLv, bslot(it), dU, us, N, L, Lv, st, s);
    }
    if (kernel)  // the one-pass kernel gradient's partial rows hold all iterations
        for (int k = 0; k < T; k++)
            if (m.terms[k]->num_kparams() && kg_grad_fused(L, m.terms[k]->lat.d))
                launch_kparam_final(m.kpartial.get() + (size_t)k * pstride, kg_grad_blocks(N, L),
                                    m.terms[k]->num_kparams(), m.kacc.get() + koff[k], s);
    // G_k = sum_t b_{t+1} (K~_k Q_t)^T over all iterations: the statistic rows of the
    // Potts / Diagonal terms first (they share the partial buffer with the Matrix
    // terms' products), then for Matrix terms b_{t+1} in slot t + 1 against the messages
    // of iteration t
    for (int k = 0, j = 0; k < T; k++)
        if (m.terms[k]->ckind != DCRF_COMPAT_MATRIX) {
            launch_sum_rows(m.partial.get() + (size_t)j * n * nblk * L, (long long)n * nblk, L, m.rmid.get(),
                            m.gacc.get() + goff[k], s);
            j++;
        }
    for (int k = 0, j = 0; k < T; k++)
        if (m.terms[k]->ckind == DCRF_COMPAT_MATRIX) {
            launch_grad_stat(bslot(1), Lv, NLv, m.mcache.get() + (size_t)j * NL, (size_t)nm * NL, n, N, L,
                             m.partial.get(), m.rmid.get(), m.gacc.get() + goff[k], s);
            j++;
        }
    if (dcompat || dkw) {
        size_t coff = 0;
        for (int k = 0; k < T; k++) {
            const Term& t = *m.terms[k];
            launch_compat_finish(m.gacc.get() + goff[k], t.ckind, L, t.d_compat.get(),
                                 m.train_kw ? m.train_kw + k : nullptr, dcompat ? dcompat + coff : nullptr,
                                 dkw ? dkw + k : nullptr, s);
            coff += compat_raw_len(t.ckind, L);
        }
    }
}

// Hamming's class weights (objective.cpp:51-63): the given ones, or from the class
// counts c of gt as (c / sum c)^-pow normalised by sum c w.  Checks that every label of
// gt inside [0, L) has a weight.
std::vector<float> hamming_weights(const int16_t* gt, int N, int L, float pow_, const float* cw_in, int ncw) {
    std::vector<float> w;
    if (cw_in) {
        w.assign(cw_in, cw_in + ncw);
    } else {
        int M = 0;
        for (int i = 0; i < N; i++) M = std::max(M, gt[i] + 1);
        std::vector<float> cnt(M, 0.f);
        for (int i = 0; i < N; i++)
            if (gt[i] >= 0) cnt[gt[i]] += 1.0f;
        float total = 0.f;
        for (float c : cnt) total += c;
        w.resize(M);
        float z = 0.f;
        for (int l = 0; l < M; l++) {
            w[l] = std::pow(cnt[l] / total, -pow_);
            z += cnt[l] * w[l];
        }
        for (int l = 0; l < M; l++) w[l] = w[l] / z;
    }
    for (int i = 0; i < N; i++) {
        const int g = gt[i];
        if (g >= 0 && g < L) require(g < (int)w.size(), "a ground-truth label has no class weight");
    }
    if (w.empty()) w.assign(1, 0.f);  // no labelled pixel: the kernel reads no weight
    return w;
}

// The objective's value from launch_objective's partial sums (OP: its partial array):
// LogLikelihood / Hamming add the block sums in order; IoU is sum_l in_l / un_l / L.
double objective_value(int kind, const std::vector<double>& OP, int L) {
    double r = 0.0;
    if (kind == DCRF_OBJECTIVE_IOU) {
        const double* st = OP.data() + OP.size() - 2 * (size_t)L;
        for (int l = 0; l < L; l++) r += st[2 * l] / st[2 * l + 1];
        return r / L;
    }
    for (double v : OP) r += v;
    return r;
}

// ---- allocation-free inference (dcrf_inference_device_noalloc)
// The filter's vertex rows (splat output, partial rows, both blur buffers) in one static
// device array per GPU instead of the model's buffers.  Host code must not use the
// array's name as an address: the address comes from hipGetSymbolAddress, once per
// device, and is kept in scratch_dev.
// The limit (kNoAllocRowBytes) counts rows of L floats; the array holds them padded (at
// most 8 floats for 5 labels) and the second buffer's alignment.
constexpr size_t kNoAllocScratchBytes = kNoAllocRowBytes / 5 * 8 + 4096;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];
float* scratch_dev[kMaxDevices] = {};
std::mutex scratch_mu;

float* scratch_for_current_device() {
    int dev = 0;
    DCRF_HIP_CHECK(hipGetDevice(&dev));
    require(dev >= 0 && dev < kMaxDevices, "device index out of range for the allocation-free inference");
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_dev[dev]) {
        void* p = nullptr;
        DCRF_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        require(p != nullptr, "the scratch array has no device address");
        scratch_dev[dev] = static_cast<float*>(p);
    }
    return scratch_dev[dev];
}

// Points the model's two vertex-row buffers at other memory for its lifetime (nothing
// may reserve or release them meanwhile), then gives the model its own back.
struct BorrowedRows {
    dcrf_model& m;
    float* own_p[2];
    size_t own_n[2];
    BorrowedRows(dcrf_model& m_, float* r0, size_t n0, float* r1, size_t n1) : m(m_) {
        for (int i = 0; i < 2; i++) {
            own_p[i] = m.vals[i].p;
            own_n[i] = m.vals[i].n;
        }
        m.vals[0].p = r0;
        m.vals[0].n = n0;
        m.vals[1].p = r1;
        m.vals[1].n = n1;
    }
    ~BorrowedRows() {
        for (int i = 0; i < 2; i++) {
            m.vals[i].p = own_p[i];
            m.vals[i].n = own_n[i];
        }
    }
    BorrowedRows(const BorrowedRows&) = delete;
    BorrowedRows& operator=(const BorrowedRows&) = delete;
};

dcrf_model* new_model(const std::vector<int>& N, const std::vector<int>* W, const std::vector<int>* H, int L) {
    require(!N.empty(), "a model needs at least one instance");
    require(L >= 1 && L <= DCRF_MAX_LABELS, "number of labels must be between 1 and " +
                                                std::to_string(DCRF_MAX_LABELS));
    auto m = std::make_unique<dcrf_model>();
    m->L = L;
    Geometry& g = m->geo;
    g.n_inst = (int)N.size();
    g.N = N;
    g.pix_base.assign(1, 0);
    g.pad_base.assign(1, 0);
    long long pix = 0, pad = 0;
    for (int n : N) {
        require(n >= 1, "number of variables must be positive");
        pix += n;
        pad += (n + 3) / 4 * 4;
        require(pix * L < (1ll << 31) && pad * (DCRF_MAX_DIM + 1) < (1ll << 31),
                "model too large for 32-bit indexing");
        g.pix_base.push_back((int)pix);
        g.pad_base.push_back((int)pad);
    }
    if (W) {
        g.is2d = true;
        g.W = *W;
        g.H = *H;
    }
    return m.release();
}

}  // namespace

// =====================================================================================
extern "C" {

const char* dcrf_last_error(void) { return g_last_error.c_str(); }

int dcrf_release_cached_memory(size_t* bytes) {
    return guard([&] {
        const size_t b = pool_release_all() + release_host_stage() + release_pinned();
        if (bytes) *bytes = b;
    });
}

int dcrf_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int dcrf_create(int N, int L, dcrf_model** out) {
    return guard([&] {
        require(out != nullptr, "null output pointer");
        *out = new_model({N}, nullptr, nullptr, L);
    });
}

int dcrf_create_2d(int W, int H, int L, dcrf_model** out) {
    return guard([&] {
        require(out != nullptr, "null output pointer");
        require(W >= 1 && H >= 1, "width and height must be positive");
        require((long long)W * H < (1ll << 31), "image too large");
        std::vector<int> w{W}, h{H};
        *out = new_model({W * H}, &w, &h, L);
    });
}

int dcrf_create_batch(int n, const int* N, int L, dcrf_model** out) {
    return guard([&] {
        require(out != nullptr && N != nullptr && n >= 1, "bad batch description");
        *out = new_model(std::vector<int>(N, N + n), nullptr, nullptr, L);
    });
}

int dcrf_create_batch_2d(int n, const int* W, const int* H, int L, dcrf_model** out) {
    return guard([&] {
        require(out != nullptr && W != nullptr && H != nullptr && n >= 1, "bad batch description");
        std::vector<int> w(W, W + n), h(H, H + n), N(n);
        for (int i = 0; i < n; i++) {
            require(w[i] >= 1 && h[i] >= 1 && (long long)w[i] * h[i] < (1ll << 31), "bad image size");
            N[i] = w[i] * h[i];
        }
        *out = new_model(N, &w, &h, L);
    });
}

void dcrf_destroy(dcrf_model* m) {
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    delete m;
}

int dcrf_set_unary(dcrf_model* m, const float* U) {
    return guard([&] {
        require(m && U, "null argument");
        const size_t n = (size_t)m->N() * m->L;
        finish_unary_upload(*m);
        // one instance: page-locked memory, from which the upload is one asynchronous copy
        // (several instances may be set one by one later, beside this call's values)
        if (m->geo.n_inst == 1 && m->unary_pin.take(sizeof(float) * n)) {
            host_copy(m->unary_pin.p, U, sizeof(float) * n);
        } else {
            m->unary_pin.give();
            m->unary_host.resize(n);
            host_copy(m->unary_host.data(), U, sizeof(float) * n);
        }
        m->unary_unset.clear();
        m->has_unary = true;
        m->unary_dirty = true;
        m->logistic = false;
    });
}

int dcrf_set_logistic_unary(dcrf_model* m, const float* Lmat, int F, const float* feat) {
    return guard([&] {
        require(m && Lmat && feat, "null argument");
        require(F >= 1, "the logistic unary needs at least one feature");
        const int N = m->N(), L = m->L;
        require((long long)N * F < (1ll << 31), "logistic unary features too large for 32-bit indexing");
        ensure_device(*m);
        hipStream_t s = m->stream;
        m->lL.assign(Lmat, Lmat + (size_t)L * F);
        // features (F, N) row-major, kept as given and as [N][F]
        m->lfFN.reserve((size_t)N * F);
        m->lf.reserve((size_t)N * F);
        DCRF_HIP_CHECK(hipMemcpyAsync(m->lfFN.get(), feat, sizeof(float) * N * F, hipMemcpyHostToDevice, s));
        launch_transpose(m->lfFN.get(), m->lf.get(), F, N, s);
        DCRF_HIP_CHECK(hipStreamSynchronize(s));
        finish_unary_upload(*m);
        m->unary_pin.give();
        m->lF = F;
        m->logistic = true;
        m->has_unary = true;
        m->unary_dirty = true;
        m->ugrad_param.clear();
    });
}

int dcrf_num_unary_params(const dcrf_model* m) { return m && m->logistic ? m->L * m->lF : 0; }

int dcrf_get_unary_params(const dcrf_model* m, float* params) {
    return guard([&] {
        require(m && params, "null argument");
        // LogisticUnaryEnergy::parameters (unary.cpp:53-57): L packed column-major
        const int L = m->L, F = m->lF;
        if (!m->logistic) return;
        for (int c = 0; c < F; c++)
            for (int r = 0; r < L; r++) params[(size_t)c * L + r] = m->lL[(size_t)r * F + c];
    });
}

int dcrf_set_unary_params(dcrf_model* m, const float* params) {
    return guard([&] {
        require(m && params, "null argument");
        require(m->logistic, "the unary has no parameters (only a logistic unary does)");
        const int L = m->L, F = m->lF;
        for (int c = 0; c < F; c++)
            for (int r = 0; r < L; r++) m->lL[(size_t)r * F + c] = params[(size_t)c * L + r];
        m->unary_dirty = true;
        m->train_n = -1;
    });
}

int dcrf_unary_param_gradient(const dcrf_model* m, float* grad) {
    return guard([&] {
        require(m && grad, "null argument");
        require(m->logistic, "the unary has no parameters (only a logistic unary does)");
        require(!m->ugrad_param.empty(), "no dcrf_gradient call since the logistic unary was set");
        std::copy(m->ugrad_param.begin(), m->ugrad_param.end(), grad);
    });
}

int dcrf_set_unary_instance(dcrf_model* m, int i, const float* U) {
    return guard([&] {
        require(m && U, "null argument");
        require(!m->logistic, "the model has a logistic unary: set a full unary with dcrf_set_unary first");
        require(i >= 0 && i < m->geo.n_inst, "instance index out of range");
        const int N = m->N(), L = m->L, b = m->geo.pix_base[i], Ni = m->geo.N[i];
        finish_unary_upload(*m);
        m->unary_pin.give();  // (held by single-instance models: this call sets all of it)
        if (m->unary_host.size() != (size_t)N * L) {  // instances not set are zero at the upload
            m->unary_host.resize((size_t)N * L);
            m->unary_unset.assign(m->geo.n_inst, 1);
        }
        copy_rows(m->unary_host.data() + b, N, U, Ni, L, Ni);
        if (!m->unary_unset.empty()) m->unary_unset[i] = 0;
        m->has_unary = true;
        m->unary_dirty = true;
    });
}

int dcrf_add_pairwise(dcrf_model* m, const float* feat, int d, int ckind, const float* compat, int ktype,
                      int ntype) {
    return guard([&] {
        require(m && feat, "null argument");
        require(d >= 1 && d <= DCRF_MAX_DIM, "feature dimension must be between 1 and " + std::to_string(DCRF_MAX_DIM));
        const size_t n = (size_t)d * m->N();
        add_term(*m, d, ckind, compat, ktype, ntype, [&](float* out) {
            DevBuf<float> raw;
            raw.reserve(n);
            DCRF_HIP_CHECK(hipMemcpy(raw.get(), feat, sizeof(float) * n, hipMemcpyHostToDevice));
            features_from_dxN(m->geo, m->geod, raw.get(), d, out, m->stream);
            DCRF_HIP_CHECK(hipStreamSynchronize(m->stream));
        });
    });
}

int dcrf_add_gaussian_2d(dcrf_model* m, float sx, float sy, int ckind, const float* compat, int ktype, int ntype) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(m->geo.is2d, "addPairwiseGaussian needs a 2-D model", DCRF_ERR_STATE);
        add_term(*m, 2, ckind, compat, ktype, ntype,
                 [&](float* out) { features_gaussian_2d(m->geo, m->geod, sx, sy, out, m->stream); });
    });
}

int dcrf_add_bilateral_2d(dcrf_model* m, float sx, float sy, float sr, float sg, float sb, const uint8_t* rgb,
                          int ckind, const float* compat, int ktype, int ntype) {
    return guard([&] {
        require(m && rgb, "null argument");
        require(m->geo.is2d, "addPairwiseBilateral needs a 2-D model", DCRF_ERR_STATE);
        const size_t n = (size_t)m->N() * 3;
        add_term(*m, 5, ckind, compat, ktype, ntype, [&](float* out) {
            DevBuf<uint8_t> img;
            img.reserve(n);
            DCRF_HIP_CHECK(hipMemcpy(img.get(), rgb, n, hipMemcpyHostToDevice));
            features_bilateral_2d(m->geo, m->geod, sx, sy, sr, sg, sb, img.get(), out, m->stream);
            DCRF_HIP_CHECK(hipStreamSynchronize(m->stream));
        });
    });
}

int dcrf_inference(dcrf_model* m, int n_iter, float* Q) {
    return guard([&] {
        require(m && Q, "null argument");
        require(n_iter >= 0, "number of iterations must be non-negative");
        prepare(*m);
        const float* U = m->has_unary ? m->unary.get() : nullptr;
        run_inference(*m, n_iter, U, m->Q.get(), m->stream);
        copy_to_host(Q, m->Q.get(), sizeof(float) * (size_t)m->N() * m->L, m->stream);
        if (m->timing) collect_timing(*m);
    });
}

int dcrf_map(dcrf_model* m, int n_iter, int16_t* labels) {
    return guard([&] {
        require(m && labels, "null argument");
        require(n_iter >= 0, "number of iterations must be non-negative");
        prepare(*m);
        const float* U = m->has_unary ? m->unary.get() : nullptr;
        run_inference(*m, n_iter, U, m->Q.get(), m->stream);
        m->labels.reserve(m->N());
        launch_argmax(m->Q.get(), m->L, m->N(), m->L, m->labels.get(), m->stream);
        copy_to_host(labels, m->labels.get(), sizeof(int16_t) * m->N(), m->stream);
        if (m->timing) collect_timing(*m);
    });
}

int dcrf_current_map(dcrf_model* m, const float* Q, int16_t* labels) {
    return guard([&] {
        require(m && Q && labels, "null argument");
        ensure_device(*m);
        const size_t n = (size_t)m->N() * m->L;
        m->work.reserve(n);
        m->labels.reserve(m->N());
        copy_to_device(m->work.get(), Q, sizeof(float) * n, m->stream);
        launch_argmax(m->work.get(), m->L, m->N(), m->L, m->labels.get(), m->stream);
        copy_to_host(labels, m->labels.get(), sizeof(int16_t) * m->N(), m->stream);
    });
}

int dcrf_current_map_device(dcrf_model* m, const float* Q_dev, int16_t* labels_dev, void* stream) {
    return guard([&] {
        require(m && Q_dev && labels_dev, "null argument");
        ensure_device(*m);
        launch_argmax(Q_dev, m->L, m->N(), m->L, labels_dev, (hipStream_t)stream);
    });
}

int dcrf_inference_device(dcrf_model* m, int n_iter, const float* U_dev, float* Q_dev, void* stream) {
    return guard([&] {
        require(m && Q_dev, "null argument");
        require(n_iter >= 0, "number of iterations must be non-negative");
        prepare(*m);
        hipStream_t s = (hipStream_t)stream;  // 0 is the null stream, as in HIP
        const float* U = U_dev ? U_dev : (m->has_unary ? m->unary.get() : nullptr);
        run_inference(*m, n_iter, U, Q_dev, s);
    });
}

int dcrf_capture_inference(dcrf_model* m, int n_iter, const float* U_dev, float* Q_dev) {
    return guard([&] {
        require(m && Q_dev, "null argument");
        require(n_iter >= 0, "number of iterations must be non-negative");
        require(!m->timing, "disable kernel timing before capturing a graph", DCRF_ERR_STATE);
        prepare(*m);
        m->drop_graph();
        const float* U = U_dev ? U_dev : (m->has_unary ? m->unary.get() : nullptr);
        DCRF_HIP_CHECK(hipStreamSynchronize(m->stream));
        DCRF_HIP_CHECK(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
        try {
            run_inference(*m, n_iter, U, Q_dev, m->stream);
        } catch (...) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(m->stream, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        DCRF_HIP_CHECK(hipStreamEndCapture(m->stream, &m->graph));
        DCRF_HIP_CHECK(hipGraphInstantiate(&m->graph_exec, m->graph, nullptr, nullptr, 0));
        m->graph_own_unary = U_dev == nullptr;
        m->graph_unary = U_dev ? nullptr : U;
        m->graph_kw = m->kw_set ? m->kw.get() : nullptr;
        m->graph_valid = true;
    });
}

int dcrf_launch_graph(dcrf_model* m, void* stream) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(m->graph_valid && m->layout_valid, "no captured inference (or the model changed since)",
                DCRF_ERR_STATE);
        // The graph reads the unary and term-weight buffers it was captured with: new
        // values in the same buffers are picked up (a unary set since the capture is
        // uploaded first), a buffer that appeared, went or moved needs a new capture.
        if (m->graph_own_unary) {
            require(m->has_unary == (m->graph_unary != nullptr),
                    "the unary was set or removed since the capture: capture again", DCRF_ERR_STATE);
            if (m->has_unary) {
                ensure_unary(*m);
                require(m->unary.get() == m->graph_unary, "the unary buffer moved since the capture: capture again",
                        DCRF_ERR_STATE);
            }
        }
        require((m->kw_set ? m->kw.get() : nullptr) == m->graph_kw,
                "term weights were set or removed since the capture: capture again", DCRF_ERR_STATE);
        DCRF_HIP_CHECK(hipGraphLaunch(m->graph_exec, (hipStream_t)stream));
    });
}

int dcrf_inference_device_noalloc(dcrf_model* m, int n_iter, const float* U_dev, float* Q_dev, void* stream) {
    return guard([&] {
        require(m && Q_dev, "null argument");
        require(n_iter >= 0, "number of iterations must be non-negative");
        require(m->dev_ready && m->layout_valid,
                "the model's layout is not built: run dcrf_inference_device (or dcrf_inference) on it once first",
                DCRF_ERR_STATE);
        require(!m->timing, "disable kernel timing for the allocation-free inference", DCRF_ERR_STATE);
        require(!m->tiled && !m->runs,
                "the allocation-free inference runs the default splat and mean-field kernels only", DCRF_ERR_STATE);
        require(m->ldv == m->L || m->Qp.n >= (size_t)m->N() * m->ldv, "the layout has no buffer for the padded iterate",
                DCRF_ERR_STATE);
        require(U_dev || !m->has_unary || !m->unary_dirty,
                "the unary changed since the last call: upload it with dcrf_inference_device first, or pass U_dev",
                DCRF_ERR_STATE);
        const size_t n0 = (size_t)m->rows0 * m->ldv, n1 = (size_t)(m->V_total + 1) * m->ldv;
        const size_t off1 = (n0 + 63) / 64 * 64;  // second buffer 256-byte aligned
        const size_t need = off1 + n1;
        const size_t bytes = m->noalloc_rows * m->L * sizeof(float);
        if (bytes > kNoAllocRowBytes || need > kNoAllocScratchBytes / sizeof(float))
            throw Error{DCRF_ERR_VALUE, "the model needs " + std::to_string(bytes) +
                                            " bytes of vertex rows; the allocation-free inference holds at most " +
                                            std::to_string(kNoAllocRowBytes) + " (use dcrf_inference_device)"};
        float* base = scratch_for_current_device();
        hipStream_t s = (hipStream_t)stream;
        // the rows start at zero, as the layout leaves the model's own buffers (the
        // missing-neighbour row is read as zero); the array keeps the last call's rows
        launch_fill(base, 0.f, need, s);
        BorrowedRows rows(*m, base, n0, base + off1, n1);
        const float* U = U_dev ? U_dev : (m->has_unary ? m->unary.get() : nullptr);
        run_inference(*m, n_iter, U, Q_dev, s);
    });
}

int dcrf_start_inference(dcrf_model* m, float* Q) {
    return guard([&] {
        require(m && Q, "null argument");
        const size_t n = (size_t)m->N() * m->L;
        if (!m->has_unary) {  // densecrf.cpp:180-184: zeros without a unary
            std::memset(Q, 0, sizeof(float) * n);
            return;
        }
        ensure_device(*m);
        ensure_unary(*m);
        m->Q.reserve(n);
        launch_softmax_neg(m->unary.get(), m->Q.get(), m->L, m->N(), m->L, padded_labels(m->L), m->stream);
        copy_to_host(Q, m->Q.get(), sizeof(float) * n, m->stream);
    });
}

int dcrf_step_inference(dcrf_model* m, float* Q, float* tmp1, float* tmp2) {
    return guard([&] {
        require(m && Q, "null argument");
        prepare(*m);
        const size_t n = (size_t)m->N() * m->L;
        m->tmp1.reserve(n);
        m->tmp2.reserve(n);
        hipStream_t s = m->stream;
        copy_to_device(m->Q.get(), Q, sizeof(float) * n, s);
        if (m->terms.empty()) launch_fill(m->tmp2.get(), 0.f, n, s);
        run_filter(*m, splat_rows(*m, m->Q.get(), s), false, s);
        launch_meanfield(m->has_unary ? m->unary.get() : nullptr, m->Q.get(), m->L, m->N(), m->L, m->ldv,
                         slice_table(*m, false, m->kw_set ? m->kw.get() : nullptr), m->tmp1.get(), m->terms.empty() ? nullptr : m->tmp2.get(), s);
        copy_to_host(Q, m->Q.get(), sizeof(float) * n, s);
        if (tmp1) copy_to_host(tmp1, m->tmp1.get(), sizeof(float) * n, s);
        if (tmp2) copy_to_host(tmp2, m->tmp2.get(), sizeof(float) * n, s);
        if (m->timing) collect_timing(*m);
    });
}

int dcrf_kl_divergence(dcrf_model* m, const float* Q, double* kl) {
    return guard([&] {
        require(m && Q && kl, "null argument");
        prepare(*m);
        const size_t n = (size_t)m->N() * m->L;
        m->work.reserve(n);
        hipStream_t s = m->stream;
        copy_to_device(m->work.get(), Q, sizeof(float) * n, s);
        run_filter(*m, splat_rows(*m, m->work.get(), s), false, s);
        const int nb = kl_blocks(m->N(), m->ldv);
        DevBuf<double> part;
        part.reserve(nb);
        launch_kl(m->work.get(), m->has_unary ? m->unary.get() : nullptr, m->N(), m->L, m->ldv,
                  slice_table(*m, false, m->kw_set ? m->kw.get() : nullptr), part.get(), s);
        std::vector<double> h(nb);
        DCRF_HIP_CHECK(hipMemcpyAsync(h.data(), part.get(), sizeof(double) * nb, hipMemcpyDeviceToHost, s));
        DCRF_HIP_CHECK(hipStreamSynchronize(s));
        double acc = 0.0;
        for (double v : h) acc += v;
        *kl = acc;
        if (m->timing) collect_timing(*m);
    });
}

int dcrf_apply_pairwise(dcrf_model* m, int term, const float* Q, float* out, int transpose) {
    return guard([&] {
        require(m && Q && out, "null argument");
        require(term >= 0 && term < (int)m->terms.size(), "pairwise term index out of range");
        prepare(*m);
        const size_t n = (size_t)m->N() * m->L;
        m->work.reserve(n);
        m->tmp1.reserve(n);
        hipStream_t s = m->stream;
        copy_to_device(m->work.get(), Q, sizeof(float) * n, s);
        run_filter(*m, splat_rows(*m, m->work.get(), s), transpose != 0, s);
        launch_slice_term(m->tmp1.get(), m->N(), m->L, m->ldv,
                          slice_table(*m, transpose != 0, m->kw_set ? m->kw.get() : nullptr), term, s);
        copy_to_host(out, m->tmp1.get(), sizeof(float) * n, s);
        if (m->timing) collect_timing(*m);
    });
}

int dcrf_unary_from_softmax_device(const float* sm, int L, int N, double scale, double clip, float* U, void* stream) {
    return guard([&] {
        require(sm && U, "null argument");
        require(L >= 1 && N >= 0, "bad shape");
        require(!(scale > 1.0), "scale needs to be in (0, 1]");
        launch_unary_from_softmax(sm, L, N, scale, scale > 0.0, clip, clip > 0.0, U, (hipStream_t)stream);
    });
}

int dcrf_unary_from_labels_device(const int32_t* labels, int N, int L, double gt_prob, int zero_unsure, float* U,
                                  void* stream) {
    return guard([&] {
        require(labels && U, "null argument");
        require(gt_prob > 0.0 && gt_prob < 1.0, "gt_prob must be in (0, 1)");
        require(L >= 2, "at least two labels");
        // the energies as numpy forms them: float64 logs stored to float32
        const double n_e = -std::log((1.0 - gt_prob) / (L - 1));
        const double p_e = -std::log(gt_prob);
        const double u_e = -std::log(1.0 / L);
        launch_unary_from_labels(labels, N, L, (float)p_e, (float)n_e, (float)u_e, zero_unsure != 0, U,
                                 (hipStream_t)stream);
    });
}

int dcrf_unary_energy(dcrf_model* m, const int16_t* labels, float* out) {
    return guard([&] {
        require(m && labels && out, "null argument");
        const int N = m->N(), L = m->L;
        // DenseCRF::unaryEnergy (densecrf.cpp:141-152): U(l_i, i), 0 for a label outside
        // [0, L) or without a unary
        std::fill(out, out + N, 0.0f);
        if (!m->has_unary) return;
        ensure_device(*m);
        ensure_unary(*m);
        std::vector<float> U((size_t)N * L);
        DCRF_HIP_CHECK(hipMemcpy(U.data(), m->unary.get(), sizeof(float) * U.size(), hipMemcpyDeviceToHost));
        for (int i = 0; i < N; i++)
            if (labels[i] >= 0 && labels[i] < L) out[i] = U[(size_t)i * L + labels[i]];
    });
}

int dcrf_pairwise_energy(dcrf_model* m, const int16_t* labels, int term, float* out) {
    return guard([&] {
        require(m && labels && out, "null argument");
        const int T = (int)m->terms.size();
        require(term == -1 || (term >= 0 && term < T), "pairwise term index out of range");
        const int N = m->N(), L = m->L;
        const size_t n = (size_t)N * L;
        std::fill(out, out + N, 0.0f);
        if (!T) return;
        // DenseCRF::pairwiseEnergy (densecrf.cpp:153-177): the one-hot labelling Q
        // through the term's message, -0.5 Q'(l_i, i); term -1 sums the terms in order
        prepare(*m);
        std::vector<float> Q(n, 0.0f), x(n);
        for (int i = 0; i < N; i++)
            if (labels[i] >= 0 && labels[i] < L) Q[(size_t)i * L + labels[i]] = 1.0f;
        m->work.reserve(n);
        m->tmp1.reserve(n);
        hipStream_t s = m->stream;
        copy_to_device(m->work.get(), Q.data(), sizeof(float) * n, s);
        run_filter(*m, splat_rows(*m, m->work.get(), s), false, s);
        const SliceTable st = slice_table(*m, false, m->kw_set ? m->kw.get() : nullptr);
        for (int k = term < 0 ? 0 : term; k < (term < 0 ? T : term + 1); k++) {
            launch_slice_term(m->tmp1.get(), N, L, m->ldv, st, k, s);
            copy_to_host(x.data(), m->tmp1.get(), sizeof(float) * n, s);
            for (int i = 0; i < N; i++) {
                const float e = labels[i] >= 0 && labels[i] < L ? -0.5f * x[(size_t)i * L + labels[i]] : 0.0f;
                out[i] = out[i] + e;
            }
        }
    });
}

int dcrf_set_compat(dcrf_model* m, int term, const float* params) {
    return guard([&] {
        require(m && params, "null argument");
        require(term >= 0 && term < (int)m->terms.size(), "pairwise term index out of range");
        Term& t = *m->terms[term];
        const int L = m->L;
        if (t.ckind == DCRF_COMPAT_MATRIX) {
            for (int a = 0; a < L; a++)
                for (int b = 0; b < L; b++) {
                    const float sum = params[a * L + b] + params[b * L + a];
                    t.compat[(size_t)a * L + b] = 0.5f * sum;
                }
        } else {
            t.compat.assign(params, params + compat_raw_len(t.ckind, L));
        }
        ensure_device(*m);
        DCRF_HIP_CHECK(hipMemcpy(t.d_compat.get(), t.compat.data(), sizeof(float) * t.compat.size(),
                                 hipMemcpyHostToDevice));
    });
}

int dcrf_set_kernel_weights(dcrf_model* m, const float* w) {
    return guard([&] {
        require(m != nullptr, "null model");
        const int T = (int)m->terms.size();
        if (!w) {
            m->kw_set = false;
            return;
        }
        ensure_device(*m);
        m->kw.reserve(std::max(T, 1));
        DCRF_HIP_CHECK(hipMemcpy(m->kw.get(), w, sizeof(float) * T, hipMemcpyHostToDevice));
        m->kw_set = true;
    });
}

int dcrf_num_compat_params(const dcrf_model* m) {
    if (!m) return 0;
    int n = 0;
    for (const auto& t : m->terms) n += compat_packed_len(t->ckind, m->L);
    return n;
}

int dcrf_get_compat_params(const dcrf_model* m, float* p) {
    return guard([&] {
        require(m && p, "null argument");
        const int L = m->L;
        for (const auto& tp : m->terms) {
            std::vector<float> c(tp->compat.size());
            if (m->dev_ready)
                DCRF_HIP_CHECK(hipMemcpy(c.data(), tp->d_compat.get(), sizeof(float) * c.size(), hipMemcpyDeviceToHost));
            else
                c = tp->compat;
            if (tp->ckind == DCRF_COMPAT_MATRIX) {
                for (int i = 0; i < L; i++)
                    for (int j = i; j < L; j++) *p++ = c[(size_t)i * L + j];
            } else {
                for (float v : c) *p++ = v;
            }
        }
    });
}

int dcrf_set_compat_params(dcrf_model* m, const float* p) {
    return guard([&] {
        require(m && p, "null argument");
        ensure_device(*m);
        const int L = m->L;
        // setLabelCompatibilityParameters (densecrf.cpp:329-341): Potts w, Diagonal w[L],
        // Matrix upper triangle w(i, j>=i) written to both w(i,j) and w(j,i)
        // (labelcompatibility.cpp:95-100)
        for (auto& tp : m->terms) {
            Term& t = *tp;
            if (t.ckind == DCRF_COMPAT_MATRIX) {
                for (int i = 0; i < L; i++)
                    for (int j = i; j < L; j++) {
                        const float v = *p++;
                        t.compat[(size_t)i * L + j] = v;
                        t.compat[(size_t)j * L + i] = v;
                    }
            } else {
                for (float& v : t.compat) v = *p++;
            }
            DCRF_HIP_CHECK(hipMemcpy(t.d_compat.get(), t.compat.data(), sizeof(float) * t.compat.size(),
                                     hipMemcpyHostToDevice));
        }
    });
}

int dcrf_num_kernel_params(const dcrf_model* m) { return m ? num_kernel_params(*m) : 0; }

int dcrf_get_kernel_params(const dcrf_model* m, float* params) {
    return guard([&] {
        require(m && params, "null argument");
        for (const auto& t : m->terms) {
            std::copy(t->kparams.begin(), t->kparams.begin() + t->num_kparams(), params);
            params += t->num_kparams();
        }
    });
}

int dcrf_set_kernel_params(dcrf_model* m, const float* params) {
    return guard([&] {
        require(m && params, "null argument");
        const int np = num_kernel_params(*m);
        for (int i = 0; i < np; i++) require(std::isfinite(params[i]), "kernel parameters must be finite");
        ensure_device(*m);
        hipStream_t s = m->stream;
        // new lattices of every scaled term first, then commit them all
        struct Rebuilt {
            Term* t;
            Term tmp;
            std::vector<float> kp;
        };
        std::vector<std::unique_ptr<Rebuilt>> done;
        const float* p = params;
        const int npad = m->geo.npad_total();
        for (auto& tp : m->terms) {
            Term& t = *tp;
            const int n = t.num_kparams();
            if (!n) continue;
            auto r = std::make_unique<Rebuilt>();
            r->t = &t;
            r->kp.assign(p, p + n);
            p += n;
            const int d = t.lat.d;
            DevBuf<float> P, feat;
            upload(P, r->kp, s);
            feat.reserve((size_t)npad * d);
            launch_scale_features(t.feat0.get(), npad, d, t.ktype == DCRF_FULL_KERNEL, P.get(), feat.get(), s);
            r->tmp.ntype = t.ntype;
            build_lattice(m->geo, m->geod, m->tiles, feat.get(), d, r->tmp.lat, m->hash_load, s);
            if (r->tmp.lat.overflow)
                throw Error{DCRF_ERR_OVERFLOW, "a scaled lattice coordinate exceeds the int16 range of the lattice "
                                               "keys; scale the kernel parameters down"};
            done.push_back(std::move(r));
        }
        for (auto& r : done) {
            r->t->lat = std::move(r->tmp.lat);
            r->t->kparams = std::move(r->kp);
        }
        if (!done.empty()) {
            m->layout_valid = false;
            m->lat_gen++;
            m->train_n = -1;
            m->drop_graph();
        }
    });
}

int dcrf_gradient(dcrf_model* m, int n_iter, const int16_t* gt, float robust, double* objective, float* unary_grad,
                  float* compat_grad, float* kweight_grad, float* kernel_grad) {
    return dcrf_gradient_objective(m, n_iter, DCRF_OBJECTIVE_LOG_LIKELIHOOD, gt, robust, nullptr, 0, objective,
                                   unary_grad, compat_grad, kweight_grad, kernel_grad);
}

int dcrf_gradient_objective(dcrf_model* m, int n_iter, int objective_kind, const int16_t* gt, float param,
                            const float* class_weight, int n_class_weight, double* objective, float* unary_grad,
                            float* compat_grad, float* kweight_grad, float* kernel_grad) {
    return guard([&] {
        require(m && gt, "null argument");
        require(n_iter >= 0, "number of iterations must be non-negative");
        require(objective_kind >= DCRF_OBJECTIVE_LOG_LIKELIHOOD && objective_kind <= DCRF_OBJECTIVE_IOU,
                "unknown objective");
        require(!class_weight || n_class_weight >= 0, "negative class-weight count");
        prepare(*m);
        const int N = m->N(), L = m->L, T = (int)m->terms.size();
        const size_t NL = (size_t)N * L;
        hipStream_t s = m->stream;
        const float* U = m->has_unary ? m->unary.get() : nullptr;
        const float* kw = m->kw_set ? m->kw.get() : nullptr;
        // Hamming's class weights come from the host's ground truth (objective.cpp:51-63)
        std::vector<float> hw;
        if (objective_kind == DCRF_OBJECTIVE_HAMMING) hw = hamming_weights(gt, N, L, param, class_weight,
                                                                              n_class_weight);
        forward_train(*m, n_iter, U, nullptr, kw, s);
        m->work.reserve(NL);
        m->tmp1.reserve(NL);
        m->gt_dev.reserve(N);
        DCRF_HIP_CHECK(hipMemcpyAsync(m->gt_dev.get(), gt, sizeof(int16_t) * N, hipMemcpyHostToDevice, s));
        if (!hw.empty()) {
            m->obj_w.reserve(hw.size());
            DCRF_HIP_CHECK(hipMemcpyAsync(m->obj_w.get(), hw.data(), sizeof(float) * hw.size(),
                                          hipMemcpyHostToDevice, s));
        }
        const int npart = objective_partials(objective_kind, N, L);
        m->obj_partial.reserve(npart);
        launch_objective(objective_kind, m->qcache.get() + (size_t)n_iter * N * m->ldv, m->gt_dev.get(), N, L, param,
                         hw.empty() ? nullptr : m->obj_w.get(), m->work.get(), m->obj_partial.get(), s);
        std::vector<double> OP(npart);
        DCRF_HIP_CHECK(hipMemcpyAsync(OP.data(), m->obj_partial.get(), sizeof(double) * npart,
                                      hipMemcpyDeviceToHost, s));
        const int nkp = num_kernel_params(*m);
        backward(*m, m->work.get(), m->tmp1.get(), nullptr, nullptr, s, kernel_grad && nkp > 0);
        std::vector<double> KG(nkp, 0.0);
        if (kernel_grad && nkp && n_iter > 0)
            DCRF_HIP_CHECK(hipMemcpyAsync(KG.data(), m->kacc.get(), sizeof(double) * nkp, hipMemcpyDeviceToHost, s));
        if (unary_grad)
            copy_to_host(unary_grad, m->tmp1.get(), sizeof(float) * NL, s);
        std::vector<double> UG;
        if (m->logistic) {
            // LogisticUnaryEnergy::gradient summed over the iterations (densecrf.cpp:261-262,
            // 293-294; unary.cpp:64-68): sum_t b_t f^T = (dL/dU) f^T, one gram product
            const int F = m->lF;
            m->partial.reserve(std::max(m->partial.n, gram_partial_floats(L, F, N)));
            m->gacc2.reserve((size_t)L * F);
            launch_gram(m->tmp1.get(), L, m->lf.get(), F, N, m->partial.get(), m->gacc2.get(), s);
            UG.resize((size_t)L * F);
            DCRF_HIP_CHECK(hipMemcpyAsync(UG.data(), m->gacc2.get(), sizeof(double) * L * F, hipMemcpyDeviceToHost, s));
        }
        size_t glen = 0;
        for (auto& t : m->terms) glen += stat_len(t->ckind, L);
        std::vector<double> G(glen);
        DCRF_HIP_CHECK(hipMemcpyAsync(G.data(), m->gacc.get(), sizeof(double) * glen, hipMemcpyDeviceToHost, s));
        std::vector<float> w(T, 1.0f);
        if (kw) DCRF_HIP_CHECK(hipMemcpyAsync(w.data(), kw, sizeof(float) * T, hipMemcpyDeviceToHost, s));
        // the compatibilities the forward used: the device copies (a training forward with
        // raw compatibilities, dcrf_forward_device, writes them there only)
        std::vector<std::vector<float>> cw(T);
        for (int k = 0; k < T; k++) {
            const Term& t = *m->terms[k];
            cw[k].resize(compat_raw_len(t.ckind, L));
            DCRF_HIP_CHECK(hipMemcpyAsync(cw[k].data(), t.d_compat.get(), sizeof(float) * cw[k].size(),
                                          hipMemcpyDeviceToHost, s));
        }
        DCRF_HIP_CHECK(hipStreamSynchronize(s));
        if (objective) *objective = objective_value(objective_kind, OP, L);
        // pack like DenseCRF::gradient (labelcompatibility.cpp:57-61, 76-78, 101-108)
        size_t go = 0;
        float* cp = compat_grad;
        for (int k = 0; k < T; k++) {
            const Term& t = *m->terms[k];
            const double* g = G.data() + go;
            double kg = 0.0;
            if (t.ckind == DCRF_COMPAT_POTTS) {
                double sd = 0.0;
                for (int a = 0; a < L; a++) sd += g[a];
                if (cp) *cp++ = (float)(-w[k] * sd);
                kg = -(double)cw[k][0] * sd;
            } else if (t.ckind == DCRF_COMPAT_DIAGONAL) {
                for (int a = 0; a < L; a++) {
                    if (cp) *cp++ = (float)(w[k] * g[a]);
                    kg += (double)cw[k][a] * g[a];
                }
            } else {
                for (int i = 0; i < L; i++)
                    for (int j = i; j < L; j++) {
                        const double v = i == j ? g[i * L + i] : g[i * L + j] + g[j * L + i];
                        if (cp) *cp++ = (float)(w[k] * v);
                    }
                for (int j = 0; j < L * L; j++) kg += (double)cw[k][j] * g[j];
            }
            if (kweight_grad) kweight_grad[k] = (float)kg;
            go += stat_len(t.ckind, L);
        }
        if (kernel_grad)
            for (int i = 0; i < nkp; i++) kernel_grad[i] = (float)KG[i];
        if (m->logistic) {
            const int F = m->lF;
            m->ugrad_param.resize((size_t)L * F);
            for (int c = 0; c < F; c++)
                for (int r = 0; r < L; r++) m->ugrad_param[(size_t)c * L + r] = (float)UG[(size_t)r * F + c];
        }
        if (m->timing) collect_timing(*m);
    });
}

int dcrf_forward_device(dcrf_model* m, int n_iter, const float* U_dev, const float* compat_dev, const float* kw_dev,
                        float* Q_dev, void* stream) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(n_iter >= 0, "number of iterations must be non-negative");
        prepare(*m);
        hipStream_t s = (hipStream_t)stream;
        const float* U = U_dev ? U_dev : (m->has_unary ? m->unary.get() : nullptr);
        const float* kw = kw_dev ? kw_dev : (m->kw_set ? m->kw.get() : nullptr);
        forward_train(*m, n_iter, U, compat_dev, kw, s);
        if (Q_dev) {
            const size_t NL = (size_t)m->N() * m->L;
            DCRF_HIP_CHECK(hipMemcpyAsync(Q_dev, m->qcache.get() + (size_t)n_iter * m->N() * m->ldv, sizeof(float) * NL,
                                          hipMemcpyDeviceToDevice, s));
        }
    });
}

int dcrf_backward_device(dcrf_model* m, const float* dQ_dev, float* dU_dev, float* dcompat_dev, float* dkw_dev,
                         float* dkernel_dev, void* stream) {
    return guard([&] {
        require(m && dQ_dev && dU_dev, "null argument");
        hipStream_t s = (hipStream_t)stream;
        const int nkp = num_kernel_params(*m);
        const bool kernel = dkernel_dev && nkp > 0;
        backward(*m, dQ_dev, dU_dev, dcompat_dev, dkw_dev, s, kernel);
        if (kernel) {
            if (m->train_n > 0)
                launch_kparam_store(m->kacc.get(), nkp, dkernel_dev, s);
            else
                launch_fill(dkernel_dev, 0.f, nkp, s);
        }
    });
}

int dcrf_num_variables(const dcrf_model* m) { return m ? m->N() : 0; }
int dcrf_num_labels(const dcrf_model* m) { return m ? m->L : 0; }
int dcrf_num_terms(const dcrf_model* m) { return m ? (int)m->terms.size() : 0; }
int dcrf_num_instances(const dcrf_model* m) { return m ? m->geo.n_inst : 0; }

int dcrf_term_info(const dcrf_model* m, int term, int* d, int* V) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(term >= 0 && term < (int)m->terms.size(), "pairwise term index out of range");
        if (d) *d = m->terms[term]->lat.d;
        if (V) *V = m->terms[term]->lat.V;
    });
}

int dcrf_term_instance_vertices(const dcrf_model* m, int term, int inst, int* V) {
    return guard([&] {
        require(m && V, "null argument");
        require(term >= 0 && term < (int)m->terms.size(), "pairwise term index out of range");
        require(inst >= 0 && inst < m->geo.n_inst, "instance index out of range");
        const auto& vb = m->terms[term]->lat.inst_vbase;
        *V = vb[inst + 1] - vb[inst];
    });
}

int dcrf_get_lattice(const dcrf_model* m, int term, int inst, int* offset, int* rank, float* bary, int* nbr,
                     int16_t* keys, float* norm) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(term >= 0 && term < (int)m->terms.size(), "pairwise term index out of range");
        require(inst >= 0 && inst < m->geo.n_inst, "instance index out of range");
        const Term& t = *m->terms[term];
        const TermLattice& lat = t.lat;
        const int d1 = lat.d + 1;
        const int pb = m->geo.pix_base[inst], Ni = m->geo.N[inst];
        const int vb = lat.inst_vbase[inst], Vi = lat.inst_vbase[inst + 1] - vb;
        const size_t ne = (size_t)Ni * d1;
        if (offset) {
            DCRF_HIP_CHECK(hipMemcpy(offset, lat.vtx.get() + (size_t)pb * d1, sizeof(int) * ne, hipMemcpyDeviceToHost));
            for (size_t i = 0; i < ne; i++) offset[i] -= vb;
        }
        if (rank) DCRF_HIP_CHECK(hipMemcpy(rank, lat.rank.get() + (size_t)pb * d1, sizeof(int) * ne, hipMemcpyDeviceToHost));
        if (bary) DCRF_HIP_CHECK(hipMemcpy(bary, lat.bary.get() + (size_t)pb * d1, sizeof(float) * ne, hipMemcpyDeviceToHost));
        if (nbr) {
            std::vector<int> all((size_t)2 * d1 * lat.V);
            DCRF_HIP_CHECK(hipMemcpy(all.data(), lat.nbr.get(), sizeof(int) * all.size(), hipMemcpyDeviceToHost));
            for (int j = 0; j < d1; j++)
                for (int v = 0; v < Vi; v++)
                    for (int c = 0; c < 2; c++) {
                        const int x = all[2 * ((size_t)j * lat.V + vb + v) + c];
                        nbr[2 * ((size_t)j * Vi + v) + c] = x < 0 ? -1 : x - vb;
                    }
        }
        if (keys)
            DCRF_HIP_CHECK(hipMemcpy(keys, lat.keys.get() + (size_t)vb * lat.d, sizeof(int16_t) * (size_t)Vi * lat.d,
                                     hipMemcpyDeviceToHost));
        if (norm) {
            DevBuf<float> own;  // the layout, which holds the normalisers, is not built for them
            if (!m->layout_valid) term_norm(*m, t, own);
            const float* src = m->layout_valid ? t.norm.get() : own.get();
            DCRF_HIP_CHECK(hipMemcpy(norm, src + pb, sizeof(float) * Ni, hipMemcpyDeviceToHost));
        }
    });
}

int dcrf_set_splat_chunk(dcrf_model* m, int chunk) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(chunk >= 0 && chunk <= (1 << 20), "chunk length out of range");
        if (chunk != m->splat_chunk) {
            m->splat_chunk = chunk;
            m->layout_valid = false;
        }
    });
}

int dcrf_set_splat_tile(dcrf_model* m, int side) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(side >= 0 && side <= 4096, "tile side must be in [0, 4096]");
        require(m->terms.empty(), "set the splat tile before adding pairwise terms", DCRF_ERR_STATE);
        m->tile_side = side;
        m->tiles_ready = false;
    });
}

int dcrf_set_meanfield_kernel(dcrf_model* m, int mode, int run_rows) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(mode >= 0 && mode <= 3, "mean-field kernel mode must be 0 (auto), 1, 2 or 3");
        require(run_rows >= 0 && run_rows <= 64, "run rows must be in [0, 64]");
        const int rr = run_rows ? run_rows : 16;
        if (mode != m->mf_mode || rr != m->run_rows) {
            m->mf_mode = mode;
            m->run_rows = rr;
            m->layout_valid = false;
        }
    });
}

int dcrf_set_blur_lanes(dcrf_model* m, int labels_per_lane, int below_vertices) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(labels_per_lane >= 0 && labels_per_lane <= 4, "labels per lane must be 0 (default) or 1 to 4");
        require(labels_per_lane == 0 || m->L % labels_per_lane == 0, "labels per lane must divide the label count");
        require(labels_per_lane == 0 || shape_for_r(m->L, labels_per_lane).wave,
                "too few labels per lane for a lane group within one wave");
        m->blur_r = labels_per_lane;
        m->blur_small_v = below_vertices;
        m->drop_graph();
    });
}

int dcrf_set_q_blocks(dcrf_model* m, int on) {
    return guard([&] {
        require(m != nullptr, "null model");
        if (m->qblocks != (on != 0)) {
            m->qblocks = on != 0;
            m->qblocks_ready = false;
            m->drop_graph();
        }
    });
}

int dcrf_set_blur_steps(dcrf_model* m, int steps) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(steps == 2 || steps == 3, "blur steps per pass: 2 or 3");
        if (m->blur_steps != steps) {
            m->blur_steps = steps;
            m->layout_valid = false;
            m->train_n = -1;
        }
    });
}

int dcrf_set_blur_pairs(dcrf_model* m, int on) {
    return guard([&] {
        require(m != nullptr, "null model");
        if (m->pairs != (on != 0)) {
            m->pairs = on != 0;
            m->layout_valid = false;
            m->train_n = -1;
        }
    });
}

int dcrf_set_hash_load(dcrf_model* m, float load) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(load > 0.0f && load <= 0.5f, "hash load factor must be in (0, 0.5]");
        m->hash_load = load;
    });
}

int dcrf_enable_timing(dcrf_model* m, int on) {
    return guard([&] {
        require(m != nullptr, "null model");
        if (m->timing && !on) collect_timing(*m);
        m->timing = on != 0;
        for (int c = 0; c < KC_COUNT; c++) {
            m->kc_launches[c] = 0;
            m->kc_ms[c] = 0.0;
            m->kc_bytes[c] = 0.0;
        }
    });
}

int dcrf_kernel_stats(dcrf_model* m, int kernel, long long* launches, double* ms, double* bytes) {
    return guard([&] {
        require(m != nullptr, "null model");
        require(kernel >= 0 && kernel < KC_COUNT, "unknown kernel class");
        collect_timing(*m);
        if (launches) *launches = m->kc_launches[kernel];
        if (ms) *ms = m->kc_ms[kernel];
        if (bytes) *bytes = m->kc_bytes[kernel];
    });
}

int dcrf_splat_layout(dcrf_model* m, int* tiled, int* tile_side, int* n_tiles, int* segments, int* partials,
                      int* meanfield) {
    return guard([&] {
        require(m && tiled && tile_side && n_tiles && segments && partials && meanfield, "null argument");
        ensure_device(*m);
        ensure_layout(*m);
        *tiled = m->tiled ? 1 : 0;
        *tile_side = m->tiles.side;
        *n_tiles = m->tiles.n_tiles();
        *segments = m->seg.nch;
        *partials = m->rows0 - m->V_total - 1;
        *meanfield = m->runs ? 2 : (m->fused ? 1 : 0);
    });
}

int dcrf_iteration_bytes(const dcrf_model* m, double* bytes) {
    return guard([&] {
        require(m && bytes, "null argument");
        const double N = m->N(), L = m->L;
        double b = 3.0 * N * L * 4.0;
        for (const auto& t : m->terms) {
            const double d1 = t->lat.d + 1, V = t->lat.V;
            b += 2.0 * N * d1 * 8.0 + 2.0 * N * 4.0 + V * L * 4.0 * (2.0 + 2.0 * d1) + d1 * V * 8.0;
        }
        *bytes = b;
    });
}

}  // extern "C"
