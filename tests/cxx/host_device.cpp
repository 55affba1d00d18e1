// The library's host code on a device of host memory: this program defines the
// HIP calls that libmwgreen.so imports (the executable's definitions come
// first), with memory that is counted against a capacity, streams and events
// that keep account of what waits for what, and kernels that do nothing (norms
// are all one, and a search finds no slot) but can be made to fail.  So the host's error paths and its use of memory are
// checked without a GPU (tests/test_host_device.py).
//
//   host_device <scenario>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#define _Float16 short  // (g++ has none; only pointers to it are declared)
#include "mw_apply.hpp"
#undef _Float16
#include "mwgreen.h"

namespace {

std::recursive_mutex g_mtx;
size_t g_capacity = (size_t)4 << 30, g_used = 0, g_peak = 0, g_copy_max = ~(size_t)0;
long long g_mallocs = 0;
std::map<void *, size_t> g_mem;
// by host function (registered before this program's own objects are made)
std::map<const void *, std::string> &kernels() {
    static std::map<const void *, std::string> k;
    return k;
}
std::map<std::string, long long> g_groups;  // workgroups (x) launched, by kernel
std::string g_fail;  // launches of kernels with this in their names fail
int g_failed = 0;
hipError_t g_last = hipSuccess;

// A stream: items enqueued, items finished, and how far into each other stream
// its own next item waits.
struct Stream {
    long long queued = 0, done = 0;
    std::map<Stream *, long long> after;
};
struct Event {
    Stream *s = nullptr;
    long long at = 0;
    std::map<Stream *, long long> after;
};
std::vector<Stream *> g_streams;

Stream *of(hipStream_t s) { return reinterpret_cast<Stream *>(s); }
Event *of(hipEvent_t e) { return reinterpret_cast<Event *>(e); }

void finish(Stream *s, long long at, const std::map<Stream *, long long> &after) {
    s->done = std::max(s->done, at);
    for (const auto &a : after) a.first->done = std::max(a.first->done, a.second);
}

// Items of the second and later streams that are neither finished nor waited
// for by the first stream (the context's).
long long unjoined() {
    long long n = 0;
    for (size_t i = 1; i < g_streams.size(); i++) {
        Stream *s = g_streams[i], *main = g_streams[0];
        n += s->queued - std::max(s->done, main->after.count(s) ? main->after[s] : 0);
    }
    return n;
}

hipError_t result(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}

}  // namespace

extern "C" {

struct Dim {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
};
static thread_local std::vector<Dim> t_config;

void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
    kernels()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream) {
    t_config.push_back(Dim{grid, block, shmem, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, hipStream_t *stream) {
    const Dim d = t_config.back();
    t_config.pop_back();
    *grid = d.grid;
    *block = d.block;
    *shmem = d.shmem;
    *stream = d.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t s) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    // the work items of a launch are counted in 32 bits
    if ((unsigned long long)grid.x * block.x >= (1ull << 32) || grid.x == 0 || grid.y == 0 || grid.y > 65535)
        return result(hipErrorInvalidConfiguration);
    if (!g_fail.empty() && kernels()[f].find(g_fail) != std::string::npos) {
        g_failed++;
        return result(hipErrorLaunchFailure);
    }
    const std::string &name = kernels()[f];
    auto ones = [&](int s2) {
        for (int a = s2; a < s2 + 2; a++)
            if (double *p = *static_cast<double **>(args[a])) std::fill_n(p, grid.x, 1.0);
    };
    if (name.find("k_node_norms") != std::string::npos) ones(3);
    if (name.find("k_move_norms") != std::string::npos) ones(2);
    if (name.find("k_band_clear") != std::string::npos)
        std::fill_n(static_cast<mwg::BandArgs *>(args[0])->cnt, mwg::kBandCounts, 0u);
    g_groups[name] += grid.x;
    of(s)->queued++;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 2;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}

hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    *p = nullptr;
    if (g_used + n > g_capacity) return result(hipErrorOutOfMemory);
    *p = std::calloc(n, 1);
    g_mallocs++;
    g_mem[*p] = n;
    g_used += n;
    g_peak = std::max(g_peak, g_used);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    if (!p) return hipSuccess;
    auto it = g_mem.find(p);
    if (it == g_mem.end()) {
        std::printf("FAIL: free of memory that is not allocated\n");
        std::exit(1);
    }
    for (Stream *s : g_streams) s->done = s->queued;  // waits for the device
    g_used -= it->second;
    g_mem.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(n, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *scratch = std::calloc((size_t)128 << 20, 1);
    *p = scratch;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t s) {
    if (n <= g_copy_max) std::memcpy(dst, src, n);
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    of(s)->queued++;
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int v, size_t n, hipStream_t s) {
    std::memset(dst, v, n);
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    of(s)->queued++;
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    g_streams.push_back(new Stream);
    *s = reinterpret_cast<hipStream_t>(g_streams.back());
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    finish(of(s), of(s)->queued, of(s)->after);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    auto wait = [&](Stream *o, long long at) {
        if (o && o != of(s)) of(s)->after[o] = std::max(of(s)->after[o], at);
    };
    wait(of(e)->s, of(e)->at);
    for (const auto &a : of(e)->after) wait(a.first, a.second);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    delete of(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    *of(e) = Event{of(s), of(s)->queued, of(s)->after};
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::recursive_mutex> g(g_mtx);
    if (of(e)->s) finish(of(e)->s, of(e)->at, of(e)->after);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.f;
    return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return result(hipErrorNotSupported); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return result(hipErrorNotSupported); }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    return result(hipErrorNotSupported);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return result(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"

namespace {

int g_bad = 0;
void check(bool ok, const char *what) {
    if (ok) return;
    std::printf("FAIL: %s (%s)\n", what, mwg_last_error());
    g_bad++;
}

mwg_mra world(int order, int depth) {
    const int corner[3] = {-1, -1, -1}, boxes[3] = {2, 2, 2};
    mwg_mra m = nullptr;
    check(mwg_mra_create(order, 0, -4, corner, boxes, 1.25, depth, &m) == MWG_OK, "MRA");
    return m;
}

mwg_tree gaussian(mwg_mra m, double prec, double a) {
    mwg_tree t = nullptr;
    const double c = 1.0, pos[3] = {0.3, -0.2, 0.1};
    check(mwg_tree_create(m, &t) == MWG_OK, "tree");
    check(mwg_tree_project_gaussians(t, prec, 0, -1, 1, &c, &a, pos) == MWG_OK, "projection");
    return t;
}

// A step of the split mode that fails after its FP64 class went to the second
// stream leaves nothing there that the context's stream does not wait for.
void split_step_fails() {
    mwg_mra m = world(3, 8);
    mwg_context ctx = nullptr;
    check(mwg_context_create(0, &ctx) == MWG_OK, "context");
    check(mwg_context_set_precision(ctx, MWG_MODE_SPLIT16, 65536.0) == MWG_OK, "mode");
    mwg_operator P = nullptr;
    check(mwg_poisson_create(m, 1e-2, &P) == MWG_OK, "operator");
    mwg_tree f = gaussian(m, 1e-2, 4.0), V = nullptr;
    check(mwg_tree_create(m, &V) == MWG_OK, "tree");
    g_fail = "k_apply_h";
    check(mwg_apply(ctx, 1e-2, V, P, f, -1, 1) == MWG_ERR_DEVICE, "the apply reports the failed launch");
    std::printf("%zu streams, %lld items on the second, %d launches failed, %lld items not joined\n", g_streams.size(),
                g_streams[1]->queued, g_failed, unjoined());
    check(g_failed == 1 && g_streams[1]->queued > 0, "the split launch failed behind the fork");
    check(unjoined() == 0, "the second stream is joined");
}

// Memory that lies idle in a context's pool is given back for every kind of
// allocation, and a block whose size class does not fit is tried at its size.
void idle_memory_is_given_back() {
    mwg_mra m = world(7, 8);
    mwg_context a = nullptr, b = nullptr;
    check(mwg_context_create(0, &a) == MWG_OK && mwg_context_create(0, &b) == MWG_OK, "contexts");
    mwg_tree f = gaussian(m, 1e-4, 40.0);
    int n = 0;
    check(mwg_tree_size(f, &n) == MWG_OK, "size");
    const size_t bytes = (size_t)n * 8 * 512 * sizeof(double);
    long long size = 0;
    check(mwg_tree_pack_size(f, &size) == MWG_OK, "pack size");
    std::vector<char> packed(size);
    // (each uploads the blocks and puts them back)
    for (mwg_context c : {a, b}) check(mwg_tree_pack_device(f, c, packed.data(), size) == MWG_OK, "pack");
    std::printf("%d nodes, %zu bytes of blocks, %zu held by the pools\n", n, bytes, g_used);
    check(g_used >= 2 * bytes, "both pools hold their blocks");
    // room for the tree's blocks once, but not beside what lies idle
    g_capacity = g_used + bytes / 2;
    void *buf = nullptr;
    check(mwg_device_buffer_create(a, (long long)bytes, &buf) == MWG_OK, "a caller's buffer");
    check(mwg_device_buffer_destroy(a, buf) == MWG_OK, "destroy");
    // room for the blocks to the byte, less than their class
    g_capacity = g_used + bytes;
    check(mwg_tree_pack_device(f, a, packed.data(), size) == MWG_OK, "blocks on a card they just fit");
    check(g_used <= g_capacity, "within the card");
}

// What the contexts of a device hold idle is bounded for all of them together,
// and a context that works after many others still keeps its own.
void idle_memory_is_bounded() {
    mwg_mra m = world(11, 4);
    g_capacity = (size_t)64 << 30;
    g_copy_max = (size_t)1 << 20;  // larger transfers move nothing
    const size_t bound = (size_t)8 << 30;
    mwg_tree f = nullptr;
    const double c = 1.0, e = 0.05, pos[3] = {0.3, -0.2, 0.1};
    check(mwg_tree_create(m, &f) == MWG_OK, "tree");
    check(mwg_tree_project_gaussians(f, 1e-30, 1, 3, 1, &c, &e, pos) == MWG_OK, "projection");
    int n = 0;
    long long size = 0;
    check(mwg_tree_size(f, &n) == MWG_OK && mwg_tree_pack_size(f, &size) == MWG_OK, "size");
    const size_t bytes = (size_t)n * 8 * 1728 * sizeof(double);
    char *dst = static_cast<char *>(std::malloc(size));
    size_t most = 0;
    long long last = 0;
    const int contexts = (int)(bound / bytes) + 4;
    for (int i = 0; i < contexts; i++) {
        mwg_context ctx = nullptr;
        check(mwg_context_create(0, &ctx) == MWG_OK, "context");
        check(mwg_tree_pack_device(f, ctx, dst, size) == MWG_OK, "pack");
        most = std::max(most, g_used);
        last = g_mallocs;
        check(mwg_tree_pack_device(f, ctx, dst, size) == MWG_OK, "pack again");
        last = g_mallocs - last;
    }
    std::printf("%d nodes, %zu bytes of blocks, %d contexts: at most %zu bytes idle\n", n, bytes, contexts, most);
    check(most > bound / 2 && most <= bound, "idle memory of all contexts");
    check(last == 0, "the last context's block is kept for its next call");
}

// An apply to a host tree holds its output's blocks on the device once.
void host_output_memory() {
    mwg_mra m = world(5, 4);
    mwg_context ctx = nullptr;
    check(mwg_context_create(0, &ctx) == MWG_OK, "context");
    mwg_operator P = nullptr;
    check(mwg_poisson_create(m, 1e-2, &P) == MWG_OK, "operator");
    mwg_tree f = gaussian(m, 1e-2, 1.0), V = nullptr;
    check(mwg_tree_create(m, &V) == MWG_OK, "tree");
    g_copy_max = (size_t)16 << 20;  // larger transfers move nothing
    // every wavelet norm is one: the grid grows to the full depth
    check(mwg_apply(ctx, 0.1, V, P, f, -1, 1) == MWG_OK, "apply");
    int n = 0;
    check(mwg_tree_size(V, &n) == MWG_OK, "size");
    const size_t bytes = (size_t)n * 8 * 216 * sizeof(double);
    std::printf("%d nodes, %zu bytes of blocks, at most %zu bytes on the device\n", n, bytes, g_peak);
    check(n == 8 * 4681, "the whole grid");
    check(g_peak < bytes + bytes * 4 / 5, "blocks on the device once, and a part of them to copy from");
}

// The stages of an apply's plan make up its plan time, each under its own name.
void apply_stages() {
    mwg_mra m = world(3, 3);
    mwg_context ctx = nullptr;
    check(mwg_context_create(0, &ctx) == MWG_OK, "context");
    mwg_operator P = nullptr;
    check(mwg_poisson_create(m, 1e-2, &P) == MWG_OK, "operator");
    mwg_tree f = gaussian(m, 1e-2, 4.0), V = nullptr;
    check(mwg_tree_create(m, &V) == MWG_OK, "tree");
    check(mwg_apply(ctx, 1e-2, V, P, f, -1, 1) == MWG_OK, "apply");
    double st[16];
    check(mwg_last_apply_stats(ctx, st, 16) == MWG_OK, "stats");
    std::printf("plan %g ms = bands %g + pools %g + counts %g; create %g + run %g of %g; apply %g\n", st[4], st[13],
                st[14], st[15], st[11], st[12], st[7], st[10]);
    for (int i : {11, 12, 13, 14, 15}) check(st[i] > 0.0, "every stage takes time");
    const double sum = st[13] + st[14] + st[15];
    check(sum > st[4] * (1.0 - 1e-12) && sum < st[4] * (1.0 + 1e-12), "bands, pools and counts are the plan");
    check(st[11] + st[12] <= st[7] && st[4] + st[7] + st[8] + st[9] <= st[10], "no time counted twice");
}

// More nodes and slots than one launch has work items for: the launches are
// split, and together hold a workgroup for each.
void more_than_a_launch() {
    hipStream_t stream = nullptr;
    check(hipStreamCreateWithFlags(&stream, 0) == hipSuccess, "stream");
    std::string err;
    const int n = 20 << 20;  // times 256 threads: past 32 bits
    auto groups = [](const char *kernel) {
        long long sum = 0;
        for (const auto &g : g_groups)
            if (g.first.find(kernel) != std::string::npos) sum += g.second;
        return sum;
    };
    mwg::BandArgs b{};
    std::vector<unsigned> cnt(mwg::kBandCounts);
    b.n_out = n;
    b.cap = 1024;
    b.cnt = cnt.data();
    check(mwg::dev_band_find(stream, b, 27, err) == 0 && groups("k_band_find") == n, "bands");
    mwg::CountArgs c;
    c.n_out = n;
    c.widest = 27;
    for (bool bounds : {false, true}) {
        g_groups.clear();
        check(mwg::dev_count_terms(stream, c, bounds, err) == 0 && groups("k_count") == n, "counts");
        check(mwg::dev_cut_segments(stream, c, bounds, err) == 0 && groups("k_cut") == (bounds ? 2LL : 1LL) * n, "cuts");
    }
    check(mwg::dev_pool_fill(stream, 2, nullptr, nullptr, {0, n, 2 * n}, nullptr, n, err) == 0 &&
              groups("k_gen_fill") == 2LL * n && groups("k_pool_fill") == 2LL * n,
          "pool");
    std::printf("%d nodes: %s\n", n, err.c_str());
}

}  // namespace

int main(int argc, char **argv) {
    const std::map<std::string, void (*)()> scenarios = {{"split_step_fails", split_step_fails},
                                                            {"idle_memory_is_given_back", idle_memory_is_given_back},
                                                            {"idle_memory_is_bounded", idle_memory_is_bounded},
                                                            {"host_output_memory", host_output_memory},
                                                            {"apply_stages", apply_stages},
                                                            {"more_than_a_launch", more_than_a_launch}};
    const auto it = argc > 1 ? scenarios.find(argv[1]) : scenarios.end();
    if (it == scenarios.end()) return 2;
    it->second();
    std::fflush(stdout);
    std::_Exit(g_bad ? 1 : 0);
}
