// Interface between the host driver and the HIP apply kernels.
#pragma once

#include <string>
#include <vector>

#include "mw_internal.hpp"

namespace mwg {

struct DeviceCtx;

// Workgroups of `threads` that one launch can hold: its work items are counted
// in 32 bits.  Launches of a workgroup per node, slot or segment run in parts
// of that many.
constexpr long long launch_room(int threads) { return ((1LL << 32) - 1) / threads; }
// launch(first, count) over [0, n) in parts a launch can hold.
template <typename F>
int in_launches(long long n, int threads, F &&launch) {
    const long long room = launch_room(threads);
    for (long long i = 0; i < n; i += room)
        if (const int rc = launch(i, n - i < room ? n - i : room)) return rc;
    return 0;
}

// Returns 0 on success; on failure a negative code and a message in err
// (-1: invalid argument, -2: device error).
int dev_create(int device, DeviceCtx **out, std::string &err);
void dev_destroy(DeviceCtx *c);
// Drop the device copy of an operator's tables (called when it is destroyed).
void dev_forget_operator(DeviceCtx *c, const void *key);

// One apply of a (possibly batched) device plan: the operator (its host
// tables, keyed for the context's resident copy), the host plan, the input
// tree and its blocks on the device (tree order).
struct PlanPart {
    const void *op_key;
    const OperFlat *flat;
    const ApplyPlan *plan;
    const Tree *tree;
    const double *inp;
};

// A plan resident in device memory: band tables, input slots and output
// blocks of one or more applies, run together in each launch.
struct DevicePlan;
// Uploads the host plans and makes the rest on the device: the bands and input
// slots (dev_band_find), the input pool (dev_pool_fill), the norm and
// pre-screen tables, the exact counts and the work segments (the fine
// single-component ones only for a mode with an FP64 class beside a
// low-precision one).  mode: the arithmetic the plan will run.
// With once (a plan that is run once) the host does not wait for the counts:
// the run reads the number of segments on the device.
// plan_ms (optional): the host's time for bands and slots, for the pool, and
// for counts and segments is added to plan_ms[0..2] (device work that the host
// does not wait for is in the run's time).
// first_cells: cells of the slot search's first table, a power of two (0: twice
// what the bands can hold); a table that is too small is doubled.
int dev_plan_create(DeviceCtx *c, const MRA &mra, const std::vector<PlanPart> &parts, int mode, bool once,
                    DevicePlan **out, std::string &err, double *plan_ms = nullptr, long long first_cells = 0);
// Term-applications counted with the screening rule when the plan was made,
// and its pair segments.
void dev_plan_counts(const DevicePlan *p, unsigned long long *term_apps, int *segments);
// Input slots of the plan, and how many of them are generated nodes.
void dev_plan_slots(const DevicePlan *p, long long *slots, long long *generated);
// Run the per-node calculator over the resident plan.  kernel_ms receives the
// device time of the launches, term_apps the number of term-applications that
// passed screening.
// mode 0: every term in FP64.  mode 1: terms with bound > tau * thr in FP64,
// the rest on FP32 MFMA, their sum added to the FP64 output.  lp_apps
// receives the number of FP32 term-applications.
// split_ms (optional, 2 values): device time of the FP64-class launch and of
// the low-precision launch (they run concurrently, on two streams).
// With post (after dev_plan_set_post) the post transforms and the node
// norms run in place on the output blocks after the calculator, inside the
// timed region; post_ms receives their device time.
// With graph the step (zeroing, class launches, post) replays a hipGraph
// captured on the plan for (mode, tau, post) after one eager run; a replay
// reports the whole device time only (split_ms and post_ms stay 0).
// norms2 (optional, 2 n_out values): the squared norms of the scaling part,
// then of the wavelet parts, of every raw output block.
int dev_plan_run(DevicePlan *p, int mode, double tau, double *kernel_ms, unsigned long long *term_apps,
                 unsigned long long *lp_apps, std::string &err, double *split_ms = nullptr, bool post = false,
                 double *post_ms = nullptr, bool graph = false, double *norms2 = nullptr);
// Post transforms of the plan's output grid: levels[d] holds the (branch
// node, first child) pairs at depth d as indices into the plan's output
// nodes.  Uploads the pairs with their device addresses and the filter.
int dev_plan_set_post(DevicePlan *p, const MRA &mra, const std::vector<std::vector<std::pair<long long, long long>>> &levels,
                      std::string &err);
// Tunable knobs of a plan: the split class's single-rounding cut (items with
// bound <= single_ratio x thr_cls round their intermediates once) and the
// work-queue order (0: segment order, 1: largest passing-term count first).
int dev_plan_set_knobs(DevicePlan *p, double single_ratio, int order, std::string &err);
void dev_plan_knobs(const DevicePlan *p, double *single_ratio, int *order);
// A device copy of the plan's output blocks (freed with dev_free), and the
// largest |output - ref| and |ref| over all output values.
int dev_plan_snapshot(DevicePlan *p, double **copy, std::string &err);
int dev_plan_max_diff(DevicePlan *p, const double *ref, double *max_diff, double *max_ref, std::string &err);
// Squared norms (scaling, wavelet) of every output node after a run with post.
int dev_plan_download_norms(DevicePlan *p, double *s2, double *w2, std::string &err);
// Copy the raw non-standard blocks of every part, in part order
// (sum of n_out x 8(k+1)^3), to the host.
int dev_plan_download(DevicePlan *p, double *out_ns, std::string &err);
// The plan's output blocks (all applies' output nodes, 8(k+1)^3 each),
// detached from the plan: the caller frees them with dev_free.
double *dev_plan_take_output(DevicePlan *p);
// A device copy of the plan's output blocks (freed with dev_free).
int dev_plan_clone_output(DevicePlan *p, double **out, std::string &err);
// Output blocks [first, first + count) of the plan's concatenated output nodes.
int dev_plan_download_range(DevicePlan *p, long long first, long long count, double *dst, std::string &err);
void dev_plan_destroy(DevicePlan *p);

// Device construction of operator tables (mw_opbuild.hip).  Each job holds an
// operator prepared by prepare_operator (terms, no tables); the build fills
// its L and norms on the host, its flat table header (f.blocks stays empty,
// f.device_blocks counts the device values) and registers the device tables
// in the context under `key`.
struct OpBuildJob {
    Operator *op;
    OperFlat *flat;
    const void *key;
};
// Largest error |fit - K| r of every candidate fit on its grid of kFitPoints
// points (kernel_fit_error on the device).
struct FitCand {
    const std::vector<GaussTerm> *terms;
    double mu, r_min, r_max;
};
int dev_fit_errors(DeviceCtx *c, const std::vector<FitCand> &cands, std::vector<double> &errs, std::string &err);
int dev_build_operators(DeviceCtx *c, const MRA &mra, const std::vector<OpBuildJob> &jobs, std::string &err);
// Copy the device table of a device-built operator (f.device_blocks values).
int dev_download_operator_blocks(DeviceCtx *c, const void *key, double *out, long long n, std::string &err);

// An output node of a product or sum: depth and world_translation.
struct NodeAt {
    int d, l[3];
};

// Node-wise products for the multiplication (mw_multiply.hip).  For one
// output node: each input's source node (its deepest node on the path, block
// offset in the input's coefficient pool), the levels from it down to the
// output node and the child index of each level (3 bits per level, the first
// level below the source in the lowest bits), and h^{-3/2} of the output
// node's children.
struct MulNode {
    long long src_a, src_b;
    int dep_a, dep_b;
    unsigned path_a, path_b;
    double hfac;
};
struct DevMulSession;
// noalloc: every device buffer of the session is carved from the device's
// scratch array (dev_noalloc_init); no device memory is allocated, and
// inputs that do not fit are an argument error.
// a_on_device / b_on_device: that pool is device memory, used in place (or,
// with noalloc, copied into the scratch array); otherwise it is host memory
// and uploaded.
int dev_mul_begin(DeviceCtx *c, const MRA &mra, const Tree &a, const double *pool_a, size_t n_a, const Tree &b,
                  const double *pool_b, size_t n_b, DevMulSession **out, std::string &err, bool noalloc = false,
                  bool a_on_device = false, bool b_on_device = false);
// The product at every node of nodes, the inputs' sources found on the device
// (every node at most 10 levels below them: a 32-bit path; neither input
// empty).  out_blocks: nodes.size() x 8(k+1)^3, on the host, or on the device
// with out_on_device (then launches only: nodes must live until the stream has
// run them, as for dev_add_nodes).
int dev_mul_at(DevMulSession *m, const std::vector<NodeAt> &nodes, double coef, double *out_blocks, std::string &err,
               bool out_on_device = false);
// The same of an allocation-free session, from the host's descriptors into host
// memory.
int dev_mul_nodes(DevMulSession *m, const std::vector<MulNode> &nodes, double coef, double *out_blocks,
                  std::string &err);
void dev_mul_end(DevMulSession *m);

// A device copy of n doubles (freed with dev_free).
int dev_upload(DeviceCtx *c, const double *src, size_t n, double **dst, std::string &err);
// n doubles of device memory (freed with dev_free).
int dev_alloc(DeviceCtx *c, size_t n, double **dst, std::string &err);
// Block src_idx[i] of src to block i of dst, on the device.
int dev_gather_blocks(DeviceCtx *c, const double *src, const std::vector<int> &src_idx, int blk, double *dst,
                      std::string &err);
// p[0, n) *= f on the device, finished on return.
int dev_scale(DeviceCtx *c, double *p, size_t n, double f, std::string &err);
// n doubles from host memory into device memory at dst, finished on return.
int dev_upload_into(DeviceCtx *c, const double *src, size_t n, double *dst, std::string &err);

// Node blocks resident on the device (mw_multiply.hip).  Per node of
// blocks[0, n): its scaling part's and wavelet parts' squared norms.
int dev_node_norms(DeviceCtx *c, int kp1, const double *blocks, long long n, double *host_s2, double *host_w2,
                   std::string &err);
// Per node of blocks[0, n): the norms of its 8 components (8 per node).
int dev_component_norms(DeviceCtx *c, int kp1, const double *blocks, long long n, double *host8, std::string &err);
// A branch node's block and its 8 children's blocks (consecutive).
struct PostPair {
    double *node, *child0;
};
// Post transforms of an NS output tree whose blocks are on the device, the
// branch nodes grouped by depth (levels[d]): TopDown (each branch's
// reconstruction added into its children's scaling parts, shallow to deep),
// then BottomUp (each branch's block recomputed from its children's scaling
// parts, deep to shallow).
// Without topdown only the BottomUp steps run (a compressed tree from its
// leaves' scaling parts).
int dev_post_transform(DeviceCtx *c, const MRA &mra, const std::vector<std::vector<PostPair>> &levels,
                       std::string &err, bool topdown = true);
// The last step of a tree built level by level on the device, with one upload
// and one wait: the blocks of `before` copied, the post transforms over
// `levels` (none: empty), then the blocks of `after` copied (src == dst: left
// in place) and normed: norms2 receives after.size() squared norms of the
// scaling parts, then of the wavelet parts.
struct BlockMove {
    const double *src;
    double *dst;
};
int dev_finish_blocks(DeviceCtx *c, const MRA &mra, const std::vector<BlockMove> &before,
                      const std::vector<std::vector<PostPair>> &levels, bool topdown,
                      const std::vector<BlockMove> &after, double *norms2, std::string &err);
// Blocks on the device (8 (k+1)^3 values each), wherever they lie, one after
// another into host memory: n of them to dst, for each of `to` in turn.  They
// pass through `room`, kDownloadRoom bytes of device memory at most, which
// holds `per` blocks; the first `per` are there already.
constexpr size_t kDownloadRoom = (size_t)256 << 20;
struct HostBlocks {
    double *dst;
    size_t n;
};
int dev_download_blocks(DeviceCtx *c, const MRA &mra, const std::vector<const double *> &src, double *room, size_t per,
                        const std::vector<HostBlocks> &to, std::string &err);
// A packed tree: head (host) and n doubles of blocks (device) into device
// memory at dst, finished on return.
int dev_pack(DeviceCtx *c, void *dst, const void *head, size_t head_bytes, const double *blocks, size_t n,
             std::string &err);
// The same TopDown/BottomUp sequence over pairs already on the device:
// level d's pairs are pairs[lvl_off[d], lvl_off[d + 1]); F is the two-scale
// filter on the device.  Launches only, on `stream`.
int dev_post_launch(void *stream, int kp1, const PostPair *pairs, const std::vector<long long> &lvl_off,
                    const double *F, std::string &err, bool topdown = true);
// Squared norms of the scaling and wavelet parts of blocks[0, n) into the
// device arrays s2, w2 (a launch on `stream`).
int dev_node_norms_launch(void *stream, int kp1, const double *blocks, long long n, double *s2, double *w2,
                          std::string &err);
int dev_download(DeviceCtx *c, const double *src, size_t n, double *dst, std::string &err);
// Device-to-host copy on the context's stream, finished on return; large
// copies go through pinned staging buffers (mw_device.hip).
int dev_copy_d2h(DeviceCtx *c, void *dst, const void *src, size_t bytes, std::string &err);
// Host-to-device copy on the context's stream, finished on return; large
// copies go through the same pinned staging buffers.
int dev_copy_h2d(DeviceCtx *c, void *dst, const void *src, size_t bytes, std::string &err);
void dev_free(DeviceCtx *c, void *p);
// Device memory from the context's pool (mw_device.hip): a block put back is
// handed out again without a call to the driver.  Blocks are used by work on
// the context's stream (or joined to it), so a block may be put back while
// such work still runs: what its next holder enqueues comes after.
int dev_mem_get(DeviceCtx *c, size_t bytes, void **p, std::string &err);
void dev_mem_put(DeviceCtx *c, void *p);
template <typename T>
int dev_mem(DeviceCtx *c, size_t n, T **p, std::string &err) {
    void *v = nullptr;
    const int rc = dev_mem_get(c, sizeof(T) * (n ? n : 1), &v, err);
    *p = static_cast<T *>(v);
    return rc;
}
// Memory that callers outside the library hold (and may use on streams of
// their own): straight from and back to the driver.
int dev_raw_alloc(DeviceCtx *c, size_t bytes, void **p, std::string &err);
void dev_raw_free(DeviceCtx *c, void *p);

// Node-wise sums (mw_multiply.hip): for one output node and one input, the
// input's source node (its deepest node on the path: its block on the device,
// or null when the input has no node on the path), the levels from it down to
// the output node and the child index of each level (3 bits per level, the
// first level below the source lowest).
struct AddSrc {
    const double *p;
    int dep, pad_;
    unsigned long long path;
};
// (a 64-bit path holds 21 levels, one more than the deepest tree has)
struct DevAddSession;
// One input's blocks: n doubles at p, in host or device memory.
struct BlockSource {
    const double *p;
    size_t n;
    bool on_device;
};
// Uploads the host inputs (a device input is read in place) and the structure
// of the input trees.
int dev_add_begin(DeviceCtx *c, const MRA &mra, const std::vector<BlockSource> &inputs,
                  const std::vector<const Tree *> &trees, const std::vector<double> &coefs, DevAddSession **out,
                  std::string &err);
// The sum at every node of nodes, each input's source found on the device.
// out_blocks: nodes.size() x 8(k+1)^3, on the host, or on the device with
// out_on_device (then launches only: nodes must live until the stream has run
// them).
int dev_add_nodes(DevAddSession *m, const std::vector<NodeAt> &nodes, double *out_blocks, std::string &err,
                  bool out_on_device = false);
void dev_add_end(DevAddSession *m);

// The device's scratch array of the allocation-free entry points
// (mw_multiply.hip): its device address, taken once per context with the
// context's device current, and stored in the context.
int dev_noalloc_init(DeviceCtx *c, std::string &err);
void dev_set_noalloc(DeviceCtx *c, void *base, size_t bytes);
void *dev_noalloc_base(DeviceCtx *c);
size_t dev_noalloc_bytes(DeviceCtx *c);

// The root level as dense products (mw_root.hip): output blocks of every root
// box of `apps` from all their terms, added into out_ns.
struct RootGeo {
    int n, boxes[3];  // k + 1, root boxes per direction
};
// One apply: its operator's tables and the start of its boxes (x fastest) in
// the launch's slot_off (pool offsets of their blocks) and root_out (output
// nodes).
struct RootApp {
    const int *L;
    const long long *boff;
    const double *blocks;
    int ndepth, root0;
};
struct RootItem {
    int app, m;  // root apply, term
};
struct RootLaunch {
    RootGeo geo{};
    const RootApp *apps = nullptr;
    const RootItem *items = nullptr;  // of one apply after another
    int n_items = 0;
    const long long *slot_off = nullptr;
    const int *root_out = nullptr;
    const double *pool = nullptr;
    double *A = nullptr, *Y = nullptr;  // work areas (root_work_values)
    double *out_ns = nullptr;
    // counter += the root terms of every apply, totals[2 i + 1], i < n_totals
    unsigned long long *counter = nullptr;
    const unsigned long long *totals = nullptr;
    int n_totals = 0;
};
void root_work_values(int n, const int *boxes, long long n_items, size_t *a_values, size_t *y_values);
// Launches only, on `stream`.
int dev_root_launch(void *stream, const RootLaunch &r, std::string &err);

// Helpers shared by the HIP sources.
struct DevOperTables {
    int *L = nullptr;
    long long *boff = nullptr, *noff = nullptr;
    double *blocks = nullptr, *norms = nullptr;
};
int dev_device(DeviceCtx *c);
void *dev_stream(DeviceCtx *c);
// Allocate the device tables of f (blocks and norms cleared, L/boff/noff uploaded).
int dev_alloc_oper_tables(DeviceCtx *c, const OperFlat &f, DevOperTables &t, std::string &err);
// Make t the context's resident copy of operator `key` (ownership passes to
// the context).
int dev_register_operator(DeviceCtx *c, const void *key, const OperFlat &f, const DevOperTables &t, std::string &err);

}  // namespace mwg
