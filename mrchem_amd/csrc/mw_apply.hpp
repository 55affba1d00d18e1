// Kernel arguments of an apply plan, shared by the per-node calculators
// (mw_device.hip) and the kernels that count and cut a plan's work
// (mw_count.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "mw_device.hpp"

namespace mwg {

// Per apply of a batched plan: its operator tables (device copies resident in
// the context) and where its screening tables start.
struct AppDesc {
    const int *opL;                   // [m * ndepth + d]
    const long long *op_boff, *op_noff;
    const double *op_norms;
    const double *blk64;              // FP64 blocks
    const float *blk32;               // FP32 copy (mixed mode), or null
    const _Float16 *blk_h;            // FP16 split rows (split mode), or null
    const double *blk_hsc;            // their per-block scales
    int M, ndepth;
    long long bw_off;                 // start of this apply in bw
    int act_base;                     // start of this apply in act_off
    int mt_d0;                        // first output depth of mtab
    double thr_floor;                 // positive floor of the class threshold
    // pre-screen: per output depth d >= mt_d0, component combination
    // cmb = cx | cy << 2 | cz << 4 and translation |l| <= mt_w, the largest
    // ((N_x N_y) N_z) over the depth's active terms, [d - mt_d0][cmb][lz][ly][lx]
    const double *mtab;
    int mt_w, pad_;
};

struct KArgs {
    // output nodes (all applies, concatenated)
    const int *out_depth;
    const int *out_app;               // apply of each output node
    const double *out_thr;
    const long long *band_off;
    const int *band_w;
    const int *band;
    double *out_ns;
    // input slots (all applies, concatenated)
    const long long *slot_off;
    const double *slot_norm;
    int n_real, pad_;                 // slots [0, n_real) hold full blocks
    // screening tables: active terms per depth, and their norms (k_term_norms)
    // [c][l + w][active term] of the depth's band half-width w, from
    // tn + tn_off[act_base + d]
    const int *bw;
    const int *act_off, *act_terms;
    const double *tn;
    const long long *tn_off;
    // per active term (as act_terms): block id of component 0 at translation
    // 0, and the distance of two components' blocks
    const int2 *tb;
    const AppDesc *apps;
    // [0] term-applications passing screening (algorithmic work)
    unsigned long long *counters;
    // work segments: job = 8*out + gt, [p0, p1) with ends (8 p + ft) << 12 | e:
    // from active term e of the pair of band position p and input component ft
    // (e = 0 but in plain FP64)
    const int *seg_job, *seg_p0, *seg_p1;
};

// A generated node of an apply plan's pool (mw_multiply.hip): scaling block dst
// of child `child` of the node at src, a full block or a scaling block.
struct GenItem {
    const double *src;
    double *dst;
    int child, full;
};

// One slot of the pool: len doubles from src (an input node's full block, or a
// generated node's scaling block) to dst, and the slot's 8 component norms to
// norms (wavelet norms 0 for a generated slot).
struct SlotItem {
    const double *src;
    double *dst, *norms;
    int len;
};

// The pool from its items on the device: generated nodes level by level (of
// level lv: gen[lv_off[lv], lv_off[lv + 1]), their parents in the input tree or
// of level lv - 1), then every slot.  F: the basis' filter on the device.
// Launches only, on stream.
int dev_pool_fill(hipStream_t s, int n, const double *F, const GenItem *gen, const std::vector<int> &lv_off,
                  const SlotItem *slots, int n_slot, std::string &err);

// ---- Bands and slots of a plan (mw_band.hip) ----

// The input tree of an apply: first child of every node (-1: none; the roots
// are the first nodes, box x fastest) and the nodes' blocks.
struct BandTree {
    const int *child0;
    const double *inp;
};
// Counters of the search: [0] real slots, [1] generated slots, [2] not 0: the
// table was too small, [3 + lv] generated nodes lv generated levels below a
// node of the input tree.
constexpr int kBandLevels = 32, kBandCounts = 3 + kBandLevels;
struct BandArgs {
    const int *out_l, *out_depth, *out_app;  // out_l: 3 per output node, from the world's corner
    const long long *band_off;
    const int *band_w;
    const BandTree *trees;  // per apply
    int boxes[3];
    int n_out, q0;  // q0: output node of the launch's first workgroups
    long long n_band;
    // table of cap cells (a power of two): name of the node, slot, generation
    // level (-1: in the input tree) and, of a node in the tree, {its index, 0},
    // of a generated one {parent's cell or -(tree node + 1), position in its
    // level}
    unsigned cap;
    unsigned long long *rep;
    int *slot;
    int2 *gen;
    signed char *lv;
    int *cell;      // per band entry: its cell, or -1
    unsigned *cnt;  // kBandCounts
};
// What the search found, as items: real slots are slots [0, n_real).
struct BandItems {
    int n3, n_real, n_roots;
    int lv_off[kBandLevels];
    double *gen_s, *pool, *norms;
    GenItem *gen;
    SlotItem *slots;
    long long *slot_off;
    int *band;
    const int *root_out;  // output nodes of the dense root kernels
    long long *root_off;  // pool offsets of their own slots
};
// Launches only, on stream.  widest: entries of the widest band.
int dev_band_find(hipStream_t s, const BandArgs &a, long long widest, std::string &err);
int dev_band_items(hipStream_t s, const BandArgs &a, const BandItems &o, std::string &err);

// One depth of one apply in the norm and pre-screen tables.
struct TermLevel {
    int app, d, w;       // apply, output depth, band half-width there
    int na, a0;          // its active terms: act_terms[a0, a0 + na)
    int pad_;
    long long tn;        // start of its norms in tn
};

// What the class lists of the mixed and split modes need of a segment: passing
// terms and the smallest and largest passing bound.
struct SegRec {
    int job, p0, apps, pad_;
    double lo, hi;
};

// Work counts and segments of a plan (mw_count.hip).
struct CountArgs {
    KArgs k{};
    int n_out = 0, n_share = 1;
    int q0 = 0;                            // output node of the launch's first workgroups
    long long widest = 1;                  // positions of the widest band
    const unsigned char *dense = nullptr;  // per output node: computed by the root kernels
    // passing terms per (output component, band position) of every node,
    // node q's at 8 band_off[q] + gt nb + p; with bounds the smallest and
    // largest passing bound there
    int *cnt = nullptr;
    double *bmin = nullptr, *bmax = nullptr;
    // per apply: passing terms, and those of dense nodes
    unsigned long long *totals = nullptr;
    // segments found: [0] pair ones, [1] fine ones (also past the capacity)
    unsigned long long *n_seg = nullptr;
    int cap[2] = {0, 0};
    // pair segments at [0, cap[0]), fine ones at [cap[0], cap[0] + cap[1])
    int *seg_job = nullptr, *seg_p0 = nullptr, *seg_p1 = nullptr;
    SegRec *rec = nullptr;  // with bounds
};
// Norm, block and pre-screen tables of levels[0, n) (device array), nn the
// values of an operator block; mtab of each apply is written through
// apps[app].mtab.  Launches only, on stream.
int dev_term_tables(hipStream_t s, const KArgs &k, int nn, const TermLevel *levels, int n, double *tn, int2 *tb,
                    std::string &err);
// Counts per position (bounds: the class bounds too), then the segments.
// Launches only, on stream.
int dev_count_terms(hipStream_t s, const CountArgs &c, bool bounds, std::string &err);
int dev_cut_segments(hipStream_t s, const CountArgs &c, bool bounds, std::string &err);
// The class lists of a cut with bounds (n: their two lengths, cleared before).
// Launches only, on stream.
int dev_class_lists(hipStream_t s, const CountArgs &c, double tau, int *lo, int *hi, unsigned long long *n,
                    std::string &err);

}  // namespace mwg
