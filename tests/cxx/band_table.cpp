// A frozen FP64 plan whose slot search starts with a table of first_cells cells
// (0: the size the bands ask for): its slots, generated slots, terms and raw
// output blocks, for tests/test_gpu_band_table.py.
#include <string>
#include <vector>

#include "mw_device.hpp"

using namespace mwg;

// blocks: room for *nodes blocks of 512 values.  Returns 0, or a step's number.
extern "C" int band_table(long long first_cells, long long *slots, long long *generated, unsigned long long *terms,
                          double *blocks, int *nodes) {
    MRA mra;
    mra.basis = make_basis(3, BASIS_INTERPOLATING);
    mra.n0 = -4;
    mra.sfac = 1.25;
    mra.max_depth = 8;
    Operator op;
    build_operator(op, mra, 0.0, 1e-3, mra.max_depth);
    OperFlat flat;
    flatten_operator(op, flat);
    // a shallow input under a deep grid: chains of generated nodes
    Tree inp, out;
    inp.mra = out.mra = &mra;
    GaussSum wide{{1.0}, {0.3}, {1.0, 2.0, 1.0}}, sharp{{1.0}, {60.0}, {0.3, -0.2, 0.1}};
    project_adaptive(inp, wide, 1e-1, false, 1);
    project_adaptive(out, sharp, 1e-3, false, mra.max_depth);
    std::vector<int> all(out.size());
    std::vector<double> thr(out.size()), cn8(8 * (size_t)inp.size());
    for (int i = 0; i < out.size(); i++) {
        all[i] = i;
        thr[i] = out.keys[i].depth == 0 ? 0.0 : 1e-7;
    }
    for (int i = 0; i < inp.size(); i++) component_norms(mra, inp.node(i), cn8.data() + 8 * (size_t)i);
    ApplyPlan plan;
    build_plan(plan, op, inp, out, all, thr, 64, cn8.data());
    if (out.size() > *nodes) return 1;
    *nodes = out.size();
    std::string err;
    DeviceCtx *ctx = nullptr;
    if (dev_create(0, &ctx, err)) return 2;
    double *blk = nullptr;
    DevicePlan *dp = nullptr;
    int rc = 0;
    if (dev_upload(ctx, inp.coefs.data(), inp.coefs.size(), &blk, err)) rc = 3;
    if (!rc && dev_plan_create(ctx, mra, {PlanPart{&op, &flat, &plan, &inp, blk}}, 0, false, &dp, err, nullptr, first_cells))
        rc = 4;
    if (!rc) dev_plan_slots(dp, slots, generated);
    if (!rc && dev_plan_run(dp, 0, 1.0, nullptr, terms, nullptr, err)) rc = 5;
    if (!rc && dev_plan_download(dp, blocks, err)) rc = 6;
    dev_plan_destroy(dp);
    dev_free(ctx, blk);
    dev_destroy(ctx);
    return rc;
}
