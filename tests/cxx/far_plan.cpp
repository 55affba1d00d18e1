// Plans of one grid in two worlds, one far from the origin: what the device
// is given of the output nodes must not depend on where the world lies.  Host
// code alone (compiled with the library's host sources by
// tests/test_far_world.py).
#include <cstdio>

#include "mw_internal.hpp"

using namespace mwg;

static MRA world(int cx) {
    MRA m;
    m.basis = make_basis(1, BASIS_INTERPOLATING);
    m.n0 = -2;
    m.max_depth = 16;
    m.corner[0] = cx;
    m.corner[1] = m.corner[2] = 0;
    return m;
}

// The roots and one chain of splits down to depth 16, towards a corner that
// changes from level to level.
static void grow(Tree &t) {
    t.make_roots();
    int node = 1;
    for (int d = 0; d < 16; d++) node = t.split(node) + (5 * d + 3) % 8;
    for (size_t e = 0; e < t.coefs.size(); e++) t.coefs[e] = 1.0 / (1.0 + (double)(e % 97));
}

int main() {
    ApplyPlan plan[2];
    // the far world's translations at depth 16 pass 2^33
    const int cx[2] = {0, 200000};
    for (int w = 0; w < 2; w++) {
        const MRA m = world(cx[w]);
        Operator op;
        build_operator(op, m, 0.0, 1e-2, m.max_depth);
        Tree t;
        t.mra = &m;
        grow(t);
        std::vector<double> cn8(8 * (size_t)t.size()), thr(t.size(), 1e-6);
        std::vector<int> nodes(t.size());
        for (int i = 0; i < t.size(); i++) {
            nodes[i] = i;
            component_norms(m, t.node(i), cn8.data() + 8 * (size_t)i);
        }
        build_plan(plan[w], op, t, t, nodes, thr, 64, cn8.data());
    }
    int bad = 0;
    for (size_t i = 0; i < plan[0].out_l.size(); i++) bad += plan[0].out_l[i] != plan[1].out_l[i];
    std::printf("%zu nodes, %d of %zu translations differ\n", plan[0].out_depth.size(), bad, plan[0].out_l.size());
    return bad || plan[0].out_depth != plan[1].out_depth || plan[0].band_w != plan[1].band_w;
}
