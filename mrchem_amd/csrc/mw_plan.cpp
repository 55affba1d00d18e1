// Apply plan: output nodes, active terms and screening-derived bandwidths.  The
// bands themselves, the input slots and their pool, the slot norms, the exact
// counts and the work segments are made on the device (mw_band.hip,
// mw_multiply.hip, mw_count.hip).
//
// The band half-width is derived from the screening rule itself, so it never
// changes which terms pass: along one direction, a translation l can pass
//     N_x(l) N_y N_z ||f_ft|| > thr
// only if N(l) * Nmax^2 * Fmax > thr_min, where Nmax bounds every block norm
// of the term at that depth and Fmax bounds every input component norm there.
#include "mw_internal.hpp"

#include <algorithm>
#include <cmath>
#include <stdexcept>

namespace mwg {

double oper_norm(const Operator &op, int m, int d, int c, long long l) {
    const OperDepth &od = op.terms[m].depth[d];
    if (od.L < 0 || l < -od.L || l > od.L) return 0.0;
    return od.norms[(size_t)c * (2 * od.L + 1) + (size_t)(l + od.L)];
}

void build_plan(ApplyPlan &plan, const Operator &op, const Tree &inp, const Tree &out,
                const std::vector<int> &nodes, const std::vector<double> &thr, int max_band_w,
                const double *in_cnorm8) {
    const MRA &mra = *out.mra;
    const int M = op.size(), ndepth = op.max_depth + 1;
    if (inp.mra != out.mra || op.mra != out.mra) throw std::invalid_argument("apply: trees and operator must share one MRA");
    if (thr.size() != nodes.size()) throw std::invalid_argument("apply: one threshold per output node");
    plan = ApplyPlan();
    plan.kp1 = mra.kp1();
    plan.ndepth = ndepth;
    plan.M = M;

    int maxd = 0;
    for (int g : nodes) maxd = std::max(maxd, out.keys[g].depth);
    if (maxd >= ndepth) throw std::runtime_error("apply: output deeper than the operator tables");

    std::vector<double> thr_min(maxd + 1, 1e300), fmax(maxd + 1, 0.0);
    std::vector<char> has_depth(maxd + 1, 0);
    for (size_t q = 0; q < nodes.size(); q++) {
        int d = out.keys[nodes[q]].depth;
        thr_min[d] = std::min(thr_min[d], thr[q]);
        has_depth[d] = 1;
    }
    for (int i = 0; i < inp.size(); i++) {
        int d = inp.keys[i].depth;
        const double *nrm = in_cnorm8 + (size_t)i * 8;
        double tot = 0.0;
        for (int t = 0; t < 8; t++) {
            tot += nrm[t] * nrm[t];
            if (d <= maxd) fmax[d] = std::max(fmax[d], nrm[t]);
        }
        if (inp.child0[i] < 0)
            for (int dd = d + 1; dd <= maxd; dd++) fmax[dd] = std::max(fmax[dd], std::sqrt(tot));
    }

    plan.bw.assign((size_t)(maxd + 1) * M * 4, -1);
    plan.active_off.assign(maxd + 2, 0);
    std::vector<int> W(maxd + 1, 0);
    for (int d = 0; d <= maxd; d++) {
        plan.active_off[d] = (int)plan.active_terms.size();
        if (!has_depth[d]) continue;
        for (int m = 0; m < M; m++) {
            const OperDepth &od = op.terms[m].depth[d];
            if (od.L < 0) continue;
            // nmax bounds every block of the term at this depth, wmax every
            // wavelet-component block.  Off the root each candidate pairs at
            // least one wavelet component with the others, so an s<-s block
            // contributes at most N * nmax * wmax * Fmax.
            double nmax = 0.0, wmax = 0.0;
            for (int c = 0; c < 4; c++)
                for (long long l = -od.L; l <= od.L; l++) {
                    double nb = oper_norm(op, m, d, c, l);
                    nmax = std::max(nmax, nb);
                    if (c > 0) wmax = std::max(wmax, nb);
                }
            bool any = false;
            for (int c = 0; c < 4; c++) {
                double other = (d > 0 && c == 0) ? nmax * wmax : nmax * nmax;
                int w = -1;
                for (long long l = -od.L; l <= od.L; l++) {
                    double nb = oper_norm(op, m, d, c, l);
                    if (nb * other * fmax[d] * (1.0 + 1e-12) > thr_min[d]) w = std::max(w, (int)std::llabs(l));
                }
                plan.bw[((size_t)d * M + m) * 4 + c] = w;
                if (w >= 0) {
                    any = true;
                    W[d] = std::max(W[d], w);
                }
            }
            if (any) plan.active_terms.push_back(m);
        }
        if (W[d] > max_band_w)
            throw std::runtime_error("apply: band half-width " + std::to_string(W[d]) + " exceeds limit " +
                                     std::to_string(max_band_w));
    }
    plan.active_off[maxd + 1] = (int)plan.active_terms.size();

    // Output nodes and the sizes of their bands.
    plan.out_depth.resize(nodes.size());
    plan.out_l.resize(3 * nodes.size());
    plan.out_thr = thr;
    plan.band_off.resize(nodes.size());
    plan.band_w.resize(nodes.size());
    for (size_t q = 0; q < nodes.size(); q++) {
        const NodeKey &k = out.keys[nodes[q]];
        const int side = 2 * W[k.depth] + 1;
        plan.out_depth[q] = k.depth;
        world_translation(mra, k, &plan.out_l[3 * q]);
        plan.band_w[q] = W[k.depth];
        plan.band_off[q] = plan.n_band;
        plan.n_band += (long long)side * side * side;
    }

    // Root boxes for the dense root kernels (48: three 16-wide tiles a
    // direction, the widest they hold in registers).
    for (int d = 0; d < 3; d++) plan.boxes[d] = mra.boxes[d];
    const int n_roots = mra.boxes[0] * mra.boxes[1] * mra.boxes[2];
    if (inp.size() < n_roots) throw std::runtime_error("apply: input tree has no root covering a band node");
    if (2 * mra.kp1() * std::max(mra.boxes[0], std::max(mra.boxes[1], mra.boxes[2])) <= 48) {
        plan.root_q.assign(n_roots, -1);
        int found = 0;
        for (size_t q = 0; q < nodes.size(); q++) {
            const NodeKey &k = out.keys[nodes[q]];
            if (k.depth != 0 || thr[q] != 0.0) continue;
            long long b[3];
            for (int d = 0; d < 3; d++) b[d] = k.l[d] - mra.corner[d];
            const int r = (int)((b[2] * mra.boxes[1] + b[1]) * mra.boxes[0] + b[0]);
            if (plan.root_q[r] >= 0) continue;
            plan.root_q[r] = (int)q;
            found++;
        }
        if (found < n_roots) plan.root_q.clear();
    }

    plan.thr_floor = 0.0;
    for (double t : plan.out_thr)
        if (t > 0.0 && (plan.thr_floor == 0.0 || t < plan.thr_floor)) plan.thr_floor = t;
}

}  // namespace mwg
