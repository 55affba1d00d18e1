// Work counts and segments of an apply plan on the device (gfx950).
//
// A plan's jobs (output node, component or component pair) are cut into
// segments of about as many passing term-applications, counted exactly with
// the calculator's screening rule ((N_x N_y) N_z) ||f_ft|| > thr (the rule of
// upstream MRCPP's OperApplicationCalculator, reached from
// src/qmoperators/two_electron/CoulombPotential.cpp:131).  On the host, with
// 8 threads and sorted products per translation, this took 3-20 ms of an
// adaptive apply (a third to a half of the call at k = 7); here a level's
// tables, counts and cut are four launches of a few microseconds each, and
// the slot norms they read never leave the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "mw_apply.hpp"

namespace mwg {

#define HIP_TRY(expr)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess) {                                                            \
            err = std::string(#expr) + ": " + hipGetErrorString(e_);                       \
            return -2;                                                                     \
        }                                                                                  \
    } while (0)

namespace {

// 1D norms of one depth's active terms, [c][l + w][term] (term fastest, so
// that a wave with one term per lane reads whole lines): zero outside the
// term's bandwidth and stored width; and where its blocks lie.  One workgroup per (level, component).
__global__ __launch_bounds__(256) void k_term_norms(KArgs a, int nn, const TermLevel *levels, double *tn,
                                                    int2 *tb) {
    const TermLevel lv = levels[blockIdx.x];
    const int c = blockIdx.y, nl = 2 * lv.w + 1;
    if (lv.na == 0) return;
    const AppDesc &ad = a.apps[lv.app];
    double *dst = tn + lv.tn + (long long)c * nl * lv.na;
    if (c == 0)
        for (int ai = threadIdx.x; ai < lv.na; ai += 256) {
            const int m = a.act_terms[lv.a0 + ai], L = ad.opL[m * ad.ndepth + lv.d];
            tb[lv.a0 + ai] = int2{(int)(ad.op_boff[m * ad.ndepth + lv.d] / nn) + L, 2 * L + 1};
        }
    for (int e = threadIdx.x; e < nl * lv.na; e += 256) {
        const int li = e / lv.na, ai = e % lv.na, l = li - lv.w;
        const int m = a.act_terms[lv.a0 + ai];
        const int L = ad.opL[m * ad.ndepth + lv.d];
        const int bwc = a.bw[ad.bw_off + ((long long)lv.d * ad.M + m) * 4 + c];
        double v = 0.0;
        if (abs(l) <= bwc && abs(l) <= L)
            v = ad.op_norms[ad.op_noff[m * ad.ndepth + lv.d] + (long long)c * (2 * L + 1) + (l + L)];
        dst[e] = v;
    }
}

// Pre-screen table of one depth and component combination cmb = cx | cy << 2
// | cz << 4: per translation |l| <= mt_w the largest (N_x N_y) N_z of the
// active terms.  One wave per translation, one term per lane.
__global__ __launch_bounds__(256) void k_prescreen(KArgs a, const TermLevel *levels) {
    const TermLevel lv = levels[blockIdx.x];
    const AppDesc &ad = a.apps[lv.app];
    const int cmb = blockIdx.y, nl = 2 * lv.w + 1, W = ad.mt_w, S = 2 * W + 1, S3 = S * S * S;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const double *tn = a.tn + lv.tn;
    double *dst = const_cast<double *>(ad.mtab) + ((long long)(lv.d - ad.mt_d0) * 64 + cmb) * S3;
    for (int pos = wv; pos < S3; pos += 4) {
        const int lx = pos % S - W, ly = (pos / S) % S - W, lz = pos / (S * S) - W;
        double b = 0.0;
        if (abs(lx) <= lv.w && abs(ly) <= lv.w && abs(lz) <= lv.w) {
            const double *nx = tn + (long long)((cmb & 3) * nl + lx + lv.w) * lv.na;
            const double *ny = tn + (long long)(((cmb >> 2) & 3) * nl + ly + lv.w) * lv.na;
            const double *nz = tn + (long long)((cmb >> 4) * nl + lz + lv.w) * lv.na;
            for (int e = lane; e < lv.na; e += 64) b = fmax(b, (nx[e] * ny[e]) * nz[e]);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) b = fmax(b, __shfl_xor(b, o));
        if (lane == 0) dst[pos] = b;
    }
}

// An output node as the screening sees it.
struct NodeView {
    int q, d, w, side, nb, na, mt_w, mt_s;
    double thr;
    const int *band;
    const double *tn, *mt;
};
__device__ __forceinline__ NodeView node_view(const KArgs &a, int q) {
    NodeView v;
    const AppDesc &ad = a.apps[a.out_app[q]];
    v.q = q;
    v.d = a.out_depth[q];
    v.w = a.band_w[q];
    v.side = 2 * v.w + 1;
    v.nb = v.side * v.side * v.side;
    v.na = a.act_off[ad.act_base + v.d + 1] - a.act_off[ad.act_base + v.d];
    v.mt_w = ad.mt_w;
    v.mt_s = 2 * ad.mt_w + 1;
    v.thr = a.out_thr[q];
    v.band = a.band + a.band_off[q];
    v.tn = a.tn + a.tn_off[ad.act_base + v.d];
    v.mt = ad.mtab + (long long)(v.d - ad.mt_d0) * 64 * v.mt_s * v.mt_s * v.mt_s;
    return v;
}

// The norms of the three directions for output component gt and input
// component ft of band position p, one value per active term.
struct PairNorms {
    const double *nx, *ny, *nz;
};
__device__ __forceinline__ PairNorms pair_norms(const NodeView &v, int gt, int p, int ft) {
    const int lx = p % v.side, ly = (p / v.side) % v.side, lz = p / (v.side * v.side);
    const int cx = 2 * (gt & 1) + (ft & 1), cy = (gt & 2) + ((ft >> 1) & 1), cz = 2 * (gt >> 2) + (ft >> 2);
    return PairNorms{v.tn + (long long)(cx * v.side + lx) * v.na, v.tn + (long long)(cy * v.side + ly) * v.na,
                     v.tn + (long long)(cz * v.side + lz) * v.na};
}

// Passing terms of the pair (norm fn of ft), counted by the whole wave (one
// term per lane); the smallest and largest passing bound are folded into this
// lane's lo and hi.
__device__ __forceinline__ int pair_terms(const NodeView &v, int gt, int p, int ft, double fn, int lane, double &lo,
                                          double &hi) {
    const PairNorms n = pair_norms(v, gt, p, ft);
    int c = 0;
    for (int e0 = 0; e0 < v.na; e0 += 64) {
        const int e = e0 + lane;
        bool pass = false;
        if (e < v.na) {
            const double b = ((n.nx[e] * n.ny[e]) * n.nz[e]) * fn;
            pass = b > v.thr;
            if (pass) {
                lo = fmin(lo, b);
                hi = fmax(hi, b);
            }
        }
        c += __popcll(__ballot(pass));
    }
    return c;
}

// Whether output component gt may hold a passing term of input component ft
// (norm fn) of band position p: the depth's largest product against thr.
__device__ __forceinline__ bool pair_candidate(const NodeView &v, int gt, int p, int ft, double fn) {
    if (!(fn > 0.0) || (v.d > 0 && ft == 0 && gt == 0)) return false;
    const int lx = p % v.side - v.w, ly = (p / v.side) % v.side - v.w, lz = p / (v.side * v.side) - v.w;
    const long long li = ((long long)(lz + v.mt_w) * v.mt_s + (ly + v.mt_w)) * v.mt_s + (lx + v.mt_w);
    const int cmb = (2 * (gt & 1) + (ft & 1)) | (((gt & 2) + ((ft >> 1) & 1)) << 2) |
                    ((2 * (gt >> 2) + (ft >> 2)) << 4);
    return v.mt[(long long)cmb * v.mt_s * v.mt_s * v.mt_s + li] * fn > v.thr;
}

__device__ __forceinline__ void wave_range(double &lo, double &hi) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, o));
        hi = fmax(hi, __shfl_xor(hi, o));
    }
}

// Counts of one output node: one wave per output component.  Up to 64
// (position, ft) pairs at a time (step: a multiple of 8) are pre-screened against the depth's largest products
// (rounding is monotone, so a pair whose largest bound does not pass holds no
// passing term); the terms of each candidate are then counted by ballot, one
// after the other: a microsecond of load latency each, which a launch of few
// nodes shortens by sharing a node's steps among workgroups (grid y; with the
// parts of k_cut 2.11 -> 1.96 ms for a Coulomb apply at k = 7).
template <bool BOUNDS>
__global__ __launch_bounds__(512) void k_count(CountArgs c, int step) {
    const KArgs &a = c.k;
    const NodeView v = node_view(a, c.q0 + (int)blockIdx.x);
    const int gt = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long long base = 8 * a.band_off[v.q] + (long long)gt * v.nb;
    __shared__ unsigned long long part[8];
    unsigned long long total = 0;
    for (int pi = step * blockIdx.y; pi < 8 * v.nb; pi += step * gridDim.y) {
        const int p = (pi + lane) >> 3, ft = lane & 7;
        bool cand = false;
        double fn = 0.0;
        if (lane < step && p < v.nb) {
            const int s = v.band[p];
            if (s >= 0) {
                fn = a.slot_norm[(long long)s * 8 + ft];
                cand = pair_candidate(v, gt, p, ft, fn);
            }
        }
        int my = 0;  // lane i < 8: terms of position pi / 8 + i
        double mlo = HUGE_VAL, mhi = 0.0;
        unsigned long long cm = __ballot(cand);
        while (cm) {
            const int k = __builtin_ctzll(cm);
            cm &= cm - 1;
            double lo = HUGE_VAL, hi = 0.0;
            const int n = pair_terms(v, gt, (pi + k) >> 3, k & 7, __shfl(fn, k), lane, lo, hi);
            if (BOUNDS) wave_range(lo, hi);
            total += n;
            if (lane == (k >> 3)) {
                my += n;
                mlo = fmin(mlo, lo);
                mhi = fmax(mhi, hi);
            }
        }
        if (lane < step >> 3 && (pi >> 3) + lane < v.nb) {
            const long long e = base + (pi >> 3) + lane;
            c.cnt[e] = my;
            if (BOUNDS) {
                c.bmin[e] = mlo;
                c.bmax[e] = mhi;
            }
        }
    }
    if (lane == 0) part[gt] = total;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int i = 0; i < 8; i++) t += part[i];
        const int app = a.out_app[v.q];
        if (t) atomicAdd(&c.totals[2 * app], t);
        if (t && c.dense[v.q]) atomicAdd(&c.totals[2 * app + 1], t);
    }
}

// Segment cut of one output node: one wave per job, the pair (gt, gt | 4)
// (PAIR) or one component.  The positions are taken in order and a segment
// closes at the first that brings it to the target; segments without passing
// terms are left out.  A segment's ends are (8 p + ft) << 12 | term.  In the
// mixed and split modes (BOUNDS) a small launch also cuts a position that
// holds more than a segment at input-component boundaries.  Plain FP64 always
// does, and inside a component at every 16th term: a (position, component)
// pair of a coarse node holds all the depth's terms, and one wave working
// through a hundred of them alone was the end of every level's launch.  (The
// low-precision classes sum a segment in 32 bits and keep their segments.)
// Lane i keeps the i-th segment found; every 64 the wave, and at the end the
// workgroup, takes places for them with one addition (to one address they take
// about 10 ns each, the time of a launch of some thousand waves) and they are
// written side by side.  Grid y: parts
// of a node's positions, each cut by itself (never for the low-precision
// classes' segments).
constexpr int kSegTarget = 256;      // passing terms of a segment
constexpr int kSegFloor = 32;        // the least in a small launch
constexpr int kSegWanted = 2048;     // segments a small launch is cut into
// plain FP64, whose segments are single waves (2048 of them resident)
constexpr int kSegTarget64 = 64, kSegFloor64 = 16, kSegWanted64 = 8192;

template <bool PAIR, bool BOUNDS>
__global__ __launch_bounds__(PAIR ? 256 : 512) void k_cut(CountArgs c) {
    const KArgs &a = c.k;
    if (c.dense[c.q0 + (int)blockIdx.x]) return;
    const NodeView v = node_view(a, c.q0 + (int)blockIdx.x);
    const int gt = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int app = a.out_app[v.q], kind = PAIR ? 0 : 1;
    // A launch with fewer than kSegWanted x kSegTarget passing terms (this
    // apply's count times the applies that share it) is cut into about
    // kSegWanted segments, so that it still has work for every compute unit.
    const unsigned long long launch = (c.totals[2 * app] - c.totals[2 * app + 1]) * (unsigned long long)c.n_share;
    const unsigned long long most = BOUNDS ? kSegTarget : kSegTarget64, least = BOUNDS ? kSegFloor : kSegFloor64;
    const int whole = (int)min(most, max(least, launch / (BOUNDS ? kSegWanted : kSegWanted64)));
    const bool split = !BOUNDS || whole < kSegTarget;
    const int target = PAIR ? whole : max(1, whole / 8);
    const int *c0 = c.cnt + 8 * a.band_off[v.q] + (long long)gt * v.nb, *c1 = c0 + 4LL * v.nb;
    const double *l0 = BOUNDS ? c.bmin + 8 * a.band_off[v.q] + (long long)gt * v.nb : nullptr;
    const double *h0 = BOUNDS ? c.bmax + 8 * a.band_off[v.q] + (long long)gt * v.nb : nullptr;
    const int part0 = (int)((long long)v.nb * blockIdx.y / gridDim.y);
    const int part1 = (int)((long long)v.nb * (blockIdx.y + 1) / gridDim.y);
    int u0 = (8 * part0) << 12, acc = 0, n = 0;
    double lo = HUGE_VAL, hi = 0.0;
    int my_p0 = 0, my_p1 = 0, my_acc = 0;  // the segment this lane keeps
    double my_lo = 0.0, my_hi = 0.0;
    auto write = [&](int at) {  // the wave's n segments to places at, at + 1, ...
        at += lane;
        if (lane < n && at < c.cap[kind]) {
            const int e = (PAIR ? 0 : c.cap[0]) + at;
            c.seg_job[e] = v.q * 8 + gt;
            c.seg_p0[e] = my_p0;
            c.seg_p1[e] = my_p1;
            if (BOUNDS) c.rec[e] = SegRec{v.q * 8 + gt, my_p0, my_acc, 0, my_lo, my_hi};
        }
        n = 0;
    };
    auto flush = [&]() {
        int at = 0;
        if (lane == 0) at = (int)atomicAdd(&c.n_seg[kind], (unsigned long long)n);
        write(__shfl(at, 0));
    };
    auto close = [&](int u1) {  // u1 = end << 12 | term
        if (acc > 0) {
            if (lane == n) {
                my_p0 = u0;
                my_p1 = u1;
                my_acc = acc;
                my_lo = lo;
                my_hi = hi;
            }
            if (++n == 64) flush();
        }
        u0 = u1;
        acc = 0;
        lo = HUGE_VAL;
        hi = 0.0;
    };
    for (int pb = part0; pb < part1; pb += 64) {
        const int pl = pb + lane;
        const int mine = pl < part1 ? c0[pl] + (PAIR ? c1[pl] : 0) : 0;
        unsigned long long m = __ballot(mine > 0);
        while (m) {
            const int k = __builtin_ctzll(m), p = pb + k;
            m &= m - 1;
            const int pc = __shfl(mine, k);
            if (split && pc > target) {
                // lane ft (and, for gt | 4, lane 8 + ft): the norm of ft and
                // whether the pair is a candidate
                const double fl = a.slot_norm[(long long)v.band[p] * 8 + (lane & 7)];
                const unsigned long long cm =
                    __ballot(lane < (PAIR ? 16 : 8) && pair_candidate(v, gt | (lane & 8 ? 4 : 0), p, lane & 7, fl));
                for (int ft = 0; ft < 8; ft++) {
                    if (!((cm >> ft) & 0x101)) continue;
                    const double fn = __shfl(fl, ft);
                    if constexpr (!BOUNDS) {
                        const bool p0 = (cm >> ft) & 1, p1 = PAIR && ((cm >> (8 + ft)) & 1);
                        const PairNorms q = pair_norms(v, gt, p, ft);
                        const double *nz1 = q.nz + (long long)2 * v.side * v.na;
                        for (int b0 = 0; b0 < v.na; b0 += 64) {
                            const int e = b0 + lane;
                            const bool in = e < v.na;
                            const double xy = in ? q.nx[e] * q.ny[e] : 0.0;
                            const unsigned long long m0 = __ballot(in && p0 && (xy * q.nz[in ? e : 0]) * fn > v.thr);
                            const unsigned long long m1 = __ballot(in && p1 && (xy * nz1[in ? e : 0]) * fn > v.thr);
                            for (int sb = 0; sb < 64; sb += 16) {
                                acc += __popcll((m0 >> sb) & 0xffff) + __popcll((m1 >> sb) & 0xffff);
                                if (acc >= target) {
                                    const bool end = b0 + sb + 16 >= v.na;
                                    close(((8 * p + ft + (end ? 1 : 0)) << 12) | (end ? 0 : b0 + sb + 16));
                                }
                            }
                        }
                        continue;
                    }
                    double l = HUGE_VAL, h = 0.0;
                    int t = 0;
                    if ((cm >> ft) & 1) t = pair_terms(v, gt, p, ft, fn, lane, l, h);
                    if (PAIR && ((cm >> (8 + ft)) & 1)) t += pair_terms(v, gt | 4, p, ft, fn, lane, l, h);
                    if (t == 0) continue;
                    if (BOUNDS) wave_range(l, h);
                    acc += t;
                    lo = fmin(lo, l);
                    hi = fmax(hi, h);
                    if (acc >= target) close((8 * p + ft + 1) << 12);
                }
            } else {
                acc += pc;
                if (BOUNDS) {
                    lo = fmin(lo, PAIR ? fmin(l0[p], l0[4 * v.nb + p]) : l0[p]);
                    hi = fmax(hi, PAIR ? fmax(h0[p], h0[4 * v.nb + p]) : h0[p]);
                }
                if (acc >= target) close((8 * (p + 1)) << 12);
            }
        }
    }
    close((8 * part1) << 12);
    // what is left, with one addition for the workgroup
    constexpr int WAVES = PAIR ? 4 : 8;
    __shared__ int left[WAVES], base;
    if (lane == 0) left[gt] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;
        for (int w = 0; w < WAVES; w++) sum += left[w];
        base = sum ? (int)atomicAdd(&c.n_seg[kind], (unsigned long long)sum) : 0;
    }
    __syncthreads();
    int at = base;
    for (int w = 0; w < gt; w++) at += left[w];
    write(at);
}

// The class lists of the low-precision modes (pair segments with a term of the
// low class to lo, fine ones with a term of the FP64 class to hi), widened by a
// relative 1e-9 so that rounding can only add segments: the calculators' own
// class test decides each term.  n[0], n[1] receive their lengths, zero where
// the segments outgrew their room.  One thread per place, one addition per wave
// and list; the segments stay near the order they were cut in.  A level's lists
// made on the host cost a wait, a download of 32 bytes per segment, two sorts
// and two uploads: 4.4 of 8.8 ms of a split FP16 Helmholtz apply at k = 9.
__global__ __launch_bounds__(256) void k_class_lists(CountArgs c, double tau, int *lo, int *hi,
                                                     unsigned long long *n) {
    const unsigned long long n0 = c.n_seg[0], n1 = c.n_seg[1];
    if (n0 > (unsigned long long)c.cap[0] || n1 > (unsigned long long)c.cap[1]) return;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x, j = i - c.cap[0];
    const bool pair = i < c.cap[0], in = pair ? i < (long long)n0 : j < (long long)n1;
    bool take = false;
    if (in) {
        const SegRec r = c.rec[i];
        const int q = r.job >> 3;
        const double thr = fmax(c.k.out_thr[q], c.k.apps[c.k.out_app[q]].thr_floor);
        take = pair ? r.lo <= tau * thr * (1.0 + 1e-9) : r.hi > tau * thr * (1.0 - 1e-9);
    }
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const unsigned long long m = __ballot(take && pair == (k == 0));
        if (!m) continue;
        const int lead = __ffsll(m) - 1;
        int at = 0;
        if (lane == lead) at = (int)atomicAdd(&n[k], (unsigned long long)__popcll(m));
        at = __shfl(at, lead);
        if ((m >> lane) & 1) (k ? hi : lo)[at + __popcll(m & ((1ull << lane) - 1))] = (int)i;
    }
}

}  // namespace

int dev_class_lists(hipStream_t s, const CountArgs &c, double tau, int *lo, int *hi, unsigned long long *n,
                    std::string &err) {
    const long long places = (long long)c.cap[0] + c.cap[1];
    hipLaunchKernelGGL(k_class_lists, dim3((unsigned)((places + 255) / 256)), dim3(256), 0, s, c, tau, lo, hi, n);
    HIP_TRY(hipGetLastError());
    return 0;
}

int dev_term_tables(hipStream_t s, const KArgs &k, int nn, const TermLevel *levels, int n, double *tn, int2 *tb,
                    std::string &err) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_term_norms, dim3(n, 4), dim3(256), 0, s, k, nn, levels, tn, tb);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_prescreen, dim3(n, 64), dim3(256), 0, s, k, levels);
    HIP_TRY(hipGetLastError());
    return 0;
}

int dev_count_terms(hipStream_t s, const CountArgs &c, bool bounds, std::string &err) {
    if (c.n_out == 0) return 0;
    // a node's steps shared among as many workgroups as keep a launch below
    // 768 of them (each adds to its apply's total, 10 ns for an addition to
    // one address: 17 -> 15 us a level at k = 9 against 2048), shorter steps
    // where whole ones leave less than 1024
    const long long pairs = 8 * c.widest;
    const int step = c.n_out * ((pairs + 63) / 64) < 1024 ? 16 : 64;
    const int y = (int)std::max<long long>(1, std::min<long long>((pairs + step - 1) / step, 768 / c.n_out));
    return in_launches(c.n_out, 512, [&](long long first, long long n) {
        CountArgs part = c;
        part.q0 = (int)first;
        if (bounds)
            hipLaunchKernelGGL((k_count<true>), dim3((unsigned)n, y), dim3(512), 0, s, part, step);
        else
            hipLaunchKernelGGL((k_count<false>), dim3((unsigned)n, y), dim3(512), 0, s, part, step);
        HIP_TRY(hipGetLastError());
        return 0;
    });
}

int dev_cut_segments(hipStream_t s, const CountArgs &c, bool bounds, std::string &err) {
    if (c.n_out == 0) return 0;
    // three positions a part at the least, and no more parts than fill the
    // chip: each ends a segment
    const int y = (int)std::max<long long>(1, std::min<long long>(c.widest / 3, 1024 / c.n_out));
    return in_launches(c.n_out, 512, [&](long long first, long long n) {
        CountArgs part = c;
        part.q0 = (int)first;
        if (bounds) {
            hipLaunchKernelGGL((k_cut<true, true>), dim3((unsigned)n), dim3(256), 0, s, part);
            HIP_TRY(hipGetLastError());
            hipLaunchKernelGGL((k_cut<false, true>), dim3((unsigned)n, y), dim3(512), 0, s, part);
        } else {
            hipLaunchKernelGGL((k_cut<true, false>), dim3((unsigned)n, y), dim3(256), 0, s, part);
        }
        HIP_TRY(hipGetLastError());
        return 0;
    });
}

}  // namespace mwg
