// The root level of an apply as three dense products per kernel term (gfx950).
//
// The first refinement level of mrcpp::apply has no output norm yet, so its
// thresholds are zero and every term of every (output box, input box,
// component pair) passes the screening rule (reached from
// src/qmoperators/two_electron/CoulombPotential.cpp:131).  All root boxes
// together are then one dense tensor of D_x x D_y x D_z values, D_d = 2 N
// boxes_d (the box, its scaling or wavelet part, the N coefficients), and a
// term acts on it as A_z (x) A_y (x) A_x, where A_d holds the term's blocks
// [box g][out component][i] x [box f][in component][j] of the translations
// f - g: 6 D^4 operations a term where the calculator's per-component items
// need 64 x 6 N^4 for each of the box pairs (16 times as many at 2 x 2 x 2
// boxes).
//
// The sums over the terms run in three launches per chunk of terms: the
// matrices A (k_root_ops), both in-plane passes of every z plane
// (k_root_xy, Y = A_y F_p A_x^T) and the z pass, one long sum over (term,
// plane) (k_root_z).  The work is a few Gflop, so the 16 x 16 x 4 FP64 MFMA
// with the dimensions padded to 16 is near enough to its bound; what the
// launches wait for is Y (8 D^3 bytes a term, written once and read once,
// from the memory-side cache): a SIMD holds one or two waves, so both passes
// have their next operands on the way while they work (matrices through LDS,
// Y in registers).  Device time of the root level, per-component items ->
// these kernels: one apply at k = 7 (171 terms) 1.64 -> 0.06 ms (0.08 with
// operands loaded as they are needed), ten exchange densities 5.96 -> 0.38 ms
// (0.54), six orbitals at k = 11 (145 terms each) 11.2 -> 0.95 ms (1.7).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "mw_device.hpp"

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

typedef double root_d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ root_d4 root_mfma(double a, double b, root_d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Items (term m of root apply app) of one chunk, [item0, item0 + n).
// Matrices of an item: nd of them (1 when the box counts agree in all
// directions, so that one matrix serves x, y and z; else 3, x first), each
// T x 4T operand pieces of 64 lanes: element (16 t + lane % 16, 4 k +
// lane / 16) at [(t 4T + k) 64 + lane], zero outside D x D.  As the A operand
// of a 16 x 16 x 4 MFMA a piece gives rows of A, as the B operand columns of
// its transpose.
template <int T>
__global__ __launch_bounds__(256) void k_root_ops(RootGeo geo, const RootApp *apps, const RootItem *items, int nd,
                                                  double *A) {
    constexpr int SZ = T * 4 * T * 64;
    const RootItem it = items[blockIdx.x];
    const RootApp ap = apps[it.app];
    const int dim = blockIdx.y, N = geo.n, D = 2 * N * geo.boxes[dim];
    const int L = ap.L[it.m * ap.ndepth];
    const double *blk = ap.blocks + (L >= 0 ? ap.boff[it.m * ap.ndepth] : 0);
    double *dst = A + ((size_t)blockIdx.x * nd + dim) * SZ;
    for (int e = threadIdx.x; e < SZ; e += 256) {
        const int lane = e & 63, k = (e >> 6) % (4 * T), t = (e >> 6) / (4 * T);
        const int row = 16 * t + (lane & 15), col = 4 * k + (lane >> 4);
        double v = 0.0;
        if (row < D && col < D) {
            const int l = col / (2 * N) - row / (2 * N);
            const int c = 2 * ((row / N) & 1) + ((col / N) & 1);
            if (L >= 0 && abs(l) <= L) v = blk[((size_t)c * (2 * L + 1) + (l + L)) * N * N + (row % N) * N + col % N];
        }
        dst[e] = v;
    }
}

// Position q of a direction (box, component, coefficient) as its parts.
struct RootPos {
    int box, comp, i;
};
__device__ __forceinline__ RootPos root_pos(int n, int q) { return RootPos{q / (2 * n), (q / n) & 1, q % n}; }

// In-plane passes: one wave per (plane p, group of kRootItems items).  The
// plane's values stay in registers as A operands for all its items (and are
// reloaded where the apply changes); the x pass leaves X[jy][ix] in exactly
// the lanes in which the y pass reads it as its B operand (D row lane / 16 +
// 4 r of register r = the operand's row of step r), so no value passes
// through LDS.  The four waves of a workgroup take four planes with the same
// items, whose matrices they share in LDS.
constexpr int kRootItems = 4;

template <int T, bool SAME>
__global__ __launch_bounds__(256) void k_root_xy(RootGeo geo, const RootApp *apps, const RootItem *items, int n_items,
                                                 const long long *slot_off, const double *pool, const double *A,
                                                 double *Y) {
    constexpr int K = 4 * T, SZ = T * K * 64, DP = 16 * T, nd = SAME ? 1 : 3;
    const int N = geo.n, N3 = N * N * N;
    const int D[3] = {2 * N * geo.boxes[0], 2 * N * geo.boxes[1], 2 * N * geo.boxes[2]};
    const int lane = threadIdx.x & 63, lc = lane & 15, lq = lane >> 4;
    const int p = min(4 * blockIdx.y + (int)(threadIdx.x >> 6), D[2] - 1);  // the last: maybe twice, same values
    const RootPos pz = root_pos(N, p);
    double fa[T][K];
    int cur = -1;
    const int i0 = blockIdx.x * kRootItems, i1 = min(i0 + kRootItems, n_items);
    // the items' matrices (x, then y) in LDS, the next item's on its way in
    // registers meanwhile
    constexpr int NM = SAME ? 1 : 2, PER = NM * SZ / 256;
    __shared__ double As[2][NM * SZ];
    double next[PER];
    auto fetch = [&](int it) {
        const double *a = A + (size_t)it * nd * SZ + threadIdx.x;
#pragma unroll
        for (int e = 0; e < PER; e++) next[e] = a[256 * e];
    };
    auto keep = [&](int buf) {
#pragma unroll
        for (int e = 0; e < PER; e++) As[buf][threadIdx.x + 256 * e] = next[e];
    };
    fetch(i0);
    keep(0);
    __syncthreads();
    for (int it = i0; it < i1; it++) {
        if (it + 1 < i1) fetch(it + 1);
        const int app = items[it].app, buf = (it - i0) & 1;
        if (app != cur) {
            cur = app;
            const long long *so = slot_off + apps[app].root0;
#pragma unroll
            for (int a = 0; a < T; a++) {
                const int jy = 16 * a + lc;
                const RootPos py = root_pos(N, jy);
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int jx = 4 * k + lq;
                    const RootPos px = root_pos(N, jx);
                    double v = 0.0;
                    if (jy < D[1] && jx < D[0])
                        v = pool[so[(pz.box * geo.boxes[1] + py.box) * geo.boxes[0] + px.box] +
                                 (px.comp | (py.comp << 1) | (pz.comp << 2)) * N3 + (pz.i * N + py.i) * N + px.i];
                    fa[a][k] = v;
                }
            }
        }
        const double *Ax = As[buf], *Ay = SAME ? Ax : Ax + SZ;
        double *y = Y + ((size_t)it * D[2] + p) * DP * DP;
#pragma unroll 1
        for (int h = 0; h < T; h++) {
            double op[K];
#pragma unroll
            for (int k = 0; k < K; k++) op[k] = Ax[(h * K + k) * 64 + lane];
            root_d4 x[T], d[T];
#pragma unroll
            for (int a = 0; a < T; a++) x[a] = d[a] = root_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < K; k++)
#pragma unroll
                for (int a = 0; a < T; a++) x[a] = root_mfma(fa[a][k], op[k], x[a]);
#pragma unroll
            for (int a = 0; a < T; a++)
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int b = 0; b < T; b++) d[b] = root_mfma(Ay[(b * K + 4 * a + r) * 64 + lane], x[a][r], d[b]);
#pragma unroll
            for (int b = 0; b < T; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) y[(16 * b + 4 * r + lq) * DP + 16 * h + lc] = d[b][r];
        }
        if (it + 1 < i1) keep(buf ^ 1);
        __syncthreads();
    }
}

// The z pass: out[iz][(iy, ix)] += sum over items and planes of A_z Y.  One
// wave per (64 columns, run of per items); the accumulators are added into
// the roots' output blocks (zeroed before) when the apply changes and at the
// end of the run.  totals: per apply of the plan its term-applications and
// those of the roots; the latter are added to the plan's counter (n_totals 0:
// not by this launch).
template <int T, bool SAME>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_root_z(
    RootGeo geo, const RootApp *apps, const RootItem *items, int n_items, int per, const int *root_out, const double *A,
    const double *Y, double *out_ns, unsigned long long *counter, const unsigned long long *totals, int n_totals) {
    constexpr int K = 4 * T, SZ = T * K * 64, DP = 16 * T, nd = SAME ? 1 : 3;
    const int N = geo.n, N3 = N * N * N;
    const int D[3] = {2 * N * geo.boxes[0], 2 * N * geo.boxes[1], 2 * N * geo.boxes[2]};
    const int lane = threadIdx.x & 63, lc = lane & 15, lq = lane >> 4;
    if (blockIdx.x == 0 && blockIdx.y == 0)
        for (int i = threadIdx.x; i < n_totals; i += 256) atomicAdd(counter, totals[2 * i + 1]);
    const int cg = 4 * blockIdx.y + (threadIdx.x >> 6);  // DP DP / 64 groups: a multiple of 4
    const int i0 = blockIdx.x * per, i1 = min(i0 + per, n_items);
    root_d4 acc[4][T];
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int t = 0; t < T; t++) acc[c][t] = root_d4{0.0, 0.0, 0.0, 0.0};
    auto flush = [&](int app) {
        const int *ro = root_out + apps[app].root0;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            int cv = 16 * c + lc;  // (not to be worked out ahead of the steps)
            asm volatile("" : "+v"(cv));
            const int col = 64 * cg + cv, iy = col / DP, ix = col % DP;
            const RootPos py = root_pos(N, iy), px = root_pos(N, ix);
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int iz = 16 * t + 4 * r + lq;
                    if (iz < D[2] && iy < D[1] && ix < D[0]) {
                        const RootPos pz = root_pos(N, iz);
                        const int g = ro[(pz.box * geo.boxes[1] + py.box) * geo.boxes[0] + px.box];
                        atomicAdd(&out_ns[((size_t)g * 8 + (px.comp | (py.comp << 1) | (pz.comp << 2))) * N3 +
                                          (pz.i * N + py.i) * N + px.i],
                                  acc[c][t][r]);
                    }
                    acc[c][t][r] = 0.0;
                }
        }
    };
    // Steps (item, k) in order, the operands of the next AHEAD steps on their
    // way: a SIMD holds one of these waves, and a step's loads come from the
    // memory-side cache.
    constexpr int AHEAD = 4;
    const int ks = (D[2] + 3) / 4;
    double a[AHEAD][T], b[AHEAD][4];
    for (int s0 = i0; s0 < i1;) {
        const int app = items[s0].app;
        int s1 = s0 + 1;
        while (s1 < i1 && items[s1].app == app) s1++;
        int nit = s0, nk = 0;  // the next step to load (past the end: the last again)
        auto load = [&](double (&a)[T], double (&b)[4]) {
            const double *Az = A + ((size_t)nit * nd + (SAME ? 0 : 2)) * SZ + nk * 64 + lane;
            // rows past the last plane meet zero columns of A: any finite row
            const double *y = Y + ((size_t)nit * D[2] + min(4 * nk + lq, D[2] - 1)) * DP * DP + 64 * cg + lc;
#pragma unroll
            for (int t = 0; t < T; t++) a[t] = Az[t * K * 64];
#pragma unroll
            for (int c = 0; c < 4; c++) b[c] = y[16 * c];
            const bool wrap = nk + 1 == ks, end = wrap && nit + 1 == s1;
            nk = end ? nk : wrap ? 0 : nk + 1;
            nit += wrap && !end ? 1 : 0;
        };
#pragma unroll
        for (int u = 0; u < AHEAD; u++) load(a[u], b[u]);
        auto step = [&](int u) {
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int t = 0; t < T; t++) acc[c][t] = root_mfma(a[u][t], b[u][c], acc[c][t]);
        };
        int left = (s1 - s0) * ks;
        for (; left >= AHEAD; left -= AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                step(u);
                load(a[u], b[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < AHEAD; u++)
            if (u < left) step(u);
        flush(app);
        s0 = s1;
    }
}

template <int T, bool SAME>
hipError_t root_chunk(hipStream_t s, const RootLaunch &r, int item0, int n) {
    const int nd = SAME ? 1 : 3, dz = 2 * r.geo.n * r.geo.boxes[2], groups = 16 * T * T / 4;
    const RootItem *items = r.items + item0;
    hipLaunchKernelGGL((k_root_ops<T>), dim3(n, nd), dim3(256), 0, s, r.geo, r.apps, items, nd, r.A);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_root_xy<T, SAME>), dim3((n + kRootItems - 1) / kRootItems, (dz + 3) / 4), dim3(256), 0, s,
                       r.geo, r.apps, items, n, r.slot_off, r.pool, r.A, r.Y);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    // runs of at least 4 items (every run ends in D^3 atomic adds), about
    // 1024 waves where the chunk holds enough items
    const int runs = std::max(1, std::min((n + 3) / 4, 1024 / groups));
    const int per = (n + runs - 1) / runs;
    hipLaunchKernelGGL((k_root_z<T, SAME>), dim3((n + per - 1) / per, groups / 4), dim3(256), 0, s, r.geo, r.apps,
                       items, n, per, r.root_out, r.A, r.Y, r.out_ns, r.counter, r.totals, item0 == 0 ? r.n_totals : 0);
    return hipGetLastError();
}

int root_tiles(int n, const int *boxes) {
    const int b = std::max(boxes[0], std::max(boxes[1], boxes[2]));
    return (2 * n * b + 15) / 16;
}

bool root_same(const int *boxes) { return boxes[0] == boxes[1] && boxes[1] == boxes[2]; }

// Terms of one chunk: Y of a chunk stays within 128 MB, so that the z pass
// finds it in the memory-side cache (with 64 MB the k = 11 chunks hold 75 terms
// and half fill the chip: 0.74 against 0.51 ms of z passes).
long long root_chunk_items(int n, const int *boxes, long long n_items) {
    const long long dp = 16 * root_tiles(n, boxes), y = 8LL * 2 * n * boxes[2] * dp * dp;
    return std::max(1LL, std::min(n_items, (128LL << 20) / y));
}

}  // namespace

void root_work_values(int n, const int *boxes, long long n_items, size_t *a_values, size_t *y_values) {
    const size_t t = root_tiles(n, boxes), dp = 16 * t, c = (size_t)root_chunk_items(n, boxes, n_items);
    *a_values = c * (root_same(boxes) ? 1 : 3) * dp * dp;
    *y_values = c * 2 * n * boxes[2] * dp * dp;
}

int dev_root_launch(void *stream, const RootLaunch &r, std::string &err) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int t = root_tiles(r.geo.n, r.geo.boxes);
    const bool same = root_same(r.geo.boxes);
    const int chunk = (int)root_chunk_items(r.geo.n, r.geo.boxes, r.n_items);
    for (int i = 0; i < r.n_items; i += chunk) {
        const int n = std::min(chunk, r.n_items - i);
        hipError_t e = hipErrorInvalidValue;
        if (t == 1) e = same ? root_chunk<1, true>(s, r, i, n) : root_chunk<1, false>(s, r, i, n);
        if (t == 2) e = same ? root_chunk<2, true>(s, r, i, n) : root_chunk<2, false>(s, r, i, n);
        if (t == 3) e = same ? root_chunk<3, true>(s, r, i, n) : root_chunk<3, false>(s, r, i, n);
        HIP_TRY(e);
    }
    return 0;
}

}  // namespace mwg
