// Bands and input slots of an apply plan, made on the device.
//
// Upstream MRCPP's OperApplicationCalculator::makeOperBand gathers, for each
// output node g at scale n, the input nodes f with |l_f - l_g|_inf <= w(n),
// generating missing ones by reconstruction from their deepest ancestor
// (MWTree::getNode with node generation).  Here one thread per band entry
// finds the entry's node in an open-addressed table shared by the whole plan;
// the thread that enters a node walks the input tree from its root box to it
// and so knows whether it is there or which ancestor it is generated from, and
// enters the generated nodes in between.  A second launch, with the numbers of
// slots and generated nodes known, writes the copy and generation items of the
// pool and the band table.
//
// Nothing here moves more than the table and the band entries (21 and 8 bytes
// each): both launches are bound by the latency of dependent loads and
// compare-and-swaps, so every entry has its own thread, and a node that is in
// the table costs its later finders one load.  Hash maps on the host took 330 us
// a refinement level at 74,500 entries in 10 levels (Helmholtz, k = 9: 9.9 ms
// the call, 7.0 ms with these launches; the exchange applies of 4 orbitals in
// one batch: 10.5 and 7.9 ms).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "mw_apply.hpp"

#define HIP_TRY(expr)                                                       \
    do {                                                                    \
        hipError_t e_ = (expr);                                             \
        if (e_ != hipSuccess) {                                             \
            err = std::string(#expr) + ": " + hipGetErrorString(e_);        \
            return -2;                                                      \
        }                                                                   \
    } while (0)

namespace mwg {
namespace {
constexpr unsigned long long kEmpty = ~0ull;
// Probes before a full table is assumed (the caller then comes back with a
// larger one); at most half of the cells are taken, where chains of this length
// are not expected.
constexpr int kMaxProbe = 256;

struct Key {
    int app, d, l[3];
};

// A cell is named by the band entry that took it: output node, position in its
// band and the number of levels above the entry's node.
__device__ __forceinline__ unsigned long long rep_of(int q, int p, int up) {
    return (unsigned long long)q << 27 | (unsigned long long)p << 5 | (unsigned)up;
}

__device__ __forceinline__ Key entry_key(const BandArgs &a, int q, int p, int up) {
    const int w = a.band_w[q], side = 2 * w + 1;
    const int t = p / side, x = p - t * side, z = t / side, y = t - z * side;
    Key k;
    k.app = a.out_app[q];
    k.d = a.out_depth[q] - up;
    k.l[0] = (a.out_l[3 * q] + x - w) >> up;
    k.l[1] = (a.out_l[3 * q + 1] + y - w) >> up;
    k.l[2] = (a.out_l[3 * q + 2] + z - w) >> up;
    return k;
}

__device__ __forceinline__ Key rep_key(const BandArgs &a, unsigned long long r) {
    return entry_key(a, (int)(r >> 27), (int)(r >> 5) & 0x3fffff, (int)r & 31);
}

__device__ __forceinline__ unsigned long long hash_of(const Key &k) {
    unsigned long long h = ((unsigned long long)k.app << 5 | (unsigned)k.d) * 0x9E3779B97F4A7C15ull;
    h = (h ^ (h >> 29) ^ (unsigned)k.l[0]) * 0xC2B2AE3D27D4EB4Full;
    h = (h ^ (h >> 31) ^ (unsigned)k.l[1]) * 0x165667B19E3779F9ull;
    h = (h ^ (h >> 30) ^ (unsigned)k.l[2]) * 0x27D4EB2F165667C5ull;
    return h ^ (h >> 32);
}

// The cell of node k, taken under the name rep if no cell holds it yet (fresh);
// found: the name it has.  -1: no cell within the probes.  A plain value of a
// cell may be stale only as "empty", which the compare-and-swap then corrects;
// no thread waits for another.
__device__ __forceinline__ int locate(const BandArgs &a, const Key &k, unsigned long long rep, bool &fresh,
                                      unsigned long long &found) {
    fresh = false;
    unsigned h = (unsigned)hash_of(k) & (a.cap - 1);
    for (int i = 0; i < kMaxProbe; i++, h = (h + 1) & (a.cap - 1)) {
        unsigned long long cur = __hip_atomic_load(&a.rep[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (cur == kEmpty) {
            cur = atomicCAS(&a.rep[h], kEmpty, rep);
            if (cur == kEmpty) {
                fresh = true;
                found = rep;
                return (int)h;
            }
        }
        const Key o = rep_key(a, cur);
        if (o.app == k.app && o.d == k.d && o.l[0] == k.l[0] && o.l[1] == k.l[1] && o.l[2] == k.l[2]) {
            found = cur;
            return (int)h;
        }
    }
    atomicOr(&a.cnt[2], 1u);
    return -1;
}

// Ids for the lanes with want, one addition to *n per wave.
__device__ __forceinline__ int take_ids(bool want, unsigned *n) {
    const unsigned long long m = __ballot(want);
    if (!m) return 0;
    const int lane = threadIdx.x & 63, lead = __ffsll(m) - 1;
    unsigned at = 0;
    if (lane == lead) at = atomicAdd(n, (unsigned)__popcll(m));
    return (int)__shfl(at, lead) + (int)__popcll(m & ((1ull << lane) - 1));
}

__global__ __launch_bounds__(256) void k_band_clear(BandArgs a) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < a.cap) {
        a.rep[i] = kEmpty;
        a.slot[i] = -1;
    }
    if (i < kBandCounts) a.cnt[i] = 0;
}

// Workgroups (q, y): the band entries of output node q.  slot of a cell: a real
// slot's id (>= 0), -(id + 3) for a generated slot, -2 while its id is being
// taken, -1 for a node that is no slot (a generated ancestor).
__global__ __launch_bounds__(256) void k_band_find(BandArgs a) {
    const int q = a.q0 + (int)blockIdx.x, side = 2 * a.band_w[q] + 1, nb = side * side * side;
    const BandTree &t = a.trees[a.out_app[q]];
    int *cells = a.cell + a.band_off[q];
    __shared__ int taken[2][4], first[2];
    for (int p0 = 256 * blockIdx.y; p0 < nb; p0 += 256 * gridDim.y) {
        const int p = p0 + threadIdx.x;
        int c = -1;
        bool fresh = false, claim = false, real = false;
        unsigned long long found = 0;
        Key k{};
        if (p < nb) {
            k = entry_key(a, q, p, 0);
            bool in = true;
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int b = k.l[d] >> k.d;
                in = in && b >= 0 && b < a.boxes[d];
            }
            if (in) c = locate(a, k, rep_of(q, p, 0), fresh, found);
            cells[p] = c;
            claim = fresh;
            // entered before as an ancestor: the first entry to find it makes
            // it a slot as well
            if (c >= 0 && !fresh && (found & 31)) claim = atomicCAS(&a.slot[c], -1, -2) == -1;
        }
        int node = -1, da = 0;
        if (fresh) {
            // (the roots are a tree's first nodes, box x fastest)
            node = ((k.l[2] >> k.d) * a.boxes[1] + (k.l[1] >> k.d)) * a.boxes[0] + (k.l[0] >> k.d);
            for (; da < k.d; da++) {
                const int c0 = t.child0[node], b = k.d - 1 - da;
                if (c0 < 0) break;
                node = c0 + ((k.l[0] >> b) & 1) + 2 * ((k.l[1] >> b) & 1) + 4 * ((k.l[2] >> b) & 1);
            }
            real = da == k.d;
        }
        // slot ids, one addition a workgroup (to one address they take about
        // 10 ns each from all over the chip: 34 -> 23 us a launch on the
        // exchange applies of 4 orbitals against one a wave and node)
        const unsigned long long mr = __ballot(claim && real), mg = __ballot(claim && !real);
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        if (lane == 0) {
            taken[0][wv] = (int)__popcll(mr);
            taken[1][wv] = (int)__popcll(mg);
        }
        __syncthreads();
        if (threadIdx.x < 2) {
            int sum = 0;
            for (int w = 0; w < 4; w++) sum += taken[threadIdx.x][w];
            first[threadIdx.x] = sum ? (int)atomicAdd(&a.cnt[threadIdx.x], (unsigned)sum) : 0;
        }
        __syncthreads();
        if (claim) {
            int id = first[real ? 0 : 1] + (int)__popcll((real ? mr : mg) & ((1ull << lane) - 1));
            for (int w = 0; w < wv; w++) id += taken[real ? 0 : 1][w];
            a.slot[c] = real ? id : -(id + 3);
        }
        __syncthreads();  // read before the next entries' are written
        if (fresh && real) {
            a.lv[c] = -1;
            a.gen[c] = make_int2(node, 0);
        }
        // positions of the entries' own generated nodes, a level at a time
        const int lv0 = fresh && !real ? k.d - da - 1 : -1;
        int pos = 0;
        unsigned long long todo = __ballot(lv0 >= 0);
        while (todo) {
            const int lv = __builtin_amdgcn_readlane(lv0, __ffsll(todo) - 1);
            const int id = take_ids(lv0 == lv, &a.cnt[3 + lv]);
            if (lv0 == lv) pos = id;
            todo &= ~__ballot(lv0 == lv);
        }
        if (fresh && !real) {
            // the generated nodes from the entry's up to the child of the
            // ancestor that is there; a known one has the rest of its own
            int lv = lv0, at = c;
            for (int up = 1;; up++, lv--) {
                a.lv[at] = (signed char)lv;
                if (up > 1) pos = (int)atomicAdd(&a.cnt[3 + lv], 1u);
                if (lv == 0) {
                    a.gen[at] = make_int2(-(node + 1), pos);
                    break;
                }
                k.d--;
#pragma unroll
                for (int d = 0; d < 3; d++) k.l[d] >>= 1;
                bool more;
                const int par = locate(a, k, rep_of(q, p, up), more, found);
                a.gen[at] = make_int2(par, pos);
                if (!more) break;
                at = par;
            }
        }
    }
}

// Threads [0, cap): a cell's generation item and pool item; then one thread per
// band entry: its slot; then per root box of the dense root kernels: the pool
// offset of its slot.
__global__ __launch_bounds__(256) void k_band_items(BandArgs a, BandItems o) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const size_t n3 = o.n3, blk = 8 * n3;
    if (i < a.cap) {
        const unsigned long long r = a.rep[i];
        if (r == kEmpty) return;
        const double *inp = a.trees[a.out_app[(int)(r >> 27)]].inp;
        const int lv = a.lv[i], s = a.slot[i];
        const int2 g = a.gen[i];
        const double *src = nullptr;
        if (lv >= 0) {
            const Key k = rep_key(a, r);
            double *dst = o.gen_s + (size_t)(o.lv_off[lv] + g.y) * n3;
            src = dst;
            o.gen[o.lv_off[lv] + g.y] =
                GenItem{g.x < 0 ? inp + (size_t)(-g.x - 1) * blk
                                : o.gen_s + (size_t)(o.lv_off[lv - 1] + a.gen[g.x].y) * n3,
                        dst, (k.l[0] & 1) | (k.l[1] & 1) << 1 | (k.l[2] & 1) << 2, g.x < 0};
        }
        if (s == -1) return;
        const int id = s >= 0 ? s : o.n_real - s - 3;
        const long long off = s >= 0 ? (long long)(id * blk) : (long long)(o.n_real * blk + (id - o.n_real) * n3);
        o.slot_off[id] = off;
        o.slots[id] = SlotItem{s >= 0 ? inp + (size_t)g.x * blk : src, o.pool + off, o.norms + 8 * (size_t)id,
                               (int)(s >= 0 ? blk : n3)};
        return;
    }
    i -= a.cap;
    if (i < a.n_band) {
        const int c = a.cell[i];
        int s = -1;
        if (c >= 0) {
            s = a.slot[c];
            if (s < 0) s = o.n_real - s - 3;
        }
        o.band[i] = s;
        return;
    }
    i -= a.n_band;
    if (i < o.n_roots) {
        const int q = o.root_out[i], side = 2 * a.band_w[q] + 1;
        o.root_off[i] = (long long)(a.slot[a.cell[a.band_off[q] + (side * side * side - 1) / 2]] * blk);
    }
}
}  // namespace

int dev_band_find(hipStream_t s, const BandArgs &a, long long widest, std::string &err) {
    hipLaunchKernelGGL(k_band_clear, dim3((unsigned)((std::max(a.cap, (unsigned)kBandCounts) + 255) / 256)), dim3(256),
                       0, s, a);
    HIP_TRY(hipGetLastError());
    const unsigned y = (unsigned)std::min<long long>((widest + 255) / 256, 64);
    return in_launches(a.n_out, 256, [&](long long first, long long n) {
        BandArgs part = a;
        part.q0 = (int)first;
        hipLaunchKernelGGL(k_band_find, dim3((unsigned)n, y), dim3(256), 0, s, part);
        HIP_TRY(hipGetLastError());
        return 0;
    });
}

int dev_band_items(hipStream_t s, const BandArgs &a, const BandItems &o, std::string &err) {
    const long long n = (long long)a.cap + a.n_band + o.n_roots;
    hipLaunchKernelGGL(k_band_items, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, o);
    HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace mwg
