// Neighbour update, local-sync flag, extra check and FP64 order parameter
// (EGG_SynC.cu:551-763, 767-1203; SynC.cpp:30-56), gfx950.
//
// The EGG kernels work on runs -- maximal stretches of bitwise-equal
// consecutive positions in the cell-sorted order: every point of a run has
// the same inputs and hence the same result, and every scan over a cell's
// points can visit its runs once, counting each with its length.  One
// wavefront handles a tile of <= 64 runs of one cell (tiles come from a work
// queue), so the walk over candidate cells and every cell load are
// wave-uniform while each lane runs the reference's per-point tests on its
// run's position.  A scatter pass copies each run's result to its points.
// Candidate cells come from the outer-cell box of radius R (as the
// reference), pruned in the remaining dimensions to |dg| <= R+1 by a binary
// search over the column's cells (sorted by g_od): cells farther than that
// fail the reference's box test by more than a cell side, so results do not
// change.  Up to kStreamMaxD dimensions the tests and masked sums over streamed runs
// run on the matrix cores (egg_stream.h), in the same order of FP32 additions.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "egg_candidates.h"
#include "egg_internal.h"
#include "egg_scan.h"
#include "egg_stream.h"

namespace egg {

// Odometer over the outer-cell offsets [-R, R]^od, dim 0 fastest (the
// enumeration order of EGG_SynC.cu:407-451), for per-thread walks.
template <int D>
struct Odo {
    int idx[D];
    bool finished;
    __device__ __forceinline__ void init(int od, int R) {
#pragma unroll
        for (int l = 0; l < D; l++) idx[l] = (l < od) ? -R : 0;
        finished = false;
    }
    __device__ __forceinline__ void next(int od, int R) {
        bool carry = true;
#pragma unroll
        for (int l = 0; l < D; l++) {
            if (l < od && carry) {
                idx[l]++;
                if (idx[l] > R) {
                    if (l == od - 1) finished = true;
                    else idx[l] = -R;
                } else {
                    carry = false;
                }
            }
        }
    }
    // outer cell id of the current offset, or -1 if outside the grid
    __device__ __forceinline__ int outer(const int *g0, const Geo &g) const {
        int o = 0;
        bool ok = true;
#pragma unroll
        for (int l = 0; l < D; l++) {
            if (l < g.od) {
                const int v = g0[l] + idx[l];
                if (v < 0 || v >= g.w) ok = false;
                o += v * g.wpow[l];
            }
        }
        return ok ? o : -1;
    }
};

// Walks the non-empty outer cells of the box [g0 - R, g0 + R]^od in the same
// order as Odo, cooperatively: the 2R+1 outer cells of a row along dim 0 have
// adjacent ids, so lane k loads the cell range of offset k and the wavefront
// visits the non-empty ones in lane order.  f(cb, ce) receives each cell
// range.  Called by a whole wavefront with wave-uniform g0 and R (2R+1 <= 64).
template <int D, typename Fn>
__device__ __forceinline__ void walk_columns(const int *g0, int R, const Geo &g,
                                             const int *__restrict__ ob,
                                             const int *__restrict__ oe, Fn &&f) {
    const int od = g.od, lane = __lane_id();
    int idx[D];
#pragma unroll
    for (int l = 0; l < D; l++) idx[l] = -R;
    for (;;) {
        bool ok = true;
        int base = 0;
#pragma unroll
        for (int l = 1; l < D; l++) {
            if (l < od) {
                const int v = g0[l] + idx[l];
                if (v < 0 || v >= g.w) ok = false;
                base += v * g.wpow[l];
            }
        }
        if (ok) {
            int cb = 0, ce = 0;
            const int v0 = g0[0] - R + lane;
            if (lane <= 2 * R && v0 >= 0 && v0 < g.w) {
                cb = ob[base + v0];
                ce = oe[base + v0];
            }
            unsigned long long m = __ballot(ce > cb);
            while (m) {
                const int k = __ffsll((long long)m) - 1;
                m &= m - 1;
                f(__builtin_amdgcn_readlane(cb, k), __builtin_amdgcn_readlane(ce, k));
            }
        }
        bool carry = true;
#pragma unroll
        for (int l = 1; l < D; l++) {
            if (l < od && carry) {
                if (++idx[l] > R) idx[l] = -R;
                else carry = false;
            }
        }
        if (carry) break;
    }
}

template <int D>
__device__ __forceinline__ int select_dim(const int *v, int k) {
    int r = 0;
#pragma unroll
    for (int l = 0; l < D; l++)
        if (l == k) r = v[l];
    return r;
}

template <int D>
__device__ __forceinline__ float dist2_to(const float *x, const float *__restrict__ Xs, int n,
                                          int j, float *xq) {
    float s = 0.f;
#pragma unroll
    for (int l = 0; l < D; l++) {
        xq[l] = Xs[(long long)l * n + j];
        const float df = x[l] - xq[l];
        s += df * df;
    }
    return s;
}

// Loads the D coordinates of cell c, returns false when the cell lies outside
// the pruning window of the remaining dimensions (*stop: past the window in
// g_od, so later cells of the column are outside too).
template <int D>
__device__ __forceinline__ bool cell_in_window(const int *__restrict__ cell_g, int n, int c,
                                               const int *g0, int od, int rad, int g0od,
                                               int *gc, bool *stop) {
#pragma unroll
    for (int l = 0; l < D; l++) gc[l] = cell_g[(long long)l * n + c];
    *stop = od < D && select_dim<D>(gc, od) > g0od + rad;
    bool in = true;
#pragma unroll
    for (int l = 0; l < D; l++)
        if (l > od && (gc[l] - g0[l] > rad || g0[l] - gc[l] > rad)) in = false;
    return in && !*stop;
}

// A source run of a cell staged in LDS: its position and, for its offset v
// from the tile's anchor, sin v and cos v - 1 (in cv).
template <int D>
struct SrcPt {
    static constexpr int P = (D + 3) / 4 * 4;
    float x[P], sv[P], cv[P];
};

// Group of tile t: the largest k with tile_off[k] <= t.
__device__ __forceinline__ int tile_group(const int *__restrict__ tile_off, int G, int t) {
    int lo = 0, hi = G - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tile_off[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// A tile seen by one lane: the tile's group (cells [gc0, gc1), all in one
// outer cell, equal in every inner coordinate but the last), the lane's run
// r (active if it belongs to the tile), its first sorted position i and its
// cell cl.
struct TileLane {
    int gc0, gc1, r, i, cl;
    bool active;
};

__device__ __forceinline__ TileLane tile_lane(int t, const int *__restrict__ tile_off, int G,
                                              const int *__restrict__ grp_cell,
                                              const int *__restrict__ cell_run,
                                              const int *__restrict__ run_start,
                                              const int *__restrict__ point_cell) {
    TileLane L;
    const int k = tile_group(tile_off, G, t);
    L.gc0 = grp_cell[k];
    L.gc1 = grp_cell[k + 1];
    L.r = cell_run[L.gc0] + (t - tile_off[k]) * kTile + __lane_id();
    L.active = L.r < cell_run[L.gc1];
    L.i = L.active ? run_start[L.r] : 0;
    L.cl = L.active ? point_cell[L.i] : L.gc0;
    return L;
}

// cell_in_window for a group: the window of the last dimension spans
// [g0[d-1] - rad, ghi + rad] (ghi = last coordinate of the group's last cell).
template <int D>
__device__ __forceinline__ bool cell_in_group_window(const int *__restrict__ cell_g, int n, int c,
                                                     const int *g0, int od, int rad, int ghi,
                                                     int *gc, bool *stop) {
#pragma unroll
    for (int l = 0; l < D; l++) gc[l] = cell_g[(long long)l * n + c];
    const int hi_od = od == D - 1 ? ghi : select_dim<D>(g0, od);
    *stop = od < D && select_dim<D>(gc, od) > hi_od + rad;
    bool in = true;
#pragma unroll
    for (int l = 0; l < D; l++) {
        const int hi = l == D - 1 ? ghi : g0[l];
        if (l > od && (gc[l] - hi > rad || g0[l] - gc[l] > rad)) in = false;
    }
    return in && !*stop;
}

// Bitwise OR of v over the wavefront.
__device__ __forceinline__ unsigned wave_or(unsigned v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v |= (unsigned)__shfl_xor((int)v, o, kWave);
    return v;
}

// Classifies a sub-cell for a lane at x against threshold thr (thr_in =
// thr * (1 - 64 * 2^-24), thr_out = thr * (1 + 64 * 2^-24)): 1 if every
// point of it has FP32 squared distance <= thr, 0 if none has, 2 otherwise.
// The box is the bounding box of the sub-cell's points (smin / smax); this
// FP32 distance to the box and the reference's FP32 distance of any point in
// it are each within (d + 2) * 2^-24 relative of their exact values, so for
// d <= 20 the margin of 64 * 2^-24 covers both.
template <int D>
__device__ __forceinline__ int sub_class_box(const float *blo, const float *bhi, const float *x,
                                             float thr_in, float thr_out) {
    static_assert(2 * D + 4 < 64, "classification margin");
    float mn = 0.f, mx = 0.f;
#pragma unroll
    for (int l = 0; l < D; l++) {
        const float lo = blo[l], hi = bhi[l];
        const float ta = lo - x[l], tb = hi - x[l];
        const float a = ta * ta, b = tb * tb;
        mx += fmaxf(a, b);
        mn += x[l] < lo ? a : (x[l] > hi ? b : 0.f);
    }
    if (mx <= thr_in) return 1;
    if (mn >= thr_out) return 0;
    return 2;
}

// The boxes of sub-cells s0 .. s0 + ns - 1 (ns <= 64) into LDS, box k in
// src[k] (lower corner in x, upper in sv), so that every lane reads them as
// broadcasts instead of loading them one after another.
template <int D>
__device__ __forceinline__ void stage_boxes(const unsigned *__restrict__ smin,
                                            const unsigned *__restrict__ smax, int n, int s0,
                                            int ns, SrcPt<D> *src) {
    const int lane = __lane_id();
    if (lane < ns) {
#pragma unroll
        for (int l = 0; l < D; l++) {
            src[lane].x[l] = ord_val(smin[(long long)l * n + s0 + lane]);
            src[lane].sv[l] = ord_val(smax[(long long)l * n + s0 + lane]);
        }
    }
    wave_sync();
}

// Run of index q in a streamed range: runs [r0, r0 + total) if smask is 0,
// else the runs of the sub-cells s0 + k of the bits k of smask, in order;
// -1 past the end.
__device__ __forceinline__ int stream_run(int q, int total, int r0, int s0, unsigned smask,
                                          const int *__restrict__ sub_run) {
    if (!smask) return q < total ? r0 + q : -1;
    int before = 0, rr = -1;
    for (unsigned mm = smask; mm; mm &= mm - 1) {
        const int k = __builtin_ctz(mm);
        const int a = sub_run[s0 + k], b = sub_run[s0 + k + 1];
        if (q >= before && q < before + (b - a)) rr = a + q - before;
        before += b - a;
    }
    return rr;
}

// Runs in a streamed range.
__device__ __forceinline__ int stream_total(int r0, int r1, int s0, unsigned smask,
                                            const int *__restrict__ sub_run) {
    if (!smask) return r1 - r0;
    int total = 0;
    for (unsigned mm = smask; mm; mm &= mm - 1) {
        const int k = __builtin_ctz(mm);
        total += sub_run[s0 + k + 1] - sub_run[s0 + k];
    }
    return total;
}

// Calls f(a, b) for the maximal stretches of runs [a, b) of a streamed range, in
// order.
template <typename Fn>
__device__ __forceinline__ void each_stretch(int r0, int r1, int s0, unsigned smask,
                                             const int *__restrict__ sub_run, Fn &&f) {
    if (!smask) {
        f(r0, r1);
        return;
    }
    for (unsigned long long mm = smask; mm;) {
        const int k = __builtin_ctzll(mm), len = __builtin_ctzll(~(mm >> k));
        f(__builtin_amdgcn_readfirstlane(sub_run[s0 + k]),
          __builtin_amdgcn_readfirstlane(sub_run[s0 + k + len]));
        mm &= ~(((1ull << len) - 1) << k);
    }
}

// Notes runs [lo, hi) of a streamed range (counted from its start, at most 17
// stretches) for the lanes of mask.
template <int D>
__device__ __forceinline__ void stream_add(Stream<D> &sm, int lo, int hi, int r0, int r1, int s0,
                                           unsigned smask, unsigned long long mask,
                                           const int *__restrict__ sub_run,
                                           bool count_near = false) {
    int before = 0;
    each_stretch(r0, r1, s0, smask, sub_run, [&](int a, int b) {
        const int ca = max(a, a + lo - before), cb = min(b, a + hi - before);
        before += b - a;
        if (ca < cb) sm.add(ca, cb, mask, count_near);
    });
}

// One chunk of a streamed range: runs [base, base + 64) of it go through
// LDS (each lane loads one run and computes sin v and cos v - 1 of its
// offset v from the anchor a0); lanes with `acc` test each run against eps
// and accumulate it, weighted by its length (one rounding per run instead of
// one per point).
template <int D>
__device__ __forceinline__ void stream_chunk(int base, int total, int r0, int s0, unsigned smask,
                                             const int *__restrict__ sub_run,
                                             const int *__restrict__ run_start,
                                             const float *__restrict__ Xs, int n,
                                             const float (&a0)[D], const float (&x)[D],
                                             float thr, bool acc, bool any_acc, SrcPt<D> *src,
                                             int *len, float (&ssv)[D], float (&scm)[D],
                                             int &m_part) {
    const int lane = __lane_id();
    const int rr = stream_run(base + lane, total, r0, s0, smask, sub_run);
    int my_len = 1;
    if (rr >= 0) {
        const int j = run_start[rr];
        my_len = run_start[rr + 1] - j;
        len[lane] = my_len;
#pragma unroll
        for (int l = 0; l < D; l++) {
            const float xq = Xs[(long long)l * n + j];
            src[lane].x[l] = xq;
            if (any_acc) sincosm1_small(xq - a0[l], src[lane].sv[l], src[lane].cv[l]);
        }
    }
    const bool multi = __any(my_len > 1);
    wave_sync();
    const int m = min(kWave, total - base);
    if (acc && !multi) {
        // single-point runs: four sources per step so their LDS reads overlap
        int k = 0;
        for (; k + 4 <= m; k += 4) {
            float sq[4];
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                float qx[D];
#pragma unroll
                for (int l = 0; l < D; l++) qx[l] = src[k + jj].x[l];
                sq[jj] = 0.f;
#pragma unroll
                for (int l = 0; l < D; l++) {
                    const float df = x[l] - qx[l];
                    sq[jj] += df * df;
                }
            }
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                if (sq[jj] <= thr) {
#pragma unroll
                    for (int l = 0; l < D; l++) {
                        ssv[l] += src[k + jj].sv[l];
                        scm[l] += src[k + jj].cv[l];
                    }
                    m_part += 1;
                }
            }
        }
        for (; k < m; k++) {
            const SrcPt<D> &qq = src[k];
            float sq = 0.f;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float df = x[l] - qq.x[l];
                sq += df * df;
            }
            if (sq <= thr) {
#pragma unroll
                for (int l = 0; l < D; l++) {
                    ssv[l] += qq.sv[l];
                    scm[l] += qq.cv[l];
                }
                m_part += 1;
            }
        }
    } else if (acc) {
        for (int k = 0; k < m; k++) {
            const SrcPt<D> &qq = src[k];
            float sq = 0.f;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float df = x[l] - qq.x[l];
                sq += df * df;
            }
            if (sq <= thr) {
                const int lk = len[k];
                const float w = (float)lk;  // of 2^24 points on within 2^-24; the count is exact
#pragma unroll
                for (int l = 0; l < D; l++) {
                    const float a = w * qq.sv[l];
                    const float b = w * qq.cv[l];
                    ssv[l] += a;
                    scm[l] += b;
                }
                m_part += lk;
            }
        }
    }
    wave_sync();
}

// Heavy ranges are summed in fixed point (2^-30 units, int64): integer
// additions commute, so a run's sums do not depend on which wavefront adds
// which unit, or in what order.  |sum| <= 2n <= 2^31 keeps within 2^61.
constexpr double kFix = 0x1p30;

__device__ __forceinline__ unsigned long long to_fix(float v) {
    return (unsigned long long)__double2ll_rn((double)v * kFix);
}

__device__ __forceinline__ float from_fix(long long v) { return (float)((double)v / kFix); }

template <int D>
__device__ __forceinline__ void add_fixed(long long *__restrict__ hacc, int n, int r,
                                          const float (&ps)[D], const float (&pc)[D], int pm) {
    unsigned long long *h = (unsigned long long *)hacc;
#pragma unroll
    for (int l = 0; l < D; l++) {
        atomicAdd(h + (long long)l * n + r, to_fix(ps[l]));
        atomicAdd(h + (long long)(D + l) * n + r, to_fix(pc[l]));
    }
    atomicAdd(h + (long long)(2 * D) * n + r, (unsigned long long)(long long)pm);
}

// The tile's per-lane setup: position (the anchor for lanes without a run),
// anchor a0 (tile_anchor) and sin / cos of u = x - a0.
template <int D>
__device__ __forceinline__ void tile_setup(const TileLane &tl, const float *__restrict__ Xs,
                                           const int *__restrict__ cell_g, const Geo &g,
                                           int (&g0)[D], float (&a0)[D], float (&x)[D],
                                           float (&su)[D], float (&cu)[D]) {
    const int n = g.n;
#pragma unroll
    for (int l = 0; l < D; l++) {
        g0[l] = cell_g[(long long)l * n + tl.gc0];
        a0[l] = tile_anchor(g0[l], l, g);
        x[l] = tl.active ? Xs[(long long)l * n + tl.i] : a0[l];
        sincos_small(x[l] - a0[l], su[l], cu[l]);
    }
}

// Final step of a run's update (EGG_SynC.cu:701-709): new position into
// rres, diagnostics; returns the local-sync test.
template <int D>
__device__ __forceinline__ bool finish_run(const float (&x)[D], const float (&su)[D],
                                           const float (&cu)[D], const float (&sum)[D],
                                           const float (&ssv)[D], const float (&scm)[D], int N,
                                           int m_part, int half, bool border, int own, int n,
                                           int r, float *__restrict__ rres,
                                           int *__restrict__ rdbg) {
    N += m_part;
    float xo[D];
#pragma unroll
    for (int l = 0; l < D; l++) {
        const float p1 = ssv[l] * cu[l];
        const float p2 = ((float)m_part + scm[l]) * su[l];
        const float sml = p1 - p2;
        float tt = sum[l] + sml;
        tt = tt / (float)N;
        xo[l] = x[l] + tt;
    }
    const bool synced = !((!border && N != own) || (border && N != half));
#pragma unroll
    for (int l = 0; l < D; l++) rres[(long long)l * n + r] = xo[l];
    if (rdbg) {
        rdbg[4 * (long long)r + 0] = N;
        rdbg[4 * (long long)r + 1] = half;
        rdbg[4 * (long long)r + 2] = border ? 1 : 0;
        rdbg[4 * (long long)r + 3] = synced ? 1 : 0;
    }
    return synced;
}

// The matrix path (egg_stream.h) serves up to kStreamMaxD dimensions and n < 2^24.
constexpr int kStreamMaxD = 5;
static_assert(kStreamMaxD <= kHeavyMaxD, "k_update_dense defers heavy ranges at every d");

// A wavefront's LDS in k_update_heavy: sources of the scalar paths, or the matrix
// path's chunk.
template <int D, bool MM>
struct TileLds {
    union {
        SrcPt<D> src[kWave];
        std::conditional_t<MM, StreamLds<D>, int> stream;
    };
    int len[kWave];
};

// kernel_itr_grid_STAD5_5_1 (EGG_SynC.cu:551-763).  Per lane: full cells add
// the cell totals (EGG_SynC.cu:648-663); partial cells are streamed through
// LDS in chunks of 64 runs -- each lane loads one run and computes sin v and
// cos v - 1 of v = x_q - a0 (a0 = the tile's anchor, near the tile's cells) --
// and every lane reads each run as a broadcast and, for runs within eps,
// accumulates sin v and cos v - 1 times the run's length.  At the end of
// the tile, sum_q sin(x_q - x) = cos u * sum sin v - sin u * (m + sum (cos v - 1)),
// u = x - a0, m = number of such points.  All angles stay within a few cell
// sides of the anchor, and both sums grow like the sum of sin(x_q - x) does,
// so the result keeps the accuracy of a direct sum of sinf(x_q - x).  Border
// lanes count their eps/2-neighbours in other full cells from the same
// chunks (EGG_SynC.cu:666-681).
// This form serves more than kStreamMaxD dimensions and n >= 2^24; k_update_dense
// the others.
template <int D>
__global__ __launch_bounds__(kBlock) void k_update_tile(
    const float *__restrict__ Xs, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const float *__restrict__ Ts, const float *__restrict__ Tc,
    const int *__restrict__ ob, const int *__restrict__ oe, const int *__restrict__ run_start,
    const int *__restrict__ cell_run, const int *__restrict__ grp_cell,
    const int *__restrict__ point_cell, const int *__restrict__ tile_off,
    const int *__restrict__ cell_sub, const int *__restrict__ sub_start,
    const unsigned *__restrict__ smin, const unsigned *__restrict__ smax,
    const int *__restrict__ sub_run, const float *__restrict__ TsS,
    const float *__restrict__ TcS, float *__restrict__ rres, int *__restrict__ rdbg,
    long long *__restrict__ hacc,
    HeavyDesc *__restrict__ hdesc, int *__restrict__ dtiles, int *__restrict__ dsave, Geo g,
    DevState *st) {
    if (st->done) return;
    // heavy ranges go to k_update_heavy only up to kHeavyMaxD dimensions
    // (the deferral code costs registers)
    constexpr bool kDefer = D <= kHeavyMaxD;
    __shared__ SrcPt<D> s_src[kBlock / kWave][kWave];
    __shared__ int s_len[kBlock / kWave][kWave];
    const int n = g.n, R = g.R, od = g.od;
    const int G = st->G, T = st->TU;
    const float thr = g.thr_eps, thr_half = g.thr_half;
    // sub-cell classification bounds (sub_class); their own rounding keeps a
    // margin of at least 63 * 2^-24
    const float thr_in = thr * (1.0f - 64.0f * 0x1p-24f);
    const float thr_out = thr * (1.0f + 64.0f * 0x1p-24f);
    const float thr_half_in = thr_half * (1.0f - 64.0f * 0x1p-24f);
    const float thr_half_out = thr_half * (1.0f + 64.0f * 0x1p-24f);
    const int lane = __lane_id();
    SrcPt<D> *src = s_src[threadIdx.x / kWave];
    int *len = s_len[threadIdx.x / kWave];
    const int *cg_od = cell_g + (long long)od * n;
    bool unsynced = false;
    // tiles of the non-sparse groups only (tile_off: their scan); sparse
    // groups go to k_update_pairs
    for (int t = wave_index(); t < T; t = wave_count() + next_tile(&st->tile_next)) {
        const TileLane tl = tile_lane(t, tile_off, G, grp_cell, cell_run, run_start, point_cell);
        const int cl = tl.cl, r = tl.r;
        const bool active = tl.active;
        const int own = cell_start[cl + 1] - cell_start[cl];
        const int ghi = cell_g[(long long)(D - 1) * n + tl.gc1 - 1];
        float x[D], a0[D], sx[D], cx[D], su[D], cu[D], sum[D], ssv[D], scm[D];
        int g0[D];
        tile_setup<D>(tl, Xs, cell_g, g, g0, a0, x, su, cu);
        bool border = false;
#pragma unroll
        for (int l = 0; l < D; l++) {
            sum[l] = 0.f;
            ssv[l] = 0.f;
            scm[l] = 0.f;
            sx[l] = sinf(x[l]);
            cx[l] = cosf(x[l]);
            border |= active && on_border(x[l], g.cs);
        }
        const int g0od = select_dim<D>(g0, od);
        int N = 0, half = 0, m_part = 0;
        bool deferred = false;  // some range went to k_update_heavy
        int cur_c = 0;          // candidate cell of the range being streamed
        auto defer_tile = [&]() __attribute__((always_inline)) {
            if (!deferred) {
                deferred = true;
                if (active) {
#pragma unroll
                    for (int k = 0; k < 2 * D + 2; k++) hacc[(long long)k * n + r] = 0;
                }
                if (lane == 0) dtiles[atomicAdd(&st->ndt, 1)] = t;
            }
        };
        // queues a heavy range; false if the queue is full
        auto queue_range = [&](int r0, int s0, unsigned smask, int total,
                               int half_kind) __attribute__((always_inline)) {
            const int nunits = (total + kUnitRuns - 1) / kUnitRuns;
            unsigned long long old = 0;
            if (lane == 0)
                old = atomicAdd(&st->heavy_pack, (1ull << 32) | (unsigned long long)nunits);
            const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)old);
            const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(old >> 32));
            if (hi >= (unsigned)kHeavyCap) return false;
            if (lane == 0)
                hdesc[hi] = HeavyDesc{t, cur_c, r0, s0, smask, total, (int)lo, nunits, half_kind};
            return true;
        };
        // Streams a range of runs (stream_run) through LDS, 64 per chunk.  A
        // range of kHeavyRuns runs or more is queued for k_update_heavy
        // instead, in units any wavefront can take; the tile's runs then
        // finish in k_update_finish.
        auto scan_runs = [&](int r0, int r1, int s0, unsigned smask,
                             bool acc) __attribute__((always_inline)) {
            const bool any_acc = __any(acc);
            const int total = stream_total(r0, r1, s0, smask, sub_run);
            const bool heavy = kDefer && hacc && total >= kHeavyRuns;
            if (heavy) {
                defer_tile();
                // the float sums so far go to hacc now, so that what follows
                // does not depend on who sums the range (all sums are additive)
                if (active) add_fixed<D>(hacc, n, r, ssv, scm, m_part);
#pragma unroll
                for (int l = 0; l < D; l++) ssv[l] = scm[l] = 0.f;
                m_part = 0;
                if (queue_range(r0, s0, smask, total, 0)) return;
                // queue full: this wavefront sums the range itself, unit by
                // unit in fixed point, as k_update_heavy would
            }
            for (int base = 0; base < total; base += kWave) {
                stream_chunk<D>(base, total, r0, s0, smask, sub_run, run_start, Xs, n, a0, x,
                                thr, acc, any_acc, src, len, ssv, scm, m_part);
                if (heavy && (base + kWave == total || (base + kWave) % kUnitRuns == 0 ||
                              base + kWave > total)) {
                    if (active) add_fixed<D>(hacc, n, r, ssv, scm, m_part);
#pragma unroll
                    for (int l = 0; l < D; l++) ssv[l] = scm[l] = 0.f;
                    m_part = 0;
                }
            }
        };
        // Lanes with `hcnt` count the points of a range of runs (stream_run)
        // within eps/2.
        auto half_scan = [&](int r0, int r1, int s0, unsigned smask,
                             bool hcnt) __attribute__((always_inline)) {
            const int total = stream_total(r0, r1, s0, smask, sub_run);
            if (kDefer && hacc && total >= kHeavyRuns) {
                // a count: exact in any order, so k_update_heavy may take it
                defer_tile();
                if (queue_range(r0, s0, smask, total, 1)) return;
            }
            for (int base = 0; base < total; base += kWave) {
                const int rr = stream_run(base + lane, total, r0, s0, smask, sub_run);
                if (rr >= 0) {
                    const int j = run_start[rr];
                    len[lane] = run_start[rr + 1] - j;
#pragma unroll
                    for (int l = 0; l < D; l++) src[lane].x[l] = Xs[(long long)l * n + j];
                }
                wave_sync();
                const int m = min(kWave, total - base);
                if (hcnt) {
                    for (int k = 0; k < m; k++) {
                        float sq = 0.f;
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            const float df = x[l] - src[k].x[l];
                            sq += df * df;
                        }
                        if (sq <= thr_half) half += len[k];
                    }
                }
                wave_sync();
            }
        };
        walk_columns<D>(g0, R, g, ob, oe, [&](int cb, const int ce) {
            if (od < D) cb = column_lower(cg_od, cb, ce, g0od - R - 1);
            for (int c = cb; c < ce; c++) {
                int gc[D];
                bool stop;
                const bool in =
                    cell_in_group_window<D>(cell_g, n, c, g0, od, R + 1, ghi, gc, &stop);
                if (stop) break;
                if (!in) continue;
                float sm, lg;
                box_dist<D>(gc, x, g.cs, sm, lg);
                const bool full = active && lg <= thr;
                const bool part = active && !full && sm <= thr;
                if (full) {
#pragma unroll
                    for (int l = 0; l < D; l++) {
                        const float a = Ts[(long long)l * n + c] * cx[l];
                        const float b = Tc[(long long)l * n + c] * sx[l];
                        const float tt = a - b;
                        sum[l] += tt;
                    }
                    const int cnt = cell_start[c + 1] - cell_start[c];
                    N += cnt;
                    if (border && c == cl) half += cnt;
                }
                const bool need_half = full && border && c != cl;
                const bool any_part = __any(part), any_half = __any(need_half);
                if (!any_part && !any_half) continue;
                if (any_half) {
                    cur_c = c;
                    // eps/2-neighbours in another full cell: sub-cells wholly
                    // within eps/2 of a lane count whole, those straddling
                    // eps/2 for some lane are streamed for the wavefront
                    const int hs0 = cell_sub[c], hns = cell_sub[c + 1] - hs0;
                    if (g.sub_bits && hns <= 32) {
                        unsigned hin = 0, hst = 0;
                        stage_boxes<D>(smin, smax, n, hs0, hns, src);
                        if (need_half) {
                            for (int k = 0; k < hns; k++) {
                                const int cls = sub_class_box<D>(src[k].x, src[k].sv, x,
                                                                 thr_half_in, thr_half_out);
                                if (cls == 1) hin |= 1u << k;
                                else if (cls == 2) hst |= 1u << k;
                            }
                        }
                        wave_sync();
                        const unsigned hu = wave_or(hst);
                        const unsigned ht = hin & ~hu;
                        for (unsigned mm = wave_or(ht); mm; mm &= mm - 1) {
                            const int k = __builtin_ctz(mm);
                            if ((ht >> k) & 1u) half += sub_start[hs0 + k + 1] - sub_start[hs0 + k];
                        }
                        if (hu) half_scan(0, 0, hs0, hu, need_half);
                    } else {
                        half_scan(cell_run[c], cell_run[c + 1], 0, 0u, need_half);
                    }
                }
                if (!any_part) continue;
                const int s0 = cell_sub[c], ns = cell_sub[c + 1] - s0;
                unsigned umask = 0;
                if (g.sub_bits && ns <= 32) {
                    // sub-cells of a partial cell: each lane classifies them
                    // (wholly within eps / wholly beyond / straddling); the
                    // sub-cells some lane straddles are streamed once for the
                    // wavefront and tested point by point by every lane with
                    // a partial cell; other sub-cells wholly within eps add
                    // their totals
                    unsigned imask = 0, smask = 0;
                    stage_boxes<D>(smin, smax, n, s0, ns, src);
                    if (part) {
                        for (int k = 0; k < ns; k++) {
                            const int cls =
                                sub_class_box<D>(src[k].x, src[k].sv, x, thr_in, thr_out);
                            if (cls == 1) imask |= 1u << k;
                            else if (cls == 2) smask |= 1u << k;
                        }
                    }
                    wave_sync();
                    umask = wave_or(smask);
                    const unsigned tmask = imask & ~umask;
                    for (unsigned mm = wave_or(tmask); mm; mm &= mm - 1) {
                        const int k = __builtin_ctz(mm);
                        const int sc = s0 + k;
                        if ((tmask >> k) & 1u) {
#pragma unroll
                            for (int l = 0; l < D; l++) {
                                const float a = TsS[(long long)l * n + sc] * cx[l];
                                const float b = TcS[(long long)l * n + sc] * sx[l];
                                const float tt = a - b;
                                sum[l] += tt;
                            }
                            N += sub_start[sc + 1] - sub_start[sc];
                        }
                    }
                    if (!umask) continue;
                }
                cur_c = c;
                scan_runs(cell_run[c], cell_run[c + 1], s0, umask, part);
            }
        });
        if (deferred) {
            // the sums so far wait for the heavy ranges: full-cell totals in
            // rres, N / half / border in dsave, streamed sums into hacc
            if (active) {
#pragma unroll
                for (int l = 0; l < D; l++) rres[(long long)l * n + r] = sum[l];
                dsave[4 * (long long)r + 0] = N;
                dsave[4 * (long long)r + 1] = half;
                dsave[4 * (long long)r + 2] = border ? 1 : 0;
                add_fixed<D>(hacc, n, r, ssv, scm, m_part);
            }
            continue;
        }
        if (active) {
            if (!finish_run<D>(x, su, cu, sum, ssv, scm, N, m_part, half, border, own, n, r, rres,
                               rdbg))
                unsynced = true;
        }
    }
    if (__any(unsynced) && lane == 0) atomicAnd(&st->flag, 0);
}

// v, without the compiler's knowledge of it: keeps addresses made from it from
// being formed ahead of a rare branch, and held in registers until then.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A wavefront's LDS in k_update_dense: the records of a batch of cells, those of the
// sub-cells of the next few of them, and, not at the same time, boxes for the eps/2
// counts or the matrix path's chunk.
template <int D>
struct DenseLds {
    struct Cell {
        float lo[D], hi[D], ts[D], tc[D];
        int c, pts, sub0, nsub, run0, run1;
    } cell[kWave];
    struct Box {
        float lo[D], hi[D], ts[D], tc[D];
        int pts, run0;
    };
    Box box[kWave];
    union {
        SrcPt<D> src[kWave];
        StreamLds<D> stream;
    };
};

// k_update_tile for up to kStreamMaxD dimensions and n < 2^24: the same tests and
// the same sums in the same order, arranged for the time a tile takes by itself (a
// pass ends with its densest tile) and for the VALU.
//   Candidate cells come 64 at a time.  A lane finds the window of one column by
// itself, a lane of the next step takes one cell, loads its record and tests it
// against the box of the tile's targets: cells beyond eps of the whole box are
// dropped and cells within eps of all of it are marked, by the formula each target
// would use (FP32 rounding is monotone, so the box bounds every target's result).
// The rest of the work on a cell reads its record from LDS: no global load is waited
// for.  Sub-cells are treated alike, their records loaded a cell ahead.
//   Streamed ranges are noted and summed together on the matrix cores (Stream), from
// one place in the code: the loop over the cells returns to its head for it.
// Bound by the VALU: per cell some 250 instructions of tests, per 8 sources 37 beside
// the matrix instructions.  Up to d = 3 held to three wavefronts a SIMD (165 registers
// at d = 3, and 171 spilled scalar ones): with four the spills cost more than the
// fourth hides (100 ms against 81 in one state of it).  At d = 4 and 5 a workgroup's
// 60 and 74 KB of LDS leave a CU two of them, two wavefronts a SIMD (193 and 207
// registers).
// Against k_update_tile (which had the sums alone on the matrix cores), whole solve,
// n = 1,000,000, d = 3, eps = 0.02: 88 -> 70 ms; one pass of n = 100,003, d = 3: 4.0 ->
// 3.4 ms; n = 100,000, d = 2: 5.1 -> 3.9; d = 5 passes of a batch 116 -> 75 us.
template <int D>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(D <= 3 ? 3 : 2)))
void k_update_dense(GridBufs b, int *__restrict__ rdbg, Geo g, DevState *st) {
    if (st->done) return;
    __shared__ DenseLds<D> s_lds[kBlock / kWave];
    DenseLds<D> &lds = s_lds[threadIdx.x / kWave];
    const float *__restrict__ Xs = b.Xs;
    const int *__restrict__ run_start = b.run_start;
    const int n = g.n, R = g.R, od = g.od, lane = __lane_id();
    const int G = st->G, T = st->TU;
    const float thr = g.thr_eps, thr_half = g.thr_half;
    const float thr_in = thr * (1.0f - 64.0f * 0x1p-24f);
    const float thr_out = thr * (1.0f + 64.0f * 0x1p-24f);
    const float thr_half_in = thr_half * (1.0f - 64.0f * 0x1p-24f);
    const float thr_half_out = thr_half * (1.0f + 64.0f * 0x1p-24f);
    const int *cg_od = b.cell_g + (long long)od * n;
    bool unsynced = false;
    for (int t = wave_index(); t < T; t = wave_count() + next_tile(&st->tile_next)) {
        const TileLane tl =
            tile_lane(t, b.utile_off, G, b.grp_cell, b.cell_run, run_start, b.point_cell);
        const int cl = tl.cl, r = tl.r;
        const bool active = tl.active;
        float x[D], sx[D], cx[D], sum[D];
        float tlo[D], thi[D], ux = 0.f;  // box of the targets, bound on |u_x|^2 (Stream)
        int g0[D];
        bool border = false, nan = false;
#pragma unroll
        for (int l = 0; l < D; l++) {
            g0[l] = __builtin_amdgcn_readfirstlane(b.cell_g[(long long)l * n + tl.gc0]);
            x[l] = active ? Xs[(long long)l * n + tl.i] : tile_anchor(g0[l], l, g);
            sum[l] = 0.f;
            sx[l] = sinf(x[l]);
            cx[l] = cosf(x[l]);
            border |= active && on_border(x[l], g.cs);
            nan |= active && !(x[l] == x[l]);
            float lo = active ? x[l] : INFINITY, hi = active ? x[l] : -INFINITY;
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) {
                lo = fminf(lo, __shfl_xor(lo, o, kWave));
                hi = fmaxf(hi, __shfl_xor(hi, o, kWave));
            }
            tlo[l] = uniform(lo);
            thi[l] = uniform(hi);
            const float ctr = cell_mid(g0[l], g.cs);
            const float far = fmaxf(fabsf(lo - ctr), fabsf(hi - ctr));
            ux += far * far;
        }
        if (__any(nan)) {  // in no box: let nothing be decided by it
#pragma unroll
            for (int l = 0; l < D; l++) {
                tlo[l] = -INFINITY;
                thi[l] = INFINITY;
            }
        }
        Stream<D> sm;
        sm.init(ux, g);
        int N = 0, half = 0;
        bool deferred = false;  // some range went to k_update_heavy
        auto defer_tile = [&]() __attribute__((always_inline)) {
            if (!deferred) {
                deferred = true;
                if (active) {
                    const int hr = opaque(r);
#pragma unroll
                    for (int k = 0; k < 2 * D + 2; k++) b.hacc[(long long)k * n + hr] = 0;
                }
                if (lane == 0) b.dtiles[atomicAdd(&st->ndt, 1)] = t;
            }
        };
        // queues a heavy range of cell c; false if the queue is full
        auto queue_range = [&](int c, int r0, int s0, unsigned smask, int total,
                               int half_kind) __attribute__((always_inline)) {
            const int nunits = (total + kUnitRuns - 1) / kUnitRuns;
            unsigned long long old = 0;
            if (lane == 0)
                old = atomicAdd(&st->heavy_pack, (1ull << 32) | (unsigned long long)nunits);
            const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)old);
            const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(old >> 32));
            const bool queued = hi < (unsigned)kHeavyCap;
            if (queued && lane == 0)
                b.hdesc[hi] = HeavyDesc{t, c, r0, s0, smask, total, (int)lo, nunits, half_kind};
            // one lane's branch must not make the loop's state look like the lanes' own
            return __builtin_amdgcn_readfirstlane(queued) != 0;
        };
        // a heavy range of streamed runs waiting for the loop's head: next unit, -1
        // before it was offered to the queue
        bool heavy = false;
        int hu = 0, hc = 0, hr0 = 0, hr1 = 0, hs0 = 0;
        unsigned hmask = 0;
        unsigned long long haccs = 0;

        // the columns of the box [g0 - R, g0 + R]^od inside the grid, dim 0 fastest,
        // 64 at a time: lane k's first cell in the window and the cells before it
        int rows = 1, row0 = 0, ccell = 0, coff = 0, ctotal = 0, f0 = 0;
        int ghi[D];  // the tile's group: coordinates g0 .. ghi
#pragma unroll
        for (int l = 0; l < D; l++) {
            ghi[l] = l < D - 1 ? g0[l] : b.cell_g[(long long)l * n + tl.gc1 - 1];
            if (l < od) rows *= min(g.w - 1, g0[l] + R) - max(0, g0[l] - R) + 1;
        }
        const int win_lo = select_dim<D>(g0, od) - R - 1, win_hi = select_dim<D>(ghi, od) + R + 1;
        unsigned long long keep = 0, all_full = 0;  // of the cells in lds.cell
        // lane k: sub-cells of cell k if they are to be looked at, and those before
        int scnt = 0, soff = 0;
        // cells whose sub-cells are in lds.box, from place sbase on; of those, by
        // the targets' box: wholly within eps, straddling it
        unsigned long long staged = 0, sub_in = 0, sub_mixed = 0;
        int sbase = 0;
        auto stage_subs = [&](int k) __attribute__((always_inline)) {
            sbase = __builtin_amdgcn_readlane(soff, k);
            staged = __ballot(scnt > 0 && soff >= sbase && soff + scnt <= sbase + kWave);
            const int i = sbase + lane;
            int q = 0;  // the cell of place i: the last that starts at or before it
#pragma unroll
            for (int st = kWave / 2; st > 0; st >>= 1) q += __shfl(soff, q + st) <= i ? st : 0;
            const int at = i - __shfl(soff, q);
            int cls = 0;
            if (at < __shfl(scnt, q) && (staged >> q & 1)) {
                typename DenseLds<D>::Box sub;
                const int s = lds.cell[q].sub0 + at;
                float mx = 0.f, mn = 0.f;
#pragma unroll
                for (int l = 0; l < D; l++) {
                    sub.lo[l] = ord_val(b.smin[(long long)l * n + s]);
                    sub.hi[l] = ord_val(b.smax[(long long)l * n + s]);
                    sub.ts[l] = b.TsS[(long long)l * n + s];
                    sub.tc[l] = b.TcS[(long long)l * n + s];
                    const float dl = sub.lo[l] - thi[l], dh = sub.hi[l] - tlo[l];
                    const float el = sub.lo[l] - tlo[l], eh = sub.hi[l] - thi[l];
                    mx += fmaxf(fmaxf(dl * dl, dh * dh), fmaxf(el * el, eh * eh));
                    mn += thi[l] < sub.lo[l] ? dl * dl : (tlo[l] > sub.hi[l] ? dh * dh : 0.f);
                }
                sub.pts = b.sub_start[s + 1] - b.sub_start[s];
                sub.run0 = b.sub_run[s];
                lds.box[lane] = sub;
                cls = mx <= thr_in ? 1 : (mn >= thr_out ? 0 : 2);
            }
            sub_in = __ballot(cls == 1);
            sub_mixed = __ballot(cls == 2);
            wave_sync();
        };
        // Lanes with `hcnt` count the points of a range of runs (stream_run) of cell
        // c within eps/2.
        auto half_scan = [&](int c, int r0, int r1, int s0, unsigned smask,
                             bool hcnt) __attribute__((always_inline)) {
            const int total = stream_total(r0, r1, s0, smask, b.sub_run);
            if (total >= kHeavyRuns) {
                // a count: exact in any order, so k_update_heavy may take it
                defer_tile();
                if (queue_range(c, r0, s0, smask, total, 1)) return;
            }
            stream_add<D>(sm, 0, total, r0, r1, s0, smask, __ballot(hcnt), b.sub_run, true);
        };
        for (;;) {
            bool last = false;
            if (!keep && !heavy) {
                if (f0 >= ctotal) {
                    if (row0 < rows) {
                        int rest = row0 + lane, o = 0, cb = 0, ce = 0;
                        const bool on = rest < rows;
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            if (l < od) {
                                const int lo = max(0, g0[l] - R);
                                const int ext = min(g.w - 1, g0[l] + R) - lo + 1;
                                o += (lo + rest % ext) * g.wpow[l];
                                rest /= ext;
                            }
                        }
                        if (on) {
                            cb = b.ob[o];
                            ce = b.oe[o];
                        }
                        if (od < D) {
                            // first cells at or above win_lo, above win_hi
                            int l1 = cb, h1 = ce, l2 = cb, h2 = ce;
                            while (l1 < h1 || l2 < h2) {
                                const int m1 = (l1 + h1) >> 1, m2 = (l2 + h2) >> 1;
                                const int v1 = l1 < h1 ? cg_od[m1] : 0;
                                const int v2 = l2 < h2 ? cg_od[m2] : 0;
                                if (l1 < h1) {
                                    if (v1 < win_lo) l1 = m1 + 1;
                                    else h1 = m1;
                                }
                                if (l2 < h2) {
                                    if (v2 <= win_hi) l2 = m2 + 1;
                                    else h2 = m2;
                                }
                            }
                            cb = l1;
                            ce = max(l1, l2);
                        }
                        const int cnt = ce - cb;
                        const int incl = wave_incl_scan(cnt);
                        ccell = cb;
                        coff = incl - cnt;
                        ctotal = __builtin_amdgcn_readlane(incl, kWave - 1);
                        row0 += kWave;
                        f0 = 0;
                        continue;
                    }
                    last = true;
                } else {
                    const int f = f0 + lane;
                    const bool on = f < ctotal;
                    int q = 0;  // last column that starts at or before f
#pragma unroll
                    for (int s = kWave / 2; s > 0; s >>= 1) q += __shfl(coff, q + s) <= f ? s : 0;
                    const int c = __shfl(ccell, q) + f - __shfl(coff, q);
                    bool in = on, all = on;
                    int nsub = 0;
                    if (on) {
                        typename DenseLds<D>::Cell rec;
                        rec.c = c;
                        const int p0 = b.cell_start[c], s0 = b.cell_sub[c];
                        rec.pts = b.cell_start[c + 1] - p0;
                        rec.sub0 = s0;
                        rec.nsub = nsub = b.cell_sub[c + 1] - s0;
                        rec.run0 = b.cell_run[c];
                        rec.run1 = b.cell_run[c + 1];
                        float near = 0.f, far = 0.f;
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            const int gc = b.cell_g[(long long)l * n + c];
                            rec.ts[l] = b.Ts[(long long)l * n + c];
                            rec.tc[l] = b.Tc[(long long)l * n + c];
                            if (l > od && (gc - ghi[l] > R + 1 || g0[l] - gc > R + 1)) in = false;
                            const float lo = (float)gc * g.cs, hi = (float)(gc + 1) * g.cs;
                            rec.lo[l] = lo;
                            rec.hi[l] = hi;
                            // bounds of box_dist over the targets' box
                            const float dl = lo - thi[l], dh = hi - tlo[l];
                            near += dl > 0.f ? dl * dl : (dh < 0.f ? dh * dh : 0.f);
                            const float el = lo - tlo[l], eh = hi - thi[l];
                            far += fmaxf(fmaxf(dl * dl, dh * dh), fmaxf(el * el, eh * eh));
                        }
                        in = in && !(near > thr);
                        all = far <= thr;
                        lds.cell[lane] = rec;
                    }
                    wave_sync();
                    keep = __ballot(in);
                    all_full = __ballot(all);
                    f0 += kWave;
                    staged = 0;
                    if (!keep) continue;
                    scnt = in && !all && g.sub_bits && nsub <= 32 ? nsub : 0;
                    soff = wave_incl_scan(scnt) - scnt;
                }
            }
            if (last || heavy || __builtin_amdgcn_readfirstlane(sm.nseg) > kWave - 34) {  // a cell adds two ranges
                sm.flush(lds.stream, x, active, g0, g, Xs, run_start);
                if (heavy) {
                    // the float sums so far go to hacc, so that what follows does
                    // not depend on who sums the range (all sums are additive)
                    float ssv[D], scm[D];
#pragma unroll
                    for (int l = 0; l < D; l++) {
                        ssv[l] = sm.sin_sum(l);
                        scm[l] = sm.cos_sum(l);
                    }
                    if (active) add_fixed<D>(b.hacc, n, opaque(r), ssv, scm, sm.count());
                    sm.clear_sums();
                    const int total = stream_total(hr0, hr1, hs0, hmask, b.sub_run);
                    if (hu < 0) {
                        hu = 0;
                        heavy = !queue_range(hc, hr0, hs0, hmask, total, 0);
                    }
                    if (heavy) {
                        // queue full: this wavefront sums the range itself, unit by
                        // unit in fixed point, as k_update_heavy would
                        heavy = hu < total;
                        if (heavy)
                            stream_add<D>(sm, hu, min(total, hu + kUnitRuns), hr0, hr1, hs0,
                                          hmask, haccs, b.sub_run);
                        hu += kUnitRuns;
                    }
                    continue;
                }
                if (last) break;
            }
            const int k = __builtin_ctzll(keep);
            keep &= keep - 1;
            const typename DenseLds<D>::Cell &rec = lds.cell[k];
            bool full = active, part = false;
            if (!(all_full >> k & 1)) {
                float near = 0.f, far = 0.f;  // box_dist
#pragma unroll
                for (int l = 0; l < D; l++) {
                    float lo = rec.lo[l] - x[l], hi = rec.hi[l] - x[l];
                    lo *= lo;
                    hi *= hi;
                    near += lo < hi ? lo : hi;
                    far += lo < hi ? hi : lo;
                }
                full = active && far <= thr;
                part = active && !full && near <= thr;
            }
            const int c = __builtin_amdgcn_readfirstlane(rec.c);
            if (full) {
#pragma unroll
                for (int l = 0; l < D; l++) {
                    const float p = rec.ts[l] * cx[l];
                    const float q = rec.tc[l] * sx[l];
                    const float tt = p - q;
                    sum[l] += tt;
                }
                N += rec.pts;
                if (border && c == cl) half += rec.pts;
            }
            if (all_full >> k & 1 && !__any(border && c != cl)) continue;
            const int s0 = __builtin_amdgcn_readfirstlane(rec.sub0);
            const int ns = __builtin_amdgcn_readfirstlane(rec.nsub);
            const int r0 = __builtin_amdgcn_readfirstlane(rec.run0);
            const int r1 = __builtin_amdgcn_readfirstlane(rec.run1);
            const bool by_subs = g.sub_bits && ns <= 32;
            const bool need_half = full && border && c != cl;
            if (__any(need_half)) {
                // eps/2-neighbours in another full cell: sub-cells wholly
                // within eps/2 of a lane count whole, those straddling
                // eps/2 for some lane are streamed for the wavefront
                if (by_subs) {
                    unsigned hin = 0, hst = 0;
                    stage_boxes<D>(b.smin, b.smax, n, s0, ns, lds.src);
                    if (need_half) {
                        for (int i = 0; i < ns; i++) {
                            const int cls = sub_class_box<D>(lds.src[i].x, lds.src[i].sv, x,
                                                             thr_half_in, thr_half_out);
                            if (cls == 1) hin |= 1u << i;
                            else if (cls == 2) hst |= 1u << i;
                        }
                    }
                    wave_sync();
                    const unsigned hu32 = wave_or(hst);
                    const unsigned ht = hin & ~hu32;
                    for (unsigned mm = wave_or(ht); mm; mm &= mm - 1) {
                        const int i = __builtin_ctz(mm);
                        if ((ht >> i) & 1u) half += b.sub_start[s0 + i + 1] - b.sub_start[s0 + i];
                    }
                    if (hu32) half_scan(c, 0, 0, s0, hu32, need_half);
                } else {
                    half_scan(c, r0, r1, 0, 0u, need_half);
                }
            }
            if (all_full >> k & 1) continue;
            const unsigned long long parts = __ballot(part);
            unsigned umask = 0;
            int at = 0;  // place of the cell's sub-cells in lds.box
            if (parts && by_subs) {
                // sub-cells of a partial cell: wholly within eps, wholly beyond or
                // straddling it, for all targets by their box where that decides, else
                // for each; those some lane straddles are streamed once for the
                // wavefront and tested point by point by every lane with a partial
                // cell; others wholly within eps add their totals
                if (!(staged >> k & 1)) stage_subs(k);
                at = __builtin_amdgcn_readlane(soff, k) - sbase;
                const typename DenseLds<D>::Box *box = lds.box + at;
                const unsigned below = ns < 32 ? (1u << ns) - 1u : ~0u;
                unsigned in_some = (unsigned)(sub_in >> at) & below;
                const unsigned mixed = (unsigned)(sub_mixed >> at) & below;
                unsigned imask = part ? in_some : 0u;
                for (unsigned mm = mixed; mm; mm &= mm - 1) {
                    const int i = __builtin_ctz(mm);
                    const int cl2 = part ? sub_class_box<D>(box[i].lo, box[i].hi, x, thr_in, thr_out)
                                         : 0;
                    if (cl2 == 1) imask |= 1u << i;
                    if (__any(cl2 == 1)) in_some |= 1u << i;
                    if (__any(cl2 == 2)) umask |= 1u << i;
                }
                for (unsigned mm = in_some & ~umask; mm; mm &= mm - 1) {
                    const int i = __builtin_ctz(mm);
                    if ((imask >> i) & 1u) {
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            const float p = box[i].ts[l] * cx[l];
                            const float q = box[i].tc[l] * sx[l];
                            const float tt = p - q;
                            sum[l] += tt;
                        }
                        N += box[i].pts;
                    }
                }
            }
            if (!parts || (by_subs && !umask)) continue;
            if (r1 - r0 >= kHeavyRuns && stream_total(r0, r1, s0, umask, b.sub_run) >= kHeavyRuns) {
                defer_tile();
                heavy = true;
                hu = -1;
                hc = c;
                hr0 = r0;
                hr1 = r1;
                hs0 = s0;
                hmask = umask;
                haccs = parts;
            } else if (!umask) {
                sm.add(r0, r1, parts);
            } else {
                for (unsigned long long mm = umask; mm;) {
                    const int i = __builtin_ctzll(mm), len = __builtin_ctzll(~(mm >> i));
                    sm.add(lds.box[at + i].run0, i + len < ns ? lds.box[at + i + len].run0 : r1,
                           parts);
                    mm &= ~(((1ull << len) - 1) << i);
                }
            }
        }
        float su[D], cu[D], ssv[D], scm[D];
#pragma unroll
        for (int l = 0; l < D; l++) {
            sincos_small(x[l] - tile_anchor(g0[l], l, g), su[l], cu[l]);
            ssv[l] = sm.sin_sum(l);
            scm[l] = sm.cos_sum(l);
        }
        const int m_part = sm.count();
        half += (int)sm.near;
        const int ro = opaque(r);
        if (deferred) {
            // the sums so far wait for the heavy ranges: full-cell totals in
            // rres, N / half / border in dsave, streamed sums into hacc
            if (active) {
#pragma unroll
                for (int l = 0; l < D; l++) b.rres[(long long)l * n + ro] = sum[l];
                b.rdbg[4 * (long long)ro + 0] = N;
                b.rdbg[4 * (long long)ro + 1] = half;
                b.rdbg[4 * (long long)ro + 2] = border ? 1 : 0;
                add_fixed<D>(b.hacc, n, ro, ssv, scm, m_part);
            }
            continue;
        }
        if (active) {
            const int own = b.cell_start[cl + 1] - b.cell_start[cl];
            if (!finish_run<D>(x, su, cu, sum, ssv, scm, N, m_part, half, border, own, n, ro,
                               b.rres, rdbg))
                unsynced = true;
        }
    }
    if (__any(unsynced) && lane == 0) atomicAnd(&st->flag, 0);
}

// Work units of the heavy ranges (kUnitRuns runs each), from a queue over
// all of them: every wavefront rebuilds the tile's lanes, tests the unit's
// runs as the tile kernel would and adds its sums in fixed point.
template <int D, bool MM>
__global__ __launch_bounds__(kBlock) void k_update_heavy(
    const float *__restrict__ Xs, const int *__restrict__ cell_g,
    const int *__restrict__ run_start, const int *__restrict__ cell_run,
    const int *__restrict__ grp_cell, const int *__restrict__ point_cell,
    const int *__restrict__ tile_off, const int *__restrict__ sub_run,
    const HeavyDesc *__restrict__ hdesc, long long *__restrict__ hacc, Geo g, DevState *st) {
    if (st->done) return;
    const int nd = (int)min((unsigned long long)kHeavyCap, st->heavy_pack >> 32);
    if (nd == 0) return;
    __shared__ TileLds<D, MM> s_lds[kBlock / kWave];
    TileLds<D, MM> &lds = s_lds[threadIdx.x / kWave];
    SrcPt<D> *src = lds.src;
    int *len = lds.len;
    const int n = g.n, G = st->G;
    const float thr = g.thr_eps;
    // descriptors k < nd hold consecutive unit ranges in the order of k
    const int end = hdesc[nd - 1].ubase + hdesc[nd - 1].nunits;
    for (int u = wave_index(); u < end; u = wave_count() + next_tile(&st->unit_next)) {
        int lo = 0, hi = nd - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (hdesc[mid].ubase <= u) lo = mid;
            else hi = mid - 1;
        }
        const HeavyDesc hd = hdesc[lo];
        const TileLane tl = tile_lane(hd.t, tile_off, G, grp_cell, cell_run, run_start,
                                      point_cell);
        float x[D], a0[D], su[D], cu[D];
        int g0[D], gc[D];
        tile_setup<D>(tl, Xs, cell_g, g, g0, a0, x, su, cu);
#pragma unroll
        for (int l = 0; l < D; l++) gc[l] = cell_g[(long long)l * n + hd.c];
        float sm, lg;
        box_dist<D>(gc, x, g.cs, sm, lg);
        const int k = u - hd.ubase;
        const int b1 = min(hd.total, (k + 1) * kUnitRuns);
        const bool acc = tl.active && !(lg <= thr) && sm <= thr;
        // border lanes of the tile, a half range's cell full for them and not
        // their own: points within eps/2
        bool border = false;
#pragma unroll
        for (int l = 0; l < D; l++) border |= on_border(x[l], g.cs);
        const bool hcnt = tl.active && lg <= thr && border && hd.c != tl.cl;
        float ps[D], pc[D];
        int pm = 0, cnt = 0;
#pragma unroll
        for (int l = 0; l < D; l++) ps[l] = pc[l] = 0.f;
        if constexpr (MM) {
            float ux = 0.f;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float v = tl.active ? x[l] - cell_mid(g0[l], g.cs) : 0.f;
                ux += v * v;
            }
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) ux = fmaxf(ux, __shfl_xor(ux, o, kWave));
            Stream<D> q;
            q.init(ux, g);
            stream_add<D>(q, k * kUnitRuns, b1, hd.r0, hd.r0 + hd.total, hd.s0, hd.smask,
                          __ballot(hd.half ? hcnt : acc), sub_run, hd.half != 0);
            q.flush(lds.stream, x, tl.active, g0, g, Xs, run_start);
#pragma unroll
            for (int l = 0; l < D; l++) {
                ps[l] = q.sin_sum(l);
                pc[l] = q.cos_sum(l);
            }
            pm = q.count();
            cnt = (int)q.near;
        } else if (hd.half) {
            for (int base = k * kUnitRuns; base < b1; base += kWave) {
                const int rr =
                    stream_run(base + __lane_id(), b1, hd.r0, hd.s0, hd.smask, sub_run);
                if (rr >= 0) {
                    const int j = run_start[rr];
                    len[__lane_id()] = run_start[rr + 1] - j;
#pragma unroll
                    for (int l = 0; l < D; l++) src[__lane_id()].x[l] = Xs[(long long)l * n + j];
                }
                wave_sync();
                const int m = min(kWave, b1 - base);
                if (hcnt) {
                    for (int q = 0; q < m; q++) {
                        float sq = 0.f;
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            const float df = x[l] - src[q].x[l];
                            sq += df * df;
                        }
                        if (sq <= g.thr_half) cnt += len[q];
                    }
                }
                wave_sync();
            }
        } else {
            for (int base = k * kUnitRuns; base < b1; base += kWave)
                stream_chunk<D>(base, b1, hd.r0, hd.s0, hd.smask, sub_run, run_start, Xs, n, a0,
                                x, thr, acc, __any(acc), src, len, ps, pc, pm);
        }
        if (hd.half) {
            if (hcnt)
                atomicAdd((unsigned long long *)hacc + (long long)(2 * D + 1) * n + tl.r,
                          (unsigned long long)cnt);
        } else if (acc) {
            add_fixed<D>(hacc, n, tl.r, ps, pc, pm);
        }
    }
}

// The runs of tiles with heavy ranges: their sums from hacc, then the
// tile kernel's final step.
template <int D>
__global__ __launch_bounds__(kBlock) void k_update_finish(
    const float *__restrict__ Xs, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const int *__restrict__ run_start,
    const int *__restrict__ cell_run, const int *__restrict__ grp_cell,
    const int *__restrict__ point_cell, const int *__restrict__ tile_off,
    const int *__restrict__ dtiles, const int *__restrict__ dsave,
    const long long *__restrict__ hacc, float *__restrict__ rres, int *__restrict__ rdbg, Geo g,
    DevState *st) {
    if (st->done) return;
    const int ndt = st->ndt, n = g.n, G = st->G;
    const int waves = gridDim.x * (blockDim.x / kWave);
    bool unsynced = false;
    for (int w = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; w < ndt; w += waves) {
        const TileLane tl = tile_lane(dtiles[w], tile_off, G, grp_cell, cell_run, run_start,
                                      point_cell);
        if (!tl.active) continue;
        const int r = tl.r;
        float x[D], a0[D], su[D], cu[D], sum[D], ssv[D], scm[D];
        int g0[D];
        tile_setup<D>(tl, Xs, cell_g, g, g0, a0, x, su, cu);
#pragma unroll
        for (int l = 0; l < D; l++) {
            sum[l] = rres[(long long)l * n + r];
            ssv[l] = from_fix(hacc[(long long)l * n + r]);
            scm[l] = from_fix(hacc[(long long)(D + l) * n + r]);
        }
        const int m_part = (int)hacc[(long long)(2 * D) * n + r];
        const int own = cell_start[tl.cl + 1] - cell_start[tl.cl];
        const int half = dsave[4 * (long long)r + 1] + (int)hacc[(long long)(2 * D + 1) * n + r];
        if (!finish_run<D>(x, su, cu, sum, ssv, scm, dsave[4 * (long long)r], m_part, half,
                           dsave[4 * (long long)r + 2] != 0, own, n, r, rres, rdbg))
            unsynced = true;
    }
    if (__any(unsynced) && __lane_id() == 0) atomicAnd(&st->flag, 0);
}

// Every point takes its run's result and carries its id over to the next
// iteration's order.
template <int D>
__global__ __launch_bounds__(kBlock) void k_scatter_runs(
    const int *__restrict__ point_run, const float *__restrict__ rres,
    const int *__restrict__ rdbg, const int *__restrict__ perm_s, float *__restrict__ Xout,
    int *__restrict__ perm_out, int n, DevState *st, DebugOut dbg) {
    if (st->done) return;
    // the local-sync flag as the update left it, before the extra check
    if (blockIdx.x == 0 && threadIdx.x == 0) st->flag_local = st->flag;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        perm_out[i] = perm_s[i];
        const int r = point_run[i];
#pragma unroll
        for (int l = 0; l < D; l++) Xout[(long long)l * n + i] = rres[(long long)l * n + r];
        if (rdbg) {
            if (dbg.N) dbg.N[i] = rdbg[4 * (long long)r + 0];
            if (dbg.half) dbg.half[i] = rdbg[4 * (long long)r + 1];
            if (dbg.border) dbg.border[i] = rdbg[4 * (long long)r + 2];
            if (dbg.synced) dbg.synced[i] = rdbg[4 * (long long)r + 3];
        }
    }
}

// MBR_in_eps (EGG_SynC.cu:1037-1159) for the pair (p, q), one thread: per
// dimension the coordinate, among q and q's eps/2-neighbours, closest to p;
// true if that point is within eps of p.  Used only when the pair queue of
// the extra check overflows.
template <int D>
__device__ bool mbr_in_eps(const float *xp, const float *xq, const float *__restrict__ Xs,
                           const int *__restrict__ cell_g, const int *__restrict__ ob,
                           const int *__restrict__ oe, const int *__restrict__ run_start,
                           const int *__restrict__ cell_run, const Geo &g) {
    const int n = g.n, od = g.od, R = g.R_half;
    float mbr[D];
    int g0[D];
#pragma unroll
    for (int l = 0; l < D; l++) {
        mbr[l] = xq[l];
        g0[l] = cell_coord(xq[l], g.cs, g.w);
    }
    const int g0od = select_dim<D>(g0, od);
    const int *cg_od = cell_g + (long long)od * n;
    Odo<D> odo;
    odo.init(od, R);
    while (!odo.finished) {
        const int o = odo.outer(g0, g);
        if (o >= 0) {
            int cb = ob[o];
            const int ce = oe[o];
            if (od < D) cb = column_lower(cg_od, cb, ce, g0od - R - 1);
            for (int c = cb; c < ce; c++) {
                int gc[D];
                bool stop;
                const bool in = cell_in_window<D>(cell_g, n, c, g0, od, R + 1, g0od, gc, &stop);
                if (stop) break;
                if (!in) continue;
                float sm, lg;
                box_dist<D>(gc, xq, g.cs, sm, lg);
                if (!(sm <= g.thr_half)) continue;
                for (int rr = cell_run[c]; rr < cell_run[c + 1]; rr++) {
                    float x2[D];
                    if (dist2_to<D>(xq, Xs, n, run_start[rr], x2) <= g.thr_half) {
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            float od_ = mbr[l] - xp[l];
                            od_ *= od_;
                            float nd = x2[l] - xp[l];
                            nd *= nd;
                            if (nd < od_) mbr[l] = x2[l];
                        }
                    }
                }
            }
        }
        odo.next(od, R);
    }
    float dd = 0.f;
#pragma unroll
    for (int l = 0; l < D; l++) {
        float t = mbr[l] - xp[l];
        t *= t;
        dd += t;
    }
    return dd <= g.thr_eps;
}

// kernel_float_grid_extra_check_part1 (EGG_SynC.cu:900-1034), per tile: each
// lane looks for partners q with eps < |p-q| <= eps_extra in cells that are
// not fully within eps of it, reading the cells' points from LDS chunks, and
// queues the pairs for k_extra_mbr.  Pairs are deduplicated by position (the
// MBR test depends on x_p and x_q only): a point equal to its predecessor in
// the cell is skipped, and so is a partner equal to the lane's last queued
// one.  Should the queue overflow, the lane tests the pair itself.  Runs only
// when every point is locally synced; any hit clears the flag.
template <int D>
__global__ __launch_bounds__(kBlock) void k_extra_tile(
    const float *__restrict__ Xs, const int *__restrict__ cell_g, const int *__restrict__ ob,
    const int *__restrict__ oe, const int *__restrict__ run_start,
    const int *__restrict__ cell_run, const int *__restrict__ grp_cell,
    const int *__restrict__ point_cell, const int *__restrict__ tile_off,
    int *__restrict__ pairs, int pair_cap, Geo g, DevState *st) {
    if (st->done || st->flag == 0) return;
    __shared__ float s_x[kBlock / kWave][kWave][SrcPt<D>::P];
    __shared__ int s_pos[kBlock / kWave][kWave];
    const int n = g.n, od = g.od, R = g.R_extra;
    const int G = st->G, T = st->T;
    const int lane = __lane_id();
    float(*src)[SrcPt<D>::P] = s_x[threadIdx.x / kWave];
    int *src_pos = s_pos[threadIdx.x / kWave];
    const int *cg_od = cell_g + (long long)od * n;
    bool hit = false;
    for (int t = wave_index(); t < T; t = wave_count() + next_tile(&st->xtile_next)) {
        if (__hip_atomic_load(&st->flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) break;
        const TileLane tl = tile_lane(t, tile_off, G, grp_cell, cell_run, run_start, point_cell);
        const int c0 = tl.gc0, i = tl.i;
        const bool active = tl.active;
        const int ghi = cell_g[(long long)(D - 1) * n + tl.gc1 - 1];
        float xp[D];
        int g0[D];
#pragma unroll
        for (int l = 0; l < D; l++) {
            g0[l] = cell_g[(long long)l * n + c0];
            xp[l] = active ? Xs[(long long)l * n + i] : 0.f;
        }
        float lq[D];
        bool have_lq = false;
        const int g0od = select_dim<D>(g0, od);
        auto consider = [&](const float *xq, int j) {
            bool rep = have_lq;
#pragma unroll
            for (int l = 0; l < D; l++) rep = rep && __float_as_uint(lq[l]) == __float_as_uint(xq[l]);
            if (rep) return;
#pragma unroll
            for (int l = 0; l < D; l++) lq[l] = xq[l];
            have_lq = true;
            const int slot = atomicAdd(&st->pair_count, 1);
            if (slot < pair_cap) {
                pairs[2 * slot] = i;
                pairs[2 * slot + 1] = j;
            } else if (mbr_in_eps<D>(xp, xq, Xs, cell_g, ob, oe, run_start, cell_run, g)) {
                hit = true;
            }
        };
        walk_columns<D>(g0, R, g, ob, oe, [&](int cb, const int ce) {
            if (od < D) cb = column_lower(cg_od, cb, ce, g0od - R - 1);
            for (int c = cb; c < ce; c++) {
                int gc[D];
                bool stop;
                const bool in =
                    cell_in_group_window<D>(cell_g, n, c, g0, od, R + 1, ghi, gc, &stop);
                if (stop) break;
                if (!in) continue;
                float sm, lg;
                box_dist<D>(gc, xp, g.cs, sm, lg);
                const bool need = active && !(lg <= g.thr_eps) && sm <= g.thr_extra;
                if (!__any(need)) continue;
                const int r0 = cell_run[c], r1 = cell_run[c + 1];
                for (int base = r0; base < r1; base += kWave) {
                    const int rr = base + lane;
                    if (rr < r1) {
                        const int j = run_start[rr];
                        src_pos[lane] = j;
#pragma unroll
                        for (int l = 0; l < D; l++) src[lane][l] = Xs[(long long)l * n + j];
                    }
                    wave_sync();
                    const int m = min(kWave, r1 - base);
                    if (need) {
                        for (int k = 0; k < m; k++) {
                            float xq[D], s = 0.f;
#pragma unroll
                            for (int l = 0; l < D; l++) {
                                xq[l] = src[k][l];
                                const float df = xp[l] - xq[l];
                                s += df * df;
                            }
                            if (!(s <= g.thr_eps) && s <= g.thr_extra) consider(xq, src_pos[k]);
                        }
                    }
                    wave_sync();
                }
            }
        });
    }
    if (__any(hit) && lane == 0) atomicAnd(&st->flag, 0);
}

// kernel_float_grid_extra_check_part2 + MBR_in_eps (EGG_SynC.cu:1037-1203),
// one wavefront per queued pair: the lanes share the scan of q's
// eps/2-neighbourhood and keep, per dimension, the smallest squared distance
// to p of a candidate coordinate (the reference keeps the coordinate with the
// smallest one, so its MBR distance is the sum of these minima); a lane-min
// reduction then gives the same value as the sequential scan.
template <int D>
__global__ __launch_bounds__(kBlock) void k_extra_mbr(
    const float *__restrict__ Xs, const int *__restrict__ cell_g, const int *__restrict__ ob,
    const int *__restrict__ oe, const int *__restrict__ run_start,
    const int *__restrict__ cell_run, const int *__restrict__ pairs, int pair_cap, Geo g,
    DevState *st) {
    if (st->done || st->flag == 0) return;
    const int n = g.n, od = g.od, R = g.R_half;
    const int npairs = min(st->pair_count, pair_cap);
    const int lane = __lane_id();
    const int waves = gridDim.x * (blockDim.x / kWave);
    const int *cg_od = cell_g + (long long)od * n;
    for (int k = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; k < npairs;
         k += waves) {
        if (__hip_atomic_load(&st->flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) break;
        const int ip = pairs[2 * k], iq = pairs[2 * k + 1];
        float xp[D], xq[D], best[D];
        int g0[D];
#pragma unroll
        for (int l = 0; l < D; l++) {
            xp[l] = Xs[(long long)l * n + ip];
            xq[l] = Xs[(long long)l * n + iq];
            g0[l] = cell_coord(xq[l], g.cs, g.w);
            float t = xq[l] - xp[l];  // the MBR starts at q
            t *= t;
            best[l] = t;
        }
        const int g0od = select_dim<D>(g0, od);
        walk_columns<D>(g0, R, g, ob, oe, [&](int cb, const int ce) {
            if (od < D) cb = column_lower(cg_od, cb, ce, g0od - R - 1);
            for (int c = cb; c < ce; c++) {
                int gc[D];
                bool stop;
                const bool in = cell_in_window<D>(cell_g, n, c, g0, od, R + 1, g0od, gc, &stop);
                if (stop) break;
                if (!in) continue;
                float sm, lg;
                box_dist<D>(gc, xq, g.cs, sm, lg);
                if (!(sm <= g.thr_half)) continue;
                for (int rr = cell_run[c] + lane; rr < cell_run[c + 1]; rr += kWave) {
                    float x2[D];
                    if (dist2_to<D>(xq, Xs, n, run_start[rr], x2) <= g.thr_half) {
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            float nd = x2[l] - xp[l];
                            nd *= nd;
                            best[l] = fminf(best[l], nd);
                        }
                    }
                }
            }
        });
#pragma unroll
        for (int l = 0; l < D; l++)
            for (int o = kWave / 2; o > 0; o >>= 1)
                best[l] = fminf(best[l], __shfl_xor(best[l], o, kWave));
        float dd = 0.f;
#pragma unroll
        for (int l = 0; l < D; l++) dd += best[l];
        if (dd <= g.thr_eps && lane == 0) atomicAnd(&st->flag, 0);
    }
}

// SynC pass over the grid (SynC.cpp:16-56): every point within FP32 distance
// eps (candidates: Chebyshev radius R+1 in the outer dimensions, which contains
// every such point) contributes sinf(x_j - x) to the update and
// expf(-|x_j - x|) to r_p, in ascending sorted position.  Targets are the runs of
// equal positions, whose points have the same sums; k_sync_points hands the results to
// the points.  A target per point took 6 to 20 times as long on final positions, with
// tens to hundreds of points to a run: r_c at n = 100,000, d = 3, eps = 0.02: 7.7 ms,
// here 0.9; n = 400,000 31.9 and 3.0.
//
// A workgroup takes T consecutive targets, a wavefront each.  In a round every
// wavefront tests its target's next S candidates, one per lane, packs the
// accepted ones into LDS and evaluates their terms 64 at a time; after the
// barrier, lanes of the first wavefronts (one per target and coordinate) and of
// the last (r_p, in FP64) add the packed terms one after another -- the sums of
// a scan by one thread, bit for bit -- while the next round's go to the other
// half of the LDS.  Bound by the VALU: the terms (~45 instructions a
// coordinate) once per 64 accepted pairs, ~40 instructions per 64 tested ones.
// One thread per target ran the terms for every candidate any of 64 lanes
// accepted, and 8,000 targets filled 125 of 1,024 SIMDs: n = 8,000, d = 2,
// eps = 0.05: 3,760 us a pass, here 154.
//
// Which form (kLaneMin): k_update_sync_lane gives each target a lane, which adds its
// neighbours by itself.  It tests a candidate in fewer instructions, but its
// wavefronts run the terms of every candidate any lane accepts, and end with their
// longest list.  Wavefront / lane form, ms of a pass with its grid build, blobs as
// given, eps = 0.002 to 0.1:
//   n        d = 1      2        3        4        6
//   65,536   1.3/2.7  4.1/10   2.4/6.4  5.8/52   3.7/18
//   131,072  2.6/3.3  14/20    7.7/12   20/56    11/48
//   200,000  4.9/4.7  22/22    19/32    43/86    24/76
//   400,000  18/13    79/56    67/63    173/246  78/177
// and of r_c alone at d = 1 0.73/1.5, 1.25/1.33 (n = 100,000), 1.74/1.79, 3.4/2.2.
// From d = 3 on the line could lie higher; it is where d = 1 and 2 are even.
template <int D, bool WRITE>
struct SyncShape {
    static constexpr int NC = WRITE ? D + 1 : 1;             // terms per pair
    static constexpr int T = NC <= 17 ? 16 : 8;              // targets, and wavefronts
    static constexpr int S = NC <= 4 ? 128 : 64;             // candidates per round
    static constexpr int kThreads = T * kWave;
    // from this many targets on a lane each (k_update_sync_lane)
    static constexpr int kLaneMin = D == 1 && !WRITE ? 3 << 15 : 1 << 17;
    // row of a target's terms: 4 banks apart for the adding lanes, 2 where 4 would cost
    // the second workgroup of a CU its LDS (d = 18)
    static constexpr int kLds = 160 * 1024, kRows = 8 * T * NC;
    static constexpr int P = kLds / (kRows * (S + 4)) == kLds / (kRows * S) ? S + 4 : S + 2;
    static constexpr int kAdders = (D * T + kWave - 1) / kWave;
    static_assert(kRows * P + 8 * T <= kLds, "LDS");
    static_assert(!WRITE || kAdders < T, "the last wavefront adds r_p");
    // workgroups of at most n targets, fewer than kLaneMin
    static int blocks(int n) { return (std::min(n, kLaneMin - 1) + T - 1) / T; }
};

template <int D, bool WRITE>
__global__ __launch_bounds__((SyncShape<D, WRITE>::kThreads))
__attribute__((amdgpu_waves_per_eu(D <= 8 ? 8 : 4))) void k_update_sync(
    const float *__restrict__ Xs, const int *__restrict__ run_start,
    const int *__restrict__ point_cell, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const int *__restrict__ ob, const int *__restrict__ oe, Geo g,
    const DevState *st, float *__restrict__ rres, double *__restrict__ ratio) {
    if (WRITE && st->done) return;
    using Sh = SyncShape<D, WRITE>;
    constexpr int T = Sh::T, S = Sh::S, P = Sh::P, NC = Sh::NC;
    const int runs = st->runs;
    if ((int)blockIdx.x * T >= runs || runs >= Sh::kLaneMin) return;
    __shared__ __align__(16) float s_term[2][NC][T * P];
    __shared__ int s_cnt[2][T];
    const int n = g.n, lane = __lane_id();
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int target = blockIdx.x * T + w;  // this wavefront's run
    const int i = run_start[min(target, runs - 1)];
    float x[D];
    Candidates<D> cand;
#pragma unroll
    for (int l = 0; l < D; l++) x[l] = Xs[(long long)l * n + i];
    cand.init(g, cell_g, cell_start, ob, oe, point_cell[i], g.R + 1);
    // the adding lanes' target and coordinate; the last wavefront adds r_p
    const int at = lane % T, ac = w * (kWave / T) + lane / T;
    const bool adds = WRITE && w < Sh::kAdders && ac < D, adds_r = w == T - 1 && lane < T;
    float sum = 0.f;
    double r = 0.0;
    int N = 0;
    bool left = target < runs;
    for (int k = 0;; k++) {
        int cnt = 0;
        if (left) {
            float(*term)[T * P] = s_term[k & 1];
            for (int step = 0; step < S / kWave; step++) {
                left = cand.more();
                if (!left) break;
                const int f = cand.f0 + lane;
                const bool in_range = f < cand.total;
                const int j = cand.point(min(f, cand.total - 1), cand.f0);
                cand.f0 += kWave;
                float df[D], s = 0.f;
#pragma unroll
                for (int l = 0; l < D; l++) {
                    df[l] = Xs[(long long)l * n + j] - x[l];
                    s += df[l] * df[l];
                }
                const bool in = in_range && s <= g.thr_eps;
                const unsigned long long m = __ballot(in);
                if (in) {
                    const int e = w * P + cnt + __popcll(m & lanemask_lt());
                    if (WRITE) {
#pragma unroll
                        for (int l = 0; l < D; l++) term[l][e] = df[l];
                    }
                    term[NC - 1][e] = s;
                }
                cnt += __popcll(m);
            }
            wave_sync();
            for (int q = lane; q < cnt; q += kWave) {
                const int e = w * P + q;
                if (WRITE) {
#pragma unroll
                    for (int l = 0; l < D; l++) term[l][e] = sinf(term[l][e]);
                }
                term[NC - 1][e] = expf(-fabsf(sqrtf(term[NC - 1][e])));
            }
        }
        if (lane == 0) s_cnt[k & 1][w] = cnt;
        if (k > 0 && (adds || adds_r)) {
            const int b = (k - 1) & 1, c = s_cnt[b][at];
            const float *t = s_term[b][adds ? ac : NC - 1] + at * P;
            N += c;
            for (int q0 = 0; q0 < c; q0 += 8) {
                float v[8];
#pragma unroll
                for (int q = 0; q < 8; q++) v[q] = t[q0 + q];  // S is a multiple of 8
                if (adds) {
#pragma unroll
                    for (int q = 0; q < 8; q++)
                        if (q0 + q < c) sum += v[q];
                } else {
#pragma unroll
                    for (int q = 0; q < 8; q++)
                        if (q0 + q < c) r += (double)v[q];
                }
            }
        }
        // one more round than the longest candidate list, to add its last terms
        if (!__syncthreads_or(left || cnt > 0)) break;
    }
    const int ra = blockIdx.x * T + at;
    if (adds && ra < runs)
        rres[(long long)ac * n + ra] = Xs[(long long)ac * n + run_start[ra]] + sum / (float)N;
    if (adds_r && ra < runs) ratio[ra] = N > 0 ? r / (double)N : 1.0;
}

constexpr int kRcBlocks = 1024;

// The same pass with a lane per target, each adding its neighbours one after the
// other (SyncShape::kLaneMin).
template <int D, bool WRITE>
__global__ __launch_bounds__(kBlock) void k_update_sync_lane(
    const float *__restrict__ Xs, const int *__restrict__ run_start,
    const int *__restrict__ point_cell, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const int *__restrict__ ob, const int *__restrict__ oe, Geo g,
    const DevState *st, float *__restrict__ rres, double *__restrict__ ratio) {
    if (WRITE && st->done) return;
    const int n = g.n, od = g.od, R = g.R + 1, runs = st->runs;
    if (runs < SyncShape<D, WRITE>::kLaneMin) return;
    const int *cg_od = cell_g + (long long)od * n;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < runs; t += gridDim.x * blockDim.x) {
        const int i = run_start[t];
        float x[D], sum[D];
        int g0[D];
        const int c0 = point_cell[i];
#pragma unroll
        for (int l = 0; l < D; l++) {
            x[l] = Xs[(long long)l * n + i];
            g0[l] = cell_g[(long long)l * n + c0];
            sum[l] = 0.f;
        }
        const int g0od = select_dim<D>(g0, od);
        int N = 0;
        double r = 0.0;
        Odo<D> odo;
        odo.init(od, R);
        while (!odo.finished) {
            const int o = odo.outer(g0, g);
            if (o >= 0) {
                int cb = ob[o];
                const int ce = oe[o];
                if (od < D) cb = column_lower(cg_od, cb, ce, g0od - R);
                for (int c = cb; c < ce; c++) {
                    int gc[D];
#pragma unroll
                    for (int l = 0; l < D; l++) gc[l] = cell_g[(long long)l * n + c];
                    if (od < D && select_dim<D>(gc, od) > g0od + R) break;
                    bool skip = false;
#pragma unroll
                    for (int l = 0; l < D; l++)
                        if (l > od && (gc[l] - g0[l] > R || g0[l] - gc[l] > R)) skip = true;
                    if (skip) continue;
                    for (int j = cell_start[c]; j < cell_start[c + 1]; j++) {
                        float xq[D];
                        const float s = dist2_to<D>(x, Xs, n, j, xq);
                        if (s <= g.thr_eps) {
                            if (WRITE) {
#pragma unroll
                                for (int l = 0; l < D; l++) sum[l] += sinf(xq[l] - x[l]);
                            }
                            N++;
                            r += (double)expf(-fabsf(sqrtf(s)));
                        }
                    }
                }
            }
            odo.next(od, R);
        }
        if (WRITE) {
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float mean = sum[l] / (float)N;
                rres[(long long)l * n + t] = x[l] + mean;
            }
        }
        ratio[t] = N > 0 ? r / (double)N : 1.0;
    }
}

// A run's results to its points: with `write` the new positions (and the point ids,
// for the next grid build's order), and block partial sums of the points' r_p / N,
// combined in a fixed order by k_rc_finish, so r_c is deterministic.
__global__ __launch_bounds__(kBlock) void k_sync_points(const int *__restrict__ point_run,
                                                        const double *__restrict__ ratio,
                                                        const float *__restrict__ rres,
                                                        const int *__restrict__ perm_s, int n,
                                                        int d, bool write, const DevState *st,
                                                        float *__restrict__ Xout,
                                                        int *__restrict__ perm_out,
                                                        double *__restrict__ rc_part) {
    if (write && st->done) return;
    double racc = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int r = point_run[i];
        racc += ratio[r];
        if (write) {
            for (int l = 0; l < d; l++) Xout[(long long)l * n + i] = rres[(long long)l * n + r];
            perm_out[i] = perm_s[i];
        }
    }
    __shared__ double s_r[kBlock / kWave];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) racc += __shfl_xor(racc, o, kWave);
    if (__lane_id() == 0) s_r[threadIdx.x / kWave] = racc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < kBlock / kWave; w++) t += s_r[w];
        rc_part[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(kBlock) void k_rc_finish(const double *__restrict__ rc_part,
                                                      int nparts, int n, DevState *st,
                                                      bool guard) {
    if (guard && st->done) return;
    __shared__ double s_r[kBlock];
    double t = 0.0;
    for (int k = threadIdx.x; k < nparts; k += kBlock) t += rc_part[k];
    s_r[threadIdx.x] = t;
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) s_r[threadIdx.x] += s_r[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) st->rc = s_r[0] / (double)n;
}


__global__ void k_set_flag(DevState *st) {
    if (st->done) return;
    reset_pass_state(st);
}

static inline int grid_for(long long n) {
    long long b = (n + kBlock - 1) / kBlock;
    if (b < 1) b = 1;
    if (b > 65536) b = 65536;
    return (int)b;
}

static inline int queue_threads(const Geo &g) {
    return g.qthreads >= kWave && g.qthreads <= kBlock && g.qthreads % kWave == 0 ? g.qthreads
                                                                                 : kBlock;
}

static inline int queue_blocks(const Geo &g) {
    const long long tiles_max = (long long)g.n / kTile + g.n;  // >= n/64 + C
    const int waves = queue_threads(g) / kWave;
    const long long cap = g.qblocks > 0 ? g.qblocks : kQueueBlocks * (kBlock / kWave) / waves;
    return (int)std::max<long long>(1, std::min<long long>(cap, (tiles_max + waves - 1) / waves));
}

template <int D, bool MM>
static void launch_tiles(const Geo &g, GridBufs &b, int *rdbg, int qb, int qt, DevState *st,
                         hipStream_t s) {
    if constexpr (MM)
        k_update_dense<D><<<qb, qt, 0, s>>>(b, rdbg, g, st);
    else
        k_update_tile<D><<<qb, qt, 0, s>>>(
            b.Xs, b.cell_start, b.cell_g, b.Ts, b.Tc, b.ob, b.oe, b.run_start, b.cell_run,
            b.grp_cell, b.point_cell, b.utile_off, b.cell_sub, b.sub_start, b.smin, b.smax,
            b.sub_run, b.TsS, b.TcS, b.rres, rdbg, b.hacc, b.hdesc, b.dtiles, b.rdbg, g, st);
    if (!b.hacc) return;
    k_update_heavy<D, MM><<<qb, qt, 0, s>>>(b.Xs, b.cell_g, b.run_start, b.cell_run, b.grp_cell,
                                            b.point_cell, b.utile_off, b.sub_run, b.hdesc, b.hacc,
                                            g, st);
    k_update_finish<D><<<qb, qt, 0, s>>>(b.Xs, b.cell_start, b.cell_g, b.run_start, b.cell_run,
                                         b.grp_cell, b.point_cell, b.utile_off, b.dtiles, b.rdbg,
                                         b.hacc, b.rres, rdbg, g, st);
}

void launch_update_egg(const Geo &g, GridBufs &b, DevState *st, const DebugOut *dbg,
                       hipStream_t s) {
    DebugOut d = dbg ? *dbg : DebugOut{nullptr, nullptr, nullptr, nullptr};
    const int qb = queue_blocks(g), qt = queue_threads(g);
    int *rdbg = (d.N || d.half || d.border || d.synced) ? b.rdbg : nullptr;
#define UPD_CASE(DD)                                                                      \
    case DD:                                                                              \
        if (DD <= kStreamMaxD && g.n < (1 << 24))                                         \
            launch_tiles<DD, (DD <= kStreamMaxD)>(g, b, rdbg, qb, qt, st, s);             \
        else                                                                              \
            launch_tiles<DD, false>(g, b, rdbg, qb, qt, st, s);                           \
        launch_update_pairs(g, b, rdbg, st, s);                                           \
        k_scatter_runs<DD><<<grid_for(g.n), kBlock, 0, s>>>(b.point_run, b.rres, rdbg,    \
                                                            b.perm_s, b.X, b.perm, g.n,   \
                                                            st, d);                       \
        break;
    switch (g.d) {
        EGG_EACH_D(UPD_CASE)
    }
#undef UPD_CASE
}

void launch_extra_check(const Geo &g, GridBufs &b, DevState *st, hipStream_t s) {
    const int qb = queue_blocks(g), qt = queue_threads(g);
#define EX_CASE(DD)                                                                           \
    case DD:                                                                                  \
        k_extra_tile<DD><<<qb, qt, 0, s>>>(b.Xs, b.cell_g, b.ob, b.oe, b.run_start,       \
                                           b.cell_run, b.grp_cell, b.point_cell, b.tile_off,  \
                                           b.pairs, b.pair_cap, g, st);                       \
        k_extra_mbr<DD><<<1024, kBlock, 0, s>>>(b.Xs, b.cell_g, b.ob, b.oe, b.run_start,      \
                                                b.cell_run, b.pairs, b.pair_cap, g, st);      \
        break;
    switch (g.d) {
        EGG_EACH_D(EX_CASE)
    }
#undef EX_CASE
}

int rc_partials(int n) { return kRcBlocks; }

void launch_update_sync(const Geo &g, GridBufs &b, DevState *st, double *rc_part, bool write_pos,
                        hipStream_t s) {
    double *ratio = (double *)b.rdbg;  // [n] of its 4n ints, unused by this pass
    // the number of targets is on the device: each form returns at the other's numbers
#define SY_ARGS                                                                                   \
    b.Xs, b.run_start, b.point_cell, b.cell_start, b.cell_g, b.ob, b.oe, g, st, b.rres, ratio
#define SY_LAUNCH(DD, W)                                                                          \
    k_update_sync<DD, W><<<SyncShape<DD, W>::blocks(g.n), SyncShape<DD, W>::kThreads, 0, s>>>(     \
        SY_ARGS);                                                                                 \
    if (g.n >= SyncShape<DD, W>::kLaneMin)                                                        \
        k_update_sync_lane<DD, W><<<kRcBlocks, kBlock, 0, s>>>(SY_ARGS)
#define SY_CASE(DD)                     \
    case DD:                            \
        if (write_pos) {                \
            SY_LAUNCH(DD, true);        \
        } else {                        \
            SY_LAUNCH(DD, false);       \
        }                               \
        break;
    switch (g.d) {
        EGG_EACH_D(SY_CASE)
    }
#undef SY_CASE
#undef SY_LAUNCH
#undef SY_ARGS
    k_sync_points<<<kRcBlocks, kBlock, 0, s>>>(b.point_run, ratio, b.rres, b.perm_s, g.n, g.d,
                                               write_pos, st, b.X, b.perm, rc_part);
    k_rc_finish<<<1, kBlock, 0, s>>>(rc_part, kRcBlocks, g.n, st, write_pos);
}

void launch_set_flag(DevState *st, hipStream_t s) { k_set_flag<<<1, 1, 0, s>>>(st); }

}  // namespace egg
