// The update of sparse cell groups, point pair by point pair (gfx950).
//
// The runs of the cell groups sparse_group selects (the runs of sparse groups,
// or every run) are updated from all runs of the grid instead of cell by cell
// (EGG_SynC.cu:551-763 walks the neighbour cells).  In a sparse grid
// (high-dimensional data: 250k points in 248k cells at d = 8) the neighbour
// cells of a point are the inner cells of (2R+1)^od outer cells, almost all
// holding a point or none, and walking them costs far more than testing the
// points they hold.  Sources come in blocks of kBlkRuns consecutive runs (sorted
// order, so spatially compact) with bounding boxes, and blocks in superblocks
// of kSupBlks.  A wavefront takes a tile of 16 target runs, prunes superblocks
// and blocks whose box lies farther from the tile's box than any counted point
// can, and takes the remaining blocks one after another (k_update_pairs).
//
// A pair within eps, or with a clamped source (such a point lies outside its
// cell's box), gets the reference's cell decision for the source's cell
// (EGG_SynC.cu:612-636): a full cell adds its totals (T_s cos x - T_c sin x,
// EGG_SynC.cu:648-663) and its count once, at the cell's first run -- every run
// of a full cell is within the filter radius of the target (it lies in the
// box, whose farthest corner is within eps, and FP32 rounding is monotone), so
// that run is always met; a partial cell adds sin(x_q - x) and the length of
// each run within eps (EGG_SynC.cu:683-696); neither -> nothing.  Only cells
// whose outer coordinates are within R of the target's are candidates, as in
// the reference's neighbour list (EGG_SynC.cu:368-536).  Blocks are visited in
// increasing order, which is the reference's order of outer cells, cells and
// points, and a target's terms are added one after another in that order, so
// the sums are the oracle's order of additions (runs weighted by their
// length); N and half are exactly the reference's.
#include <algorithm>
#include <cmath>

#include "egg_internal.h"
#include "egg_wave.h"

namespace egg {

// Per run: its cell, flags (bit 0: the first run of its cell, bit 1: a
// coordinate clamped into cell w-1), position, cell coordinates and length,
// indexed by run so that the pair update stages a block with one coalesced
// load per field; per cell (at its first run): its sin and cos totals as one
// row; per block of kBlkRuns runs: the bounding box of its positions, whether
// it holds a clamped run, and its cell if all its runs share one (-1
// otherwise).  One wavefront per block.
template <int D>
__global__ __launch_bounds__(kBlock) void k_run_boxes(
    const float *__restrict__ Xs, const int *__restrict__ run_start,
    const int *__restrict__ point_cell, const int *__restrict__ cell_run,
    const int *__restrict__ cell_g, const float *__restrict__ Ts, const float *__restrict__ Tc,
    Geo g, DevState *st, float *__restrict__ totals, int *__restrict__ rcell,
    int *__restrict__ rflag, float *__restrict__ Xr, int *__restrict__ gr,
    int *__restrict__ rlen, float *__restrict__ bmin, float *__restrict__ bmax,
    int *__restrict__ bclamp, int *__restrict__ bcell) {
    if (st->done || st->sparse_count == 0) return;
    const int n = g.n, runs = st->runs;
    const int nblk = (runs + kBlkRuns - 1) / kBlkRuns, nb = n / kBlkRuns + 1;
    const float wf = (float)g.w;
    for (int b = wave_index(); b < nblk; b += wave_count()) {
        const int r = b * kBlkRuns + __lane_id();
        const bool on = r < runs;
        float lo[D], hi[D];
        int f = 0, c = -1;
        if (on) {
            const int i = run_start[r];
            c = point_cell[i];
            bool clamped = false;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float x = Xs[(long long)l * n + i];
                lo[l] = hi[l] = x;
                clamped |= x / g.cs >= wf;  // cell_coord's clamp of w to w-1
                Xr[(long long)l * n + r] = x;
                gr[(long long)l * n + r] = cell_g[(long long)l * n + c];
            }
            f = (cell_run[c] == r ? 1 : 0) | (clamped ? 2 : 0);
            rcell[r] = c;
            rflag[r] = f;
            rlen[r] = run_start[r + 1] - i;
            if (f & 1) {
#pragma unroll
                for (int l = 0; l < D; l++) {
                    totals[(long long)c * 2 * D + l] = Ts[(long long)l * n + c];
                    totals[(long long)c * 2 * D + D + l] = Tc[(long long)l * n + c];
                }
            }
        } else {
#pragma unroll
            for (int l = 0; l < D; l++) {
                lo[l] = __builtin_inff();
                hi[l] = -__builtin_inff();
            }
        }
        const bool any_clamp = __any((f & 2) != 0);
        const int c_first = __builtin_amdgcn_readfirstlane(c);
        const bool one_cell = !__any(on && c != c_first);
#pragma unroll
        for (int l = 0; l < D; l++) {
            for (int o = kWave / 2; o > 0; o >>= 1) {
                lo[l] = fminf(lo[l], __shfl_xor(lo[l], o, kWave));
                hi[l] = fmaxf(hi[l], __shfl_xor(hi[l], o, kWave));
            }
            if (__lane_id() == 0) {
                bmin[(long long)l * nb + b] = lo[l];
                bmax[(long long)l * nb + b] = hi[l];
            }
        }
        if (__lane_id() == 0) {
            bclamp[b] = any_clamp ? 1 : 0;
            bcell[b] = one_cell ? c_first : -1;
        }
    }
}

// Bounding box of every superblock of kSupBlks blocks, and whether it holds a
// clamped run.
template <int D>
__global__ __launch_bounds__(kBlock) void k_super_boxes(
    const float *__restrict__ bmin, const float *__restrict__ bmax,
    const int *__restrict__ bclamp, Geo g, DevState *st, float *__restrict__ sbmin,
    float *__restrict__ sbmax, int *__restrict__ sbclamp) {
    if (st->done || st->sparse_count == 0) return;
    const int n = g.n, runs = st->runs;
    const int nblk = (runs + kBlkRuns - 1) / kBlkRuns, nb = n / kBlkRuns + 1;
    const int nsup = (nblk + kSupBlks - 1) / kSupBlks, ns = n / (kBlkRuns * kSupBlks) + 1;
    for (int sb = wave_index(); sb < nsup; sb += wave_count()) {
        const int b = sb * kSupBlks + __lane_id();
        const bool on = b < nblk;
        const bool any_clamp = __any(on && bclamp[b] != 0);
#pragma unroll
        for (int l = 0; l < D; l++) {
            float lo = on ? bmin[(long long)l * nb + b] : __builtin_inff();
            float hi = on ? bmax[(long long)l * nb + b] : -__builtin_inff();
            for (int o = kWave / 2; o > 0; o >>= 1) {
                lo = fminf(lo, __shfl_xor(lo, o, kWave));
                hi = fmaxf(hi, __shfl_xor(hi, o, kWave));
            }
            if (__lane_id() == 0) {
                sbmin[(long long)l * ns + sb] = lo;
                sbmax[(long long)l * ns + sb] = hi;
            }
        }
        if (__lane_id() == 0) sbclamp[sb] = any_clamp ? 1 : 0;
    }
}

// Whether box k of a (lo, hi) table ([D][stride]) lies within squared
// distance thr of the box [alo, ahi] (thr_clamp if the box holds a clamped
// run).  Box distances round like the point distances they bound; the
// caller's thresholds carry a relative margin of 2^-10 for that.
template <int D>
__device__ __forceinline__ bool box_near(const float (&alo)[D], const float (&ahi)[D],
                                         const float *__restrict__ blo,
                                         const float *__restrict__ bhi, long long stride, int k,
                                         float thr) {
    float s = 0.f;
#pragma unroll
    for (int l = 0; l < D; l++) {
        const float gap = fmaxf(0.f, fmaxf(blo[l * stride + k] - ahi[l], alo[l] - bhi[l * stride + k]));
        s += gap * gap;
    }
    return s <= thr;
}

// sin v: the polynomial of sin_small for |v| <= 1 when the caller knows that
// bound holds (SMALL), else sinf.
template <bool SMALL>
__device__ __forceinline__ float sin_pair(float v) {
    if (!SMALL) return sinf(v);
    const float v2 = v * v;
    float ps = -2.50521083854417e-08f;
    ps = fmaf(ps, v2, 2.75573192239859e-06f);
    ps = fmaf(ps, v2, -1.98412698412698e-04f);
    ps = fmaf(ps, v2, 8.33333333333333e-03f);
    ps = fmaf(ps, v2, -1.66666666666667e-01f);
    return fmaf(v * v2, ps, v);
}

// Thresholds of the pair update (pair_bounds).
struct PairBounds {
    float thr_filter, thr_clamp;  // squared filter radii, of clamped sources
    float r, rounding;            // larger filter radius; relative error of the MFMA distance
    float lo, hi;                 // squared distances surely <= / > thr_eps
};

constexpr int kPairTargets = 16;  // targets of a tile, four lanes each

// Source runs of a block staged in LDS.  x and c (the cell's centre) are rows
// of 16-byte reads for the accepted pairs, where each lane reads a run of its
// own; a row stride of 4 mod 8 floats spreads the rows over all banks.  f holds
// the features of the distance product (row stride odd).
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int D>
struct PairStage {
    static constexpr int P = (D + 3) / 4 * 4;
    static constexpr int XS = P % 8 == 0 ? P + 4 : P;
    static constexpr int KS = (D + 2 + 3) / 4;  // MFMA steps of the distance product
    static constexpr int FS = 4 * KS + 1;
    alignas(16) float x[kBlkRuns * XS];
    alignas(16) float c[kBlkRuns * XS];
    alignas(16) int4 meta[kBlkRuns];  // cell, flags, length, points of the cell (first runs)
    float f[kBlkRuns * FS];
};

template <int D>
__device__ __forceinline__ void read_row(const float *row, float (&v)[PairStage<D>::P]) {
#pragma unroll
    for (int l = 0; l < PairStage<D>::P; l += 4) {
        const f32x4 q = *reinterpret_cast<const f32x4 *>(row + l);
#pragma unroll
        for (int k = 0; k < 4; k++) v[l + k] = q[k];
    }
}

// The reference's decision for the cell of source run rr as seen from target x
// in cell c0 (EGG_SynC.cu:612-634): 0 not counted (or not in the neighbour
// list), 1 full, 2 partial.
template <int D>
__device__ int pair_class(const float (&x)[D], int c0, int rr, const int *__restrict__ gr,
                          const int *__restrict__ cell_g, const Geo &g) {
    int gc[D];
    bool win = true;
#pragma unroll
    for (int l = 0; l < D; l++) {
        gc[l] = gr[(long long)l * g.n + rr];
        if (l < g.od) {
            const int dg = gc[l] - cell_g[(long long)l * g.n + c0];
            if (dg > g.R || dg < -g.R) win = false;
        }
    }
    float sm, lg;
    box_dist<D>(gc, x, g.cs, sm, lg);
    return !win ? 0 : (lg <= g.thr_eps ? 1 : (sm <= g.thr_eps ? 2 : 0));
}

// Adds lane I of each group of four lanes' v to s on all four.
template <int I>
__device__ __forceinline__ float add_quad(float s, float v) {
    return s + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), I * 0x55, 0xf, 0xf, true));
}

__device__ __forceinline__ int quad_sum(int v) {
    v += __shfl_xor(v, 1, kWave);
    return v + __shfl_xor(v, 2, kWave);
}

// One wavefront per tile of 16 targets (lanes 4t .. 4t+3 serve target t).  Per
// block of 64 source runs:
//  1. the squared distances of all 1,024 pairs by v_mfma_f32_16x16x4_f32,
//     |v|^2 - 2 u.v + (|u|^2 - thr) relative to the tile's centre; its sign bits
//     are the accepted pairs (one v_alignbit each).  thr holds the filter radius
//     and a bound on the product's rounding, so that no pair within the filter
//     is missed; what is accepted beyond it fails the tests below;
//  2. the four lanes of a target take its accepted runs in turns of four and
//     evaluate the FP32 distance, the cell's class and sin(x_q - x); the class
//     comes from the distances to the cell's near and far faces by its centre
//     (5 instructions a dimension against 8), and where those lie within
//     rounding of eps, from the reference's own box test (pair_class);
//  3. the four terms are added one after another (DPP broadcasts within the
//     four lanes), each lane keeping the target's full sum;
//  4. full cells met at their first run add their totals, each lane in its own
//     dimensions.
// 16 targets a tile instead of 64: a quarter of the idle lanes when targets'
// counts differ, boxes that prune more, and four times the wavefronts where n
// is small.  Bound by the VALU, ~200 instructions per 64 evaluated pairs.
// n = 250,000, d = 8, eps = 0.1: 65 ms a pass with a lane per target and the
// totals read (and sinf / cosf taken) inside the pair loop, here 35; n = 14,980,
// d = 14: 7.3 ms (234 wavefronts), here 1.6.
// SMALL: every pair the filter passes is closer than 1 in each coordinate
// (filter radius below 1), so sin(x_q - x) takes the polynomial.
template <int D, bool SMALL>
__global__ __launch_bounds__(kBlock) void k_update_pairs(
    const float *__restrict__ Xs, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const float *__restrict__ totals,
    const int *__restrict__ run_start, const int *__restrict__ point_cell,
    const int *__restrict__ cell_run, const int *__restrict__ list,
    const int *__restrict__ rcell, const int *__restrict__ rflag,
    const float *__restrict__ Xr, const int *__restrict__ gr, const int *__restrict__ rlen,
    const float *__restrict__ bmin, const float *__restrict__ bmax,
    const int *__restrict__ bclamp, const int *__restrict__ bcell,
    const float *__restrict__ sbmin, const float *__restrict__ sbmax,
    const int *__restrict__ sbclamp, PairBounds pb, float *__restrict__ rres,
    int *__restrict__ rdbg, Geo g, DevState *st) {
    if (st->done) return;
    const int count = st->sparse_count;
    if (count == 0) return;
    using Stage = PairStage<D>;
    constexpr int P = Stage::P, XS = Stage::XS, KS = Stage::KS, FS = Stage::FS;
    constexpr int DO = P / 4;  // dimensions of a lane's totals: 4e + sub
    __shared__ Stage s_stage[kBlock / kWave];
    Stage &S = s_stage[threadIdx.x / kWave];
    const int n = g.n, od = g.od, R = g.R, runs = st->runs, lane = __lane_id();
    const int tq = lane >> 2, sub = lane & 3;   // target and lane of the target
    const int j16 = lane & 15, kq = lane >> 4;  // MFMA column (target) and k
    const int nblk = (runs + kBlkRuns - 1) / kBlkRuns, nb = n / kBlkRuns + 1;
    const int nsup = (nblk + kSupBlks - 1) / kSupBlks, ns = n / (kBlkRuns * kSupBlks) + 1;
    const float thr = g.thr_eps, thr_half = g.thr_half, halfcs = 0.5f * g.cs;
    const float box_thr = pb.thr_filter * (1.0f + 0x1p-10f);
    const float box_thr_clamp = pb.thr_clamp * (1.0f + 0x1p-10f);
    const int ntiles = (count + kPairTargets - 1) / kPairTargets;
    bool unsynced = false;
    for (int t = wave_index(); t < ntiles; t = wave_count() + next_tile(&st->ptile_next)) {
        const int k = t * kPairTargets + tq;
        const bool active = k < count;
        const int kk = active ? k : t * kPairTargets;
        const int r = list ? list[kk] : kk;
        const int i = run_start[r];
        const int c0 = point_cell[i];
        const int own = cell_start[c0 + 1] - cell_start[c0];
        float x[D], sml[D], tlo[D], thi[D], a[D];
        float xo[DO], cxo[DO], sxo[DO], sum[DO];
        bool border = false;
        float rho = 0.f;
#pragma unroll
        for (int l = 0; l < D; l++) {
            x[l] = Xs[(long long)l * n + i];
            sml[l] = 0.f;
            border |= on_border(x[l], g.cs);
            tlo[l] = active ? x[l] : __builtin_inff();
            thi[l] = active ? x[l] : -__builtin_inff();
            for (int o = kWave / 2; o > 2; o >>= 1) {
                tlo[l] = fminf(tlo[l], __shfl_xor(tlo[l], o, kWave));
                thi[l] = fmaxf(thi[l], __shfl_xor(thi[l], o, kWave));
            }
            a[l] = 0.5f * (tlo[l] + thi[l]);
            rho = fmaf(thi[l] - tlo[l], thi[l] - tlo[l], rho);
        }
#pragma unroll
        for (int e = 0; e < DO; e++) {
            const int l = 4 * e + sub;
            xo[e] = l < D ? Xs[(long long)l * n + i] : 0.f;
            cxo[e] = cosf(xo[e]);
            sxo[e] = sinf(xo[e]);
            sum[e] = 0.f;
        }
        // the targets' side of the distance product: -2u, 1, |u|^2 - thr
        float bf[KS];
        {
            // |u| <= half the box's diagonal; the sources that matter are
            // within it plus the filter radius
            const float reach = sqrtf(rho) + pb.r;
            const float slack = pb.rounding * (reach * reach + pb.r * pb.r);
            const int from = 4 * j16;
            float u2 = 0.f;
#pragma unroll
            for (int s = 0; s < KS; s++) bf[s] = 0.f;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float u = __shfl(x[l], from, kWave) - a[l];
                u2 = fmaf(u, u, u2);
                if (kq == l % 4) bf[l / 4] = -2.f * u;
            }
            const bool on = t * kPairTargets + j16 < count;
            if (kq == D % 4) bf[D / 4] = 1.f;
            if (kq == (D + 1) % 4) bf[(D + 1) / 4] = on ? u2 - pb.thr_filter - slack : 1e30f;
        }
        int N = 0, half = 0;
        for (int sb0 = 0; sb0 < nsup; sb0 += kWave) {
            const int sbl = sb0 + lane;
            const bool sp = sbl < nsup &&
                            box_near<D>(tlo, thi, sbmin, sbmax, ns, sbl,
                                        sbclamp[sbl] ? box_thr_clamp : box_thr);
            for (unsigned long long ms = __ballot(sp); ms; ms &= ms - 1) {
                const int sb = sb0 + __ffsll((long long)ms) - 1;
                const int bl = sb * kSupBlks + lane;
                const bool bp = bl < nblk &&
                                box_near<D>(tlo, thi, bmin, bmax, nb, bl,
                                            bclamp[bl] ? box_thr_clamp : box_thr);
                for (unsigned long long mb = __ballot(bp); mb; mb &= mb - 1) {
                    const int b = sb * kSupBlks + __ffsll((long long)mb) - 1;
                    const int r0 = b * kBlkRuns;
                    // a block whose runs share one cell c (a dense cell): one
                    // box test of c per target decides for all its runs, unless
                    // c is partial for it or a border target needs its eps/2
                    // count; if no target needs the runs one by one, the block
                    // is not staged, and targets for which c is full add its
                    // totals in the block holding its first run
                    const int bc = bcell[b];
                    if (bc >= 0 && !bclamp[b]) {
                        const int cls = active ? pair_class<D>(x, c0, r0, gr, cell_g, g) : 0;
                        if (!__any(cls == 2 || (cls == 1 && border && bc != c0))) {
                            const int fr = cell_run[bc];
                            if (cls == 1 && fr >= r0 && fr < r0 + kBlkRuns) {
                                const float *row = totals + (long long)bc * 2 * D;
#pragma unroll
                                for (int e = 0; e < DO; e++) {
                                    const int l = 4 * e + sub;
                                    if (l < D) {
                                        const float p1 = row[l] * cxo[e];
                                        const float p2 = row[D + l] * sxo[e];
                                        const float tt = p1 - p2;
                                        sum[e] += tt;
                                    }
                                }
                                if (sub == 0) {
                                    const int cnt = cell_start[bc + 1] - cell_start[bc];
                                    N += cnt;
                                    if (border && bc == c0) half += cnt;
                                }
                            }
                            continue;
                        }
                    }
                    {
                        const int rr = r0 + lane;
                        const bool on = rr < runs;
                        float v2 = 0.f;
                        int fl = 0;
                        if (on) {
                            const int c = rcell[rr];
                            fl = rflag[rr];
                            S.meta[lane] = make_int4(
                                c, fl, rlen[rr], fl & 1 ? cell_start[c + 1] - cell_start[c] : 0);
                        }
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            float v = 0.f;
                            if (on) {
                                const float xq = Xr[(long long)l * n + rr];
                                S.x[lane * XS + l] = xq;
                                S.c[lane * XS + l] =
                                    ((float)gr[(long long)l * n + rr] + 0.5f) * g.cs;
                                v = xq - a[l];
                            }
                            v2 = fmaf(v, v, v2);
                            S.f[lane * FS + l] = v;
                        }
                        // a clamped run is accepted up to its wider radius
                        if (fl & 2) v2 -= pb.thr_clamp - pb.thr_filter;
                        S.f[lane * FS + D] = on ? v2 : 1e30f;
                        S.f[lane * FS + D + 1] = 1.f;
#pragma unroll
                        for (int l = D + 2; l < 4 * KS; l++) S.f[lane * FS + l] = 0.f;
                    }
                    wave_sync();
                    // lane (j16, kq): sign bits of target j16 and sources 16kq .. 16kq+15
                    unsigned bits = 0;
#pragma unroll
                    for (int tau = 3; tau >= 0; tau--) {
                        const float *row =
                            S.f + (16 * (j16 >> 2) + 4 * tau + (j16 & 3)) * FS + kq;
                        f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int s = 0; s < KS; s++)
                            d = __builtin_amdgcn_mfma_f32_16x16x4f32(row[4 * s], bf[s], d, 0, 0, 0);
#pragma unroll
                        for (int q = 3; q >= 0; q--)
                            bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(d[q]), 31);
                    }
                    unsigned long long acc =
                        (unsigned)__shfl((int)bits, tq, kWave) |
                        (unsigned)__shfl((int)bits, tq + 16, kWave) << 16;
                    acc |= (unsigned long long)((unsigned)__shfl((int)bits, tq + 32, kWave) |
                                                (unsigned)__shfl((int)bits, tq + 48, kWave) << 16)
                           << 32;
                    // this lane's runs are the sub-th, (sub+4)-th, ... of the target's
#pragma unroll
                    for (int q = 0; q < 3; q++)
                        if (sub > q) acc &= acc - 1;
                    unsigned long long fullm = 0;  // full cells' first runs
                    while (__any(acc != 0)) {
                        float term[D];
#pragma unroll
                        for (int l = 0; l < D; l++) term[l] = 0.f;
                        if (acc) {
                            const int q = __ffsll((long long)acc) - 1;
                            acc &= acc - 1;
                            acc &= acc - 1;
                            acc &= acc - 1;
                            acc &= acc - 1;
                            float xq[P], cq[P];
                            read_row<D>(S.x + q * XS, xq);
                            read_row<D>(S.c + q * XS, cq);
                            const int4 meta = S.meta[q];
                            float s = 0.f, lg = 0.f, sm = 0.f;
#pragma unroll
                            for (int l = 0; l < D; l++) {
                                xq[l] -= x[l];
                                s += xq[l] * xq[l];
                                const float d = fabsf(x[l] - cq[l]);
                                const float df = d + halfcs, dn = d - halfcs;
                                lg = fmaf(df, df, lg);
                                sm = fmaf(dn, dn, sm);
                            }
                            // sm > thr where the outer coordinates differ by more
                            // than R, up to rounding, which pair_class decides
                            int cls = lg <= pb.lo ? 1 : (sm <= pb.lo ? 2 : 0);
                            if ((lg > pb.lo && lg < pb.hi) || (sm > pb.lo && sm < pb.hi))
                                cls = pair_class<D>(x, c0, r0 + q, gr, cell_g, g);
                            if (cls == 1) {
                                if (meta.y & 1) fullm |= 1ull << q;
                                if (border && meta.x != c0 && s <= thr_half) half += meta.z;
                            } else if (cls == 2 && s <= thr) {
                                const float w = (float)meta.z;  // exact: < 2^24
#pragma unroll
                                for (int l = 0; l < D; l++) term[l] = w * sin_pair<SMALL>(xq[l]);
                                N += meta.z;
                            }
                        }
#pragma unroll
                        for (int l = 0; l < D; l++) {
                            sml[l] = add_quad<0>(sml[l], term[l]);
                            sml[l] = add_quad<1>(sml[l], term[l]);
                            sml[l] = add_quad<2>(sml[l], term[l]);
                            sml[l] = add_quad<3>(sml[l], term[l]);
                        }
                    }
                    // the target's full cells, in order, on all four lanes
                    if (__any(fullm != 0)) {
                        unsigned flo = (unsigned)fullm, fhi = (unsigned)(fullm >> 32);
                        flo |= (unsigned)__shfl_xor((int)flo, 1, kWave);
                        fhi |= (unsigned)__shfl_xor((int)fhi, 1, kWave);
                        flo |= (unsigned)__shfl_xor((int)flo, 2, kWave);
                        fhi |= (unsigned)__shfl_xor((int)fhi, 2, kWave);
                        fullm = flo | (unsigned long long)fhi << 32;
                        while (fullm) {
                            const int q = __ffsll((long long)fullm) - 1;
                            fullm &= fullm - 1;
                            const int4 meta = S.meta[q];
                            const float *row = totals + (long long)meta.x * 2 * D;
#pragma unroll
                            for (int e = 0; e < DO; e++) {
                                const int l = 4 * e + sub;
                                if (l < D) {
                                    const float p1 = row[l] * cxo[e];
                                    const float p2 = row[D + l] * sxo[e];
                                    const float tt = p1 - p2;
                                    sum[e] += tt;
                                }
                            }
                            if (sub == 0) {
                                N += meta.w;
                                if (border && meta.x == c0) half += meta.w;
                            }
                        }
                    }
                    wave_sync();
                }
            }
        }
        N = quad_sum(N);
        half = quad_sum(half);
        if (active) {
            const bool synced = !((!border && N != own) || (border && N != half));
            if (!synced) unsynced = true;
#pragma unroll
            for (int e = 0; e < DO; e++) {
                const int l = 4 * e + sub;
                float part = sml[4 * e];
#pragma unroll
                for (int q = 1; q < 4; q++)
                    if (4 * e + q < D && sub == q) part = sml[4 * e + q];
                if (l < D) {
                    float tt = sum[e] + part;
                    tt = tt / (float)N;
                    rres[(long long)l * n + r] = xo[e] + tt;
                }
            }
            if (rdbg && sub == 0) {
                rdbg[4 * (long long)r + 0] = N;
                rdbg[4 * (long long)r + 1] = half;
                rdbg[4 * (long long)r + 2] = border ? 1 : 0;
                rdbg[4 * (long long)r + 3] = synced ? 1 : 0;
            }
        }
    }
    if (__any(unsynced) && lane == 0) atomicAnd(&st->flag, 0);
}

// Filter radii of the pair update: pairs within eps, with a relative margin of
// 2^-12 for points that cell_coord's FP32 division puts one ulp outside their
// cell's box; for sources with a clamped coordinate (they lie up to 1 - w cs
// outside the box of cell w-1 in each such dimension), eps + sqrt(d)(1 - w cs).
// The MFMA distance: d + 4 FMAs on terms of at most (|u| + |v|)^2 + thr, and as
// many roundings in |u|^2 and |v|^2; 4d + 32 covers them four times over.
// The face distances: both ways of taking them (the reference's from g cs and
// (g+1) cs, here from the cell's centre) are within 2^-24 (4 sqrt(d) / eps +
// d + 10) of the exact ones, relative, near eps; four times that separates
// "surely" from pair_class.
static PairBounds pair_bounds(const Geo &g) {
    PairBounds p;
    p.thr_filter = g.thr_eps * (1.0f + 0x1p-12f);
    const double gap = std::max(0.0, 1.0 - (double)g.w * (double)g.cs);
    const double r = (double)g.eps + std::sqrt((double)g.d) * gap;
    p.thr_clamp = std::max(p.thr_filter, (float)(r * r * (1.0 + 0x1p-10)));
    p.r = (float)(std::sqrt((double)p.thr_clamp) * (1.0 + 0x1p-20));
    p.rounding = (float)((4 * g.d + 32) * 0x1p-24);
    const double m = 0x1p-24 * (16.0 * std::sqrt((double)g.d) / (double)g.eps + 4.0 * g.d + 64.0);
    p.lo = m < 0.5 ? (float)((double)g.thr_eps * (1.0 - m)) : -1.0f;
    p.hi = m < 0.5 ? (float)((double)g.thr_eps * (1.0 + m)) : INFINITY;
    return p;
}

void launch_update_pairs(const Geo &g, GridBufs &b, int *rdbg, DevState *st, hipStream_t s) {
    const long long nblk_max = g.n / kBlkRuns + 1;
    const int waves = kBlock / kWave;
    const int pb = (int)std::min<long long>(16384, (nblk_max + waves - 1) / waves);
    const int sb = (int)std::max<long long>(
        1, std::min<long long>(1024, (nblk_max / kSupBlks + waves) / waves));
    const long long tiles_max = g.n / kPairTargets + 1;
    const int pq = (int)std::min<long long>(kQueueBlocks, (tiles_max + waves - 1) / waves);
    const PairBounds bounds = pair_bounds(g);
    // the summaries' partials are free: 4 d (n + ...) floats for 2 d per cell
    float *totals = b.partial;
    // every filtered pair is closer than 1 in each coordinate
    const bool pair_small = bounds.thr_clamp < 1.0f;
#define PAIR_LAUNCH(DD, SMALL)                                                                  \
    k_update_pairs<DD, SMALL><<<pq, kBlock, 0, s>>>(                                            \
        b.Xs, b.cell_start, b.cell_g, totals, b.run_start, b.point_cell, b.cell_run,            \
        g.pair_mode == kPairAll ? nullptr : b.sparse_runs, b.rcell, b.rflag, b.Xr, b.gr,        \
        b.rlen, b.bmin, b.bmax, b.bclamp, b.bcell, b.sbmin, b.sbmax, b.sbclamp, bounds, b.rres, \
        rdbg, g, st)
#define PAIR_CASE(DD)                                                                          \
    case DD:                                                                                   \
        k_run_boxes<DD><<<pb, kBlock, 0, s>>>(b.Xs, b.run_start, b.point_cell, b.cell_run,     \
                                              b.cell_g, b.Ts, b.Tc, g, st, totals, b.rcell,    \
                                              b.rflag, b.Xr, b.gr, b.rlen, b.bmin, b.bmax,     \
                                              b.bclamp, b.bcell);                              \
        k_super_boxes<DD><<<sb, kBlock, 0, s>>>(b.bmin, b.bmax, b.bclamp, g, st, b.sbmin,      \
                                                b.sbmax, b.sbclamp);                           \
        if (pair_small) PAIR_LAUNCH(DD, true);                                                 \
        else PAIR_LAUNCH(DD, false);                                                           \
        break;
    switch (g.d) {
        EGG_EACH_D(PAIR_CASE)
    }
#undef PAIR_CASE
#undef PAIR_LAUNCH
}

}  // namespace egg
