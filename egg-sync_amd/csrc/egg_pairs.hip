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
// can, and takes the remaining blocks eight at a time (k_update_pairs).
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

typedef float f32x4 __attribute__((ext_vector_type(4)));

// What the pair update reads, by run so that a batch of sources is a few
// coalesced 16-byte loads, and where it lies.
//   rows    [NC][n][4]  position, then the centre of the run's cell: 2d floats
//                       in NC = ceil(2d / 4) chunks
//   meta    [n]         cell, flags (bit 0: first run of its cell, bit 1: a
//                       coordinate clamped into cell w-1), length, points of the
//                       cell (first runs)
//   totals  [n][2d]     sin and cos totals of a cell
//   blo/bhi [d][nb]     bounding boxes of blocks, bflag [nb] whether a block holds
//                       a clamped run, bcell [nb] its cell if its runs share one
//                       (-1 otherwise); slo/shi/sflag the same of superblocks
struct PairData {
    f32x4 *rows;
    int4 *meta;
    float *totals, *blo, *bhi, *slo, *shi;
    int *bflag, *bcell, *sflag;
    int nb, ns;  // strides of the box tables
};

// rows take the summaries' partials (16 d bytes a point of at most 16 NC), meta
// the sort's keys (16 bytes a point), the rest is pair_scratch_bytes.
static PairData pair_data(const Geo &g, const GridBufs &b) {
    const size_t n = (size_t)g.n, d = (size_t)g.d;
    PairData p;
    p.nb = g.n / kBlkRuns + 1;
    p.ns = g.n / (kBlkRuns * kSupBlks) + 1;
    p.rows = (f32x4 *)b.partial;
    p.meta = (int4 *)b.keys_a;
    char *at = b.pair;
    auto take = [&](size_t bytes) {
        char *r = at;
        at += (bytes + 255) & ~(size_t)255;
        return r;
    };
    p.totals = (float *)take(8 * d * n);
    p.blo = (float *)take(4 * d * p.nb);
    p.bhi = (float *)take(4 * d * p.nb);
    p.bflag = (int *)take(4 * (size_t)p.nb);
    p.bcell = (int *)take(4 * (size_t)p.nb);
    p.slo = (float *)take(4 * d * p.ns);
    p.shi = (float *)take(4 * d * p.ns);
    p.sflag = (int *)take(4 * (size_t)p.ns);
    return p;
}

size_t pair_scratch_bytes(size_t n, size_t d) {
    const size_t nb = n / kBlkRuns + 1, ns = n / ((size_t)kBlkRuns * kSupBlks) + 1;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    return al(8 * d * n) + 2 * al(4 * d * nb) + 2 * al(4 * nb) + 2 * al(4 * d * ns) + al(4 * ns);
}

// The runs' rows, the cells' totals (at their first runs) and the blocks' boxes;
// one wavefront per four blocks.  A coordinate that is not a number, or farther out
// than PairBounds::far, becomes `far` in its row: the pair loop evaluates rows of
// runs that its target does not count, with weight 0, which is nothing only of a
// finite term.
template <int D>
__global__ __launch_bounds__(kBlock) void k_run_boxes(
    const float *__restrict__ Xs, const int *__restrict__ run_start,
    const int *__restrict__ point_cell, const int *__restrict__ cell_run,
    const int *__restrict__ cell_start, const int *__restrict__ cell_g,
    const float *__restrict__ Ts, const float *__restrict__ Tc, Geo g, DevState *st, PairData p,
    float far) {
    if (st->done || st->sparse_count == 0) return;
    constexpr int NC = (2 * D + 3) / 4;
    const int n = g.n, runs = st->runs, lane = __lane_id();
    const float wf = (float)g.w;
    for (int b = wave_index(); b * kWave < runs; b += wave_count()) {
        const int r = b * kWave + lane;
        const bool on = r < runs;
        float lo[D], hi[D], row[4 * NC];
        int f = 0, c = -1;
#pragma unroll
        for (int l = 0; l < 4 * NC; l++) row[l] = 0.f;
        if (on) {
            const int i = run_start[r];
            c = point_cell[i];
            bool clamped = false;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float x = Xs[(long long)l * n + i];
                lo[l] = hi[l] = x;
                clamped |= x / g.cs >= wf;  // cell_coord's clamp of w to w-1
                row[l] = fabsf(x) <= far ? x : far;
                row[D + l] = ((float)cell_g[(long long)l * n + c] + 0.5f) * g.cs;
            }
            f = (cell_run[c] == r ? 1 : 0) | (clamped ? 2 : 0);
            p.meta[r] = make_int4(c, f, run_start[r + 1] - i,
                                  f & 1 ? cell_start[c + 1] - cell_start[c] : 0);
#pragma unroll
            for (int k = 0; k < NC; k++) {
                const f32x4 q = {row[4 * k], row[4 * k + 1], row[4 * k + 2], row[4 * k + 3]};
                p.rows[(long long)k * n + r] = q;
            }
            if (f & 1) {
#pragma unroll
                for (int l = 0; l < D; l++) {
                    p.totals[(long long)c * 2 * D + l] = Ts[(long long)l * n + c];
                    p.totals[(long long)c * 2 * D + D + l] = Tc[(long long)l * n + c];
                }
            }
        } else {
#pragma unroll
            for (int l = 0; l < D; l++) {
                lo[l] = __builtin_inff();
                hi[l] = -__builtin_inff();
            }
        }
        const unsigned long long mine = 0xffffull << (lane & 48);  // the block's lanes
        const bool any_clamp = (__ballot((f & 2) != 0) & mine) != 0;
        const int c_first = __shfl(c, lane & 48, kWave);
        const bool one_cell = (__ballot(on && c != c_first) & mine) == 0;
        const bool writes = on && (lane & 15) == 0;
        const int blk = r / kBlkRuns;
#pragma unroll
        for (int l = 0; l < D; l++) {
            for (int o = kBlkRuns / 2; o > 0; o >>= 1) {
                lo[l] = fminf(lo[l], __shfl_xor(lo[l], o, kWave));
                hi[l] = fmaxf(hi[l], __shfl_xor(hi[l], o, kWave));
            }
            if (writes) {
                p.blo[(long long)l * p.nb + blk] = lo[l];
                p.bhi[(long long)l * p.nb + blk] = hi[l];
            }
        }
        if (writes) {
            p.bflag[blk] = any_clamp ? 1 : 0;
            p.bcell[blk] = one_cell ? c_first : -1;
        }
    }
}

// Bounding box of every superblock of kSupBlks blocks, and whether it holds a
// clamped run.
template <int D>
__global__ __launch_bounds__(kBlock) void k_super_boxes(Geo g, DevState *st, PairData p) {
    if (st->done || st->sparse_count == 0) return;
    const int nblk = (st->runs + kBlkRuns - 1) / kBlkRuns;
    const int nsup = (nblk + kSupBlks - 1) / kSupBlks;
    for (int sb = wave_index(); sb < nsup; sb += wave_count()) {
        const int b = sb * kSupBlks + __lane_id();
        const bool on = b < nblk;
        const bool any_clamp = __any(on && p.bflag[b] != 0);
#pragma unroll
        for (int l = 0; l < D; l++) {
            float lo = on ? p.blo[(long long)l * p.nb + b] : __builtin_inff();
            float hi = on ? p.bhi[(long long)l * p.nb + b] : -__builtin_inff();
            for (int o = kWave / 2; o > 0; o >>= 1) {
                lo = fminf(lo, __shfl_xor(lo, o, kWave));
                hi = fmaxf(hi, __shfl_xor(hi, o, kWave));
            }
            if (__lane_id() == 0) {
                p.slo[(long long)l * p.ns + sb] = lo;
                p.shi[(long long)l * p.ns + sb] = hi;
            }
        }
        if (__lane_id() == 0) p.sflag[sb] = any_clamp ? 1 : 0;
    }
}

// Whether box k of a (lo, hi) table ([D][stride]) lies within squared
// distance thr of the box a (D lower, D upper bounds; thr_clamp if the box holds
// a clamped run).  Box distances round like the point distances they bound; the
// caller's thresholds carry a relative margin of 2^-10 for that.
template <int D>
__device__ __forceinline__ bool box_near(const float (&a)[2 * D], const float *__restrict__ blo,
                                         const float *__restrict__ bhi, long long stride, int k,
                                         float thr) {
    float s = 0.f;
#pragma unroll
    for (int l = 0; l < D; l++) {
        const float gap =
            fmaxf(0.f, fmaxf(blo[l * stride + k] - a[D + l], a[l] - bhi[l * stride + k]));
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
    float lo, hi;                 // face distances less D h^2 surely <= / > thr_eps
    float far;                    // points with a coordinate beyond it are near no other
};

constexpr int kPairTargets = 16;  // targets of a tile, four lanes each
constexpr int kBatchBlks = 8;     // source blocks of a batch
constexpr int kBatch = kBatchBlks * kBlkRuns;

// A batch of source runs in LDS (PairData's rows and meta), and per target the
// accepted ones of them, in order.
template <int D>
struct PairStage {
    static constexpr int NC = (2 * D + 3) / 4;
    f32x4 rows[NC][kBatch];
    int4 meta[kBatch];
    float cs[2 * D][kPairTargets];  // cos and sin of the targets
    float box[2 * D];               // the tile's box
    unsigned char list[kPairTargets][kBatch];
};

// The reference's decision for cell c as seen from the target at sorted position
// i in cell c0 (EGG_SynC.cu:612-634): 0 not counted (or not in the neighbour
// list), 1 full, 2 partial.  A loop over memory: it is taken rarely, and its
// registers would be the pair loop's.
__device__ __forceinline__ int pair_class(const float *__restrict__ Xs, int i, int c0, int c,
                                          const int *__restrict__ cell_g, const Geo &g) {
    bool win = true;
    float sm = 0.f, lg = 0.f;
#pragma unroll 1
    for (int l = 0; l < g.d; l++) {
        const float x = Xs[(long long)l * g.n + i];
        const int gc = cell_g[(long long)l * g.n + c];
        if (l < g.od) {
            const int dg = gc - cell_g[(long long)l * g.n + c0];
            if (dg > g.R || dg < -g.R) win = false;
        }
        float s1, l1;
        box_dist<1>(&gc, &x, g.cs, s1, l1);
        sm += s1;
        lg += l1;
    }
    return !win ? 0 : (lg <= g.thr_eps ? 1 : (sm <= g.thr_eps ? 2 : 0));
}

// Lane I of each group of four lanes' v, on all four.
template <int I>
__device__ __forceinline__ int quad_lane(int v) {
    return __builtin_amdgcn_mov_dpp(v, I * 0x55, 0xf, 0xf, true);
}

__device__ __forceinline__ int quad_sum(int v) {
    return quad_lane<0>(v) + quad_lane<1>(v) + quad_lane<2>(v) + quad_lane<3>(v);
}

// Adds the terms of a target's four lanes to its sum one after another; every
// lane keeps the whole sum.
__device__ __forceinline__ float add_quad(float s, float v) {
    const int t = __float_as_int(v);
    s += __int_as_float(quad_lane<0>(t));
    s += __int_as_float(quad_lane<1>(t));
    s += __int_as_float(quad_lane<2>(t));
    return s + __int_as_float(quad_lane<3>(t));
}

// One wavefront per tile of 16 targets; lanes 4t .. 4t + 3 serve target t.  Blocks
// that survive the pruning are collected; per batch of eight (128 source runs):
//  1. the squared distances of all 2,048 pairs by v_mfma_f32_16x16x4_f32,
//     sum_l (-2 u_l v_l + v_l^2) + (|u|^2 - thr) relative to the tile's centre;
//     its sign bits are the accepted pairs (one v_alignbit each).  thr holds the
//     filter radius and a bound on the product's rounding, so that no pair within
//     the filter is missed; what is accepted beyond it fails the tests below;
//  2. every target's accepted runs are listed in LDS, in order; its four lanes
//     take them in turns of four and evaluate the FP32 distance, the cell's class
//     and sin(x_q - x).  The class comes from the distances to the cell's far and
//     near faces by its centre, sum d^2 + D h^2 +- 2 h sum |d| (h half the side),
//     and where those lie within rounding of eps, from the reference's own box
//     test (pair_class);
//  3. the four terms are added one after another (DPP broadcasts within the four
//     lanes).  The matrix cores can do it too, bit for bit (four FMAs in ascending
//     k), but v_mfma_f32_16x16x4_f32 takes 32 cycles of the same SIMD for what the
//     four adds of a dimension take 16 for: +20% time;
//  4. full cells met at their first run add their totals the same way.
// Blocks of 16 runs prune better than blocks of 64, batches of 128 keep a target's
// lanes busier, and 16 targets a tile give a wavefront per 16 runs where n is
// small.  Bound by the VALU: ~190 instructions at d = 8 per 64 evaluated pairs, of
// which 37 are in use on average in the first pass (the targets' counts differ).
// n = 250,000, d = 8, eps = 0.1: 65 ms a pass with a lane per target and the
// totals read (and sinf / cosf taken) inside the pair loop, 35 with blocks of 64,
// 28 here; n = 14,980, d = 14: 7.3 ms (234 wavefronts), 1.6, 1.1.
// SMALL: every pair the filter passes is closer than 1 in each coordinate
// (filter radius below 1), so sin(x_q - x) takes the polynomial.
// The register budget keeps 4 wavefronts a SIMD up to d = 3, 3 up to d = 8.
template <int D, bool SMALL>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(D <= 3 ? 4 : (D <= 8 ? 3 : 1)))) void k_update_pairs(
    const float *__restrict__ Xs, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const int *__restrict__ run_start,
    const int *__restrict__ point_cell, const int *__restrict__ cell_run,
    const int *__restrict__ list, PairData p, PairBounds pb, float *__restrict__ rres,
    int *__restrict__ rdbg, Geo g, DevState *st) {
    if (st->done) return;
    const int count = st->sparse_count;
    if (count == 0) return;
    using Stage = PairStage<D>;
    constexpr int NC = Stage::NC;
    constexpr int KD = (D + 3) / 4;  // MFMA steps over the dimensions
    __shared__ Stage s_stage[kBlock / kWave];
    Stage &S = s_stage[threadIdx.x / kWave];
    const float *S_f = reinterpret_cast<const float *>(S.rows);
    const int n = g.n, runs = st->runs, lane = __lane_id();
    const int tq = lane >> 2, sub = lane & 3;   // target and lane of the target
    const int j16 = lane & 15, kq = lane >> 4;  // MFMA column (target) and k
    const int nblk = (runs + kBlkRuns - 1) / kBlkRuns;
    const int nsup = (nblk + kSupBlks - 1) / kSupBlks;
    // the pair loop's constants, kept in vector registers: the scalar ones are
    // short, and a spilled one costs the loop a v_readlane
    float thr = g.thr_eps, thr_half = g.thr_half, lo = pb.lo, hi = pb.hi, cs = g.cs;
    __asm__ volatile("" : "+v"(thr), "+v"(thr_half), "+v"(lo), "+v"(hi), "+v"(cs));
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
        // full cells' totals and partial cells' terms, on each of the four lanes
        float x[D], sum[D], sml[D];
        bool border = false, near = active;  // near: not a target that counts nothing
        float rho = 0.f;
#pragma unroll
        for (int l = 0; l < D; l++) {
            x[l] = Xs[(long long)l * n + i];
            sum[l] = sml[l] = 0.f;
            border |= on_border(x[l], g.cs);
            near = near && fabsf(x[l]) <= pb.far;
        }
#pragma unroll
        for (int l = 0; l < D; l++) {
            float tlo = near ? x[l] : __builtin_inff();
            float thi = near ? x[l] : -__builtin_inff();
            for (int o = kWave / 2; o > 2; o >>= 1) {
                tlo = fminf(tlo, __shfl_xor(tlo, o, kWave));
                thi = fmaxf(thi, __shfl_xor(thi, o, kWave));
            }
            S.box[l] = tlo;  // every lane, the same value
            S.box[D + l] = thi;
            rho = fmaf(thi - tlo, thi - tlo, rho);
        }
        wave_sync();
        if (sub == 0) {
#pragma unroll
            for (int l = 0; l < D; l++) {
                S.cs[l][tq] = cosf(x[l]);
                S.cs[D + l][tq] = sinf(x[l]);
            }
        }
        const bool any_border = __any(border);
        // the distance product: anchors af of the lane's dimensions 4s + kq, the
        // targets' side -2u, and its constant |u|^2 - thr (on lanes kq = 0)
        float af[KD], bf[KD], b1 = 0.f;
        {
            // |u| <= half the box's diagonal; the sources that matter are
            // within it plus the filter radius
            const float reach = sqrtf(rho) + pb.r;
            const float slack = pb.rounding * (reach * reach + pb.r * pb.r);
            float u2 = 0.f;
#pragma unroll
            for (int s = 0; s < KD; s++) af[s] = bf[s] = 0.f;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float al = 0.5f * (S.box[l] + S.box[D + l]);
                const float u = __shfl(x[l], 4 * j16, kWave) - al;
                u2 = fmaf(u, u, u2);
                if (kq == l % 4) {
                    af[l / 4] = al;
                    bf[l / 4] = -2.f * u;
                }
            }
            const bool on = __shfl(near, 4 * j16, kWave);
            if (kq == 0) b1 = on ? u2 - pb.thr_filter - slack : 1e30f;
        }
        const float one_last = 4 * (KD - 1) + kq < D ? 1.f : 0.f;
        int N = 0, half = 0;
        // blocks still to come: superblocks of ms, blocks of mb; `pend` holds on
        // lane k the k-th block collected (bit 30: it has a clamped run)
        unsigned long long ms = 0, mb = 0;
        int sb_next = 0, sbase = 0, bbase = 0;
        // the last cell whose runs filled a whole block: the targets' classes
        int last_bc = -1, last_cls = 0;
        bool last_need = false;
        for (;;) {
            int np = 0, pend = 0;
            while (np < kBatchBlks) {
                if (!mb) {
                    while (!ms && sb_next < nsup) {
                        const int sbl = sb_next + lane;
                        const bool sp = sbl < nsup &&
                                        box_near<D>(S.box, p.slo, p.shi, p.ns, sbl,
                                                    p.sflag[sbl] ? box_thr_clamp : box_thr);
                        ms = __ballot(sp);
                        sbase = sb_next;
                        sb_next += kWave;
                    }
                    if (!ms) break;
                    bbase = (sbase + __ffsll((long long)ms) - 1) * kSupBlks;
                    ms &= ms - 1;
                    const int bl = bbase + lane;
                    const bool bp = bl < nblk &&
                                    box_near<D>(S.box, p.blo, p.bhi, p.nb, bl,
                                                p.bflag[bl] ? box_thr_clamp : box_thr);
                    mb = __ballot(bp);
                    continue;
                }
                const int b = bbase + __ffsll((long long)mb) - 1;
                mb &= mb - 1;
                const int bc = p.bcell[b], clamped = p.bflag[b];
                if (bc >= 0 && !clamped) {
                    // a block whose runs share one cell (a dense cell): one box
                    // test per target decides for all its runs, unless the cell
                    // is partial for it or a border target needs its eps/2 count.
                    // If no target needs the runs one by one, the block is passed
                    // by, unless the cell's first run is in it and some target is
                    // to add the cell's totals there
                    if (bc != last_bc) {
                        last_bc = bc;
                        last_cls = active ? pair_class(Xs, i, c0, bc, cell_g, g) : 0;
                        last_need = __any(last_cls == 2 || (last_cls == 1 && border && bc != c0));
                    }
                    if (!last_need) {
                        const int fr = cell_run[bc] - b * kBlkRuns;
                        if (fr < 0 || fr >= kBlkRuns || !__any(last_cls == 1)) continue;
                    }
                }
                if (lane == np) pend = b | (clamped ? 1 << 30 : 0);
                np++;
            }
            if (np == 0) break;
            // the batch to LDS; slots past the last block or run repeat run
            // runs - 1 and are masked out below
#pragma unroll
            for (int h = 0; h < kBatch / kWave; h++) {
                const int slot = h * 4 + kq;
                const int b = __shfl(pend, slot, kWave) & 0x3fffffff;
                const unsigned rr = (unsigned)min(b * kBlkRuns + j16, runs - 1);
#pragma unroll
                for (int q = 0; q < NC; q++)
                    S.rows[q][h * kWave + lane] = (p.rows + (long long)q * n)[rr];
                S.meta[h * kWave + lane] = p.meta[rr];
            }
            wave_sync();
            // lane (j16, kq): bit 4 s + q = target j16 accepts run 4 kq + q of
            // block s
            unsigned bits = 0;
#pragma unroll
            for (int s = kBatchBlks - 1; s >= 0; s--) {
                if (s >= np) continue;
                f32x4 d = {0.f, 0.f, 0.f, 0.f};
                float v[KD];
#pragma unroll
                for (int q = 0; q < KD; q++) {
                    v[q] = S_f[(q * kBatch + s * kBlkRuns + j16) * 4 + kq] - af[q];
                    d = __builtin_amdgcn_mfma_f32_16x16x4f32(v[q], bf[q], d, 0, 0, 0);
                }
#pragma unroll
                for (int q = 0; q < KD; q++)
                    d = __builtin_amdgcn_mfma_f32_16x16x4f32(v[q] * v[q], q + 1 < KD ? 1.f : one_last,
                                                             d, 0, 0, 0);
                // a block with a clamped run is accepted up to the wider radius
                const bool wide = __builtin_amdgcn_readlane(pend, s) >> 30;
                const float wider = wide && kq == 0 ? pb.thr_clamp - pb.thr_filter : 0.f;
                d = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, b1 - wider, d, 0, 0, 0);
#pragma unroll
                for (int q = 3; q >= 0; q--)
                    bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(d[q]), 31);
            }
            // lane (tq, sub): the target's bits of blocks 2 sub and 2 sub + 1
            unsigned own_bits = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const unsigned two = (unsigned)__shfl((int)bits, tq + 16 * q, kWave) >> (8 * sub);
                own_bits |= (two & 15u) << (4 * q) | ((two >> 4) & 15u) << (16 + 4 * q);
            }
            {
                // runs past the end of the last block
                const int r0 = runs - (__shfl(pend, 2 * sub, kWave) & 0x3fffffff) * kBlkRuns;
                const int r1 = runs - (__shfl(pend, 2 * sub + 1, kWave) & 0x3fffffff) * kBlkRuns;
                if (r0 < kBlkRuns) own_bits &= ~0u << 16 | ((1u << r0) - 1u);
                if (r1 < kBlkRuns) own_bits &= 0xffffu | ((1u << r1) - 1u) << 16;
            }
            // the target's list of accepted places in the batch
            const int mine = __popc(own_bits);
            const int n0 = quad_lane<0>(mine), n1 = quad_lane<1>(mine), n2 = quad_lane<2>(mine);
            const int tot = n0 + n1 + n2 + quad_lane<3>(mine);
            int at = (sub > 0 ? n0 : 0) + (sub > 1 ? n1 : 0) + (sub > 2 ? n2 : 0);
            while (own_bits) {
                S.list[tq][at++] = (unsigned char)(32 * sub + __builtin_ctz(own_bits));
                own_bits &= own_bits - 1;
            }
            wave_sync();
            // the accepted pairs, straight-line code: lanes past the end of their
            // list evaluate some staged run with weight 0
            int nfull = 0;  // full cells' first runs met; listed in place of read entries
            for (int rank = sub; __any(rank < tot); rank += 4) {
                const bool in = rank < tot;
                const int q = S.list[tq][min(rank, kBatch - 1)] & (kBatch - 1);
                float row[4 * NC];
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    const f32x4 v = S.rows[c][q];
#pragma unroll
                    for (int e = 0; e < 4; e++) row[4 * c + e] = v[e];
                }
                const int4 meta = S.meta[q];
                float s = 0.f, d2 = 0.f, d1 = 0.f;
#pragma unroll
                for (int l = 0; l < D; l++) {
                    row[l] -= x[l];
                    s += row[l] * row[l];
                    const float d = row[D + l] - x[l];
                    d2 = fmaf(d, d, d2);
                    d1 += fabsf(d);
                }
                const float lg = fmaf(cs, d1, d2), sm = fmaf(-cs, d1, d2);
                bool full = lg <= lo, part = !full && sm <= lo;
                // sm > thr where the outer coordinates differ by more than R, up to
                // rounding, which pair_class decides
                const bool unsure = in && ((lg > lo && lg < hi) || (sm > lo && sm < hi));
                if (__any(unsure)) {
                    if (unsure) {
                        const int cls = pair_class(Xs, i, c0, meta.x, cell_g, g);
                        full = cls == 1;
                        part = cls == 2;
                    }
                }
                const int len = in && part && s <= thr ? meta.z : 0;
                N += len;
                if (__any(len > 0)) {
                    const float w = (float)len;  // exact: < 2^24
#pragma unroll
                    for (int l = 0; l < D; l++)
                        sml[l] = add_quad(sml[l], w * sin_pair<SMALL>(row[l]));
                }
                full = full && in;
                if (any_border) {
                    if (full && border && meta.x != c0 && s <= thr_half) half += meta.z;
                }
                const bool first = full && (meta.y & 1);
                const unsigned quad = (unsigned)(__ballot(first) >> (lane & 60)) & 15u;
                if (first)
                    S.list[tq][nfull + __popc(quad & ((1u << sub) - 1u))] = (unsigned char)q;
                nfull += __popc(quad);
            }
            // the target's full cells, in order, its lanes in turns of four
            for (int rank = sub; __any(rank < nfull); rank += 4) {
                float term[D];
#pragma unroll
                for (int l = 0; l < D; l++) term[l] = 0.f;
                if (rank < nfull) {
                    const int4 meta = S.meta[S.list[tq][rank]];
                    const float *row = p.totals + (long long)meta.x * 2 * D;
#pragma unroll
                    for (int l = 0; l < D; l++) {
                        const float p1 = row[l] * S.cs[l][tq];
                        const float p2 = row[D + l] * S.cs[D + l][tq];
                        term[l] = p1 - p2;
                    }
                    N += meta.w;
                    if (border && meta.x == c0) half += meta.w;
                }
#pragma unroll
                for (int l = 0; l < D; l++) sum[l] = add_quad(sum[l], term[l]);
            }
            wave_sync();
        }
        N = quad_sum(N);
        half = quad_sum(half);
        if (active) {
            const bool synced = !((!border && N != own) || (border && N != half));
            if (!synced) unsynced = true;
            if (sub == 0) {
#pragma unroll
                for (int l = 0; l < D; l++) {
                    float tt = sum[l] + sml[l];
                    tt = tt / (float)N;
                    rres[(long long)l * n + r] = x[l] + tt;
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
// The face distances: the reference takes them from g cs and (g+1) cs, the pair
// loop from the cell's centre as sum d^2 +- 2 h sum |d| + D h^2.  Near eps both are
// within 2^-24 (4 sqrt(d) / eps + 3 d + 10) of the exact ones, relative (positions
// round by 2^-24, and sum d^2 + 2 h sum |d| stays below 2.3 eps^2 where the near
// distance is eps); four times that separates "surely" from pair_class.  lo and hi
// bound the distances less D h^2.
static PairBounds pair_bounds(const Geo &g) {
    PairBounds p;
    p.thr_filter = g.thr_eps * (1.0f + 0x1p-12f);
    const double gap = std::max(0.0, 1.0 - (double)g.w * (double)g.cs);
    const double r = (double)g.eps + std::sqrt((double)g.d) * gap;
    p.thr_clamp = std::max(p.thr_filter, (float)(r * r * (1.0 + 0x1p-10)));
    p.r = (float)(std::sqrt((double)p.thr_clamp) * (1.0 + 0x1p-20));
    // what a target counts lies in the grid, or within the filter radius of a target
    // within eps of it
    p.far = 2.0f + 2.0f * (g.eps + p.r);
    p.rounding = (float)((4 * g.d + 32) * 0x1p-24);
    const double m = 0x1p-24 * (16.0 * std::sqrt((double)g.d) / (double)g.eps + 12.0 * g.d + 64.0);
    const double dh2 = 0.25 * g.d * (double)g.cs * (double)g.cs;
    p.lo = m < 0.5 ? (float)((double)g.thr_eps * (1.0 - m) - dh2) : -INFINITY;
    p.hi = m < 0.5 ? (float)((double)g.thr_eps * (1.0 + m) - dh2) : INFINITY;
    return p;
}

void launch_update_pairs(const Geo &g, GridBufs &b, int *rdbg, DevState *st, hipStream_t s) {
    const int waves = kBlock / kWave;
    const int pb = (int)std::min<long long>(16384, ((long long)g.n / kWave + waves) / waves);
    const long long nsup_max = g.n / (kBlkRuns * kSupBlks) + 1;
    const int sb = (int)std::min<long long>(1024, (nsup_max + waves - 1) / waves);
    const long long tiles_max = g.n / kPairTargets + 1;
    const int pq = (int)std::min<long long>(kQueueBlocks, (tiles_max + waves - 1) / waves);
    const PairBounds bounds = pair_bounds(g);
    const PairData data = pair_data(g, b);
    // every filtered pair is closer than 1 in each coordinate
    const bool pair_small = bounds.thr_clamp < 1.0f;
#define PAIR_LAUNCH(DD, SMALL)                                                                \
    k_update_pairs<DD, SMALL><<<pq, kBlock, 0, s>>>(                                          \
        b.Xs, b.cell_start, b.cell_g, b.run_start, b.point_cell, b.cell_run,                  \
        pairs_take_all(g.pair_mode, g.d) ? nullptr : b.sparse_runs, data, bounds, b.rres, rdbg, g, st)
#define PAIR_CASE(DD)                                                                          \
    case DD:                                                                                   \
        k_run_boxes<DD><<<pb, kBlock, 0, s>>>(b.Xs, b.run_start, b.point_cell, b.cell_run,     \
                                              b.cell_start, b.cell_g, b.Ts, b.Tc, g, st,       \
                                              data, bounds.far);                               \
        k_super_boxes<DD><<<sb, kBlock, 0, s>>>(g, st, data);                                  \
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
