// Grid build and per-cell summaries (EGG_SynC.cu:248-366), gfx950.
//
// build_the_grid of the reference (two-level counting sort with atomic slot
// order and linear slot searches) becomes: per-point bit-field cell keys ->
// stable sort -> one pass that gathers the positions into cell-sorted SoA order,
// finds and counts the heads, and writes the cell table and the outer-cell ranges.  Cells and the
// points within a cell come out in a deterministic order.
//
// kernel_inner_grid_stats (float atomics) becomes a deterministic wave-level
// Kahan-compensated reduction per cell chunk (<= 256 points), with a second
// pass combining the chunks of large cells (one wavefront per cell).
//
// An iteration's build is a handful of launches (keys, sort, tables, summaries,
// groups), because a launch costs 4 to 5 us whatever it does: for the data sets of
// a few thousand points, and for every data set's last iterations, that is most of
// the time.
#include <algorithm>

#include "egg_internal.h"
#include "egg_scan.h"
#include "egg_wave.h"

namespace egg {

__global__ void k_aos_to_soa(const float *__restrict__ aos, float *__restrict__ soa,
                             int *__restrict__ perm, int n, int d) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        for (int l = 0; l < d; l++) soa[(long long)l * n + i] = aos[i * d + l];
        if (perm) perm[i] = (int)i;
    }
}

__global__ void k_soa_to_aos_by_perm(const float *__restrict__ soa, const int *__restrict__ perm,
                                     float *__restrict__ aos, int n, int d) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const long long p = perm[i];
        for (int l = 0; l < d; l++) aos[p * d + l] = soa[(long long)l * n + i];
    }
}

static inline int grid_for(long long n, int per_block = kBlock, int cap = 65536) {
    long long b = (n + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (int)b;
}

void launch_aos_to_soa(const float *aos, float *soa, int *perm, int n, int d, hipStream_t s) {
    k_aos_to_soa<<<grid_for(n), kBlock, 0, s>>>(aos, soa, perm, n, d);
}

void launch_soa_to_aos_by_perm(const float *soa, const int *perm, float *aos, int n, int d,
                               hipStream_t s) {
    k_soa_to_aos_by_perm<<<grid_for(n), kBlock, 0, s>>>(soa, perm, aos, n, d);
}

// Key bit fields: [outer | g_od | ... | g_{d-1} | sub_0 ... sub_{d-1} | hash],
// least significant last, so numeric key order = lexicographic (outer, g_od,
// ..., g_{d-1}, sub_0, ..., sub_{d-1}, position hash); the split bits and the
// hash are present when sub_bits / hash_bits > 0.
__device__ __forceinline__ void put_bits(uint64_t (&w)[kMaxKW], uint64_t v, int shift,
                                         int width) {
    const int q = shift >> 6, o = shift & 63;
#pragma unroll
    for (int k = 0; k < kMaxKW; k++) {
        if (k == q) w[k] |= v << o;
        if (k == q + 1 && o + width > 64) w[k] |= v >> (64 - o);  // o > 0 here: width <= 32
    }
}

// Sort keys of the grid build, one per element: per run of the previous
// grid when its runs are valid (every point of a run has the run's key, and
// runs are contiguous in X's order, so a stable sort of the runs expands to
// the stable sort of the points), else per point.
template <int D>
__global__ __launch_bounds__(kBlock) void k_keys(const float *__restrict__ X, Geo g,
                                                 const int *__restrict__ run_start,
                                                 uint64_t *__restrict__ keys,
                                                 int *__restrict__ ob, int *__restrict__ oe,
                                                 DevState *st, const DevState *st_loop,
                                                 bool begin) {
    if (st_loop && st_loop->done) return;
    const int n = g.n;
    // the outer cells' ranges start empty (k_tables fills the occupied ones)
    for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < g.O; o += gridDim.x * blockDim.x) {
        ob[o] = 0;
        oe[o] = 0;
    }
    const bool valid = st->runs_valid != 0;
    const int m = valid ? st->runs : n;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (begin) reset_pass_state(st);
        st->sort_m = m;
        st->sort_hist = 256 * max(1, (m + kSortTile - 1) / kSortTile);
        // m == n: every run is one point, run r is point r, as in a point sort
        st->lens_m = m < n ? m : 0;
    }
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < m; e += gridDim.x * blockDim.x) {
        const int i = valid ? run_start[e] : e;
        int c[D];
        float x[D];
#pragma unroll
        for (int l = 0; l < D; l++) {
            x[l] = X[(long long)l * n + i];
            c[l] = cell_coord(x[l], g.cs, g.w);
        }
        uint64_t kw[kMaxKW] = {};
        int shift = 0;
        if (g.hash_bits) {
            uint32_t h = 0x9E3779B9u;
#pragma unroll
            for (int l = 0; l < D; l++) h = pos_hash_step(h, __float_as_uint(x[l]));
            h = pos_hash_final(h);
            put_bits(kw, (uint64_t)(h & ((1u << g.hash_bits) - 1u)), 0, g.hash_bits);
            shift = g.hash_bits;
        }
        if (g.sub_bits) {
            // split bits, sub_{d-1} least significant
#pragma unroll
            for (int l = D - 1; l >= 0; l--) {
                put_bits(kw, x[l] >= cell_mid(c[l], g.cs) ? 1u : 0u, shift, 1);
                shift += 1;
            }
        }
#pragma unroll
        for (int l = D - 1; l >= 0; l--) {
            if (l >= g.od) {
                put_bits(kw, (uint64_t)c[l], shift, g.bits_w);
                shift += g.bits_w;
            }
        }
        uint64_t outer = 0;
#pragma unroll
        for (int l = 0; l < D; l++)
            if (l < g.od) outer += (uint64_t)c[l] * (uint64_t)g.wpow[l];
        put_bits(kw, outer, shift, g.bits_o);
#pragma unroll
        for (int k = 0; k < kMaxKW; k++)
            if (k < g.kw) keys[(long long)k * n + e] = kw[k];
    }
}

// Where each sorted run's points go: sorted position q holds run sidx[q] of the
// previous grid; off[q] is the scan of the lengths, src[q] its first old position.
struct RunScan {
    const int *sidx, *run_start;
    int *off, *src;
    const DevState *st;
    __device__ int count() const { return st->lens_m; }
    __device__ void load(int q, int (&v)[1]) const {
        const int r = sidx ? sidx[q] : q;
        v[0] = run_start[r + 1] - run_start[r];
    }
    __device__ void store(int q, const int (&)[1], const int (&ex)[1]) const {
        off[q] = ex[0];
        src[q] = run_start[sidx ? sidx[q] : q];
    }
    __device__ void finish(const int (&)[1]) const {}
};

// The last of the m sorted offsets off[0 .. m) (off[0] = 0) that is <= i; one
// wavefront, uniform i, 64 probes a step.
__device__ __forceinline__ int wave_last_le(const int *__restrict__ off, int m, int i) {
    const int lane = __lane_id();
    int lo = 0, hi = m;
    while (hi - lo > 1) {
        const int step = (hi - lo + kWave - 1) / kWave;
        const long long q = lo + (long long)lane * step;
        const int below = __popcll(__ballot(q < hi && off[min(q, (long long)hi - 1)] <= i));
        lo += (below - 1) * step;
        hi = min(hi, lo + step);
    }
    return lo;
}

// The grid's tables, from the sort to the first position of every cell, sub-cell
// and run, in one pass over the points (a scan tile of sorted positions a
// workgroup, kRows rows of 64 a wavefront).  The sort ordered st->sort_m elements: runs of
// the previous grid (st->lens_m > 0; sorted run q's points go to [off[q], off[q] +
// length) in their previous order) or points.  First the rows are gathered into
// sorted order, and a position is a head where it differs from the one before it:
// in a cell coordinate (cell), in a cell coordinate or a split bit (sub-cell; the
// sort key holds both above the hash, so equal ones are neighbours), bitwise (run).
// Ballots count the heads, look-back joins the tiles, and each head then writes its
// row of the tables: cells' first position, coordinates, outer id, first run and
// sub-cell; sub-cells' first position, fine coordinates 2g + split bit, first run;
// runs' first position; and the cell ranges of the outer cells where the outer id
// changes.  Bound by the gather on a first pass in random order (a memory line per
// coordinate and point), by latency and the launch on small grids.  In place of nine
// launches that passed flags and scans through memory (about 290 us at n = 1,000,000,
// d = 3, 45 us of launches alone at n = 2,000): 87 us and 11 us.
template <int D, int kRows>
__global__ __launch_bounds__(kBlock) void k_tables(GridBufs b, const int *__restrict__ sidx,
                                                   Geo g, DevState *st, const DevState *st_loop,
                                                   bool keep_runs) {
    if (st_loop && st_loop->done) return;
    constexpr int kWaves = kBlock / kWave;
    constexpr int kUnroll = D <= 4 ? 4 : 1;  // rows in flight
    __shared__ unsigned long long s_mask[kWaves][kRows][3];
    __shared__ int s_outer[kWaves][kRows * kWave + 1];  // from the position before the wave's first
    __shared__ int s_cnt[kWaves][3], s_tot[3], s_pre[3], s_tile;
    const float *__restrict__ X = b.X;
    const int n = g.n, nb = gridDim.x, lane = __lane_id(), wave = threadIdx.x / kWave;
    const bool subs = g.sub_bits != 0;
    int tile = 0;
    unsigned seq = 0;
    if (nb > 1) tile = lb_begin(b.scan_tmp, &s_tile, seq);
    const int base = __builtin_amdgcn_readfirstlane((tile * kWaves + wave) * kRows * kWave);
    const int m = st->lens_m;  // 0: the sort ordered points
    int qlo = 0, qhi = 0;      // sorted runs of the wave's positions and the one before
    if (m > 0 && base < n) {
        qlo = wave_last_le(b.run_off, m, max(base - 1, 0));
        qhi = wave_last_le(b.run_off, m, min(base + kRows * kWave, n) - 1);
    }
    auto source = [&](int i) {
        if (m == 0) return sidx ? sidx[i] : i;
        int lo = qlo, hi = qhi;  // the last q with off[q] <= i
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (b.run_off[mid] <= i) lo = mid;
            else hi = mid - 1;
        }
        return b.run_src[lo] + (i - b.run_off[lo]);
    };
    // fine coordinate 2 cell + split bit
    auto fine = [&](float x) {
        const int c = cell_coord(x, g.cs, g.w);
        return 2 * c + (x >= cell_mid(c, g.cs) ? 1 : 0);
    };
    int cnt[3] = {0, 0, 0};
    if (base < n) {
        float xl[D];  // the position before the row's first
        int fl[D];
        int ol = 0;
        {
            const int j = source(max(base - 1, 0));
#pragma unroll
            for (int l = 0; l < D; l++) {
                xl[l] = X[(long long)l * n + j];
                fl[l] = fine(xl[l]);
                if (l < g.od) ol += (fl[l] >> 1) * g.wpow[l];
            }
        }
        if (lane == 0) s_outer[wave][0] = ol;
#pragma unroll kUnroll
        for (int k = 0; k < kRows; k++) {
            const int i = base + k * kWave + lane;
            const bool on = i < n;
            const int j = source(on ? i : n - 1);
            bool dc = i == 0, ds = dc, dr = dc;
            int o = 0;
#pragma unroll
            for (int l = 0; l < D; l++) {
                const float x = X[(long long)l * n + j];
                const int f = fine(x);
                if (on) b.Xs[(long long)l * n + i] = x;
                float xp = __shfl_up(x, 1);
                int fp = __shfl_up(f, 1);
                if (lane == 0) {
                    xp = xl[l];
                    fp = fl[l];
                }
                dc |= f >> 1 != fp >> 1;
                ds |= f != fp;
                dr |= __float_as_uint(x) != __float_as_uint(xp);
                if (l < g.od) o += (f >> 1) * g.wpow[l];
                xl[l] = __shfl(x, kWave - 1);
                fl[l] = __shfl(f, kWave - 1);
            }
            if (on) b.perm_s[i] = b.perm[j];
            s_outer[wave][k * kWave + lane + 1] = o;
            const unsigned long long mc = __ballot(on && dc), ms = __ballot(on && subs && ds),
                                     mr = __ballot(on && dr);
            if (lane == 0) {
                s_mask[wave][k][0] = mc;
                s_mask[wave][k][1] = ms;
                s_mask[wave][k][2] = mr;
            }
            cnt[0] += __popcll(mc);
            cnt[1] += __popcll(ms);
            cnt[2] += __popcll(mr);
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int c = 0; c < 3; c++) s_cnt[wave][c] = cnt[c];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        int t = 0;
        for (int w = 0; w < kWaves; w++) t += s_cnt[w][threadIdx.x];
        s_tot[threadIdx.x] = t;
        s_pre[threadIdx.x] = 0;
    }
    __syncthreads();
    if (nb > 1) lb_join<3>(b.scan_tmp, tile, nb, seq, s_tot, s_pre);
    int at[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        at[c] = s_pre[c];
        for (int w = 0; w < wave; w++) at[c] += s_cnt[w][c];
    }
    const unsigned long long lt = lanemask_lt(), bit = 1ull << lane;
    for (int k = 0; k < kRows; k++) {
        const int i = base + k * kWave + lane;
        const unsigned long long mc = s_mask[wave][k][0], ms = s_mask[wave][k][1],
                                 mr = s_mask[wave][k][2];
        if (i < n) {
            const bool hc = mc & bit, hs = ms & bit, hr = mr & bit;
            const int c = at[0] + __popcll(mc & lt) + hc - 1;
            const int sp = at[1] + __popcll(ms & lt) + hs - 1;
            const int r = at[2] + __popcll(mr & lt) + hr - 1;
            b.point_cell[i] = c;
            b.point_run[i] = r;
            if (subs) b.point_sub[i] = sp;
            if (hc) {
                const int op = s_outer[wave][k * kWave + lane], o = s_outer[wave][k * kWave + lane + 1];
                b.cell_start[c] = i;
                b.cell_outer[c] = o;
                b.cell_run[c] = r;
                b.cell_sub[c] = sp;
                if (i == 0 || o != op) {
                    b.ob[o] = c;
                    if (i > 0) b.oe[op] = c;
                }
            }
            if (hs) {
                b.sub_start[sp] = i;
                b.sub_run[sp] = r;
            }
            if (hc || hs) {
#pragma unroll
                for (int l = 0; l < D; l++) {
                    const int f = fine(b.Xs[(long long)l * n + i]);
                    if (hc) b.cell_g[(long long)l * n + c] = f >> 1;
                    if (hs) b.sub_g[(long long)l * n + sp] = f;
                }
            }
            if (hr) b.run_start[r] = i;
            if (i == n - 1) {
                b.cell_start[c + 1] = n;
                b.cell_run[c + 1] = r + 1;
                b.run_start[r + 1] = n;
                b.oe[s_outer[wave][k * kWave + lane + 1]] = c + 1;
                st->C = c + 1;
                st->runs = r + 1;
                if (keep_runs) st->runs_valid = 1;
                if (subs) {
                    b.sub_start[sp + 1] = n;
                    b.sub_run[sp + 1] = r + 1;
                    b.cell_sub[c + 1] = sp + 1;
                    st->S = sp + 1;
                }
            }
        }
        at[0] += __popcll(mc);
        at[1] += __popcll(ms);
        at[2] += __popcll(mr);
    }
    if (nb > 1) lb_end(b.scan_tmp, nb, seq);
}

void build_grid(const Geo &g, GridBufs &b, DevState *st_loop, DevState *st, hipStream_t s,
                bool keep_runs, bool small, bool begin) {
    const int n = g.n;
    const bool wide = n > kTablesNarrowMax;
    const int gb = grid_for(n), sb = scan_blocks(n, wide);
#define KEYS_CASE(DD)                                                                          \
    case DD:                                                                                   \
        k_keys<DD><<<gb, kBlock, 0, s>>>(b.X, g, b.run_start, b.keys_a, b.ob, b.oe, st, st_loop, \
                                         begin);                                               \
        break;
    switch (g.d) {
        EGG_EACH_D(KEYS_CASE)
    }
#undef KEYS_CASE
    const int *sidx = b.vals_b;
    if (small) {
        rank_sort(b.keys_a, b.vals_b, n, g.kw, b.run_start, b.run_off, b.run_src, st, st_loop, s);
    } else {
        const int where = radix_sort(b.keys_a, b.keys_b, b.vals_a, b.vals_b, n, g.kw, g.sort_bits,
                                     b.hist, b.scan_tmp, st_loop, s, &st->sort_m, &st->sort_hist);
        sidx = where == 1 ? b.vals_b : (where == 0 ? b.vals_a : nullptr);
        launch_scan<1>(RunScan{sidx, b.run_start, b.run_off, b.run_src, st}, n, b.scan_tmp,
                       st_loop, s);
    }
#define TABLES_CASE(DD)                                                                        \
    case DD:                                                                                   \
        if (wide)                                                                              \
            k_tables<DD, kScanItems><<<sb, kBlock, 0, s>>>(b, sidx, g, st, st_loop, keep_runs); \
        else                                                                                   \
            k_tables<DD, kScanNarrow><<<sb, kBlock, 0, s>>>(b, sidx, g, st, st_loop, keep_runs); \
        break;
    switch (g.d) {
        EGG_EACH_D(TABLES_CASE)
    }
#undef TABLES_CASE
}

// Whether cell c heads a group of the update tiles.  Cells are sorted by
// (outer id, g_od, ..., g_{d-1}), so cells that share the outer cell and every
// inner coordinate but the last are adjacent; such a cell starts a new group
// when its last coordinate leaves the previous cell's block of gw cells.  With
// no inner dimension (od == d) or gw <= 1 every cell is its own group.
__device__ __forceinline__ bool group_head(const int *__restrict__ cell_g,
                                           const int *__restrict__ cell_outer, const Geo &g,
                                           int c) {
    const int n = g.n, last = g.d - 1;
    const bool grouped = g.gw > 1 && g.od < g.d;
    bool h = c == 0 || !grouped;
    if (!h) {
        h = cell_outer[c] != cell_outer[c - 1];
        for (int l = g.od; l < last && !h; l++)
            h = cell_g[(long long)l * n + c] != cell_g[(long long)l * n + c - 1];
        if (!h)
            h = cell_g[(long long)last * n + c] / g.gw != cell_g[(long long)last * n + c - 1] / g.gw;
    }
    return h;
}

// ------------------------------------------------------------- summaries --

// Compensated sum of two (sum, err) pairs over the wavefront by butterflies,
// combined in lane order so every lane ends with the same bits.
__device__ __forceinline__ void wave_two_sum(float &s1, float &e1, float &s2, float &e2) {
    const int lane = __lane_id();
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const float os1 = __shfl_xor(s1, o, kWave), oe1 = __shfl_xor(e1, o, kWave);
        const float os2 = __shfl_xor(s2, o, kWave), oe2 = __shfl_xor(e2, o, kWave);
        if (lane & o) {
            float a1 = os1, b1 = oe1, a2 = os2, b2 = oe2;
            two_sum_add(a1, b1, s1, e1);
            two_sum_add(a2, b2, s2, e2);
            s1 = a1; e1 = b1; s2 = a2; e2 = b2;
        } else {
            two_sum_add(s1, e1, os1, oe1);
            two_sum_add(s2, e2, os2, oe2);
        }
    }
}

// Slot of chunk k's partial sums of the group that starts at point c0.  Only
// groups of more than kSumChunk points have slots, a chunk for every kSumChunk
// points or part of them: at kSumChunk / 2 points a slot no two groups meet.
__device__ __forceinline__ int summary_slot(int c0, int k) { return c0 / (kSumChunk / 2) + k; }

// Totals of groups of consecutive sorted points: cells, or sub-cells (with
// bounding boxes).  Sums are relative to sin and cos of the group's anchor
// coords * cs.
struct SumGroups {
    const int *of, *starts, *coords;  // point -> group, first points, [d][n] coordinates
    float cs;
    float *Ts, *Tc;                   // [d][n]
    unsigned *mnk, *mxk;              // [d][n], nullptr without boxes
    float *partial;                   // [slots][6 d], kept for the second pass
};

// A sub-cell's box from the keys of its points' bounds.  A point that is not a
// number sorts beyond the infinities; its box then reaches to infinity, so that no
// test takes the sub-cell as a whole.
__device__ __forceinline__ void store_box(const SumGroups &q, long long at, unsigned kmin,
                                          unsigned kmax) {
    q.mnk[at] = max(kmin, 0x007FFFFFu);  // ord_key(-inf)
    q.mxk[at] = min(kmax, 0xFF800000u);  // ord_key(inf)
}

// Per dim: S_sin = sum(sinf(x) - sinf(g*cs)), S_cos likewise (EGG_SynC.cu:362-363),
// Kahan-compensated per lane, combined across lanes by compensated butterflies,
// then T_sin = sinf(g*cs)*cnt + S_sin (the bracket of EGG_SynC.cu:651-654).  A
// chunk is <= kSumChunk points of a group, lane e summing points e, e + 64, ...;
// groups of more than one chunk leave (sum, err) partials.
template <int D>
__device__ __forceinline__ void sum_chunk(const float *__restrict__ Xs, int n,
                                          const SumGroups &q, int grp, int c0, int c1, int j0) {
    const int lane = __lane_id();
    const int j1 = min(c1, j0 + kSumChunk);
    const bool whole = c1 - c0 <= kSumChunk;
#pragma unroll D <= 4 ? D : 1
    for (int l = 0; l < D; l++) {
        const float a = (float)q.coords[(long long)l * n + grp] * q.cs;
        const float sa = sinf(a), ca = cosf(a);
        float ss = 0.f, sc_ = 0.f, cs_ = 0.f, cc = 0.f;  // (sum, comp) for sin and cos
        unsigned kmin = 0xFFFFFFFFu, kmax = 0u;          // bounding box
        for (int j = j0 + lane; j < j1; j += kWave) {
            const float x = Xs[(long long)l * n + j];
            kmin = min(kmin, ord_key(x));
            kmax = max(kmax, ord_key(x));
            const float ts = sinf(x) - sa;
            const float tc = cosf(x) - ca;
            float y = ts - sc_;
            float t = ss + y;
            sc_ = (t - ss) - y;
            ss = t;
            y = tc - cc;
            t = cs_ + y;
            cc = (t - cs_) - y;
            cs_ = t;
        }
        // Kahan keeps sum - comp; switch to (sum, +err) form for the butterflies
        float s1 = ss, e1 = -sc_, s2 = cs_, e2 = -cc;
        wave_two_sum(s1, e1, s2, e2);
        if (q.mnk) {
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) {
                kmin = min(kmin, (unsigned)__shfl_xor((int)kmin, o, kWave));
                kmax = max(kmax, (unsigned)__shfl_xor((int)kmax, o, kWave));
            }
        }
        if (lane == 0) {
            if (whole) {
                const float cnt = (float)(c1 - c0);
                const float t1 = sa * cnt;
                const float t2 = ca * cnt;
                q.Ts[(long long)l * n + grp] = t1 + (s1 + e1);
                q.Tc[(long long)l * n + grp] = t2 + (s2 + e2);
                if (q.mnk) store_box(q, (long long)l * n + grp, kmin, kmax);
            } else {
                float *pp = &q.partial[((long long)summary_slot(c0, (j0 - c0) / kSumChunk) * D + l) * 6];
                pp[0] = s1; pp[1] = e1; pp[2] = s2; pp[3] = e2;
                pp[4] = __uint_as_float(kmin);
                pp[5] = __uint_as_float(kmax);
            }
        }
    }
}

// Summaries of the cells and, with sub-cells, of the sub-cells.  A wavefront owns
// the chunks and groups that start in a window of 32 sorted positions, which
// leaves no work list to build and search: groups of at most 32 points lie whole
// in the 64 positions from the window's start and are summed side by side, a lane
// per point (butterflies over a lane's place in its group: the same sums, in the
// same order, as a wavefront to itself would form, whose lanes beyond the count
// add zeros); larger ones one after the other (sum_chunk).  Bound by the VALU (sin
// and cos of every coordinate and both anchors, compensated adds).  A wavefront per
// group, each found by a search, took 364 us at n = 1,000,000, d = 3; this 71 us.
template <int D>
__global__ __launch_bounds__(kBlock) void k_summary(const float *__restrict__ Xs, Geo g,
                                                    SumGroups cells, SumGroups subs,
                                                    const DevState *st_loop) {
    if (st_loop && st_loop->done) return;
    const int n = g.n, lane = __lane_id();
    const int windows = (n + kSumSmall - 1) / kSumSmall;
    const int kinds = g.sub_bits ? 2 : 1;
    for (int w = wave_index(); w < windows; w += wave_count()) {
        const int w0 = w * kSumSmall, i = w0 + lane;
        const bool on = i < n;
        int grp[2], first[2], cnt[2], steps[2];
        bool small[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            grp[k] = first[k] = cnt[k] = steps[k] = 0;
            small[k] = false;
            if (k >= kinds) continue;
            const SumGroups &q = k ? subs : cells;
            int c1 = 0;
            if (on) {
                grp[k] = q.of[i];
                first[k] = q.starts[grp[k]];
                c1 = q.starts[grp[k] + 1];
                cnt[k] = c1 - first[k];
                small[k] = cnt[k] <= kSumSmall && first[k] >= w0 && first[k] < w0 + kSumSmall;
            }
            // butterfly steps of the window's largest small group
            while (__any(small[k] && cnt[k] > 1 << steps[k])) steps[k]++;
            unsigned long long big = __ballot(on && lane < kSumSmall && cnt[k] > kSumSmall &&
                                              (i - first[k]) % kSumChunk == 0);
            while (big) {
                const int at = __builtin_amdgcn_readfirstlane(__ffsll((long long)big) - 1);
                big &= big - 1;
                sum_chunk<D>(Xs, n, q, __builtin_amdgcn_readlane(grp[k], at),
                             __builtin_amdgcn_readlane(first[k], at),
                             __builtin_amdgcn_readlane(c1, at), w0 + at);
            }
        }
        if (!__any(small[0] || small[1])) continue;
#pragma unroll D <= 4 ? D : 1
        for (int l = 0; l < D; l++) {
            const float x = on ? Xs[(long long)l * n + i] : 0.f;
            const float sx = sinf(x), cx = cosf(x);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (!__any(small[k])) continue;
                const SumGroups &q = k ? subs : cells;
                const int e = i - first[k];
                const float a = (float)q.coords[(long long)l * n + grp[k]] * q.cs;
                const float sa = sinf(a), ca = cosf(a);
                float s1 = 0.f + (sx - sa), e1 = 0.f, s2 = 0.f + (cx - ca), e2 = 0.f;
                unsigned kmin = ord_key(x), kmax = kmin;
                for (int o = 1 << steps[k] >> 1; o > 0; o >>= 1) {
                    const int pe = e ^ o, from = lane - e + pe;
                    const bool has = small[k] && pe < cnt[k];
                    float a1 = __shfl(s1, from), b1 = __shfl(e1, from);
                    float a2 = __shfl(s2, from), b2 = __shfl(e2, from);
                    a1 = has ? a1 : 0.f;
                    b1 = has ? b1 : 0.f;
                    a2 = has ? a2 : 0.f;
                    b2 = has ? b2 : 0.f;
                    const bool after = e & o;
                    float p1 = after ? a1 : s1, r1 = after ? b1 : e1;
                    float p2 = after ? a2 : s2, r2 = after ? b2 : e2;
                    two_sum_add(p1, r1, after ? s1 : a1, after ? e1 : b1);
                    two_sum_add(p2, r2, after ? s2 : a2, after ? e2 : b2);
                    s1 = p1; e1 = r1; s2 = p2; e2 = r2;
                    if (k) {
                        const unsigned omin = __shfl((int)kmin, from), omax = __shfl((int)kmax, from);
                        kmin = has ? min(kmin, omin) : kmin;
                        kmax = has ? max(kmax, omax) : kmax;
                    }
                }
                if (small[k] && e == 0) {
                    const float c = (float)cnt[k];
                    const float t1 = sa * c;
                    const float t2 = ca * c;
                    q.Ts[(long long)l * n + grp[k]] = t1 + (s1 + e1);
                    q.Tc[(long long)l * n + grp[k]] = t2 + (s2 + e2);
                    if (k) store_box(q, (long long)l * n + grp[k], kmin, kmax);
                }
            }
        }
    }
}

// Totals of one group of more than one chunk, one wavefront: lane k sums the
// partials k, k + 64, ... in order, then the lanes combine by butterflies.
template <int D>
__device__ __forceinline__ void sum_partials(int n, const SumGroups &q, int grp, int c0, int c1) {
    const int lane = __lane_id();
    const int nch = (c1 - c0 + kSumChunk - 1) / kSumChunk;
    const float cnt = (float)(c1 - c0);
#pragma unroll D <= 4 ? D : 1
    for (int l = 0; l < D; l++) {
        float s1 = 0.f, e1 = 0.f, s2 = 0.f, e2 = 0.f;
        unsigned kmin = 0xFFFFFFFFu, kmax = 0u;
        for (int k = lane; k < nch; k += kWave) {
            const float *pp = &q.partial[((long long)summary_slot(c0, k) * D + l) * 6];
            two_sum_add(s1, e1, pp[0], pp[1]);
            two_sum_add(s2, e2, pp[2], pp[3]);
            kmin = min(kmin, __float_as_uint(pp[4]));
            kmax = max(kmax, __float_as_uint(pp[5]));
        }
        wave_two_sum(s1, e1, s2, e2);
        if (q.mnk) {
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) {
                kmin = min(kmin, (unsigned)__shfl_xor((int)kmin, o, kWave));
                kmax = max(kmax, (unsigned)__shfl_xor((int)kmax, o, kWave));
            }
        }
        if (lane == 0) {
            const float a = (float)q.coords[(long long)l * n + grp] * q.cs;
            const float t1 = sinf(a) * cnt;
            const float t2 = cosf(a) * cnt;
            q.Ts[(long long)l * n + grp] = t1 + (s1 + e1);
            q.Tc[(long long)l * n + grp] = t2 + (s2 + e2);
            if (q.mnk) store_box(q, (long long)l * n + grp, kmin, kmax);
        }
    }
}

// Per cell group: its tiles of 64 runs (every group: the extra check's table),
// the same for the groups updated by tiles (none for sparse groups), and
// the runs of sparse groups (k_update_pairs), listed at the offsets of their
// scan.  cell_groups: every cell is its own group.
struct GroupScan {
    const int *cell_run;
    int *grp_cell, *tile_off, *utile_off, *list;
    int mode, d;
    bool cell_groups;
    DevState *st;
    __device__ int count() const { return cell_groups ? st->C : st->G; }
    __device__ int first(int k) const { return cell_run[cell_groups ? k : grp_cell[k]]; }
    __device__ void load(int k, int (&v)[3]) const {
        const int runs = first(k + 1) - first(k);
        const int t = (runs + kTile - 1) / kTile;
        const bool sp = sparse_group(runs, st->runs, st->C, mode, d);
        v[0] = t;
        v[1] = sp ? 0 : t;
        v[2] = sp ? runs : 0;
    }
    __device__ void store(int k, const int (&v)[3], const int (&ex)[3]) const {
        tile_off[k] = ex[0];
        utile_off[k] = ex[1];
        if (!pairs_take_all(mode, d)) {  // else the list would be every run, in order
            const int r0 = v[2] ? first(k) : 0;
            for (int r = 0; r < v[2]; r++) list[ex[2] + r] = r0 + r;
        }
        if (cell_groups) {
            grp_cell[k] = k;
            if (k == st->C - 1) grp_cell[k + 1] = k + 1;
        }
    }
    __device__ void finish(const int (&tot)[3]) const {
        st->T = tot[0];
        st->TU = tot[1];
        st->sparse_count = tot[2];
        if (cell_groups) st->G = st->C;
    }
};

// First cell of every group of more than one cell; grp_cell[G] = C.
struct HeadScan {
    const int *cell_g, *cell_outer;
    Geo g;
    int *grp_cell;
    DevState *st;
    __device__ int count() const { return st->C; }
    __device__ void load(int c, int (&v)[1]) const {
        v[0] = group_head(cell_g, cell_outer, g, c) ? 1 : 0;
    }
    __device__ void store(int c, const int (&v)[1], const int (&ex)[1]) const {
        if (v[0]) grp_cell[ex[0]] = c;
        if (c == st->C - 1) grp_cell[ex[0] + v[0]] = c + 1;
    }
    __device__ void finish(const int (&tot)[1]) const { st->G = tot[0]; }
};

// The groups' scan (the first `scan` workgroups), and by the others the totals of
// the cells and sub-cells of several chunks: both follow k_summary and k_tables and
// precede the update.
template <int D, int ITEMS>
__global__ __launch_bounds__(kBlock) void k_groups(GroupScan io, int *lb, int scan, int n,
                                                   SumGroups cells, SumGroups subs,
                                                   const DevState *st, const DevState *st_loop) {
    if (st_loop && st_loop->done) return;
    if ((int)blockIdx.x < scan) {
        scan_tiles<3, ITEMS>(io, lb, scan);
        return;
    }
    const int lane = __lane_id(), skip = scan * (kBlock / kWave);
    const int waves = wave_count() - skip;
    for (int k = 0; k < 2; k++) {
        const SumGroups &q = k ? subs : cells;
        if (!q.of) continue;
        const int count = k ? st->S : st->C;
        // neighbouring groups go to different wavefronts
        for (int c0 = wave_index() - skip; c0 < count; c0 += waves * kWave) {
            const long long c = c0 + (long long)lane * waves;
            int p0 = 0, p1 = 0;
            if (c < count) {
                p0 = q.starts[c];
                p1 = q.starts[c + 1];
            }
            unsigned long long multi = __ballot(p1 - p0 > kSumChunk);
            while (multi) {
                const int at = __builtin_amdgcn_readfirstlane(__ffsll((long long)multi) - 1);
                multi &= multi - 1;
                sum_partials<D>(n, q, c0 + at * waves, __builtin_amdgcn_readlane(p0, at),
                                __builtin_amdgcn_readlane(p1, at));
            }
        }
    }
}

void cell_summaries(const Geo &g, GridBufs &b, DevState *st_loop, DevState *st, hipStream_t s) {
    const int n = g.n;
    const bool wide = n > kTablesNarrowMax;
    const int sb = scan_blocks(n, wide);
    const int wb = grid_for(((long long)n + kSumSmall - 1) / kSumSmall * kWave, kBlock, 16384);
    const bool cell_groups = !(g.gw > 1 && g.od < g.d);
    // slots: one for every kSumChunk / 2 points, cells' first
    const long long slots = n / (kSumChunk / 2) + 2;
    const SumGroups cells{b.point_cell, b.cell_start, b.cell_g, g.cs, b.Ts, b.Tc, nullptr, nullptr,
                          b.partial};
    SumGroups subs{};
    if (g.sub_bits)  // anchors on the half-side grid
        subs = SumGroups{b.point_sub, b.sub_start, b.sub_g, g.cs * 0.5f, b.TsS, b.TcS, b.smin,
                         b.smax, b.partial + slots * 6 * g.d};
    if (!cell_groups)
        launch_scan<1>(HeadScan{b.cell_g, b.cell_outer, g, b.grp_cell, st}, n, b.scan_tmp, st_loop,
                       s);
    // workgroups for the totals of several chunks: none can be without kSumChunk points
    const int tb = n > kSumChunk ? std::min(512, n / 1024 + 1) : 0;
    const GroupScan groups{b.cell_run, b.grp_cell, b.tile_off, b.utile_off, b.sparse_runs,
                           g.pair_mode, g.d, cell_groups, st};
#define SUM_CASE(DD)                                                                          \
    case DD:                                                                                  \
        k_summary<DD><<<wb, kBlock, 0, s>>>(b.Xs, g, cells, subs, st_loop);                   \
        if (wide)                                                                             \
            k_groups<DD, kScanItems><<<sb + tb, kBlock, 0, s>>>(groups, b.scan_tmp, sb, n,    \
                                                                cells, subs, st, st_loop);    \
        else                                                                                  \
            k_groups<DD, kScanNarrow><<<sb + tb, kBlock, 0, s>>>(groups, b.scan_tmp, sb, n,   \
                                                                 cells, subs, st, st_loop);   \
        break;
    switch (g.d) {
        EGG_EACH_D(SUM_CASE)
    }
#undef SUM_CASE
}

}  // namespace egg
