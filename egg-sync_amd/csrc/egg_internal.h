// Host-side launchers shared by the translation units of the library.
#pragma once

#include "egg_common.h"

namespace egg {

// Exclusive scan of n int32 values; `tmp` needs scan_tmp_ints(n) ints.  The
// sum of all values is written to *total if total != nullptr.  In-place allowed.
size_t scan_tmp_ints(int n);
void scan_exclusive(const int *in, int *out, int n, int *tmp, int *total, hipStream_t s);
// The grid build's scans (egg_scan.h) keep their shared state, up to
// kMaxScanCh channels, in scan_tmp_ints(n) ints of their own.  It must be zero
// before the first of them (scan_tmp_reset, not for graph capture); each scan
// leaves it ready for the next on the same stream.
constexpr int kMaxScanCh = 3;
int scan_tmp_reset(int *tmp, int n, hipStream_t s);
// Nonzero if a scan using tmp gave up waiting (an internal error).
int scan_tmp_error(const int *tmp, hipStream_t s, int *err);

// Stable order of the grid build's keys, st->sort_m <= kRankSortMax of them, by
// comparing every pair: sorted position q holds element sidx[q]; for runs of the
// previous grid (st->lens_m > 0) also where their points go (off, src).
constexpr int kRankSortMax = 24576;
void rank_sort(const uint64_t *keys, int *sidx, int n, int kw, const int *run_start, int *off,
               int *src, const DevState *st, const DevState *st_loop, hipStream_t s);

// Stable LSD radix sort of (key, position) pairs by key bits [0, key_bits),
// 8 bits per pass.  keys_a/keys_b: [kw][n] u64; vals_a/vals_b: [n] int32.
// On entry keys are in keys_a and vals are implicit (0..m-1), m = *n_dev
// (<= n); *hist_n_dev must hold 256 * max(1, ceil(m / kSortTile)) (the
// histogram entries of the tiles that hold elements).  Returns 0 if the sorted
// result is in the *_a buffers, 1 if in *_b, -1 if no pass was needed (identity
// order).
size_t sort_tmp_ints(int n);
int radix_sort(uint64_t *keys_a, uint64_t *keys_b, int *vals_a, int *vals_b, int n, int kw,
               int key_bits, int *hist, int *scan_tmp, const DevState *st, hipStream_t s,
               const int *n_dev, const int *hist_n_dev);

// A heavy streamed range of an update tile: tile t, candidate cell c, the
// range's runs (runs [r0, r0 + total) if smask is 0, else the runs of
// sub-cells s0 + k for the bits k of smask), and its work units
// [ubase, ubase + nunits) of kUnitRuns runs.
struct HeavyDesc {
    int t, c, r0, s0;
    unsigned smask;
    int total, ubase, nunits;
    int half;  // 1: an eps/2 count over a full cell (border lanes), 0: the update's sums
};

// Grid build, cell summaries (egg_grid.hip).
struct GridBufs {
    float *X;            // [d][n] current positions (state)
    int *perm;           // [n]
    float *Xs;           // [d][n] sorted positions
    int *perm_s;         // [n]
    uint64_t *keys_a, *keys_b;
    int *vals_a, *vals_b;
    int *hist;           // [256][ntiles]
    int *scan_tmp;
    int *point_cell;     // [n]
    int *point_run;      // [n] run and sub-cell of each sorted position
    int *point_sub;      // [n]
    int *run_off;        // [n] sorted runs of the previous grid: first new position,
    int *run_src;        // [n] first old position
    int *scratch;        // [n] of the label passes
    int *cell_start;     // [n+1]
    int *cell_g;         // [d][n]
    int *cell_outer;     // [n]
    int *ob, *oe;        // [O]
    // runs: maximal stretches of bitwise-equal consecutive positions (sorted order)
    int *run_start;      // [n+1] first sorted position of each run
    int *cell_run;       // [n+1] first run of each cell
    // sub-cells (see cell_mid): first sorted position, first sub-cell of each
    // cell, fine coordinates 2g + split bit, first run, totals as Ts / Tc
    int *sub_start;      // [n+1]
    int *cell_sub;       // [n+1]
    int *sub_g;          // [d][n]
    int *sub_run;        // [n+1]
    float *TsS, *TcS;    // [d][n]
    unsigned *smin, *smax;  // [d][n] bounding box of each sub-cell's points (ord_key)
    // update tiles: cells are grouped (consecutive cells of one outer cell,
    // equal inner coordinates but the last, last one in the same block of gw
    // cells); a tile holds <= 64 runs of one group
    int *grp_cell;       // [n+1] first cell of each group, grp_cell[G] = C
    int *tile_off;       // [n] first tile of each group (every group: extra check)
    int *utile_off;      // [n] the same for the groups updated by tiles (not sparse)
    float *rres;         // [d][n] new position of each run
    int *sparse_runs;    // [n]   runs of sparse cell groups
    // pair update (egg_pairs.hip): memory of its own (pair_scratch_bytes); it
    // also uses keys_a / keys_b and partial, free between the summaries and the
    // next grid build
    char *pair;
    int *rdbg;           // [4n]  N / half / border / synced of each run (diagnostics;
                         //       also the saved N / half / border of deferred runs)
    // heavy streamed ranges (k_update_heavy): their sums, per run, in
    // fixed point (2^-30): sum w sin v [d], sum w (cos v - 1) [d], count,
    // and the eps/2 count; nullptr for d > kHeavyMaxD (no deferral)
    long long *hacc;     // [2d+2][n]
    HeavyDesc *hdesc;    // [kHeavyCap]
    int *dtiles;         // [n]   tiles whose runs finish in k_update_finish
    float *Ts, *Tc;      // [d][n]
    float *partial;      // [n + n/kSumChunk + 1][4*d]: summary partials, see summary_slot
    int *pairs;          // [2 * pair_cap] extra-check (p, q) sorted positions
    int pair_cap;
};

void launch_aos_to_soa(const float *aos, float *soa, int *perm, int n, int d, hipStream_t s);
void launch_soa_to_aos_by_perm(const float *soa, const int *perm, float *aos, int n, int d,
                               hipStream_t s);
// Sort and grid tables; writes st->C.  st_loop (nullable): nothing runs once
// its loop has stopped; with `begin` the build opens a loop iteration (the pass
// state is reset).  keep_runs: the update moves each run of equal positions
// alike, so the next build may sort runs.  small: at most kRankSortMax elements
// to sort (rank_sort).
void build_grid(const Geo &g, GridBufs &b, DevState *st_loop, DevState *st, hipStream_t s,
                bool keep_runs, bool small = false, bool begin = false);
void cell_summaries(const Geo &g, GridBufs &b, DevState *st_loop, DevState *st, hipStream_t s);

// Update / extra check / r_c (egg_update.hip).
struct DebugOut {
    int *N, *half, *border, *synced;  // [n] per sorted position, nullable
};
void launch_update_egg(const Geo &g, GridBufs &b, DevState *st, const DebugOut *dbg,
                       hipStream_t s);
// The groups sparse_group selects, point pair by point pair (egg_pairs.hip).
size_t pair_scratch_bytes(size_t n, size_t d);
void launch_update_pairs(const Geo &g, GridBufs &b, int *rdbg, DevState *st, hipStream_t s);
void launch_extra_check(const Geo &g, GridBufs &b, DevState *st, hipStream_t s);
// SynC pass: positions (write_pos) and r_c in FP64 -> st->rc.
void launch_update_sync(const Geo &g, GridBufs &b, DevState *st, double *rc_part, bool write_pos,
                        hipStream_t s);
int rc_partials(int n);
void launch_set_flag(DevState *st, hipStream_t s);

// Labels (egg_labels.hip).
void launch_labels_egg(const Geo &g, GridBufs &b, int *labels, DevState *st, hipStream_t s);
void launch_labels_sync(const Geo &g, GridBufs &b, int *labels, DevState *st, hipStream_t s);
void launch_validate(const float *aos, long long count, int *err, hipStream_t s);

}  // namespace egg
