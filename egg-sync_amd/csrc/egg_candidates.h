// Candidate points of a position in grid order, 64 at a time (gfx950).
#pragma once

#include "egg_common.h"

namespace egg {

// First cell of [cb, ce) whose g_od is >= lo_v (cells of a column are sorted
// by g_od); the caller stops at the first cell above its range.
__device__ __forceinline__ int column_lower(const int *__restrict__ cell_g_od, int cb, int ce,
                                            int lo_v) {
    int lo = cb, hi = ce;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (cell_g_od[mid] < lo_v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// The sorted points of the outer cells within R of cell coordinates g0, cut in
// dimension od to |dg| <= R, in ascending sorted position: every point within
// eps for R = ceil(eps / cs) + 1.  One wavefront with uniform g0 walks them:
// each lane takes the point range of one outer cell, a wave scan places the 64
// ranges behind one another, and the points are then handed out 64 at a time,
// whatever the ranges' lengths.  Ranges of farther inner cells stay in; a point
// in them fails the distance test.
template <int D>
struct Candidates {
    const int *cell_start, *cell_g_od, *ob, *oe;
    int lo[D], ext[D], wpow[D];  // the box, inside the grid
    int od, g0od, R;
    int rows, row0;  // outer cells of the box, next of them to load
    int rj, rp;      // lane: its range's first point minus its offset, its offset
    int total, f0;   // points of the loaded ranges, those handed out

    __device__ __forceinline__ void init(const Geo &g, const int *cell_g, const int *starts,
                                         const int *b, const int *e, int c0, int radius) {
        cell_start = starts;
        ob = b;
        oe = e;
        od = g.od;
        R = radius;
        cell_g_od = cell_g + (long long)od * g.n;
        g0od = od < D ? cell_g_od[c0] : 0;
        rows = 1;
#pragma unroll
        for (int l = 0; l < D; l++) {
            if (l < od) {
                const int g0 = cell_g[(long long)l * g.n + c0];
                lo[l] = max(0, g0 - R);
                ext[l] = min(g.w - 1, g0 + R) - lo[l] + 1;
                wpow[l] = g.wpow[l];
                rows *= ext[l];  // <= w^od <= n, or a row of 2R + 1 cells
            }
        }
        row0 = total = f0 = 0;
    }

    // The next 64 outer cells' ranges.
    __device__ __forceinline__ void load() {
        const int lane = __lane_id();
        int rem = row0 + lane, o = 0;
        const bool ok = rem < rows;
#pragma unroll
        for (int l = 0; l < D; l++) {
            if (l < od) {
                const int q = rem / ext[l];
                o += (lo[l] + rem - q * ext[l]) * wpow[l];
                rem = q;
            }
        }
        int j0 = 0, len = 0;
        if (ok) {
            int cb = ob[o], ce = oe[o];
            if (od < D && cb < ce) {
                cb = column_lower(cell_g_od, cb, ce, g0od - R);
                ce = column_lower(cell_g_od, cb, ce, g0od + R + 1);
            }
            if (cb < ce) {
                j0 = cell_start[cb];
                len = cell_start[ce] - j0;
            }
        }
        int inc = len;
#pragma unroll
        for (int s = 1; s < kWave; s <<= 1) {
            const int t = __shfl_up(inc, s, kWave);
            if (lane >= s) inc += t;
        }
        rp = inc - len;
        rj = j0 - rp;
        total = __builtin_amdgcn_readlane(inc, kWave - 1);
        row0 += kWave;
        f0 = 0;
    }

    // Loads ranges until some points are left to hand out; false at the end.
    __device__ __forceinline__ bool more() {
        while (f0 >= total) {
            if (row0 >= rows) return false;
            load();
        }
        return true;
    }

    // Point f of the loaded ranges (f < total), of the 64 from a uniform f0 on the
    // lane's (the last lanes may share one): the last range whose offset is <= f
    // (empty ranges share their successor's offset).  In dense cells all 64 are in one.
    __device__ __forceinline__ int point(int f, int f0) const {
        const int k0 = __popcll(__ballot(rp <= f0)) - 1;
        if (k0 == kWave - 1 || __builtin_amdgcn_readlane(rp, k0 + 1) >= min(f0 + kWave, total))
            return __builtin_amdgcn_readlane(rj, k0) + f;
        int k = 0;
#pragma unroll
        for (int s = kWave / 2; s > 0; s >>= 1)
            if (__shfl(rp, k + s, kWave) <= f) k += s;
        return __shfl(rj, k, kWave) + f;
    }
};

}  // namespace egg
