// Cluster extraction (EGG_SynC.cu:1205-1227; SynC.cpp:88-129) and input
// validation, gfx950.
#include <climits>

#include "egg_candidates.h"
#include "egg_internal.h"
#include "egg_scan.h"

namespace egg {

static inline int grid_for(long long n) {
    long long b = (n + kBlock - 1) / kBlock;
    if (b < 1) b = 1;
    if (b > 65536) b = 65536;
    return (int)b;
}

// Cluster id of each cell with more than one point (the scan of such cells), -1
// for the others.
struct LabelScan {
    const int *cell_start;
    int *label;
    DevState *st;
    __device__ int count() const { return st->C; }
    __device__ void load(int c, int (&v)[1]) const {
        v[0] = cell_start[c + 1] - cell_start[c] > 1 ? 1 : 0;
    }
    __device__ void store(int c, const int (&v)[1], const int (&ex)[1]) const {
        label[c] = v[0] ? ex[0] : -1;
    }
    __device__ void finish(const int (&tot)[1]) const { st->n_clusters = tot[0]; }
};

// GPU_synCluster_float_grid: a point gets its cell's cluster id when the cell
// holds more than one point, else -1.  Ids are compacted to 0..k-1 in cell
// order (the reference leaves gaps; only the partition is meaningful).
__global__ void k_labels_egg(const int *__restrict__ point_cell,
                             const int *__restrict__ cell_label, const int *__restrict__ perm_s,
                             int n, int *__restrict__ labels) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        labels[perm_s[i]] = cell_label[point_cell[i]];
}

void launch_labels_egg(const Geo &g, GridBufs &b, int *labels, DevState *st, hipStream_t s) {
    launch_scan<1>(LabelScan{b.cell_start, b.scratch, st}, g.n, b.scan_tmp, nullptr, s);
    k_labels_egg<<<grid_for(g.n), kBlock, 0, s>>>(b.point_cell, b.scratch, b.perm_s, g.n, labels);
}

__global__ void k_invert(const int *__restrict__ perm_s, int n, int *__restrict__ inv) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        inv[perm_s[i]] = i;
}

// Squared FP32 distance of sorted point j to x.
template <int D>
__device__ __forceinline__ float point_dist2(const float *x, const float *__restrict__ Xs, int n,
                                             int j) {
    float s = 0.f;
#pragma unroll
    for (int l = 0; l < D; l++) {
        const float df = x[l] - Xs[(long long)l * n + j];
        s += df * df;
    }
    return s;
}

// Points without another point within eps neither give nor get a label: they
// are marked (kLonely) before the labelling, one wavefront per point, which
// stops at the first neighbour it meets.
constexpr int kLonely = -2;

template <int D>
__global__ __launch_bounds__(kBlock) void k_lonely(
    const float *__restrict__ Xs, const int *__restrict__ perm_s,
    const int *__restrict__ point_cell, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const int *__restrict__ ob, const int *__restrict__ oe, Geo g,
    int *__restrict__ labels) {
    const int n = g.n, lane = __lane_id();
    const int i = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave);
    if (i >= n) return;
    float x[D];
#pragma unroll
    for (int l = 0; l < D; l++) x[l] = Xs[(long long)l * n + i];
    Candidates<D> cand;
    cand.init(g, cell_g, cell_start, ob, oe, point_cell[i], g.R + 1);
    bool found = false;
    while (!found && cand.more()) {
        const int f = cand.f0 + lane;
        const int j = cand.point(min(f, cand.total - 1), cand.f0);
        cand.f0 += kWave;
        found = __any(f < cand.total && j != i && point_dist2<D>(x, Xs, n, j) <= g.thr_eps);
    }
    if (lane == 0) labels[perm_s[i]] = found ? -1 : kLonely;
}

// synCluster_v2 (SynC.cpp:88-129) in one workgroup: points are visited in id
// order; an unlabelled point i gives label cl to every other point within FP32
// distance eps (overwriting earlier labels), and takes cl itself if it found
// any.  The search for the next unlabelled id is parallel over the workgroup,
// and so is each neighbour scan: every wavefront holds the same candidate
// ranges and takes every 16th step of 64 points.  n = 8,000, d = 2: 2,300 us
// with a thread per candidate cell and every lonely point visited, here
// 232 and 21 for k_lonely.
constexpr int kLabBlock = 1024;

template <int D>
__global__ __launch_bounds__(kLabBlock) void k_labels_sync(
    const float *__restrict__ Xs, const int *__restrict__ perm_s, const int *__restrict__ invperm,
    const int *__restrict__ point_cell, const int *__restrict__ cell_start,
    const int *__restrict__ cell_g, const int *__restrict__ ob, const int *__restrict__ oe,
    Geo g, int *labels, DevState *st) {
    __shared__ int s_min, s_any;
    const int n = g.n, t = threadIdx.x;
    int cl = 0, cursor = 0;
    while (cursor < n) {
        if (t == 0) s_min = INT_MAX;
        __syncthreads();
        int found = INT_MAX;
        for (int base = cursor; base < n; base += kLabBlock) {
            const int i = base + t;
            if (i < n && labels[i] == -1) atomicMin(&s_min, i);
            __syncthreads();
            found = s_min;
            __syncthreads();
            if (found != INT_MAX) break;
        }
        if (found == INT_MAX) break;
        const int si = __builtin_amdgcn_readfirstlane(invperm[found]);
        float x[D];
#pragma unroll
        for (int l = 0; l < D; l++) x[l] = Xs[(long long)l * n + si];
        if (t == 0) s_any = 0;
        __syncthreads();
        Candidates<D> cand;
        cand.init(g, cell_g, cell_start, ob, oe, point_cell[si], g.R + 1);
        bool any = false;
        while (cand.more()) {
            for (int f0 = t - __lane_id(); f0 < cand.total; f0 += kLabBlock) {
                const int f = f0 + __lane_id();
                const int j = cand.point(min(f, cand.total - 1), f0);
                if (f < cand.total && j != si && point_dist2<D>(x, Xs, n, j) <= g.thr_eps) {
                    labels[perm_s[j]] = cl;
                    any = true;
                }
            }
            cand.f0 = cand.total;
        }
        if (any) s_any = 1;
        __syncthreads();
        if (s_any) {
            if (t == 0) labels[found] = cl;
            cl++;
        }
        cursor = found + 1;
        __syncthreads();
    }
    for (int i = t; i < n; i += kLabBlock)
        if (labels[i] == kLonely) labels[i] = -1;
    if (t == 0) st->n_clusters = cl;
}

void launch_labels_sync(const Geo &g, GridBufs &b, int *labels, DevState *st, hipStream_t s) {
    int *invperm = b.scratch;
    k_invert<<<grid_for(g.n), kBlock, 0, s>>>(b.perm_s, g.n, invperm);
#define LS_CASE(DD)                                                                           \
    case DD:                                                                                  \
        k_lonely<DD><<<(g.n + kBlock / kWave - 1) / (kBlock / kWave), kBlock, 0, s>>>(        \
            b.Xs, b.perm_s, b.point_cell, b.cell_start, b.cell_g, b.ob, b.oe, g, labels);     \
        k_labels_sync<DD><<<1, kLabBlock, 0, s>>>(b.Xs, b.perm_s, invperm, b.point_cell,      \
                                                  b.cell_start, b.cell_g, b.ob, b.oe, g,      \
                                                  labels, st);                                \
        break;
    switch (g.d) {
        EGG_EACH_D(LS_CASE)
    }
#undef LS_CASE
}

__global__ void k_validate(const float *__restrict__ aos, long long count, int *err) {
    bool bad = false;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < count;
         i += (long long)gridDim.x * blockDim.x) {
        const float v = aos[i];
        if (!(v >= 0.0f && v <= 1.0f)) bad = true;
    }
    if (__any(bad) && __lane_id() == 0) atomicOr(err, 1);
}

void launch_validate(const float *aos, long long count, int *err, hipStream_t s) {
    k_validate<<<grid_for(count), kBlock, 0, s>>>(aos, count, err);
}

}  // namespace egg
