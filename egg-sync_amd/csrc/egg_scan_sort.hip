// Device-wide exclusive scan and the stable sorts of the grid build, gfx950.
//
// Scan (of callers without look-back state; the grid build's are in egg_scan.h):
// 2048-element tiles (256 threads x 8 items), wave scans with lane shuffles;
// arrays of one tile or less are scanned by one workgroup in a single launch,
// longer ones by reduce-then-scan in three.  Up to kRankSortMax elements are
// sorted by comparing every pair.  Radix sort: 8-bit digits, per-tile LDS histogram,
// exclusive scan of the digit-major histogram, then a stable scatter in which
// each wavefront ranks its 64 keys by digit with 8 ballots (lanes holding the
// same digit form a 64-bit match mask).  Stability makes the grid build
// deterministic: points that share a cell keep their previous order.
#include <algorithm>
#include <type_traits>

#include "egg_host.h"
#include "egg_internal.h"
#include "egg_scan.h"

namespace egg {

// Scans of callers without look-back state: reduce-then-scan.
__global__ __launch_bounds__(kBlock) void k_scan_reduce(const int *__restrict__ in, int n,
                                                        int *__restrict__ bsum) {
    __shared__ int s_w[kBlock / kWave];
    const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanItems;
    int v = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++)
        if (base + k < n) v += in[base + k];
    int total;
    block_excl_scan(v, s_w, total);
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

// One workgroup of kSingleBlock threads scans a whole array in chunks of
// kSingleTile, carrying the running total.  It scans the block sums of the
// three-kernel scan and, in its place, arrays of at most kScanTile values (one
// launch instead of three; integer sums, so the result is the same).  Larger
// arrays take the three kernels: one workgroup's thread-contiguous loads and
// stores cost ~0.85 us per thousand values on gfx950, so past a few thousand
// values the single launch is the slower one.  In place is allowed: each
// thread reads its own values before it writes them, and later chunks are
// read after earlier ones are written.
constexpr int kSingleBlock = 1024;
constexpr int kSingleTile = kSingleBlock * kScanItems;

__global__ __launch_bounds__(kSingleBlock) void k_scan_single(const int *in, int *out, int n,
                                                              int *total) {
    __shared__ int s_w[kSingleBlock / kWave];
    int carry = 0;
    for (int base = 0; base < n; base += kSingleTile) {
        const int idx0 = base + threadIdx.x * kScanItems;
        int vals[kScanItems];
        int v = 0;
#pragma unroll
        for (int k = 0; k < kScanItems; k++) {
            vals[k] = (idx0 + k < n) ? in[idx0 + k] : 0;
            v += vals[k];
        }
        int tot;
        int ex = block_excl_scan<kSingleBlock>(v, s_w, tot) + carry;
#pragma unroll
        for (int k = 0; k < kScanItems; k++) {
            if (idx0 + k < n) out[idx0 + k] = ex;
            ex += vals[k];
        }
        carry += tot;
    }
    if (total && threadIdx.x == 0) *total = carry;
}

__global__ __launch_bounds__(kBlock) void k_scan_down(const int *__restrict__ in,
                                                      int *__restrict__ out, int n,
                                                      const int *__restrict__ bsum) {
    __shared__ int s_w[kBlock / kWave];
    const long long tile0 = (long long)blockIdx.x * kScanTile;
    if (tile0 >= n) return;
    const long long base = tile0 + (long long)threadIdx.x * kScanItems;
    int vals[kScanItems];
    int v = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        vals[k] = (base + k < n) ? in[base + k] : 0;
        v += vals[k];
    }
    int tot;
    int ex = block_excl_scan(v, s_w, tot) + bsum[blockIdx.x];
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        if (base + k < n) out[base + k] = ex;
        ex += vals[k];
    }
}

size_t scan_tmp_ints(int n) {
    // the look-back state; the three-launch scan's block sums need less
    const int m = std::max(n, 1);
    const int nb = std::max(scan_blocks(m, true),
                            scan_blocks(std::min(m, kTablesNarrowMax), false)) + 1;
    return 4 + 2 * (size_t)kMaxScanCh * nb;
}

int scan_tmp_reset(int *tmp, int n, hipStream_t s) {
    return hip_err(hipMemsetAsync(tmp, 0, sizeof(int) * scan_tmp_ints(n), s));
}

int scan_tmp_error(const int *tmp, hipStream_t s, int *err) {
    int rc = hip_err(hipMemcpyAsync(err, tmp + 3, sizeof(int), hipMemcpyDeviceToHost, s));
    if (!rc) rc = hip_err(hipStreamSynchronize(s));
    return rc;
}

void scan_exclusive(const int *in, int *out, int n, int *tmp, int *total, hipStream_t s) {
    if (n <= kScanTile) {
        k_scan_single<<<1, kSingleBlock, 0, s>>>(in, out, n, total);
        return;
    }
    const int nb = (n + kScanTile - 1) / kScanTile;
    k_scan_reduce<<<nb, kBlock, 0, s>>>(in, n, tmp);
    k_scan_single<<<1, kSingleBlock, 0, s>>>(tmp, tmp, nb, total);
    k_scan_down<<<nb, kBlock, 0, s>>>(in, out, n, tmp);
}

// ------------------------------------------------------------ radix sort --

__device__ __forceinline__ int digit_of(const uint64_t *keys, int n, int e, int shift) {
    const uint64_t w = keys[(long long)(shift >> 6) * n + e];
    return (int)((w >> (shift & 63)) & 255ull);
}

// Keys are stored with stride n ([kw][n]); the first m = min(n, *n_dev) of
// them are sorted.
__global__ __launch_bounds__(kBlock) void k_rs_hist(const uint64_t *__restrict__ keys, int n,
                                                    const int *n_dev, int shift,
                                                    int *__restrict__ hist,
                                                    const DevState *st) {
    if (st && st->done) return;
    __shared__ int h[256];
    const int m = min(n, *n_dev);
    // tiles holding elements: the histogram's stride (its scan covers 256
    // of them per digit)
    const int nt = max(1, (m + kSortTile - 1) / kSortTile);
    if ((int)blockIdx.x >= nt) return;
    h[threadIdx.x] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x * kSortTile;
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        long long e = base + k * kBlock + threadIdx.x;
        if (e < m) atomicAdd(&h[digit_of(keys, n, (int)e, shift)], 1);
    }
    __syncthreads();
    hist[(long long)threadIdx.x * nt + blockIdx.x] = h[threadIdx.x];
}

template <int KW>
__global__ __launch_bounds__(kBlock) void k_rs_scatter(const uint64_t *__restrict__ kin,
                                                       const int *__restrict__ vin,
                                                       uint64_t *__restrict__ kout,
                                                       int *__restrict__ vout, int n,
                                                       const int *n_dev, int shift,
                                                       const int *__restrict__ hist_scan,
                                                       const DevState *st) {
    if (st && st->done) return;
    const int m = min(n, *n_dev);
    const int nt = max(1, (m + kSortTile - 1) / kSortTile);
    if ((int)blockIdx.x >= nt) return;
    __shared__ int s_off[256];
    __shared__ int s_wc[kBlock / kWave][256];
    const int t = threadIdx.x, wid = t / kWave;
    s_off[t] = hist_scan[(long long)t * nt + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kBlock / kWave; w++) s_wc[w][t] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x * kSortTile;
    const int word = shift >> 6, sh = shift & 63;
    for (int k = 0; k < kSortItems; k++) {
        const long long e = base + k * kBlock + t;
        const bool valid = e < m;
        uint64_t kv[KW];
        int val = 0, dig = 0;
        if (valid) {
#pragma unroll
            for (int q = 0; q < KW; q++) kv[q] = kin[(long long)q * n + e];
            val = vin ? vin[e] : (int)e;
            dig = (int)((kv[word] >> sh) & 255ull);
        }
        unsigned long long m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (dig >> b) & 1;
            const unsigned long long bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const int r = __popcll(m & lanemask_lt());
        if (valid && r == 0) s_wc[wid][dig] = __popcll(m);
        __syncthreads();
        long long pos = 0;
        if (valid) {
            pos = s_off[dig] + r;
            for (int w = 0; w < wid; w++) pos += s_wc[w][dig];
        }
        __syncthreads();
        int tot = 0;
#pragma unroll
        for (int w = 0; w < kBlock / kWave; w++) {
            tot += s_wc[w][t];
            s_wc[w][t] = 0;
        }
        s_off[t] += tot;
        __syncthreads();
        if (valid) {
#pragma unroll
            for (int q = 0; q < KW; q++) kout[(long long)q * n + pos] = kv[q];
            vout[pos] = val;
        }
    }
}

// Stable sort of the first m = min(n, *n_dev) keys ([kw][n] words, the most
// significant word last, as the radix sort reads them) by rank: element i goes
// to the number of keys below it plus the number of equal keys before it, the
// position a stable sort gives it.  m^2 comparisons in one launch, where the
// radix sort takes three for each 8 bits.  A workgroup ranks 64 elements, a lane
// per element, its wavefronts against a share of the keys each: those are
// uniform, so they come through scalar loads and the compares leave lane masks.
// With lengths (LENS: the elements are runs of the previous grid) the same
// compares sum the lengths of the elements before i, the sorted run's first new
// position.  Bound by the VALU: 12 us for 2,000 keys of one word, 21 for 8,192, 65 for
// 20,000, 97 for 32,768; of two words 14, 42, 163 and 269.  A radix pass takes about
// 20 us at these sizes, its three launches included, and a key of one word has 4 to 8
// of them, one of two words 9 to 16: even at about 30,000 elements for either, hence
// kRankSortMax.
constexpr int kRankWaves = 16;

// Lanes whose key k is above key j (or, with EQ, equal to it).
template <int KW, bool EQ>
__device__ __forceinline__ bool key_after(const uint64_t (&k)[KW], const uint64_t (&j)[KW]) {
    bool r = EQ ? j[0] <= k[0] : j[0] < k[0];
#pragma unroll
    for (int w = 1; w < KW; w++) r = j[w] < k[w] || (j[w] == k[w] && r);
    return r;
}

template <int KW>
__global__ __launch_bounds__(kRankWaves *kWave) void k_rank_sort(
    const uint64_t *__restrict__ keys, int n, const int *__restrict__ run_start,
    int *__restrict__ sidx, int *__restrict__ off, int *__restrict__ src, const DevState *st,
    const DevState *st_loop) {
    if (st_loop && st_loop->done) return;
    const int m = st->sort_m, i0 = blockIdx.x * kWave;
    if (i0 >= m) return;
    __shared__ int s_rank[kRankWaves][kWave], s_off[kRankWaves][kWave];
    const int lane = __lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = min(i0 + lane, m - 1);
    uint64_t ki[KW];
#pragma unroll
    for (int w = 0; w < KW; w++) ki[w] = keys[(long long)w * n + i];
    const bool lens = st->lens_m > 0;
    int rank = 0, len = 0;
    // keys [j0, j1) are this wavefront's, in groups of kG
    constexpr int kG = KW == 1 ? 16 : 8;
    const int share = ((m + kRankWaves - 1) / kRankWaves + kG - 1) / kG * kG;
    const int j0 = min(wave * share, m), j1 = min(j0 + share, m);
    auto take = [&](auto eq, int a, int b) {
        constexpr bool EQ = decltype(eq)::value;
        int j = a;
        for (; j + kG <= b; j += kG) {
            uint64_t kj[kG][KW];
            int rs[kG + 1];
#pragma unroll
            for (int t = 0; t < kG; t++)
#pragma unroll
                for (int w = 0; w < KW; w++) kj[t][w] = keys[(long long)w * n + j + t];
            if (lens) {
#pragma unroll
                for (int t = 0; t <= kG; t++) rs[t] = run_start[j + t];
#pragma unroll
                for (int t = 0; t < kG; t++) {
                    const bool c = key_after<KW, EQ>(ki, kj[t]);
                    rank += c ? 1 : 0;
                    len += c ? rs[t + 1] - rs[t] : 0;
                }
            } else {
#pragma unroll
                for (int t = 0; t < kG; t++) rank += key_after<KW, EQ>(ki, kj[t]) ? 1 : 0;
            }
        }
        for (; j < b; j++) {
            uint64_t kj[KW];
#pragma unroll
            for (int w = 0; w < KW; w++) kj[w] = keys[(long long)w * n + j];
            const bool c = key_after<KW, EQ>(ki, kj);
            rank += c ? 1 : 0;
            if (lens) len += c ? run_start[j + 1] - run_start[j] : 0;
        }
    };
    // before the workgroup's elements an equal key comes first, after them not
    const int i1 = min(i0 + kWave, m);
    take(std::true_type{}, j0, max(j0, min(j1, i0)));
    take(std::false_type{}, min(j1, max(j0, i1)), j1);
    for (int j = max(j0, i0); j < min(j1, i1); j++) {
        uint64_t kj[KW];
#pragma unroll
        for (int w = 0; w < KW; w++) kj[w] = keys[(long long)w * n + j];
        const bool c = j < i ? key_after<KW, true>(ki, kj) : key_after<KW, false>(ki, kj);
        rank += c ? 1 : 0;
        if (lens) len += c ? run_start[j + 1] - run_start[j] : 0;
    }
    s_rank[wave][lane] = rank;
    s_off[wave][lane] = len;
    __syncthreads();
    if (wave != 0 || i0 + lane >= m) return;
    rank = len = 0;
#pragma unroll
    for (int w = 0; w < kRankWaves; w++) {
        rank += s_rank[w][lane];
        len += s_off[w][lane];
    }
    sidx[rank] = i;
    if (lens) {
        off[rank] = len;
        src[rank] = run_start[i];
    }
}

void rank_sort(const uint64_t *keys, int *sidx, int n, int kw, const int *run_start, int *off,
               int *src, const DevState *st, const DevState *st_loop, hipStream_t s) {
    const int blocks = (std::min(n, kRankSortMax) + kWave - 1) / kWave;
#define RANK_CASE(KW)                                                                       \
    case KW:                                                                                \
        k_rank_sort<KW><<<blocks, kRankWaves * kWave, 0, s>>>(keys, n, run_start, sidx,     \
                                                              off, src, st, st_loop);       \
        break;
    switch (kw) {
        RANK_CASE(1) RANK_CASE(2) RANK_CASE(3) RANK_CASE(4)
    }
#undef RANK_CASE
}

struct HistScan {
    int *hist;
    const int *n;
    __device__ int count() const { return *n; }
    __device__ void load(int i, int (&v)[1]) const { v[0] = hist[i]; }
    __device__ void store(int i, const int (&)[1], const int (&ex)[1]) const { hist[i] = ex[0]; }
    __device__ void finish(const int (&)[1]) const {}
};

size_t sort_tmp_ints(int n) {
    int ntiles = (n + kSortTile - 1) / kSortTile;
    if (ntiles == 0) ntiles = 1;
    return (size_t)256 * ntiles;
}

int radix_sort(uint64_t *keys_a, uint64_t *keys_b, int *vals_a, int *vals_b, int n, int kw,
               int key_bits, int *hist, int *scan_tmp, const DevState *st, hipStream_t s,
               const int *n_dev, const int *hist_n_dev) {
    int ntiles = (n + kSortTile - 1) / kSortTile;
    if (ntiles == 0) ntiles = 1;
    const int passes = (key_bits + 7) / 8;
    uint64_t *kin = keys_a, *kout = keys_b;
    int *vin = nullptr, *vout = vals_b;
    int where = 0;
    for (int p = 0; p < passes; p++) {
        const int shift = p * 8;
        k_rs_hist<<<ntiles, kBlock, 0, s>>>(kin, n, n_dev, shift, hist, st);
        launch_scan<1>(HistScan{hist, hist_n_dev}, 256 * ntiles, scan_tmp, st, s);
#define RS_CASE(KW)                                                                          \
    case KW:                                                                                 \
        k_rs_scatter<KW><<<ntiles, kBlock, 0, s>>>(kin, vin, kout, vout, n, n_dev, shift,    \
                                                   hist, st);                                \
        break;
        switch (kw) {
            RS_CASE(1) RS_CASE(2) RS_CASE(3) RS_CASE(4)
        }
#undef RS_CASE
        where ^= 1;
        uint64_t *tk = kin; kin = kout; kout = tk;
        vin = vout;
        vout = (vout == vals_b) ? vals_a : vals_b;
    }
    if (passes == 0) {
        // a single cell: identity order (keys unchanged in keys_a)
        return -1;
    }
    return where;
}

}  // namespace egg
