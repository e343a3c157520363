// Device side of the exclusive scans (gfx950): a tile of values per workgroup,
// tiles joined by decoupled look-back (Merrill and Garland,
// "Single-pass Parallel Prefix Scan with Decoupled Look-back", 2016).
//
// Each workgroup takes a tile from a ticket counter (so a tile's predecessors
// belong to workgroups that started earlier), scans it locally and publishes
// its sums; a wavefront per channel then walks back over its predecessors'
// published words, 64 at a time, adding sums until it meets an inclusive
// prefix, and publishes its own inclusive prefix.  A tile's sums are published
// before anything of that channel is waited for, so every wait ends; the wait
// is still bounded (kLbSpins polls, then an error flag and a wrong prefix,
// reported to the host by scan_tmp_error).
//
// State in lb: [0] ticket, [1] workgroups finished, [2] scan sequence number,
// [3] error flag; from int 4 on, one 64-bit word per channel and tile: flag
// (bits 63-62: 1 sum, 2 inclusive prefix), the sequence number of the scan that
// wrote it (bits 61-32, so that words of earlier scans read as unpublished) and
// the value (bits 31-0).  The last workgroup to finish resets the counters and
// advances the sequence number.
#pragma once

#include "egg_internal.h"

namespace egg {

constexpr int kLbSpins = 1 << 20;
constexpr unsigned long long kLbSum = 1ull << 62, kLbIncl = 2ull << 62;

__device__ __forceinline__ int wave_incl_scan(int v) {
    const int lane = __lane_id();
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        int t = __shfl_up(v, o, kWave);
        if (lane >= o) v += t;
    }
    return v;
}

// Exclusive scan of one value per thread over a block of B threads; also
// returns the total.
template <int B = kBlock>
__device__ __forceinline__ int block_excl_scan(int v, int *s_w, int &total) {
    const int lane = __lane_id(), wid = threadIdx.x / kWave;
    int inc = wave_incl_scan(v);
    if (lane == kWave - 1) s_w[wid] = inc;
    __syncthreads();
    int woff = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < B / kWave; w++) {
        int t = s_w[w];
        if (w < wid) woff += t;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return woff + inc - v;
}

__device__ __forceinline__ unsigned long long lb_word(unsigned long long flag, unsigned seq,
                                                      int v) {
    return flag | ((unsigned long long)(seq & 0x3fffffffu) << 32) | (unsigned)v;
}

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

// Exclusive prefix of tile `tile` (> 0) from its predecessors' words; one
// wavefront.
__device__ __forceinline__ int lb_prefix(const unsigned long long *status, int tile, unsigned seq,
                                         int *err) {
    const int lane = __lane_id();
    const unsigned tag = seq & 0x3fffffffu;
    int pre = 0, spins = 0;
    for (int j = tile - 1;;) {
        const int idx = j - lane;
        int flag = 2, val = 0;  // before tile 0: an inclusive prefix of 0
        if (idx >= 0) {
            const unsigned long long w =
                __hip_atomic_load(status + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            flag = (unsigned)((w >> 32) & 0x3fffffffu) == tag ? (int)(w >> 62) : 0;
            val = (int)(unsigned)w;
        }
        const unsigned long long incl = __ballot(flag == 2);
        const unsigned long long none = __ballot(flag == 0);
        const int stop = incl ? __ffsll((long long)incl) - 1 : kWave - 1;
        const unsigned long long need = stop == kWave - 1 ? ~0ull : ((2ull << stop) - 1ull);
        if (none & need) {
            if (++spins > kLbSpins) {
                if (lane == 0) atomicOr(err, 1);
                return pre;
            }
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        pre += wave_sum(lane <= stop ? val : 0);
        if (incl) return pre;
        j -= kWave;
    }
}

// Tile of this workgroup and the scan's sequence number (every thread calls it).
__device__ __forceinline__ int lb_begin(int *lb, int *s_tile, unsigned &seq) {
    if (threadIdx.x == 0) *s_tile = atomicAdd(&lb[0], 1);
    __syncthreads();
    seq = __hip_atomic_load((const unsigned *)&lb[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return *s_tile;
}

// Publishes the tile's sums tot[NC] (LDS, complete) of its nb tiles and leaves
// the exclusive prefixes in pre[NC] (LDS) behind a barrier.
template <int NC>
__device__ __forceinline__ void lb_join(int *lb, int tile, int nb, unsigned seq, const int *tot,
                                        int *pre) {
    unsigned long long *status = (unsigned long long *)(lb + 4);
    const int wave = threadIdx.x / kWave;
    static_assert(NC <= kBlock / kWave, "a wavefront per channel");
    if (wave < NC) {
        unsigned long long *sc = status + (long long)wave * nb;
        const int t = tot[wave], lane = __lane_id();
        if (lane == 0)
            __hip_atomic_store(sc + tile, lb_word(tile == 0 ? kLbIncl : kLbSum, seq, t),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int p = tile == 0 ? 0 : lb_prefix(sc, tile, seq, &lb[3]);
        if (lane == 0) {
            pre[wave] = p;
            if (tile > 0)
                __hip_atomic_store(sc + tile, lb_word(kLbIncl, seq, p + t), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
}

// End of a workgroup's part (of nb); its words have been read or need no reader.
__device__ __forceinline__ void lb_end(int *lb, int nb, unsigned seq) {
    if (threadIdx.x == 0) {
        const int fin = atomicAdd(&lb[1], 1);
        if (fin == nb - 1) {
            __hip_atomic_store(&lb[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&lb[1], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store((unsigned *)&lb[2], seq + 1u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// Exclusive scan of NC channels over io.count() values (at most nb tiles of
// ITEMS * kBlock) by nb workgroups of kBlock threads.  The io object makes the values and
// takes the results, so that neither passes through memory:
//   load(i, v)        the NC values of element i
//   store(i, v, ex)   element i's values and their exclusive sums
//   finish(tot)       the totals (one thread of the grid)
// The elements pass through LDS between a coalesced order (global accesses)
// and ITEMS consecutive ones per thread (the sums); the pad of one int in 32
// keeps the latter off each other's banks.
template <int NC, int ITEMS, class IO>
__device__ __forceinline__ void scan_tiles(const IO &io, int *lb, int nb) {
    constexpr int kTileN = ITEMS * kBlock, kPad = kTileN + kTileN / 32;
    __shared__ int s_v[NC][kPad];
    __shared__ int s_w[kBlock / kWave], s_tot[NC], s_pre[NC], s_tile;
    const int m = io.count();
    // one tile at run time: workgroup 0 scans it alone, no state is touched
    const bool alone = m <= kTileN;
    if (alone && blockIdx.x != 0) return;
    int tile = 0;
    unsigned seq = 0;
    if (!alone) tile = lb_begin(lb, &s_tile, seq);
    const int base = tile * kTileN;
    if (base < m || alone) {
        int v[ITEMS][NC];
        auto at = [](int e) { return e + e / 32; };
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            const int e = k * kBlock + threadIdx.x;
#pragma unroll
            for (int c = 0; c < NC; c++) v[k][c] = 0;
            if (base + e < m) io.load(base + e, v[k]);
#pragma unroll
            for (int c = 0; c < NC; c++) s_v[c][at(e)] = v[k][c];
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NC; c++) {
            int x[ITEMS], sum = 0;
#pragma unroll
            for (int k = 0; k < ITEMS; k++) {
                x[k] = s_v[c][at(threadIdx.x * ITEMS + k)];
                sum += x[k];
            }
            int tot, ex = block_excl_scan(sum, s_w, tot);
            if (threadIdx.x == 0) {
                s_tot[c] = tot;
                s_pre[c] = 0;
            }
#pragma unroll
            for (int k = 0; k < ITEMS; k++) {
                s_v[c][at(threadIdx.x * ITEMS + k)] = ex;
                ex += x[k];
            }
        }
        __syncthreads();
        if (!alone) lb_join<NC>(lb, tile, nb, seq, s_tot, s_pre);
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            const int e = k * kBlock + threadIdx.x;
            if (base + e >= m) continue;
            int ex[NC];
#pragma unroll
            for (int c = 0; c < NC; c++) ex[c] = s_v[c][at(e)] + s_pre[c];
            io.store(base + e, v[k], ex);
        }
        if (base + kTileN >= m && threadIdx.x == 0) {
            int tot[NC];
#pragma unroll
            for (int c = 0; c < NC; c++) tot[c] = s_pre[c] + s_tot[c];
            io.finish(tot);
        }
    }
    if (!alone) lb_end(lb, nb, seq);
}

template <int NC, int ITEMS, class IO>
__global__ __launch_bounds__(kBlock) void k_scan(IO io, int *lb, const DevState *st) {
    if (st && st->done) return;
    scan_tiles<NC, ITEMS>(io, lb, gridDim.x);
}

// Workgroups of a scan of up to n values, kScanItems (wide) or kScanNarrow a
// thread.  Wide tiles mean fewer steps of look-back, narrow ones more CUs at work:
// the radix sort's 12,500 histogram values at n = 100,000 take 5.7 us narrow and
// 7.2 wide, its 125,000 at n = 1,000,000 12.4 and 8.6; k_tables<3> takes 20 us
// narrow and 38 wide at n = 100,000, 11 and 26 at n = 2,000.  The tables' line
// (kTablesNarrowMax) lies where the forms are even: a features call at d = 3, which has
// two such scans, takes 240 us narrow and 262 wide at n = 131,072, 288 and 289 at
// 262,144, 351 and 320 at 400,000, 676 and 498 at 1,000,000; d = 2 and 5 cross between
// 200,000 and 262,144 too.
static inline int scan_blocks(int n, bool wide) {
    const int tile = kBlock * (wide ? kScanItems : kScanNarrow);
    return n > 0 ? (n + tile - 1) / tile : 1;
}

template <int NC, class IO>
static void launch_scan(const IO &io, int n, int *lb, const DevState *st, hipStream_t s) {
    const bool wide = n > kScanNarrowMax;
    const int nb = scan_blocks(n, wide);
    if (wide) k_scan<NC, kScanItems><<<nb, kBlock, 0, s>>>(io, lb, st);
    else k_scan<NC, kScanNarrow><<<nb, kBlock, 0, s>>>(io, lb, st);
}

}  // namespace egg
