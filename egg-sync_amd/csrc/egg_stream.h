// Masked sums over streamed source runs on the matrix cores (gfx950).
//
// A wavefront holds a target per lane.  Ranges of source runs, each with the
// mask of the lanes that test it, are noted as segments and worked off together
// (flush), 64 slots at a time: every lane loads one source, leaves its offset u
// from the tile's centre and w sin v, w cos v - w, w of its offset v from the
// anchor in LDS, and then two sets of v_mfma_f32_4x4x1_16b take them four sources
// (a group) at a time.  A group belongs to one segment; slots without a source add
// zeros.  As used here the instruction multiplies, for every lane, four values
// that any lane may supply (A, from LDS) by the lane's own (B) into four of the
// lane's own accumulators: 4 FMAs a lane in 8 cycles, twice the VALU's rate.
//
//   test:  t[r] = C + Q_r + sum_l u_rl X_l, a K-step per dimension and one for Q,
//          with X = 2 u_x / m, C = (eps^2 - |u_x|^2) / m, Q = -|u_q|^2 / m: the
//          margin by which source r is within eps, in units of m, and m bounds the
//          difference between this and the reference's FP32 distance.  |t| >= 1
//          therefore decides as the reference does; a group with a smaller |t|
//          (one in a hundred) takes the reference's formula instead.
//   sums:  d[c] += col_c * a with a = clamp(t) = 0 or 1, one K-step per source:
//          an FP32 addition of the value or of 0 per source, in source order, bit
//          for bit what a scalar loop over the sources within eps would add.
//
// The count column is exact while the tile's counts stay below 2^24: n < 2^24.
//
// Segments of the other kind only count their points within eps/2 (C from eps/2,
// the run lengths added up on the VALU).
//
// Per source and 64 targets at d = 3: 8 cycles of test, 6 of clamp and minimum, 16
// of sums.  Distances on the VALU, a swap to the other layout of the same MFMA and
// a pass through LDS to and from that layout in every chunk took 68 and 1,800 more
// per chunk.
#pragma once

#include "egg_wave.h"

namespace egg {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int D>
struct StreamLds {
    static constexpr int kCols = (2 * D + 1 + 3) / 4 * 4;
    static constexpr int kStride = kWave + 4;  // a row per column, 16-byte aligned
    float u[D + 1][kWave];                     // u, then Q
    float col[kCols][kStride];                 // w sin v [D], w, w (cos v - 1) [D]
    int j[kWave];                              // first position of the source, -1 without one
};

// The anchor of the streamed sums in dimension l: the centre of the tile's cell in
// the outer dimensions and of its block of kAnchorBlock cells in the inner ones, the
// same for every group width that divides kAnchorBlock.
__device__ __forceinline__ float tile_anchor(int g0, int l, const Geo &g) {
    return l < g.od ? ((float)g0 + 0.5f) * g.cs
                    : ((float)(g0 & ~(kAnchorBlock - 1)) + 0.5f * kAnchorBlock) * g.cs;
}

// A value every lane holds, in scalar registers.
__device__ __forceinline__ float uniform(float v) {
    return __uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)__float_as_uint(v)));
}

__device__ __forceinline__ unsigned long long uniform(unsigned long long v) {
    return (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 |
           (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}

template <int D>
struct Stream {
    static constexpr int kM = StreamLds<D>::kCols / 4;
    static constexpr float kNever = -1e30f;  // C of a lane that does not test, Q of no source

    f32x4 d[kM];           // sums: column 4 m + r in d[m][r]
    float near;            // points within eps/2
    float inv_m, bound_q;  // 1 / m, bound on |u_q|^2 that m was made for
    bool exact;            // no valid m: every group takes the reference's formula
    // lane k: segment k -- runs [ra, rb), first group, lanes that test it
    int ra, rb, gr;
    unsigned mlo, mhi;
    unsigned long long nears;  // segments that count within eps/2
    int nseg, ngroups;

    __device__ __forceinline__ float sin_sum(int l) const { return d[l / 4][l % 4]; }
    __device__ __forceinline__ int count() const { return (int)d[D / 4][D % 4]; }
    __device__ __forceinline__ float cos_sum(int l) const {
        return d[(D + 1 + l) / 4][(D + 1 + l) % 4];
    }
    __device__ __forceinline__ void clear_sums() {
#pragma unroll
        for (int m = 0; m < kM; m++) d[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // A tile whose targets have |u_x|^2 <= ux.  With U bounding |u_x| + |u_q|, in
    // units of 2^-24: rounding of u moves the squared distance by 2 U^2; C, Q and
    // X carry 5 U^2 + thr and another 3 U^2 + thr from their scaling; the D + 1
    // K-steps round values up to thr + 2 U^2, D + 1 <= 6 of them; the reference's
    // formula is within (D + 2) thr.  Below 24 U^2 + 16 thr together; m is
    // 40 U^2 + 24 thr.  Streamed cells are within eps of a target, so |u_q| is at
    // most |u_x| + eps + the cell's diagonal eps / 2; positions beyond that (clamped
    // cell coordinates) are found by bound_q.
    __device__ __forceinline__ void init(float ux, const Geo &g) {
        const float bx = sqrtf(ux) * (1.0f + 0x1p-10f);
        const float bq = bx + 1.5f * g.eps * (1.0f + 0x1p-10f);
        const float U = bx + bq;
        const float m = 0x1p-24f * (40.0f * U * U + 24.0f * g.thr_eps);
        static_assert(D + 1 <= 6, "K-steps the margin allows for");
        exact = __any(!(m > 1e-30f && m < 1e30f));
        inv_m = uniform(1.0f / m);
        bound_q = uniform(bq * bq);
        clear_sums();
        near = 0.f;
        nears = 0;
        nseg = ngroups = 0;
    }

    __device__ __forceinline__ void hold_uniform() {
        nseg = __builtin_amdgcn_readfirstlane(nseg);
        ngroups = __builtin_amdgcn_readfirstlane(ngroups);
        nears = uniform(nears);
    }

    // Runs [a, b), a < b, for the lanes of mask.
    __device__ __forceinline__ void add(int a, int b, unsigned long long mask,
                                        bool count_near = false) {
        a = __builtin_amdgcn_readfirstlane(a);
        b = __builtin_amdgcn_readfirstlane(b);
        const bool me = __lane_id() == nseg;
        ra = me ? a : ra;
        rb = me ? b : rb;
        gr = me ? ngroups : gr;
        mlo = me ? (unsigned)mask : mlo;
        mhi = me ? (unsigned)(mask >> 32) : mhi;
        nears |= (unsigned long long)count_near << nseg;
        nseg++;
        ngroups += (b - a + 3) / 4;
    }

    // The reference's test for the group of slots k .. k + 3.
    __device__ __forceinline__ void exact_group(const StreamLds<D> &s, int k, bool tests,
                                                const float (&x)[D], float thr,
                                                const float *__restrict__ Xs, int n,
                                                float (&a)[4]) const {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = __builtin_amdgcn_readfirstlane(s.j[k + r]);
            a[r] = 0.f;
            if (j >= 0) {
                float sq = 0.f;
#pragma unroll
                for (int l = 0; l < D; l++) {
                    const float df = x[l] - Xs[(long long)l * n + j];
                    sq += df * df;
                }
                a[r] = tests && sq <= thr ? 1.f : 0.f;
            }
        }
    }

    // Adds the segments noted so far, in order: targets x (active lanes) of a tile of
    // the cell at coordinates g0.
    __device__ __forceinline__ void flush(StreamLds<D> &s, const float (&x)[D], bool active,
                                          const int (&g0)[D], const Geo &g,
                                          const float *__restrict__ Xs,
                                          const int *__restrict__ run_start) {
        const int n = g.n;
        hold_uniform();
        if (!ngroups) return;
        float a0[D], ctr[D], X[D], u2 = 0.f;  // the anchor, the centre, see above
#pragma unroll
        for (int l = 0; l < D; l++) {
            a0[l] = tile_anchor(g0[l], l, g);
            ctr[l] = cell_mid(g0[l], g.cs);
            // a target that is not a number is within eps of nothing and tests nothing
            const float u = active && x[l] == x[l] ? x[l] - ctr[l] : 0.f;
            u2 += u * u;
            X[l] = 2.0f * u * inv_m;
        }
        const float C = (g.thr_eps - u2) * inv_m, C_near = (g.thr_half - u2) * inv_m;
        constexpr int kG = kWave / 4;  // groups per chunk
        const int lane = __lane_id(), l4 = lane & 3;
        int seg = 0;  // first segment of the next chunk to locate
        // the lane's source run in the chunk from group cb, and the groups of it
        // that start a segment
        auto locate = [&](int cb, unsigned &starts) {
            const int gi = cb + lane / 4;
            int rr = -1;
            starts = 0;
            for (; seg < nseg; seg++) {
                const int sg = __builtin_amdgcn_readlane(gr, seg);
                if (sg >= cb + kG) break;
                const int q = __builtin_amdgcn_readlane(ra, seg) + 4 * (gi - sg) + l4;
                if (gi >= sg) rr = q < __builtin_amdgcn_readlane(rb, seg) ? q : -1;
                if (sg >= cb) starts |= 1u << (sg - cb);
            }
            seg--;  // the last one may go on in the next chunk
            return rr;
        };
        unsigned starts;
        int rr = locate(0, starts);
        int j = 0, e = 0;
        float xq[D];
        if (rr >= 0) {
            j = run_start[rr];
            e = run_start[rr + 1];
        }
#pragma unroll
        for (int l = 0; l < D; l++) xq[l] = rr >= 0 ? Xs[(long long)l * n + j] : 0.f;
        int cur = -1;  // segment of the group at work
        bool tests = false, count_near = false;
        f32x4 c4 = {0.f, 0.f, 0.f, 0.f};
        for (int cb = 0; cb < ngroups; cb += kG) {
            // the next chunk's loads go out while this one is worked off
            unsigned starts_n = 0;
            int rr_n = -1, j_n = 0, e_n = 0;
            if (cb + kG < ngroups) {
                rr_n = locate(cb + kG, starts_n);
                if (rr_n >= 0) {
                    j_n = run_start[rr_n];
                    e_n = run_start[rr_n + 1];
                }
            }
            float u[D], uu = 0.f;
#pragma unroll
            for (int l = 0; l < D; l++) {
                u[l] = rr >= 0 ? xq[l] - ctr[l] : 0.f;
                uu += u[l] * u[l];
            }
            // a source that is infinite or not a number is within eps of no target
            // and takes no slot: its column times 0 would not be 0
            const bool on = rr >= 0 && uu < INFINITY;
            const float w = on ? (float)(e - j) : 0.f;  // exact: < 2^24
#pragma unroll
            for (int l = 0; l < D; l++) {
                float sv, cv;
                sincosm1_small(on ? xq[l] - a0[l] : 0.f, sv, cv);
                s.col[l][lane] = w * sv;
                s.col[D + 1 + l][lane] = w * cv;
                s.u[l][lane] = on ? u[l] : 0.f;
            }
            s.col[D][lane] = w;
            s.u[D][lane] = on ? -(uu * inv_m) : kNever;
            s.j[lane] = on ? j : -1;
            const bool all_exact = exact || __any(on && !(uu <= bound_q));
            wave_sync();
#pragma unroll
            for (int l = 0; l < D; l++) xq[l] = rr_n >= 0 ? Xs[(long long)l * n + j_n] : 0.f;
            const int groups = min(kG, ngroups - cb);
            for (int i = 0; i < groups;) {
                if (starts >> i & 1) {
                    cur++;
                    const unsigned long long mask =
                        (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)mhi, cur)
                            << 32 |
                        (unsigned)__builtin_amdgcn_readlane((int)mlo, cur);
                    tests = mask >> lane & 1;
                    count_near = nears >> cur & 1;
                    const float c = tests ? (count_near ? C_near : C) : kNever;
                    c4 = f32x4{c, c, c, c};
                }
                const int k = 4 * i;
                const float thr = count_near ? g.thr_half : g.thr_eps;
                const bool two = i + 1 < groups && !(starts >> (i + 1) & 1);
                if (two) {
                    f32x4 t0 = c4, t1 = c4;
#pragma unroll
                    for (int l = 0; l <= D; l++) {
                        const float b = l < D ? X[l] : 1.0f;
                        t0 = __builtin_amdgcn_mfma_f32_4x4x1f32(s.u[l][k + l4], b, t0, 0, 0, 0);
                        t1 = __builtin_amdgcn_mfma_f32_4x4x1f32(s.u[l][k + 4 + l4], b, t1, 0, 0, 0);
                    }
                    i += 2;
                    f32x4 v0[kM], v1[kM];
#pragma unroll
                    for (int m = 0; m < kM; m++) {
                        v0[m] = *reinterpret_cast<const f32x4 *>(&s.col[4 * m + l4][k]);
                        v1[m] = *reinterpret_cast<const f32x4 *>(&s.col[4 * m + l4][k + 4]);
                    }
                    float a[4], b[4], mn = 1e30f;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        mn = fminf(fminf(mn, fabsf(t0[r])), fabsf(t1[r]));
                        a[r] = __builtin_amdgcn_fmed3f(t0[r], 0.f, 1.f);
                        b[r] = __builtin_amdgcn_fmed3f(t1[r], 0.f, 1.f);
                    }
                    if (all_exact || __any(mn < 1.f)) {
                        exact_group(s, k, tests, x, thr, Xs, n, a);
                        exact_group(s, k + 4, tests, x, thr, Xs, n, b);
                    }
                    if (count_near) {
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            near += a[r] * s.col[D][k + r] + b[r] * s.col[D][k + 4 + r];
                        continue;
                    }
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int m = 0; m < kM; m++)
                            d[m] = __builtin_amdgcn_mfma_f32_4x4x1f32(v0[m][r], a[r], d[m], 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int m = 0; m < kM; m++)
                            d[m] = __builtin_amdgcn_mfma_f32_4x4x1f32(v1[m][r], b[r], d[m], 0, 0, 0);
                } else {
                    f32x4 t0 = c4;
#pragma unroll
                    for (int l = 0; l <= D; l++)
                        t0 = __builtin_amdgcn_mfma_f32_4x4x1f32(s.u[l][k + l4],
                                                                l < D ? X[l] : 1.0f, t0, 0, 0, 0);
                    i += 1;
                    f32x4 v0[kM];
#pragma unroll
                    for (int m = 0; m < kM; m++)
                        v0[m] = *reinterpret_cast<const f32x4 *>(&s.col[4 * m + l4][k]);
                    float a[4], mn = 1e30f;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        mn = fminf(mn, fabsf(t0[r]));
                        a[r] = __builtin_amdgcn_fmed3f(t0[r], 0.f, 1.f);
                    }
                    if (all_exact || __any(mn < 1.f))
                        exact_group(s, k, tests, x, thr, Xs, n, a);
                    if (count_near) {
#pragma unroll
                        for (int r = 0; r < 4; r++) near += a[r] * s.col[D][k + r];
                        continue;
                    }
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int m = 0; m < kM; m++)
                            d[m] = __builtin_amdgcn_mfma_f32_4x4x1f32(v0[m][r], a[r], d[m], 0, 0, 0);
                }
            }
            wave_sync();
            starts = starts_n;
            rr = rr_n;
            j = j_n;
            e = e_n;
        }
        nseg = ngroups = 0;
        nears = 0;
    }
};

}  // namespace egg
