// MLP of the learned jump: in -> hidden -> hidden -> out, ReLU, FP32.
//
// Training is expressed as small GEMMs on a batch (activations [B x width],
// row-major) with a strided FP32 GEMM kernel: 64x64 output tiles staged
// through LDS, 4x4 outputs per thread, split over K with a deterministic
// reduction of the K-slices, so gradients are reproducible bit for bit.
// The jump network itself (12-128-128-3) takes fused kernels on the FP32
// matrix cores, for inference and for the training step.
//
// Parameters live in one flat array: W1[h][in], b1[h], W2[h][h], b2[h],
// W3[out][h], b3[out].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "../../include/egg_sync.h"

namespace egg {
namespace mlp {

constexpr int kT = 64;      // output tile edge
constexpr int kKT = 16;     // K tile
constexpr int kThreads = 256;

struct Dims {
    int in, h, out;
    constexpr long long n_w1() const { return (long long)h * in; }
    constexpr long long off_b1() const { return n_w1(); }
    constexpr long long off_w2() const { return off_b1() + h; }
    constexpr long long off_b2() const { return off_w2() + (long long)h * h; }
    constexpr long long off_w3() const { return off_b2() + h; }
    constexpr long long off_b3() const { return off_w3() + (long long)out * h; }
    constexpr long long total() const { return off_b3() + out; }
};

// C_part[s][m][n] = sum_{k in slice s} A(m,k) * B(k,n), A(m,k) = A[m*sam + k*sak],
// B(k,n) = B[k*sbk + n*sbn].
__global__ __launch_bounds__(kThreads) void k_gemm_part(const float *__restrict__ A,
                                                        long long sam, long long sak,
                                                        const float *__restrict__ B,
                                                        long long sbk, long long sbn,
                                                        float *__restrict__ Cpart, int M, int N,
                                                        int K, int kslice) {
    __shared__ float sA[kKT][kT + 1];
    __shared__ float sB[kKT][kT + 1];
    const int tm = blockIdx.y * kT, tn = blockIdx.x * kT, s = blockIdx.z;
    const int k0 = s * kslice, k1 = min(K, k0 + kslice);
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    float acc[4][4] = {};
    for (int kb = k0; kb < k1; kb += kKT) {
        for (int e = threadIdx.x; e < kKT * kT; e += kThreads) {
            const int kk = e / kT, mm = e % kT;
            const int k = kb + kk;
            sA[kk][mm] = (k < k1 && tm + mm < M) ? A[(tm + mm) * sam + k * sak] : 0.f;
            sB[kk][mm] = (k < k1 && tn + mm < N) ? B[k * sbk + (tn + mm) * sbn] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kKT; kk++) {
            float a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                a[q] = sA[kk][ty * 4 + q];
                b[q] = sB[kk][tx * 4 + q];
            }
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int q = 0; q < 4; q++) acc[p][q] = fmaf(a[p], b[q], acc[p][q]);
        }
        __syncthreads();
    }
    float *C = Cpart + (long long)s * M * N;
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int m = tm + ty * 4 + p, n = tn + tx * 4 + q;
            if (m < M && n < N) C[(long long)m * N + n] = acc[p][q];
        }
}

// C[m][n] (row stride ldc) = sum_s Cpart[s][m][n] (+ bias[n]); act: 0 none, 1 ReLU.
__global__ void k_gemm_reduce(const float *__restrict__ Cpart, int S, int M, int N,
                              const float *__restrict__ bias, int act, float *__restrict__ C,
                              long long ldc) {
    const long long MN = (long long)M * N;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < MN;
         e += (long long)gridDim.x * blockDim.x) {
        float v = 0.f;
        for (int s = 0; s < S; s++) v += Cpart[s * MN + e];
        const int n = (int)(e % N);
        if (bias) v += bias[n];
        if (act == 1) v = fmaxf(v, 0.f);
        C[(e / N) * ldc + n] = v;
    }
}

// dZ = dH * (Z > 0) in place on dH (ReLU derivative).
__global__ void k_relu_mask(float *__restrict__ dH, const float *__restrict__ H, long long count) {
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < count;
         e += (long long)gridDim.x * blockDim.x)
        if (!(H[e] > 0.f)) dH[e] = 0.f;
}

// Column sums of a [rows x cols] matrix (bias gradients), fixed order.
__global__ void k_colsum(const float *__restrict__ X, int rows, int cols, float *__restrict__ out) {
    const int c = blockIdx.x;
    __shared__ float s[kThreads];
    float v = 0.f;
    for (int r = threadIdx.x; r < rows; r += kThreads) v += X[(long long)r * cols + c];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[c] = s[0];
}

// dO = 2 (O - Y) / B, loss partials per block.
__global__ void k_mse_grad(const float *__restrict__ O, const float *__restrict__ Y, long long count,
                           float inv_b, float *__restrict__ dO, double *__restrict__ loss_part) {
    __shared__ double s[kThreads];
    double l = 0.0;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < count;
         e += (long long)gridDim.x * blockDim.x) {
        const float r = O[e] - Y[e];
        dO[e] = 2.f * r * inv_b;
        l += (double)r * (double)r;
    }
    s[threadIdx.x] = l;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_part[blockIdx.x] = s[0];
}

__global__ void k_loss_finish(const double *__restrict__ part, int nparts, double inv_b,
                              double *__restrict__ loss) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < nparts; i++) t += part[i];
        *loss = t * inv_b;
    }
}

// ------------------------------------------- the jump network on MFMA --
//
// The 12-128-128-3 network (the jump's) runs on the FP32 matrix cores,
// v_mfma_f32_32x32x2_f32: lane l holds A[l & 31][l >> 5] and B[l >> 5][l & 31]
// and, of the 32 x 32 result, the rows 8g + 4h + q (register 4g + q, h = l >> 5)
// of column l & 31.  Hidden units are rows and points columns, so a layer's
// result registers are the next layer's B operands when the contraction runs
// over k = 8g + 4h + q in the order of (g, q): the activations stay in
// registers, and one 16-byte LDS read per lane holds the weights of four
// steps.
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kIn = 12, kHid = 128, kOut = 3;  // the jump network
constexpr int kCols = 32;                      // points per MFMA tile
constexpr int kTiles = kHid / 32;              // row tiles of a hidden layer
constexpr int kLdW = kHid + 4;   // row stride of W2 in LDS: 16-byte rows, and 4 banks apart, so
                                 // that a 16-byte read of 16 rows touches every bank once
constexpr int kLdW1 = kIn + 2;   // row stride of W1: 8-byte rows

__device__ __forceinline__ f32x16 mfma(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Rows 8g + 4h + q of a 32-row tile of a vector in LDS, as a result tile
// starts from its bias.
__device__ __forceinline__ f32x16 row_vector(const float *v, int h) {
    f32x16 c;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(v + 8 * g + 4 * h);
#pragma unroll
        for (int q = 0; q < 4; q++) c[4 * g + q] = b[q];
    }
    return c;
}

// Inference.  Bound by the FP32 matrix pipe: 280 MFMAs of 64 cycles per 32
// points, 0.24 ms for 2^20 points.  A wavefront takes 32 points through all
// layers; the weights (77 KB in LDS) are loaded once per workgroup, two
// workgroups of four wavefronts per CU walk the points.  The three outputs
// are a dot product per lane (a 32-row MFMA tile would be 3 rows of work).
// 2^20 points: 2,620 us with one point per thread on the vector ALUs, 289 us
// here (134 TFLOP/s; a large FP32 matrix product reaches 150).
__global__ __launch_bounds__(kThreads, 2) void k_jump_infer(const float *__restrict__ P,
                                                            const float *__restrict__ X,
                                                            long long B,
                                                            float *__restrict__ Y) {
    __shared__ __align__(16) float sW2[kHid * kLdW], sW1[kHid * kLdW1], sb1[kHid], sb2[kHid],
        sW3[kOut * kHid];
    constexpr Dims D{kIn, kHid, kOut};
#pragma unroll 16
    for (int e = threadIdx.x; e < kHid * kHid; e += kThreads)
        sW2[(e / kHid) * kLdW + e % kHid] = P[D.off_w2() + e];
    for (int e = threadIdx.x; e < kHid * kIn; e += kThreads)
        sW1[(e / kIn) * kLdW1 + e % kIn] = P[e];
    for (int e = threadIdx.x; e < kOut * kHid; e += kThreads) sW3[e] = P[D.off_w3() + e];
    for (int e = threadIdx.x; e < kHid; e += kThreads) {
        sb1[e] = P[D.off_b1() + e];
        sb2[e] = P[D.off_b2() + e];
    }
    float b3[kOut];
#pragma unroll
    for (int m = 0; m < kOut; m++) b3[m] = P[D.off_b3() + m];
    __syncthreads();
    const int lane = __lane_id(), col = lane & 31, h = lane >> 5;
    constexpr int kWaves = kThreads / 64;
    const long long tiles = (B + kCols - 1) / kCols;
    for (long long t = blockIdx.x * (long long)kWaves + threadIdx.x / 64; t < tiles;
         t += (long long)gridDim.x * kWaves) {
        // the weights are read from LDS where they are used: hoisted out of this
        // loop, or all up front, they would not fit the registers
        __asm__ volatile("" ::: "memory");
        const long long p = t * kCols + col;
        float x[kIn / 2];  // the half's six inputs of the point
#pragma unroll
        for (int s = 0; s < kIn / 2; s++) x[s] = p < B ? X[p * kIn + (kIn / 2) * h + s] : 0.f;
        f32x16 h1[kTiles], h2[kTiles];
#pragma unroll
        for (int i = 0; i < kTiles; i++) {
            h1[i] = row_vector(sb1 + 32 * i, h);
            const float *w = sW1 + (32 * i + col) * kLdW1 + (kIn / 2) * h;
#pragma unroll
            for (int s = 0; s < kIn / 2; s++) h1[i] = mfma(w[s], x[s], h1[i]);
#pragma unroll
            for (int r = 0; r < 16; r++) h1[i][r] = fmaxf(h1[i][r], 0.f);
            h2[i] = row_vector(sb2 + 32 * i, h);
        }
#pragma unroll
        for (int k = 0; k < kTiles; k++) {
            __asm__ volatile("" ::: "memory");
#pragma unroll
            for (int g = 0; g < 4; g++) {
                f32x4 w[kTiles];
#pragma unroll
                for (int i = 0; i < kTiles; i++)
                    w[i] = *reinterpret_cast<const f32x4 *>(sW2 + (32 * i + col) * kLdW + 32 * k +
                                                            8 * g + 4 * h);
#pragma unroll
                for (int q = 0; q < 4; q++)
#pragma unroll
                    for (int i = 0; i < kTiles; i++) h2[i] = mfma(w[i][q], h1[k][4 * g + q], h2[i]);
            }
        }
        __asm__ volatile("" ::: "memory");
        float o[kOut] = {};
#pragma unroll
        for (int i = 0; i < kTiles; i++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int m = 0; m < kOut; m++) {
                    const f32x4 w =
                        *reinterpret_cast<const f32x4 *>(sW3 + m * kHid + 32 * i + 8 * g + 4 * h);
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        o[m] = fmaf(w[q], fmaxf(h2[i][4 * g + q], 0.f), o[m]);
                }
#pragma unroll
        for (int m = 0; m < kOut; m++) {
            o[m] += __shfl_xor(o[m], 32, 64);
            if (h == 0 && p < B) Y[p * kOut + m] = o[m] + b3[m];
        }
    }
}

// Where column k (or point k) of a row in LDS lies: the four k = 8g + 2q + h of
// a half side by side, so that one 16-byte read serves four steps of a
// contraction in ascending k.
__device__ __forceinline__ int step_order(int k) {
    return (k & ~7) + 4 * (k & 1) + ((k & 7) >> 1);
}

// Sums of v[0 .. 15] over the 32 lanes of each half, by halving: lane k of a
// half ends with value k / 2 in v[0].
template <int N = 8>
__device__ __forceinline__ void half_sums(float (&v)[16], int lane) {
    const bool up = lane & (2 * N);
#pragma unroll
    for (int k = 0; k < N; k++) {
        const float give = up ? v[k] : v[N + k];
        const float keep = up ? v[N + k] : v[k];
        v[k] = keep + __shfl_xor(give, 2 * N, 64);
    }
    if constexpr (N > 1) half_sums<N / 2>(v, lane);
    else v[0] += __shfl_xor(v[0], 1, 64);
}

__device__ __forceinline__ f32x16 zeros() {
    f32x16 z;
#pragma unroll
    for (int r = 0; r < 16; r++) z[r] = 0.f;
    return z;
}

// A training step's forward and backward pass, workgroup k on the samples
// [k pslice, (k + 1) pslice), 32 at a time, with all gradients accumulated in
// registers.  Wavefront w owns rows 32w .. 32w + 31 of every hidden layer; the
// activations and their gradients cross between wavefronts through LDS
// ([unit][point]), where they are also the operands of the weight gradients
// (contractions over the points).  Each workgroup leaves its gradient in
// part[workgroup][total] and its loss in loss_part; points past the end have a
// zero output gradient.  Bound by the latency of a workgroup's 230 MFMAs per
// wavefront and 32 points (6 us) and its barriers, then by the partial
// gradients (19 MB at 256 workgroups).
//
// Sums are in the general path's order: v_mfma_f32_32x32x2_f32 is two FMAs in
// ascending k (bit for bit, on 204,800 random sums), so a chain of them over
// k = 2s + h is the scalar chain, cut into that path's split-K slices (kslice
// and oslice over the units, pslice over the samples).  A hidden unit within
// rounding of zero then falls on the same side of its ReLU; in another order
// a few flip per step, and each moves the gradient by ~0.1 / B.
constexpr int kLdP = kCols + 4;  // row stride of [unit][point] in LDS, as kLdW
constexpr int kTrainGroups = 256;

__global__ __launch_bounds__(kThreads, 1) void k_jump_train(
    const float *__restrict__ P, const float *__restrict__ X, const float *__restrict__ T,
    long long B, float inv_b, int kslice, int oslice, int pslice, float *__restrict__ part,
    double *__restrict__ loss_part) {
    __shared__ __align__(16) float sW2[kHid * kLdW], sH1[kHid * kLdP], sH2[kHid * kLdP],
        sZ2[kHid * kLdP], sX[(kIn + 2) * kLdP], sD[(kOut + 1) * kLdP], sb1[kHid], sb2[kHid],
        sW3[kOut * kHid];
    __shared__ float sO[kHid / kKT][kOut][kCols];
    constexpr Dims D{kIn, kHid, kOut};
#pragma unroll 16
    for (int e = threadIdx.x; e < kHid * kHid; e += kThreads)
        sW2[(e / kHid) * kLdW + step_order(e % kHid)] = P[D.off_w2() + e];
    for (int e = threadIdx.x; e < kOut * kHid; e += kThreads) sW3[e] = P[D.off_w3() + e];
    for (int e = threadIdx.x; e < kHid; e += kThreads) {
        sb1[e] = P[D.off_b1() + e];
        sb2[e] = P[D.off_b2() + e];
    }
    // rows 0-11 of sX hold the inputs, row 12 ones (the bias gradient of layer
    // 1), row 13 zeros; rows 0-2 of sD the output gradient, row 3 zeros
    for (int e = threadIdx.x; e < 2 * kLdP; e += kThreads)
        sX[kIn * kLdP + e] = e < kLdP ? 1.f : 0.f;
    for (int e = threadIdx.x; e < kLdP; e += kThreads) sD[kOut * kLdP + e] = 0.f;
    const int lane = __lane_id(), col = lane & 31, h = lane >> 5, w = threadIdx.x / 64;
    const int row = 32 * w + col;  // the lane's row of an A operand of this wavefront
    const int row_at = step_order(row), col_at = step_order(col);
    auto unit = [&](int r) { return 32 * w + 8 * (r / 4) + 4 * h + r % 4; };  // of register r
    float w1[kIn / 2], b3[kOut], gb2[16] = {}, gb3[kOut] = {};
#pragma unroll
    for (int s = 0; s < kIn / 2; s++) w1[s] = P[(long long)row * kIn + 2 * s + h];
#pragma unroll
    for (int m = 0; m < kOut; m++) b3[m] = P[D.off_b3() + m];
    f32x16 gW2[kTiles], gW1 = zeros(), gW3 = zeros();
#pragma unroll
    for (int k = 0; k < kTiles; k++) gW2[k] = zeros();
    double loss = 0.0;
    const long long p_end = min(B, (blockIdx.x + 1LL) * pslice);
    for (long long p0 = blockIdx.x * (long long)pslice; p0 < p_end; p0 += kCols) {
        __syncthreads();  // the last points' readers are done
        for (int e = threadIdx.x; e < kIn * kCols; e += kThreads) {
            const long long at = p0 * kIn + e;
            sX[(e % kIn) * kLdP + step_order(e / kIn)] = at < p_end * kIn ? X[at] : 0.f;
        }
        __syncthreads();
        // H1 = relu(W1 X + b1)
        f32x16 h1 = zeros(), bias = row_vector(sb1 + 32 * w, h);
#pragma unroll
        for (int s = 0; s < kIn / 2; s++) h1 = mfma(w1[s], sX[(2 * s + h) * kLdP + col_at], h1);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            h1[r] = fmaxf(h1[r] + bias[r], 0.f);
            sH1[unit(r) * kLdP + col_at] = h1[r];
        }
        __syncthreads();
        // H2 = relu(W2 H1 + b2)
        f32x16 h2 = zeros(), acc = zeros();
        bias = row_vector(sb2 + 32 * w, h);
#pragma unroll
        for (int g = 0; g < kHid / 8; g++) {
            const f32x4 a = *reinterpret_cast<const f32x4 *>(sW2 + row * kLdW + 8 * g + 4 * h);
#pragma unroll
            for (int q = 0; q < 4; q++)
                acc = mfma(a[q], sH1[(8 * g + 2 * q + h) * kLdP + col_at], acc);
            if (g % 2 == 1 && ((8 * g + 8) % kslice == 0 || 8 * g + 8 == kHid)) {
                h2 += acc;
                acc = zeros();
            }
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            h2[r] = fmaxf(h2[r] + bias[r], 0.f);
            sH2[unit(r) * kLdP + col_at] = h2[r];
        }
        __syncthreads();
        // the outputs: a slice of the units per wavefront, then the slices in order
        for (int s = w; s * oslice < kHid; s += kTiles) {
            float o[kOut] = {};
#pragma unroll 16
            for (int k = s * oslice; k < min(kHid, (s + 1) * oslice); k++) {
                const float v = sH2[k * kLdP + col_at];
#pragma unroll
                for (int m = 0; m < kOut; m++) o[m] = fmaf(v, sW3[m * kHid + k], o[m]);
            }
#pragma unroll
            for (int m = 0; m < kOut; m++)
                if (h == 0) sO[s][m][col] = o[m];
        }
        __syncthreads();
        const long long p = p0 + col;
        float dO[kOut];
#pragma unroll
        for (int m = 0; m < kOut; m++) {
            float v = 0.f;
            for (int s = 0; s * oslice < kHid; s++) v += sO[s][m][col];
            v += b3[m];
            const float r = p < p_end ? v - T[p * kOut + m] : 0.f;
            dO[m] = 2.f * r * inv_b;
            loss += (double)r * (double)r;
            gb3[m] += dO[m];
            if (w == 0 && h == 0) sD[m * kLdP + col_at] = dO[m];
        }
        // dZ2 = (W3^T dO) where H2 > 0
        f32x16 w3[kOut];
#pragma unroll
        for (int m = 0; m < kOut; m++) w3[m] = row_vector(sW3 + m * kHid + 32 * w, h);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            float z = w3[0][r] * dO[0];
#pragma unroll
            for (int m = 1; m < kOut; m++) z = fmaf(w3[m][r], dO[m], z);
            z = h2[r] > 0.f ? z : 0.f;
            gb2[r] += z;
            sZ2[unit(r) * kLdP + col_at] = z;
        }
        __syncthreads();
        // gradients of W2 (this wavefront's rows of dZ2 times every row of H1)
        // and W3 (transposed: its rows of H2 times dO)
#pragma unroll
        for (int g = 0; g < kCols / 8; g++) {
            const int at = 8 * g + 4 * h;
            const f32x4 a = *reinterpret_cast<const f32x4 *>(sZ2 + row * kLdP + at);
            const f32x4 a3 = *reinterpret_cast<const f32x4 *>(sH2 + row * kLdP + at);
            const f32x4 d = *reinterpret_cast<const f32x4 *>(sD + min(col, kOut) * kLdP + at);
            f32x4 b[kTiles];
#pragma unroll
            for (int k = 0; k < kTiles; k++)
                b[k] = *reinterpret_cast<const f32x4 *>(sH1 + (32 * k + col) * kLdP + at);
#pragma unroll
            for (int q = 0; q < 4; q++) {
#pragma unroll
                for (int k = 0; k < kTiles; k++) gW2[k] = mfma(a[q], b[k][q], gW2[k]);
                gW3 = mfma(a3[q], d[q], gW3);
            }
        }
        // dZ1 = (W2^T dZ2) where H1 > 0
        f32x16 z1 = zeros();
        acc = zeros();
#pragma unroll
        for (int s = 0; s < kHid / 2; s++) {
            acc = mfma(sW2[(2 * s + h) * kLdW + row_at], sZ2[(2 * s + h) * kLdP + col_at], acc);
            if (s % 8 == 7 && ((2 * s + 2) % kslice == 0 || 2 * s + 2 == kHid)) {
                z1 += acc;
                acc = zeros();
            }
        }
        __syncthreads();  // every wavefront has read H1: its place takes dZ1
#pragma unroll
        for (int r = 0; r < 16; r++) sH1[unit(r) * kLdP + col_at] = h1[r] > 0.f ? z1[r] : 0.f;
        __syncthreads();
        // gradients of W1 and (column 12) b1
#pragma unroll
        for (int g = 0; g < kCols / 8; g++) {
            const int at = 8 * g + 4 * h;
            const f32x4 a = *reinterpret_cast<const f32x4 *>(sH1 + row * kLdP + at);
            const f32x4 b = *reinterpret_cast<const f32x4 *>(sX + min(col, kIn + 1) * kLdP + at);
#pragma unroll
            for (int q = 0; q < 4; q++) gW1 = mfma(a[q], b[q], gW1);
        }
    }
    float *G = part + (long long)blockIdx.x * D.total();
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int i = unit(r);
#pragma unroll
        for (int k = 0; k < kTiles; k++) G[D.off_w2() + i * kHid + 32 * k + col] = gW2[k][r];
        if (col < kIn) G[i * kIn + col] = gW1[r];
        if (col == kIn) G[D.off_b1() + i] = gW1[r];
        if (col < kOut) G[D.off_w3() + col * kHid + i] = gW3[r];
    }
    half_sums(gb2, lane);
    if (col % 2 == 0) G[D.off_b2() + unit(col / 2)] = gb2[0];
    if (w == 0) {  // every wavefront, and both its halves, hold the same points
#pragma unroll
        for (int s = 16; s > 0; s >>= 1) {
            loss += __shfl_xor(loss, s, 64);
#pragma unroll
            for (int m = 0; m < kOut; m++) gb3[m] += __shfl_xor(gb3[m], s, 64);
        }
        if (lane == 0) {
            loss_part[blockIdx.x] = loss;
#pragma unroll
            for (int m = 0; m < kOut; m++) G[D.off_b3() + m] = gb3[m];
        }
    }
}

// One element of an Adam step (Kingma & Ba 2015).
struct AdamStep {
    float lr, b1, b2, eps, c1, c2;  // lr <= 0: no step
    __device__ __forceinline__ void apply(float *P, float *Mo, float *Ve, long long e,
                                          float g) const {
        const float m = b1 * Mo[e] + (1.f - b1) * g;
        const float v = b2 * Ve[e] + (1.f - b2) * g * g;
        Mo[e] = m;
        Ve[e] = v;
        P[e] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
    }
};

// The workgroups' gradients added in order, the Adam step on them, and the
// loss.  64 parameters per workgroup (291 for the jump network, so that the
// whole chip reads the partials' 19 MB): its four wavefronts bring the
// partials to LDS, the first adds them one after another.
__global__ __launch_bounds__(kThreads) void k_train_finish(
    const float *__restrict__ part, int nparts, float *__restrict__ G, AdamStep adam,
    float *__restrict__ P, float *__restrict__ Mo, float *__restrict__ Ve,
    const double *__restrict__ loss_part, double inv_b, double *__restrict__ loss) {
    __shared__ float s[kTrainGroups][64];
    constexpr Dims D{kIn, kHid, kOut};
    constexpr long long bias1 = D.off_b1(), bias2 = D.off_b2(), bias3 = D.off_b3();
    const long long count = D.total();
    const int lane = threadIdx.x % 64, q = threadIdx.x / 64;
    const long long e = blockIdx.x * 64LL + lane;
    if (e < count) {
#pragma unroll 16
        for (int k = q; k < nparts; k += kThreads / 64) s[k][lane] = part[k * count + e];
    }
    __syncthreads();
    if (q == 0 && e < count) {
        float g = 0.f;
        if ((e >= bias1 && e < bias1 + kHid) || (e >= bias2 && e < bias2 + kHid) || e >= bias3) {
            // in 64 bits, for the general path adds these by a tree
            double t = 0.0;
            for (int k = 0; k < nparts; k++) t += (double)s[k][lane];
            g = (float)t;
        } else {
#pragma unroll 16
            for (int k = 0; k < nparts; k++) g += s[k][lane];
        }
        G[e] = g;
        if (adam.lr > 0.f) adam.apply(P, Mo, Ve, e, g);
    }
    if (blockIdx.x == 0 && q == 1) {
        double t = 0.0;
        for (int k = lane; k < nparts; k += 64) t += loss_part[k];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        if (lane == 0) *loss = t * inv_b;
    }
}

// Adam on the flat parameter array.
__global__ void k_adam(float *__restrict__ P, const float *__restrict__ G, float *__restrict__ Mo,
                       float *__restrict__ Ve, long long count, AdamStep adam) {
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < count;
         e += (long long)gridDim.x * blockDim.x)
        adam.apply(P, Mo, Ve, e, G[e]);
}

inline int blocks_for(long long n, int cap = 4096) {
    return (int)std::max(1LL, std::min((long long)cap, (n + kThreads - 1) / kThreads));
}

// Length of the K slices of an M x N x K product (a multiple of kKT).
int split_k(int M, int N, int K, long long part_cap) {
    const int tiles = ((M + kT - 1) / kT) * ((N + kT - 1) / kT);
    int S = std::max(1, std::min(256, 1024 / std::max(tiles, 1)));
    S = std::min<long long>(S, std::max<long long>(1, part_cap / ((long long)M * N)));
    S = std::min(S, std::max(1, (K + kKT - 1) / kKT));
    const int kslice = (K + S - 1) / S;
    return (kslice + kKT - 1) / kKT * kKT;
}

// C[M x N] (ldc) = A B (+bias, act) via split-K partial tiles in `part`.
void gemm(const float *A, long long sam, long long sak, const float *B, long long sbk,
          long long sbn, float *C, long long ldc, int M, int N, int K, const float *bias, int act,
          float *part, long long part_cap, hipStream_t s) {
    const int kslice = split_k(M, N, K, part_cap);
    const int S = (K + kslice - 1) / kslice;
    // rows whose partial tiles fit `part` (all of them unless S is 1) and one grid
    const int rows = (int)std::max<long long>(1, std::min<long long>(part_cap / N, 65535LL * kT) / kT) * kT;
    for (int m0 = 0; m0 < M; m0 += rows) {
        const int m = std::min(rows, M - m0);
        dim3 grid((N + kT - 1) / kT, (m + kT - 1) / kT, S);
        k_gemm_part<<<grid, kThreads, 0, s>>>(A + m0 * sam, sam, sak, B, sbk, sbn, part, m, N, K,
                                              kslice);
        k_gemm_reduce<<<blocks_for((long long)m * N), kThreads, 0, s>>>(part, S, m, N, bias, act,
                                                                        C + m0 * ldc, ldc);
    }
}

// The loss to the host (which waits for it) if asked for; launch errors.
int loss_and_status(const double *d_loss, double *loss_out, hipStream_t s) {
    if (loss_out) {
        if (hipMemcpyAsync(loss_out, d_loss, sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess)
            return EGG_SYNC_E_HIP;
        if (hipStreamSynchronize(s) != hipSuccess) return EGG_SYNC_E_HIP;
    }
    return hipGetLastError() == hipSuccess ? EGG_SYNC_OK : EGG_SYNC_E_HIP;
}

}  // namespace mlp
}  // namespace egg

using namespace egg::mlp;

extern "C" {

int egg_mlp_param_count(int32_t in, int32_t hidden, int32_t out, int64_t *count) {
    if (in < 1 || hidden < 1 || out < 1 || !count) return EGG_SYNC_E_ARG;
    *count = Dims{in, hidden, out}.total();
    return EGG_SYNC_OK;
}

size_t egg_mlp_workspace_floats(int32_t in, int32_t hidden, int32_t out, int64_t batch) {
    const long long B = batch, h = hidden;
    // Z1/H1, Z2/H2 (B x h each, ReLU outputs kept), O, dO, dH2, dH1, split-K parts
    return (size_t)(2 * B * h + 2 * B * out + 2 * B * h + 1024LL * 64 * 64 + 4096);
}

int egg_mlp_forward_device(const float *d_params, int32_t in, int32_t hidden, int32_t out,
                           const float *d_X, int64_t batch, float *d_Y, void *stream) {
    if (!d_params || !d_X || !d_Y || batch < 0) return EGG_SYNC_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    if (batch == 0) return EGG_SYNC_OK;
    if (in == kIn && hidden == kHid && out == kOut) {
        // two workgroups fit a CU's LDS; each wavefront takes 32 points at a time
        const long long wgs = (batch + 4 * kCols - 1) / (4 * kCols);
        k_jump_infer<<<(int)std::min(512LL, wgs), kThreads, 0, s>>>(d_params, d_X, batch, d_Y);
    } else {
        return EGG_SYNC_E_ARG;
    }
    return hipGetLastError() == hipSuccess ? EGG_SYNC_OK : EGG_SYNC_E_HIP;
}

// One training step on a batch: loss, gradients (optional copy to d_grad) and,
// if lr > 0, an Adam update with step number `step` (1-based).
int egg_mlp_train_step_device(float *d_params, float *d_adam_m, float *d_adam_v, int32_t in,
                              int32_t hidden, int32_t out, const float *d_X, const float *d_T,
                              int64_t batch, float lr, int32_t step, float *d_work,
                              int64_t work_floats, float *d_grad, double *loss_out,
                              void *stream) {
    if (!d_params || !d_X || !d_T || !d_work || !d_grad || batch < 1) return EGG_SYNC_E_ARG;
    const long long B = batch, h = hidden;
    if ((size_t)work_floats < egg_mlp_workspace_floats(in, hidden, out, batch)) return EGG_SYNC_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const Dims D{in, hidden, out};
    float *H1 = d_work, *H2 = H1 + B * h, *O = H2 + B * h, *dO = O + B * out, *dH2 = dO + B * out,
          *dH1 = dH2 + B * h, *part = dH1 + B * h;
    const long long part_cap = 1024LL * 64 * 64;
    float *G = d_grad;
    const float be1 = 0.9f, be2 = 0.999f;
    AdamStep adam{lr, be1, be2, 1e-8f, 1.f, 1.f};
    if (lr > 0.f) {
        if (!d_adam_m || !d_adam_v || step < 1) return EGG_SYNC_E_ARG;
        adam.c1 = 1.f - powf(be1, (float)step);
        adam.c2 = 1.f - powf(be2, (float)step);
    }
    if (in == kIn && hidden == kHid && out == kOut) {
        // the jump network: forward, backward and weight gradients in one
        // kernel, then one that sums, steps and closes the loss.  8,192
        // samples: 418 us a step as the general path's 24 launches, 64 us as
        // these two (29 and 9 us, the rest is the caller's copies and wait).
        const int pslice = split_k(kHid, kHid, (int)B, part_cap);  // <= 256 slices
        const int wgs = (int)((B + pslice - 1) / pslice);
        double *lp = (double *)(((uintptr_t)d_work + 7) & ~(uintptr_t)7);
        float *grads = (float *)(lp + kTrainGroups + 1);
        k_jump_train<<<wgs, kThreads, 0, s>>>(d_params, d_X, d_T, B, 1.f / (float)B,
                                              split_k((int)B, kHid, kHid, part_cap),
                                              split_k((int)B, kOut, kHid, part_cap), pslice,
                                              grads, lp);
        k_train_finish<<<(int)((D.total() + 63) / 64), kThreads, 0, s>>>(
            grads, wgs, G, adam, d_params, d_adam_m, d_adam_v, lp, 1.0 / (double)B,
            lp + kTrainGroups);
        return loss_and_status(lp + kTrainGroups, loss_out, s);
    }
    double *loss_part = (double *)(part + part_cap);  // 1024 doubles fit in the 4096-float tail
    const float *W1 = d_params, *b1 = W1 + D.off_b1(), *W2 = W1 + D.off_w2(), *b2 = W1 + D.off_b2(),
                *W3 = W1 + D.off_w3(), *b3 = W1 + D.off_b3();
    // forward: H1 = relu(X W1^T + b1), H2 = relu(H1 W2^T + b2), O = H2 W3^T + b3
    gemm(d_X, in, 1, W1, 1, in, H1, h, (int)B, hidden, in, b1, 1, part, part_cap, s);
    gemm(H1, h, 1, W2, 1, h, H2, h, (int)B, hidden, hidden, b2, 1, part, part_cap, s);
    gemm(H2, h, 1, W3, 1, h, O, out, (int)B, out, hidden, b3, 0, part, part_cap, s);
    // loss and dO
    const int lb = 256;
    k_mse_grad<<<lb, kThreads, 0, s>>>(O, d_T, B * out, 1.f / (float)B, dO, loss_part);
    double *d_loss = loss_part + lb;
    k_loss_finish<<<1, 1, 0, s>>>(loss_part, lb, 1.0 / (double)B, d_loss);
    // backward
    float *gW1 = G, *gb1 = G + D.off_b1(), *gW2 = G + D.off_w2(), *gb2 = G + D.off_b2(),
          *gW3 = G + D.off_w3(), *gb3 = G + D.off_b3();
    gemm(dO, 1, out, H2, h, 1, gW3, h, out, hidden, (int)B, nullptr, 0, part, part_cap, s);  // dO^T H2
    k_colsum<<<out, kThreads, 0, s>>>(dO, (int)B, out, gb3);
    gemm(dO, out, 1, W3, h, 1, dH2, h, (int)B, hidden, out, nullptr, 0, part, part_cap, s);  // dO W3
    k_relu_mask<<<blocks_for(B * h), kThreads, 0, s>>>(dH2, H2, B * h);
    gemm(dH2, 1, h, H1, h, 1, gW2, h, hidden, hidden, (int)B, nullptr, 0, part, part_cap, s);
    k_colsum<<<hidden, kThreads, 0, s>>>(dH2, (int)B, hidden, gb2);
    gemm(dH2, h, 1, W2, h, 1, dH1, h, (int)B, hidden, hidden, nullptr, 0, part, part_cap, s);  // dH2 W2
    k_relu_mask<<<blocks_for(B * h), kThreads, 0, s>>>(dH1, H1, B * h);
    gemm(dH1, 1, h, d_X, in, 1, gW1, in, hidden, in, (int)B, nullptr, 0, part, part_cap, s);
    k_colsum<<<hidden, kThreads, 0, s>>>(dH1, (int)B, hidden, gb1);
    if (lr > 0.f)
        k_adam<<<blocks_for(D.total()), kThreads, 0, s>>>(d_params, G, d_adam_m, d_adam_v, D.total(),
                                                          adam);
    return loss_and_status(d_loss, loss_out, s);
}

// x <- clamp(x + scale * y, 0, 1) for n x d row-major positions.
__global__ void k_jump(float *__restrict__ X, const float *__restrict__ Y, long long count,
                       float scale, float clip) {
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < count;
         e += (long long)gridDim.x * blockDim.x) {
        float y = Y[e];
        if (clip > 0.f) y = fminf(fmaxf(y, -clip), clip);
        X[e] = fminf(fmaxf(X[e] + scale * y, 0.f), 1.f);
    }
}

int egg_sync_jump_device(float *d_X, const float *d_Y, int64_t n, int32_t d, float scale,
                         float clip, void *stream) {
    if ((!d_X || !d_Y) && n > 0) return EGG_SYNC_E_ARG;
    if (n == 0) return EGG_SYNC_OK;
    k_jump<<<blocks_for(n * d), kThreads, 0, (hipStream_t)stream>>>(d_X, d_Y, n * (long long)d,
                                                                     scale, clip);
    return hipGetLastError() == hipSuccess ? EGG_SYNC_OK : EGG_SYNC_E_HIP;
}

}  // extern "C"
