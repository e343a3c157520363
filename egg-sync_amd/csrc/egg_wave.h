// Wavefront helpers of the update kernels (gfx950).
#pragma once

#include "egg_common.h"

namespace egg {

// Makes the LDS writes of every lane visible to the reads of the others
// (wavefront scope; the LDS serves one wavefront's accesses in order).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int next_tile(int *counter) {
    int t = 0;
    if (__lane_id() == 0) t = atomicAdd(counter, 1);
    return __builtin_amdgcn_readfirstlane(t);
}

// Work claims of the queue kernels: wavefront w of the grid's W takes item w
// first, without an atomic, and later items from the counter, offset by W.
// A pass with fewer items than wavefronts (converged iterations) takes no
// atomic at all; with more, each wavefront takes one per extra item.
__device__ __forceinline__ int wave_index() {
    return __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave);
}

__device__ __forceinline__ int wave_count() { return gridDim.x * (blockDim.x / kWave); }

// Workgroups of the queue kernels: enough to fill the chip; they drain the tile
// queue and exit.
constexpr int kQueueBlocks = 2048;

}  // namespace egg
