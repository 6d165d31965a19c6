// Device helpers for the records that a sweep leaves in its hit chunks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gss {

__device__ __forceinline__ uint64_t wave_incl_scan(uint64_t x, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    return x;
}

// Ends of 64 chunks' records (exclusive sums from the first one's start), from
// a lane's chunk of `fill` records; the first wave writes them.
__device__ __forceinline__ void fill_ends(uint32_t fill, uint32_t *ends) {
    if (threadIdx.x < 64) ends[threadIdx.x] = (uint32_t)wave_incl_scan(fill, (int)threadIdx.x);
}

// The chunk that record i of the 64 is in: the first that ends after it.
__device__ __forceinline__ uint32_t chunk_of(const uint32_t *ends, uint32_t i) {
    uint32_t k = 0;
#pragma unroll
    for (uint32_t d = 32; d > 0; d >>= 1)
        if (ends[k + d - 1] <= i) k += d;
    return k;
}

}  // namespace gss
