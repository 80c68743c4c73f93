// bh_block.h — workgroup scans and the workgroup order shared by the sorts.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bh {

// Exclusive scan of one value per thread over a block of THREADS threads
// (a multiple of 64); *total receives the block's sum.
template <int THREADS>
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_wave_tot, uint32_t* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave_tot[wave] = x;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < THREADS / 64; w++) {
        uint32_t t = s_wave_tot[w];
        if (w < wave) off += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return off + x - v;
}

// Partition of workgroup b of a grid of g: the dispatcher deals workgroups to
// the eight XCDs in turn, so XCD x runs b = x, x + 8, ...; giving those
// workgroups consecutive partitions keeps the two halves of a 128-byte line
// that neighbouring partitions write for one digit in the same L2, where they
// merge (with partitions dealt round robin, a 1080p tile sort's first pass
// wrote 114 MB for 80 MB of pairs).  Only locality depends on this order.
__device__ __forceinline__ uint32_t xcd_partition(uint32_t b, uint32_t g) {
    const uint32_t x = b & 7u, q = g >> 3, r = g & 7u;
    return x * q + min(x, r) + (b >> 3);
}

}  // namespace bh
