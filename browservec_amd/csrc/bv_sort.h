// Workgroup-wide descending sort of u64 keys in LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bvk {
namespace {

// Descending bitonic sort of keys[0, npow) (npow a power of two), NT threads.
// Thread t takes pair t of a stage, so a wave's pairs of a stage of distance
// 64 or less lie in its own 128 keys: those stages need no workgroup barrier
// (a 1024-thread barrier per stage took 3.4 us to sort 128 keys).  Every
// thread calls it, after a barrier; it ends with one.
template <uint32_t NT> __device__ void sort_desc_lds(uint64_t *keys, uint32_t npow) {
    const uint32_t tid = threadIdx.x;
    for (uint32_t k = 2; k <= npow; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t i = tid; i < npow / 2; i += NT) {
                const uint32_t lo = ((i & ~(j - 1)) << 1) | (i & (j - 1)), hi = lo | j;
                const uint64_t x = keys[lo], y = keys[hi];
                if (((lo & k) == 0) == (x < y)) {
                    keys[lo] = y;
                    keys[hi] = x;
                }
            }
            // the next stage's pairs cross waves, or this one's did
            if (j > 64 || (j == 1 && k > 64)) {
                __syncthreads();
            } else {
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
    }
    if (npow <= 64) __syncthreads();  // (otherwise the last stage ended with one)
}

}  // namespace
}  // namespace bvk
