// Workgroup-wide descending sort of u64 keys in LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bvk {
namespace {

// Descending bitonic sort of keys[0, npow) (npow a power of two), NT threads.
// Every thread calls it, after a barrier; it ends with one.
// Up to NT keys: one per thread, in registers; stages within a wave (all but
// 3 of the 36 of 256 keys) exchange by shuffles, the others through LDS.
// Bound by the latency of a stage: 256 keys 5.2 us, against 7.1 with every
// stage's pairs read from and written to LDS.
// More keys: thread t takes pair t of a stage, so a wave's pairs of a stage of
// distance 64 or less lie in its own 128 keys and need no workgroup barrier.
template <uint32_t NT> __device__ void sort_desc_lds(uint64_t *keys, uint32_t npow) {
    const uint32_t tid = threadIdx.x;
    if (npow <= NT) {
        const uint32_t w0 = tid & ~63u;  // the wave's first key
        uint64_t x = tid < npow ? keys[tid] : 0ull;
        for (uint32_t k = 2; k <= npow; k <<= 1) {
            for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                uint64_t y = 0;
                if (j >= 64) {
                    __syncthreads();
                    if (w0 < npow) keys[tid] = x;
                    __syncthreads();
                    if (w0 < npow) y = keys[tid ^ j];
                } else if (w0 < npow) {
                    y = __shfl_xor((unsigned long long)x, (int)j);
                }
                // the lower of a pair takes the larger key where the run descends
                if ((x < y) == (((tid & j) == 0) == ((tid & k) == 0))) x = y;
            }
        }
        __syncthreads();
        if (tid < npow) keys[tid] = x;
        __syncthreads();
        return;
    }
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
}

}  // namespace
}  // namespace bvk
