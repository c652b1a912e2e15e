// Exact scores of sixteen rows per wave (Store.dotRow and, L2, Store.l2Row,
// src/store/store.ts:114-160) with coalesced row reads.
//
// Lane 4c + m runs accumulator m of candidate c over elements 4j + m in order,
// in f64 (dot: each product is exact, so fma adds it with the reference's one
// rounding; l2: the difference, its square and the sum each rounded).  Read straight from memory each lane
// would take one element in four (16 rows x 16 bytes per load instruction,
// 192 instructions at 768 dimensions: the address unit, shared by a
// workgroup's waves, bounds it); here a row's 64-element chunks come in as
// 16-byte pieces, 256 bytes of a row per 16 lanes, and go through a
// wave-private LDS tile that turns them to the accumulators' order.
#pragma once

#include "bv_device.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bvk {
namespace {

constexpr uint32_t EXACT_RS = 80;             // tile row stride in floats: 4 x 16 and 16 to spread the banks
constexpr uint32_t EXACT_TILE = 16 * EXACT_RS;  // floats of LDS per wave

constexpr uint32_t EXACT_D = 3;               // 64-element chunks in flight

// floats per accumulator of the transposed query: dim / 4 rounded up to whole
// rounds of chunks, zero-padded
__host__ __device__ inline uint32_t exact_q_stride(uint32_t dim) {
    return ((dim >> 2) + 16u * EXACT_D - 1) / (16u * EXACT_D) * (16u * EXACT_D);
}

// The query q[0, dim) as qt[m * exact_q_stride(dim) + j] = q[4j + m] (zeros
// past the last whole group), by nt threads.
__device__ __forceinline__ void exact_load_query(const float *q, uint32_t dim, float *qt, uint32_t tid, uint32_t nt) {
    const uint32_t nv = dim >> 2, st = exact_q_stride(dim);
    for (uint32_t i = tid; i < 4 * st; i += nt) {
        const uint32_t e = (i & 3u) * st + (i >> 2);  // element i = 4j + m
        qt[e] = (i >> 2) < nv ? q[i] : 0.0f;
    }
}

struct __attribute__((packed, aligned(4))) f32x4_u {
    float x, y, z, w;
};

// The (score, row) key of candidate lane >> 2 in lanes 4c; every lane of the
// wave calls it with its candidate's row (absent candidates: any valid row).
// tile: the wave's EXACT_TILE floats.  Padded elements are 0 on both sides:
// the sums are unchanged.
template <bool L2> __device__ __forceinline__ double exact_add(double acc, float x, float q) {
    if constexpr (L2) {
#pragma clang fp contract(off)
        const double d = (double)x - (double)q;
        return acc + d * d;
    } else {
        return fma((double)x, (double)q, acc);
    }
}
template <bool L2 = false>
__device__ __forceinline__ uint64_t exact_keys16(const float *rows, uint32_t dim, const float *q, const float *qt,
                                                 uint32_t row, float *tile, int lane) {
    const uint32_t vec = dim & ~3u, nch = (vec + 63) / 64, qst = exact_q_stride(dim);
    const int piece = lane & 15, m = lane & 3, c = lane >> 2;
    const float *src[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // candidate (lane >> 4) + 4i
        const uint32_t r = (uint32_t)__shfl((int)row, 4 * ((lane >> 4) + 4 * i));
        src[i] = rows + (uint64_t)r * dim + 4 * piece;
    }
    constexpr int D = (int)EXACT_D;
    f32x4_u buf[D][4];
    // (clamped to the row's first piece past its end; what comes from there is
    // zeroed when it goes to the tile, so that nothing waits for a load here)
    auto load = [&](uint32_t ch, f32x4_u (&b)[4]) {
        const int64_t off = ch * 64 + 4 * (uint32_t)piece < vec ? (int64_t)ch * 64 : -(int64_t)(4 * piece);
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = *(const f32x4_u *)(src[i] + off);
    };
    double acc = 0.0;
    const float *x = rows + (uint64_t)row * dim;
    if (vec) {
#pragma unroll
        for (int d = 0; d < D; ++d) load(d, buf[d]);
        // (whole rounds of D chunks, zeros past the row's end: an early way out
        // would make every chunk wait for all loads in flight)
        for (uint32_t c0 = 0; c0 < nch; c0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                float *w = tile + (lane >> 4) * EXACT_RS + piece;
                const bool ok = (c0 + d) * 64 + 4 * (uint32_t)piece < vec;
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float *wi = w + 4 * i * EXACT_RS;
                    wi[0] = ok ? buf[d][i].x : 0.0f;
                    wi[16] = ok ? buf[d][i].y : 0.0f;
                    wi[32] = ok ? buf[d][i].z : 0.0f;
                    wi[48] = ok ? buf[d][i].w : 0.0f;
                }
                load(c0 + d + D, buf[d]);
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                const float4 *xr = (const float4 *)(tile + c * EXACT_RS + 16 * m);
                const float4 *qr = (const float4 *)(qt + m * qst + 16 * (c0 + d));
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float4 a = xr[t], b = qr[t];
                    acc = exact_add<L2>(acc, a.x, b.x);
                    acc = exact_add<L2>(acc, a.y, b.y);
                    acc = exact_add<L2>(acc, a.z, b.z);
                    acc = exact_add<L2>(acc, a.w, b.w);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
    }
    const double a1 = __shfl_down(acc, 1), a2 = __shfl_down(acc, 2), a3 = __shfl_down(acc, 3);
    double sum = acc + a1;
    sum = sum + a2;
    sum = sum + a3;
    if (m == 0)
        for (uint32_t i = vec; i < dim; ++i) sum = exact_add<L2>(sum, x[i], q[i]);
    return make_key(ord_f32(L2 ? (float)(-sum) : (float)sum), row);
}

}  // namespace
}  // namespace bvk
