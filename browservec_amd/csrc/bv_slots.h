// The two-kernel search of short scans and small query batches: scan_slots
// scores every row for up to NQ queries per pass over the rows, pick_topk (bv_pick.hip) finds each query's best from what it left.
//
// scan_slots cuts the rows into slots of a.rw rows, one wave per slot, and
// writes every row's order word (the key's high word) and each slot's best
// key and the largest order word of each of its a.nsub parts.  The kk-th best
// of the slots' best keys bounds the kk-th best key from below, and only
// slots whose best key reaches it can hold one of the kk best, so the
// selection reads the slots' best keys, then the parts of about kk slots,
// then the rows of about kk parts.
//
// Against the fused scan_topk: no shared bound has to form while the scan
// runs, so a scan too short for it (a few steps per wave) or a fetch large
// next to it costs no more than its bytes, and the rows are read once for up
// to four queries.  The scan's launch holds no waiting workgroup and keeps no
// order between its own.
//
// Bound by HBM for large row counts (one or two queries; the dot products'
// VALU work passes the row reads at about five int8 queries), by latency
// below about 50,000 rows.
#pragma once

#include "bv_scan.h"

namespace bvk {
namespace {

// Queries per pass: the query slices share the registers (96 values).
template <int C, int UPL> constexpr int slots_nq_max() {
    return UPL * Codec<C>::QN * 4 <= 96 ? 4 : UPL * Codec<C>::QN * 2 <= 96 ? 2 : 1;
}

// Scores a loaded step for one query: order words out, the lane's best key
// kept.  C_Q1P: the order word of an upper bound of the row's exact score,
// and the best key from a lower bound (the arithmetic of compute_step_q1p).
template <int C, int LPR, int UPL>
__device__ __forceinline__ void slots_step(const SlotArgs &a, const ScanRegs<C, UPL> &R, const StepData<C, LPR, UPL> &S,
                                           uint32_t base, uint32_t lim, uint32_t *ordq, uint64_t &best, uint32_t &top, int lane) {
    using CD = Codec<C>;
    using Acc = typename CD::Acc;
    using SH = ScanShape<C, LPR, UPL>;
    constexpr int U = SH::U, G = SH::G;
    Acc acc[CD::NA][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        Acc a1[CD::NA];
#pragma unroll
        for (int m = 0; m < CD::NA; ++m) a1[m] = (Acc)0;
#pragma unroll
        for (int t = 0; t < UPL; ++t) CD::acc(Neutral<C>::get(S.d[u][t], R.qr[t], R.uok[t]), R.qr[t], a1);
#pragma unroll
        for (int m = 0; m < CD::NA; ++m) acc[m][u] = a1[m];
    }
    Acc tot[CD::NA];
#pragma unroll
    for (int m = 0; m < CD::NA; ++m) tot[m] = xreduce<U, LPR>(acc[m], lane);
    const uint32_t myrow = base + (uint32_t)(xrow<U, LPR>(lane) * G + lane / LPR);
    if (!xrep<U, LPR>(lane) || myrow >= lim) return;
    uint32_t ord = 0, low = 0;
    const float scale = S.scale * a.scale_mul;
    if constexpr (C == C_Q1P) {
        const double lev = R.fin.s1 * (double)(2 * tot[0] - R.fin.sumq1) + R.fin.s2 * (double)(2 * tot[1] - R.fin.sumq2);
        const double slack = R.fin.rsum + 4e-5 * R.fin.qabs;
        double hi = (double)scale * (lev + slack), lo = (double)scale * (lev - slack);
        hi += fabs(hi) * 1e-6;
        lo -= fabs(lo) * 1e-6;
        float hf = (float)hi, lf = (float)lo;
        if ((double)hf < hi) hf = -float_below(-hf);
        if ((double)lf > lo) lf = float_below(lf);
        ord = hf == hf ? ord_f32(hf) : 0xffffffffu;  // (NaN: kept, the exact key decides)
        low = lf == lf ? ord_f32(lf) : 0u;
    } else {
        (void)R.fin.score(tot, scale, ord);
        low = ord;
    }
    if (ord == 0) ord = 1;  // (0 marks a row the mask leaves out)
    if (a.mask && !(S.grow < a.mask_bits && ((a.mask[S.grow >> 5] >> (S.grow & 31)) & 1u))) ord = 0;
    ordq[myrow] = ord;
    if (ord == 0) return;
    const uint64_t key = make_key(low, S.grow);
    best = key > best ? key : best;
    top = ord > top ? ord : top;
}

template <int C, int LPR, int UPL, int NQ>
__global__ __launch_bounds__(SCAN_WG) void scan_slots(SlotArgs a) {
    using CD = Codec<C>;
    using QT = typename CD::QT;
    using SH = ScanShape<C, LPR, UPL>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t slot = blockIdx.x * SH::WAVES + (uint32_t)wave;
    if (slot >= a.nslots) return;
    const uint32_t q0 = blockIdx.y * NQ;
    const int p = lane % LPR;
    const uint32_t n = a.n;
    const uint32_t r0 = slot * a.rw;
    if (r0 >= n) {
#pragma unroll
        for (int k = 0; k < NQ; ++k)
            if (lane == 0 && q0 + k < a.nq) {
                a.best[(uint64_t)(q0 + k) * a.nslots + slot] = 0;  // (its parts are not read)
                if (C == C_Q1P) a.top[(uint64_t)(q0 + k) * a.nslots + slot] = 0;
            }
        return;
    }
    const uint32_t r1 = r0 + a.rw < n ? r0 + a.rw : n;
    ScanArgs la{};  // (what load_step reads)
    la.codes = a.codes;
    la.row_bytes = a.row_bytes;
    la.scales = a.scales;
    ScanRegs<C, UPL> R[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
        const uint32_t q = q0 + k < a.nq ? q0 + k : a.nq - 1;
        const QT *qb = (const QT *)((const char *)a.q + (uint64_t)q * a.q_stride);
#pragma unroll
        for (int t = 0; t < UPL; ++t) {
            const uint32_t unit = p + LPR * t;
            R[k].uok[t] = unit < a.units;
            R[k].ucl[t] = R[k].uok[t] ? unit : a.units - 1;
#pragma unroll
            for (int j = 0; j < CD::QN; ++j) {
                const QT v = qb[R[k].ucl[t] * CD::QN + j];
                R[k].qr[t][j] = R[k].uok[t] ? v : (QT)0;
            }
        }
        R[k].fin.load((const char *)qb + (uint64_t)a.units * CD::QN * sizeof(QT), a.padded_dim);
    }
    uint64_t best[NQ];
    uint32_t top[NQ], ptop[NQ];  // largest order word of the slot, of the part
    uint32_t *ordq[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
        best[k] = 0;
        top[k] = ptop[k] = 0;
        ordq[k] = a.ord + (uint64_t)(q0 + k < a.nq ? q0 + k : a.nq - 1) * a.nslots * a.rw;
    }
    const uint32_t pr = a.rw / a.nsub;  // rows per part
    uint32_t pend = r0 + pr, part = slot * a.nsub;
    // two steps' loads in flight: one is scored while the other lands (rows
    // past the slot's end load its last row and are dropped: a load under a
    // condition would make the wave wait for both)
    StepData<C, LPR, UPL> A, B;
    load_step<C, LPR, UPL, false>(la, R[0], nullptr, r0, r1, A, lane);
    for (uint32_t base = r0; base < r1; base += 2 * SH::RPS) {
        load_step<C, LPR, UPL, false>(la, R[0], nullptr, base + SH::RPS, r1, B, lane);
#pragma unroll
        for (int k = 0; k < NQ; ++k)
            slots_step<C, LPR, UPL>(a, R[k], A, base, r1, ordq[k], best[k], ptop[k], lane);
        load_step<C, LPR, UPL, false>(la, R[0], nullptr, base + 2 * SH::RPS, r1, A, lane);
        if (base + SH::RPS < r1) {
#pragma unroll
            for (int k = 0; k < NQ; ++k)
                slots_step<C, LPR, UPL>(a, R[k], B, base + SH::RPS, r1, ordq[k], best[k], ptop[k], lane);
        }
        if (base + 2 * SH::RPS >= pend || base + 2 * SH::RPS >= r1) {
#pragma unroll
            for (int k = 0; k < NQ; ++k) {
                const uint32_t m = wave_max_u32_dpp(ptop[k]);
                if (lane == 0 && q0 + k < a.nq) a.part[(uint64_t)(q0 + k) * a.nslots * a.nsub + part] = m;
                top[k] = m > top[k] ? m : top[k];
                ptop[k] = 0;
            }
            pend += pr;
            ++part;
        }
    }
    // parts wholly past the rows' end
    for (; part < (slot + 1) * a.nsub; ++part) {
#pragma unroll
        for (int k = 0; k < NQ; ++k)
            if (lane == 0 && q0 + k < a.nq) a.part[(uint64_t)(q0 + k) * a.nslots * a.nsub + part] = 0;
    }
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
        const uint64_t m = wave_max_u64(best[k]);
        if (lane == 0 && q0 + k < a.nq) {
            a.best[(uint64_t)(q0 + k) * a.nslots + slot] = m;
            if (C == C_Q1P) a.top[(uint64_t)(q0 + k) * a.nslots + slot] = top[k];
        }
    }
}

template <int C, int LPR, int UPL> hipError_t slots_go(const SlotArgs &a, hipStream_t s) {
    using SH = ScanShape<C, LPR, UPL>;
    // slots of whole steps, parts of whole step pairs; row positions in 32 bits
    if (a.rw == 0 || a.rw % SH::RPS || a.nsub == 0 || a.rw % a.nsub || (a.nsub > 1 && a.rw / a.nsub % (2 * SH::RPS)) ||
        a.cand || a.nslots == 0 || a.nq == 0 || a.nq > SLOTS_MAX_NQ ||
        (uint64_t)a.nslots * a.rw >= (1ull << 31) || (uint64_t)a.nslots * a.rw < a.n)
        return hipErrorInvalidValue;
    const uint32_t gx = (a.nslots + SH::WAVES - 1) / SH::WAVES;
    constexpr int MX = slots_nq_max<C, UPL>();
    if (MX == 1 || a.nq == 1) {
        hipLaunchKernelGGL((scan_slots<C, LPR, UPL, 1>), dim3(gx, a.nq), dim3(SCAN_WG), 0, s, a);
    } else if (MX == 2 || a.nq == 2) {
        hipLaunchKernelGGL((scan_slots<C, LPR, UPL, MX == 1 ? 1 : 2>), dim3(gx, (a.nq + 1) / 2), dim3(SCAN_WG),
                           0, s, a);
    } else {
        hipLaunchKernelGGL((scan_slots<C, LPR, UPL, MX>), dim3(gx, (a.nq + MX - 1) / MX), dim3(SCAN_WG), 0, s, a);
    }
    return hipGetLastError();
}

template <int C, int LPR, int UPL> hipError_t slots_fit(const SlotArgs &a, hipStream_t s) {
    if constexpr (UPL * Codec<C>::QN <= 64) return slots_go<C, LPR, UPL>(a, s);
    else return hipErrorInvalidValue;
}

template <int C> hipError_t slots_layout(const Layout &L, const SlotArgs &a, hipStream_t s) {
    if (L.lpr == 64) {
        switch (L.upl) {
        case 1: return slots_fit<C, 64, 1>(a, s);
        case 2: return slots_fit<C, 64, 2>(a, s);
        case 3: return slots_fit<C, 64, 3>(a, s);
        case 4: return slots_fit<C, 64, 4>(a, s);
        case 6: return slots_fit<C, 64, 6>(a, s);
        case 8: return slots_fit<C, 64, 8>(a, s);
        case 12: return slots_fit<C, 64, 12>(a, s);
        case 16: return slots_fit<C, 64, 16>(a, s);
        default: return hipErrorInvalidValue;
        }
    }
    switch (L.lpr) {
    case 4: return slots_go<C, 4, 1>(a, s);
    case 8: return slots_go<C, 8, 1>(a, s);
    case 16: return slots_go<C, 16, 1>(a, s);
    case 32: return slots_go<C, 32, 1>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace
}  // namespace bvk
