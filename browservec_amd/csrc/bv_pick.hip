// Selection of a scan_slots pass (bv_slots.h): each query's kk best keys,
// their exact re-rank, the best k_out.  One workgroup of 16 waves per query (or
// a.split, which select alike and share the re-rank).
//
//   1. The slots' best keys, in registers, give a bound: the low edge of the
//      histogram bin that holds the kk-th best (2048 bins over their range,
//      narrowed until the bin holds few others).  kk rows score at least that
//      much, so no row below it is among the kk best.
//   2. Of the slots whose best key reaches the bound (about kk) the parts that
//      reach it are read; their rows at or above it go to a list in LDS, at
//      most PICK_CAP; a list that would pass that is cut to its kk best, which
//      raises the bound.
//   3. The list is sorted and its kk best re-ranked (bv_exact.h).
//
// C_Q1P passes hold bounds instead of keys: the bound comes from the slots'
// best lower bounds and is raised to the kk-th best exact key of those rows
// (the fused scan's arithmetic); the rows whose upper bound reaches it get
// their exact keys before the list is sorted.
//
// Bound by latency: five dependent reads (best keys, slots, parts, rows, exact
// rows) of a few hundred KB, and the sorts and barriers between them: 11 us for
// 10 of 1M fp32 rows, 23 for 40 of 1M x 768 int8 rows, 34 for 200 of 4M x 1024
// Hamming rows and 60 for 200 1-bit ones, whose bounds leave 500 exact keys to
// form; all queries at once.
#include "bv_exact.h"
#include "bv_mfma.h"
#include "bv_scan.h"
#include "bv_sort.h"

namespace bvk {
namespace {

constexpr uint32_t PICK_THREADS = 1024;
constexpr uint32_t PICK_WAVES = PICK_THREADS / 64;
constexpr uint32_t PICK_CAP = 4096;                         // list entries
constexpr uint32_t PICK_BINS = 2048;
constexpr uint32_t PICK_REG = SLOTS_MAX / PICK_THREADS;     // best keys per thread
constexpr uint32_t PICK_ROUND = 8;                          // order words a thread reads at once

static_assert(PICK_BINS == 2 * PICK_THREADS, "two bins per thread");
struct PickLds {
    uint64_t keys[PICK_CAP];
    union {
        struct {
            uint32_t hist[PICK_BINS];
            uint16_t slots[SLOTS_MAX];
            uint32_t parts[PICK_CAP];
            uint32_t rows[PICK_CAP];                        // C_Q1P: the rows whose exact keys are due
        };
        float tiles[PICK_WAVES * EXACT_TILE];
    };
    uint64_t red[2][PICK_WAVES];
    uint32_t wsum[PICK_WAVES];
    uint32_t cnt, ns, np, sum, bin, excl, inbin;
};

__device__ __forceinline__ uint32_t pick_wave_sum(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan(x), 63);
}

// Lanes per row of the C_Q1P exact keys (0: another codec).
template <int LPR> __global__ __launch_bounds__(PICK_THREADS) void pick_topk(PickArgs a) {
    constexpr bool Q1P = LPR != 0;
    __shared__ PickLds L;
    extern __shared__ __align__(16) float pick_smem[];  // the transposed query, then the C_Q1P table
    const uint32_t q = blockIdx.x, tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t nslots = a.s.nslots, kk = a.kk;
    const uint32_t pr = a.s.rw / a.s.nsub, lg = 31 - __builtin_clz(pr), lgs = 31 - __builtin_clz(a.s.nsub);
    const uint64_t *best = a.s.best + (uint64_t)q * nslots;
    const uint32_t *ord = a.s.ord + (uint64_t)q * nslots * a.s.rw;
    const uint32_t *cand = a.s.cand;
    const uint32_t n = a.s.n;
    const float *rq = a.rr_src ? a.rr_q + (uint64_t)q * a.rr_q_stride : nullptr;

    uint64_t kr[PICK_REG];
#pragma unroll
    for (uint32_t j = 0; j < PICK_REG; ++j) {
        const uint32_t i = tid + j * PICK_THREADS;
        kr[j] = j * PICK_THREADS < nslots && i < nslots ? best[i] : 0ull;
    }
    // what the later steps need from memory, on its way meanwhile
    if (a.rr_src) exact_load_query(rq, a.rr_dim, pick_smem, tid, PICK_THREADS);
    float *lut = pick_smem + (a.rr_src ? 4 * exact_q_stride(a.rr_dim) : 0);
    if constexpr (Q1P)
        q1p_lut_build(a.qrot + (uint64_t)q * a.s.padded_dim, a.s.padded_dim, lut, tid, PICK_THREADS);

    // ---- the bound from the slots' best keys ----
    uint64_t th = 1;
    {
        uint64_t lo = ~0ull, hi = 0;
        uint32_t have = 0;
#pragma unroll
        for (uint32_t j = 0; j < PICK_REG; ++j) {
            if (kr[j]) {
                lo = kr[j] < lo ? kr[j] : lo;
                hi = kr[j] > hi ? kr[j] : hi;
                ++have;
            }
        }
        hi = wave_max_u64(hi);
        lo = ~wave_max_u64(~lo);
        have = pick_wave_sum(have);
        if (tid == 0) {
            L.cnt = 0;
            L.ns = 0;
            L.sum = 0;
        }
        __syncthreads();
        if (lane == 0) {
            L.red[0][wave] = lo;
            L.red[1][wave] = hi;
            atomicAdd(&L.sum, have);
        }
        __syncthreads();
        lo = L.red[0][0];
        hi = L.red[1][0];
        for (uint32_t w = 1; w < PICK_WAVES; ++w) {
            lo = L.red[0][w] < lo ? L.red[0][w] : lo;
            hi = L.red[1][w] > hi ? L.red[1][w] : hi;
        }
        if (L.sum > kk) {
            uint32_t above = 0;  // keys above [lo, hi]
            for (;;) {
                const uint64_t span = hi - lo;
                const int shift = (span >> 11) ? 64 - __clzll((long long)(span >> 11)) : 0;  // (span >> shift) < 2048
                for (uint32_t i = tid; i < PICK_BINS; i += PICK_THREADS) L.hist[i] = 0;
                __syncthreads();
#pragma unroll
                for (uint32_t j = 0; j < PICK_REG; ++j)
                    if (kr[j] && kr[j] >= lo && kr[j] <= hi) atomicAdd(&L.hist[(uint32_t)((kr[j] - lo) >> shift)], 1u);
                __syncthreads();
                // thread t: bins 2047 - 2t and 2046 - 2t, counted from the top
                const uint32_t h0 = L.hist[PICK_BINS - 1 - 2 * tid], h1 = L.hist[PICK_BINS - 2 - 2 * tid];
                const uint32_t inc = wave_incl_scan(h0 + h1);
                if (lane == 63) L.wsum[wave] = inc;
                __syncthreads();
                uint32_t run = inc - (h0 + h1);
                for (int w = 0; w < wave; ++w) run += L.wsum[w];
                if (above + run < kk && above + run + h0 + h1 >= kk) {
                    const bool first = above + run + h0 >= kk;
                    L.bin = PICK_BINS - 1 - 2 * tid - (first ? 0 : 1);
                    L.excl = first ? run : run + h0;
                    L.inbin = first ? h0 : h1;
                }
                __syncthreads();
                const uint32_t bin = L.bin, excl = L.excl, inbin = L.inbin;
                const uint64_t g = lo + ((uint64_t)bin << shift);
                th = g;
                if (shift == 0 || above + excl + inbin <= kk + kk / 4 + 16) break;
                const uint64_t w = (1ull << shift) - 1;
                hi = hi - g > w ? g + w : hi;
                above += excl;
                lo = g;
                __syncthreads();  // (hist and the found bin are rewritten)
            }
        }
    }
    uint32_t done = 0;  // (C_Q1P) entries whose exact keys stand
    // sorts the list, keeps its kk best and raises the bound to the kk-th
    auto compress = [&]() {
        __syncthreads();
        uint32_t c = L.cnt;
        if constexpr (Q1P) {
            using SH = ScanShape<C_Q1P, Q1P ? LPR : 4, 1>;
            constexpr int U = SH::U, G = SH::G, LP = Q1P ? LPR : 4;
            for (uint32_t i = done + tid; i < c; i += PICK_THREADS) L.rows[i - done] = key_row(L.keys[i]);
            __syncthreads();
            ScanRegs<C_Q1P, 1> R{};
            R.uok[0] = (uint32_t)(lane % LP) < a.s.units;
            R.ucl[0] = R.uok[0] ? (uint32_t)(lane % LP) : a.s.units - 1;
            R.qf = lut;
            ScanArgs sa{};
            sa.codes = a.s.codes;
            sa.row_bytes = a.s.row_bytes;
            sa.scales = a.s.scales;
            for (uint32_t base = (uint32_t)wave * SH::RPS; base < c - done; base += PICK_WAVES * SH::RPS) {
                StepData<C_Q1P, LP, 1> S;
                load_step<C_Q1P, LP, 1, true>(sa, R, L.rows, base, c - done, S, lane);
                float ex[U];
#pragma unroll
                for (int u = 0; u < U; ++u) ex[u] = q1p_exact_partial<LP, 1>(R, S.d[u], lane % LP);
                const float tot = xreduce<U, LP>(ex, lane);
                const uint32_t mine = base + (uint32_t)(xrow<U, LP>(lane) * G + lane / LP);
                if (xrep<U, LP>(lane) && mine < c - done)
                    L.keys[done + mine] = make_key(ord_f32(tot * (S.scale * a.s.scale_mul)), S.grow);
            }
            __syncthreads();
        }
        uint32_t npow = 2;
        while (npow < c) npow <<= 1;
        for (uint32_t i = c + tid; i < npow; i += PICK_THREADS) L.keys[i] = 0;
        __syncthreads();
        sort_desc_lds<PICK_THREADS>(L.keys, npow);
        c = c < kk ? c : kk;
        done = c;
        if (c == kk && L.keys[kk - 1] > th) th = L.keys[kk - 1];
        if (tid == 0) L.cnt = c;
        __syncthreads();
    };
    if constexpr (Q1P) {
        // the best rows of the slots that reach it: their kk-th best exact key
        // is a bound too, and above their lower bounds
        if (th > 1) {
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < PICK_REG; ++j)
                if (kr[j] >= th) L.keys[atomicAdd(&L.cnt, 1u)] = kr[j];
            compress();  // (at most kk + kk / 4 + 16 entries)
            if (tid == 0) L.cnt = 0;
            done = 0;
        }
    }
    // ---- the slots that can hold a row at or above it ----
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < PICK_REG; ++j) {
        const uint32_t i = tid + j * PICK_THREADS;
        bool take;
        if constexpr (Q1P)
            take = i < nslots && kr[j] && a.s.top[(uint64_t)q * nslots + i] >= (uint32_t)(th >> 32);
        else
            take = kr[j] >= th;
        if (take) L.slots[atomicAdd(&L.ns, 1u)] = (uint16_t)i;
    }
    __syncthreads();

    // ---- their rows at or above the bound, PICK_CAP parts at a time ----
    const uint32_t *part = a.s.part + (uint64_t)q * nslots * a.s.nsub;
    const uint32_t nparts = L.ns << lgs;  // (at most SLOTS_MAX * 64)
    for (uint32_t p0 = 0; p0 < nparts; p0 += PICK_CAP) {
        uint32_t np = nparts - p0 < PICK_CAP ? nparts - p0 : PICK_CAP;
        __syncthreads();
        if (lgs == 0) {  // one part per slot: its best key was its test
            for (uint32_t e = tid; e < np; e += PICK_THREADS) L.parts[e] = L.slots[p0 + e];
        } else {
            if (tid == 0) L.np = 0;
            uint32_t pw[PICK_CAP / PICK_THREADS], pi[PICK_CAP / PICK_THREADS];
#pragma unroll
            for (uint32_t j = 0; j < PICK_CAP / PICK_THREADS; ++j) {
                const uint32_t e = p0 + j * PICK_THREADS + tid;
                pi[j] = e < nparts ? ((uint32_t)L.slots[e >> lgs] << lgs) + (e & (a.s.nsub - 1)) : 0u;
                pw[j] = e < nparts ? part[pi[j]] : 0u;
            }
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < PICK_CAP / PICK_THREADS; ++j)
                if (pw[j] != 0 && pw[j] >= (uint32_t)(th >> 32)) L.parts[atomicAdd(&L.np, 1u)] = pi[j];
        }
        __syncthreads();
        if (lgs != 0) np = L.np;
        const uint32_t total = np << lg;
        for (uint32_t e0 = 0; e0 < total; e0 += PICK_THREADS * PICK_ROUND) {
            uint32_t o[PICK_ROUND], pos[PICK_ROUND], row[PICK_ROUND];
    #pragma unroll
            for (uint32_t j = 0; j < PICK_ROUND; ++j) {
                const uint32_t e = e0 + j * PICK_THREADS + tid;
                const bool ok = e < total;
                pos[j] = ok ? (L.parts[e >> lg] << lg) + (e & (pr - 1)) : 0u;
                o[j] = ok && pos[j] < n ? ord[pos[j]] : 0u;
            }
            uint32_t take = 0;
            const uint32_t tord = (uint32_t)(th >> 32);
    #pragma unroll
            for (uint32_t j = 0; j < PICK_ROUND; ++j) {
                row[j] = pos[j];
                if (o[j] != 0 && o[j] >= tord) {
                    if (cand) row[j] = cand[pos[j]];
                    if (Q1P || make_key(o[j], row[j]) >= th) take |= 1u << j;
                }
            }
            if (tid == 0) L.sum = 0;
            __syncthreads();
            const uint32_t w = pick_wave_sum(__popc(take));
            if (lane == 0 && w) atomicAdd(&L.sum, w);
            __syncthreads();
            const bool fits = L.cnt + L.sum <= PICK_CAP;
            __syncthreads();  // (everyone has read the count before anyone appends)
            if (fits) {
    #pragma unroll
                for (uint32_t j = 0; j < PICK_ROUND; ++j)
                    if (take & (1u << j)) L.keys[atomicAdd(&L.cnt, 1u)] = make_key(o[j], row[j]);
            } else {  // part by part, each part's room made first
    #pragma unroll
                for (uint32_t j = 0; j < PICK_ROUND; ++j) {
                    __syncthreads();
                    if (L.cnt + PICK_THREADS > PICK_CAP) compress();
                    __syncthreads();
                    if ((take & (1u << j)) && (Q1P ? o[j] >= (uint32_t)(th >> 32) : make_key(o[j], row[j]) >= th))
                        L.keys[atomicAdd(&L.cnt, 1u)] = make_key(o[j], row[j]);
                }
            }
            __syncthreads();
        }
    }
    compress();
    uint32_t m = L.cnt;

    // ---- the exact re-rank, and the results ----
    if (a.rr_src) {
        const uint32_t ns = gridDim.y;
        uint64_t *rr = ns > 1 ? a.rr_keys + (uint64_t)q * kk : nullptr;
        for (uint32_t c0 = ((uint32_t)wave * ns + blockIdx.y) * 16; c0 < m; c0 += PICK_WAVES * ns * 16) {
            const uint32_t ci = c0 + (uint32_t)(lane >> 2);
            const uint32_t row = key_row(L.keys[ci < m ? ci : c0]);
            const uint64_t ek = exact_keys16(a.rr_src, a.rr_dim, rq, pick_smem, row, L.tiles + wave * EXACT_TILE, lane);
            if ((lane & 3) == 0 && ci < m) {
                if (rr) store_shared(&rr[ci], ek);
                else L.keys[ci] = ek;  // (each entry read and written by its own lanes)
            }
        }
        if (rr) {  // the last workgroup ranks all of them
            wait_stores_done();
            __syncthreads();
            if (tid == 0) L.sum = atomicAdd(&a.tickets[q], 1u) == ns - 1;
            __syncthreads();
            if (!L.sum) return;
            if (tid == 0) a.tickets[q] = 0;
            for (uint32_t i = tid; i < m; i += PICK_THREADS) L.keys[i] = load_shared(&rr[i]);
        }
        __syncthreads();
        uint32_t npow = 2;
        while (npow < m) npow <<= 1;
        for (uint32_t i = m + tid; i < npow; i += PICK_THREADS) L.keys[i] = 0;
        __syncthreads();
        sort_desc_lds<PICK_THREADS>(L.keys, npow);
    }
    const uint32_t ko = m < a.k_out ? m : a.k_out;
    for (uint32_t i = tid; i < ko; i += PICK_THREADS) {
        const uint32_t w = (uint32_t)(L.keys[i] >> 32);
        a.out_rows[(uint64_t)q * a.k_out + i] = key_row(L.keys[i]);
        a.out_scores[(uint64_t)q * a.k_out + i] =
            a.is_int && !a.rr_src ? (float)(int32_t)(w ^ 0x80000000u) : f32_from_ord(w);
    }
    if (tid == 0) a.out_n[q] = ko;
}

// The exact score of each listed row (bv_exact.h) in scan_slots' form: one
// wave per sixteen rows, a slot of a.rw / 16 of its passes.  A listed row at
// or past nrows scores nothing and sets *bad.  Bound by the latency of one
// wave's row reads and its f64 chain (a quarter of the dimension) for lists
// of a few thousand rows, by HBM from about 50,000 (dim * 4 bytes each).
constexpr uint32_t ROWS_WAVES = 4;
template <bool L2>
__global__ __launch_bounds__(ROWS_WAVES * 64) void rows_exact(SlotArgs a, const float *q, uint64_t nrows,
                                                             uint32_t *bad) {
    extern __shared__ __align__(16) float rows_smem[];  // the transposed query
    __shared__ __align__(16) float tiles[ROWS_WAVES][EXACT_TILE];
    const uint32_t dim = a.padded_dim;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    exact_load_query(q, dim, rows_smem, threadIdx.x, ROWS_WAVES * 64);
    __syncthreads();
    const uint32_t slot = blockIdx.x * ROWS_WAVES + (uint32_t)wave;
    if (slot >= a.nslots) return;
    uint64_t best = 0;
    for (uint32_t r0 = slot * a.rw; r0 < (slot + 1) * a.rw && r0 < a.n; r0 += 16) {
        const uint32_t i = r0 + (uint32_t)(lane >> 2);
        const uint32_t row = a.cand[i < a.n ? i : r0];
        const bool ok = row < nrows;
        const uint64_t key =
            exact_keys16<L2>((const float *)a.codes, dim, q, rows_smem, ok ? row : 0u, tiles[wave], lane);
        if ((lane & 3) == 0 && i < a.n) {
            const uint32_t w = (uint32_t)(key >> 32);
            a.ord[i] = ok ? (w ? w : 1u) : 0u;
            if (ok) best = key > best ? key : best;
            else *bad = 1u;
        }
    }
    best = wave_max_u64(best);
    if (lane == 0) a.best[slot] = best;
}

}  // namespace

hipError_t launch_rows_exact(const SlotArgs &a, const float *q, uint64_t nrows, bool l2, uint32_t *bad, hipStream_t s) {
    const size_t lds = 16 * (size_t)exact_q_stride(a.padded_dim);
    if (a.n == 0 || nrows == 0 || a.nq != 1 || a.nsub != 1 || a.rw < 16 || a.rw % 16 || !a.cand ||
        (uint64_t)a.nslots * a.rw < a.n || lds + ROWS_WAVES * EXACT_TILE * 4 > 160 * 1024)
        return hipErrorInvalidValue;
    const dim3 g((a.nslots + ROWS_WAVES - 1) / ROWS_WAVES), wg(ROWS_WAVES * 64);
    if (l2) hipLaunchKernelGGL(rows_exact<true>, g, wg, lds, s, a, q, nrows, bad);
    else hipLaunchKernelGGL(rows_exact<false>, g, wg, lds, s, a, q, nrows, bad);
    return hipGetLastError();
}

bool pick_supported(int codec, uint32_t P, uint32_t rr_dim) {
    return (codec != C_Q1P || (P >= 128 && P <= 1024)) && rr_dim <= 4096;
}

hipError_t launch_pick_topk(const PickArgs &a, hipStream_t s) {
    if (a.s.nq == 0) return hipSuccess;
    if (a.kk == 0 || a.kk > (uint32_t)MAX_KPRIME || a.s.nslots == 0 || a.s.nslots > SLOTS_MAX ||
        (a.s.rw & (a.s.rw - 1)) || a.s.nsub == 0 || (a.s.nsub & (a.s.nsub - 1)) || a.s.nsub > 64 || a.s.nsub > a.s.rw ||
        (uint64_t)PICK_CAP * (a.s.rw / a.s.nsub) >= (1ull << 32) || !pick_supported(a.q1p ? C_Q1P : C_Q8, a.s.padded_dim, a.rr_src ? a.rr_dim : 0))
        return hipErrorInvalidValue;
    size_t lds = a.rr_src ? 16 * (size_t)exact_q_stride(a.rr_dim) : 0;
    if (a.q1p) lds += q1p_lut_bytes(a.s.padded_dim);
    if (lds + sizeof(PickLds) > 160 * 1024) return hipErrorInvalidValue;
    if (a.split == 0 || (a.split > 1 && (!a.rr_src || !a.rr_keys || !a.tickets))) return hipErrorInvalidValue;
    const dim3 g(a.s.nq, a.split), wg(PICK_THREADS);
    if (!a.q1p) hipLaunchKernelGGL((pick_topk<0>), g, wg, lds, s, a);
    else {
        Layout L;
        if (!a.s.top || !a.qrot || !pick_layout(a.s.units, L) || L.upl != 1) return hipErrorInvalidValue;
        if (L.lpr == 4) hipLaunchKernelGGL((pick_topk<4>), g, wg, lds, s, a);
        else if (L.lpr == 8) hipLaunchKernelGGL((pick_topk<8>), g, wg, lds, s, a);
        else return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace bvk
