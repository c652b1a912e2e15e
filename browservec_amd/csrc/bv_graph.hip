// Graph beam search over a flat fixed-degree adjacency (HNSW's layer 0), one
// workgroup of four waves per query: the searcher of src/index/hnswGpu.ts:134-206
// with the best-first beam of src/engine/wgsl/graphSearch.ts:62-259.
//
// A query is a chain of expansions, each waiting on memory twice (the node's
// links, then its neighbours' rows), so what counts is the latency of one:
//   - all rows of an expansion come in at once, 1 KB of a row per wave and
//     load (256 dimensions), two such rounds in flight; the links of the
//     node that would be next come in while they do;
//   - every lane multiplies what it loaded (products are rounded on their own,
//     so who forms them does not matter) and leaves the products in LDS; the
//     sums run in f32 in element order, one lane of wave 0 per row
//     (`acc = acc + c * q`), which is the shader's arithmetic;
//   - wave 0 keeps the whole beam in registers (lane t holds slots t, t + 64,
//     t + 128, t + 192) and finds its best and worst slots by a DPP reduction
//     and a ballot.  The shader reduces by each lane's first strict best and a
//     halving tree of strict compares: among equal distances that is the lane
//     lowest in bit-reversed order, then its lowest slot;
//   - the visited set is the shader's 2048-slot open-addressed table in LDS
//     (a run of 16 full slots sheds the id, reported unseen).  A batch of ids
//     is inserted as if in lane order: every lane probes its run at once, and
//     lanes commit together up to the first that lost its slot to a lower
//     lane, which probes again.
// 200,000 x 768, degree 32, ef 128, us a batch: 1 query 1,460 (3,024 with one
// wave per query and a lane reading each row), 64 queries 1,730 (3,681), 256
// 1,759 (3,672), 1,024 3,611 (3,962).  An expansion takes 13 us: rows 4.5, the
// 768 dependent adds 3.5 (2.8 at 8.6 clocks each), folding 3.5, marking 1.
// Eight waves with three rounds in flight: 1,725 at 64 queries, but 6,535 at
// 1,024 (one workgroup per CU).
// The end of the kernel dedups the beam (first slot of an id), sorts it by
// score (-distance) with ties in slot order, and writes the top k.
#include <hip/hip_runtime.h>

#include "bv_kernels.h"
#include "bv_scan.h"

namespace bvk {
namespace {

constexpr uint32_t GS_LANES = 64;
constexpr uint32_t GS_WAVES = 4;
constexpr uint32_t GS_WG = GS_WAVES * 64;
constexpr uint32_t GS_SLOTS = GRAPH_EF_CAP / GS_LANES;  // beam slots per lane of wave 0
constexpr uint32_t GS_HASH = 2048;
constexpr uint32_t GS_PROBES = 16;
constexpr uint32_t GS_CLAIMS = 512;  // (two slots that share a claim only make a lane probe again)
constexpr float GS_INF = 3.4e38f;
constexpr uint32_t GS_EMPTY = 0xffffffffu;
constexpr uint32_t GS_ROWS = 32;          // rows summed at once
constexpr uint32_t GS_CHUNK = 256;        // dimensions per round
constexpr int GS_DEPTH = 2;               // rounds in flight
constexpr uint32_t GS_RS = GS_CHUNK + 4;  // tile row stride (spreads the rows over the banks)

struct GraphLds {
    float tile[GS_ROWS][GS_RS];
    uint32_t vis[GS_HASH];
    uint32_t claim[GS_CLAIMS];
    float hd[GRAPH_EF_CAP];
    uint32_t hi[GRAPH_EF_CAP];
    uint32_t ids[GS_LANES];  // an expansion's rows
    float dist[GS_LANES];
    uint32_t nf;             // how many (GS_EMPTY: the search is over)
};

__device__ __forceinline__ float rdlane(float v, uint32_t l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (int)l));
}
__device__ __forceinline__ uint32_t rdlane(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// One round of a lane's four elements of a row: their products with the
// query's (L2: squared differences), zero past the dimension (adding zero
// leaves a sum as it is).
template <bool L2> __device__ __forceinline__ float4 products(float4 x, float4 y) {
#pragma clang fp contract(off)
    if (L2) {
        const float a = x.x - y.x, b = x.y - y.y, c = x.z - y.z, d = x.w - y.w;
        return make_float4(a * a, b * b, c * c, d * d);
    }
    return make_float4(x.x * y.x, x.y * y.y, x.z * y.z, x.w * y.w);
}

struct __attribute__((packed, aligned(4))) f32x4_g {
    float x, y, z, w;
};
// Elements [e, e + 4) of a row as loaded: past the dimension's end its last
// four (part4 puts them in place), so that every lane loads, nothing past the
// row is read and no lane waits for a load before it is used.
__device__ __forceinline__ float4 load4(const float *row, uint32_t e, uint32_t dim) {
    if (dim < 4) return make_float4(row[0], dim > 1 ? row[1] : 0.0f, dim > 2 ? row[2] : 0.0f, 0.0f);
    const f32x4_g v = *(const f32x4_g *)(row + (e + 4 <= dim ? e : dim - 4));
    return make_float4(v.x, v.y, v.z, v.w);
}
// Those elements in place, zeros past the end.
__device__ __forceinline__ float4 part4(float4 v, uint32_t e, uint32_t dim) {
    if (dim < 4) return e == 0 ? v : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const uint32_t sh = e + 4 <= dim ? 0u : e + 4 - dim;  // elements past the end
    return make_float4(sh == 0 ? v.x : sh == 1 ? v.y : sh == 2 ? v.z : sh == 3 ? v.w : 0.0f,
                       sh == 0 ? v.y : sh == 1 ? v.z : sh == 2 ? v.w : 0.0f, sh == 0 ? v.z : sh == 1 ? v.w : 0.0f,
                       sh == 0 ? v.w : 0.0f);
}

// L.dist[0, nf) = the distances of rows L.ids[0, nf) (smaller = closer: -dot
// for dot / cosine, the squared difference for l2).  Whole workgroup, after a
// barrier; ends with one.  qv: the query, zero-padded to whole rounds.
template <bool L2>
__device__ void row_dists(GraphLds &L, const float *corpus, const float *qv, uint32_t dim, uint32_t nf) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int PER = GS_ROWS / GS_WAVES;  // rows per wave
    const uint32_t nch = (dim + GS_CHUNK - 1) / GS_CHUNK;
    for (uint32_t base = 0; base < nf; base += GS_ROWS) {
        const uint32_t rows = nf - base < GS_ROWS ? nf - base : GS_ROWS;
        const float *src[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {  // row 4i + wave
            const uint32_t r = GS_WAVES * i + (uint32_t)wave;
            src[i] = corpus + (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(L.ids[base + (r < rows ? r : 0)]) * dim;
        }
        float4 x[GS_DEPTH][PER];
        auto load = [&](uint32_t ch, float4 (&v)[PER]) {
#pragma unroll
            for (int i = 0; i < PER; ++i)
                if (GS_WAVES * (uint32_t)i + (uint32_t)wave < rows) v[i] = load4(src[i], ch * GS_CHUNK + 4 * lane, dim);
        };
#pragma unroll
        for (int d = 0; d < GS_DEPTH; ++d)
            if ((uint32_t)d < nch) load((uint32_t)d, x[d]);
        float acc = 0.0f;
        for (uint32_t c0 = 0; c0 < nch; c0 += GS_DEPTH) {
#pragma unroll
            for (int d = 0; d < GS_DEPTH; ++d) {
                const uint32_t ch = c0 + d;
                if (ch >= nch) break;
                const uint32_t e = ch * GS_CHUNK + 4 * lane;
                const float4 y = *(const float4 *)&qv[e];
                const bool whole = (ch + 1) * GS_CHUNK <= dim;
#pragma unroll
                for (int i = 0; i < PER; ++i)
                    if (GS_WAVES * (uint32_t)i + (uint32_t)wave < rows)
                        *(float4 *)&L.tile[GS_WAVES * i + wave][4 * lane] =
                            products<L2>(whole ? x[d][i] : part4(x[d][i], e, dim), y);
                if (ch + GS_DEPTH < nch) load(ch + GS_DEPTH, x[d]);
                // (LDS only: loads stay in flight across it)
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                if (wave == 0 && (uint32_t)lane < rows) {
                    const uint32_t left = dim - ch * GS_CHUNK, n4 = ((left < GS_CHUNK ? left : GS_CHUNK) + 3) / 4;
                    const float4 *t = (const float4 *)L.tile[lane];
                    constexpr int B = 8;  // reads ahead of the sum
                    float4 v[B];
#pragma unroll
                    for (int u = 0; u < B; ++u) v[u] = t[u];
                    auto add = [&](const float4 &w) {
                        acc = acc + w.x;
                        acc = acc + w.y;
                        acc = acc + w.z;
                        acc = acc + w.w;
                    };
                    uint32_t j = 0;
                    for (; j + 2 * B <= n4; j += B) {
#pragma unroll
                        for (int u = 0; u < B; ++u) {
                            const float4 w = v[u];
                            v[u] = t[j + B + u];
                            add(w);
                        }
                    }
                    if (j + B <= n4) {
#pragma unroll
                        for (int u = 0; u < B; ++u) add(v[u]);
                        j += B;
                    }
                    for (; j < n4; ++j) add(t[j]);
                }
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
        }
        if (wave == 0 && (uint32_t)lane < rows) L.dist[base + lane] = L2 ? acc : -acc;
    }
    __syncthreads();
}

// Wave 0: the lanes in `want` insert their id into the visited set as if in
// lane order; true on a lane whose id was not there before (inserted or shed).
__device__ bool mark_batch(GraphLds &L, uint32_t id, bool want, uint32_t t) {
    bool fresh = false, pending = want;
    const uint32_t h = (id * 2654435761u) & (GS_HASH - 1u);
    while (__ballot(pending)) {
        uint32_t cur[GS_PROBES];
#pragma unroll
        for (uint32_t j = 0; j < GS_PROBES; ++j) cur[j] = L.vis[(h + j) & (GS_HASH - 1u)];
        // the first slot of the run that holds the id or is empty
        uint32_t at = GS_PROBES;
        bool seen = false;
#pragma unroll
        for (uint32_t j = GS_PROBES; j-- > 0;)
            if (cur[j] == id + 1u || cur[j] == 0u) {
                at = j;
                seen = cur[j] != 0u;
            }
        if (pending && (at == GS_PROBES || seen)) {  // stands whatever the other lanes insert
            fresh = !seen;
            pending = false;
        }
        const uint32_t pos = (h + at) & (GS_HASH - 1u);
        uint32_t *claim = &L.claim[pos & (GS_CLAIMS - 1u)];
        if (pending) atomicMin(claim, t);
        wave_sync();
        const bool won = pending && *claim == t;
        const uint64_t lost = __ballot(pending && !won);
        const uint32_t first = lost ? (uint32_t)__builtin_ctzll(lost) : GS_LANES;
        wave_sync();
        if (pending) *claim = 0xffffffffu;
        if (won && t < first) {
            L.vis[pos] = id + 1u;
            fresh = true;
            pending = false;
        }
        wave_sync();
    }
    return fresh;
}

// The wave's largest value, in every lane (no NaN among them).
__device__ __forceinline__ float wave_max_f32(float v) {
    v = fmaxf(v, dpp<DPP_XOR1>(v));
    v = fmaxf(v, dpp<DPP_XOR2>(v));
    v = fmaxf(v, dpp<DPP_HALF_MIRROR>(v));
    v = fmaxf(v, dpp<DPP_MIRROR>(v));
    const auto a = __builtin_amdgcn_permlane16_swap(as_i(v), as_i(v), false, false);
    v = fmaxf(from_i<float>(a[0]), from_i<float>(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(as_i(v), as_i(v), false, false);
    return fmaxf(from_i<float>(b[0]), from_i<float>(b[1]));
}

// Wave 0: argmax over the active slots (foldStaged's worst) or argmin over the
// unexpanded ones, in the shader's order.
template <bool MAX>
__device__ __forceinline__ void beam_arg(const float (&cd)[GS_SLOTS], const uint32_t (&ce)[GS_SLOTS], uint32_t efA,
                                         uint32_t t, float &val, uint32_t &slot) {
    float v = -GS_INF;  // (argmin: of the negated distances)
    uint32_t mi = 0;
#pragma unroll
    for (uint32_t m = 0; m < GS_SLOTS; ++m) {
        const float x = MAX ? cd[m] : -cd[m];
        if (t + GS_LANES * m < efA && (MAX || ce[m] == 0u) && x > v) {
            v = x;
            mi = m;
        }
    }
    const float top = rdlane(wave_max_f32(v), 0);
    val = MAX ? top : -top;
    if (!(top > -GS_INF)) {  // (none: the reduction's start values)
        slot = 0;
        return;
    }
    uint64_t tie = __ballot(v == top);
    uint32_t l = (uint32_t)__builtin_ctzll(tie);
    for (tie &= tie - 1; tie; tie &= tie - 1) {
        const uint32_t o = (uint32_t)__builtin_ctzll(tie);
        if (__brev(o) < __brev(l)) l = o;
    }
    slot = l + GS_LANES * rdlane(mi, l);
}

// Wave 0, foldStaged: L.dist / L.ids [0, count) in order, each replacing the
// worst active slot when it is better.
__device__ void fold(const GraphLds &L, float (&cd)[GS_SLOTS], uint32_t (&ci)[GS_SLOTS], uint32_t (&ce)[GS_SLOTS],
                     uint32_t efA, uint32_t count, uint32_t t) {
    const float sd = t < count ? L.dist[t] : GS_INF;
    const uint32_t si = t < count ? L.ids[t] : GS_EMPTY;
    float worst;
    uint32_t slot;
    beam_arg<true>(cd, ce, efA, t, worst, slot);
    // (the worst only falls: an entry not below it now never is)
    uint64_t live = __ballot(sd < GS_INF && sd < worst);
    while (live) {
        const uint32_t j = (uint32_t)__builtin_ctzll(live);
        live &= live - 1;
        const float d = rdlane(sd, j);
        if (!(d < worst)) continue;
        const uint32_t id = rdlane(si, j);
#pragma unroll
        for (uint32_t m = 0; m < GS_SLOTS; ++m)
            if (slot == t + GS_LANES * m) {
                cd[m] = d;
                ci[m] = id;
                ce[m] = 0u;
            }
        beam_arg<true>(cd, ce, efA, t, worst, slot);
    }
}

template <bool L2>
__global__ __launch_bounds__(GS_WG) void graph_beam(GraphArgs a) {
    __shared__ GraphLds L;
    extern __shared__ __align__(16) float qv[];  // the query, zero-padded to whole rounds
    const uint32_t q = blockIdx.x, tid = threadIdx.x, t = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t dim = a.dim, efA = a.efA;
    const uint32_t qpad = (dim + GS_CHUNK - 1) / GS_CHUNK * GS_CHUNK;
    for (uint32_t i = tid; i < qpad; i += GS_WG) qv[i] = i < dim ? a.queries[(uint64_t)q * dim + i] : 0.0f;
    for (uint32_t i = tid; i < GS_HASH; i += GS_WG) L.vis[i] = 0u;
    for (uint32_t i = tid; i < GS_CLAIMS; i += GS_WG) L.claim[i] = 0xffffffffu;
    float cd[GS_SLOTS];
    uint32_t ci[GS_SLOTS], ce[GS_SLOTS];
#pragma unroll
    for (uint32_t m = 0; m < GS_SLOTS; ++m) {
        cd[m] = GS_INF;
        ci[m] = GS_EMPTY;
        ce[m] = 1u;
    }
    __syncthreads();
    // wave 0 stages a batch of ids: those in the corpus and not seen before
    auto stage = [&](uint32_t id) {
        const bool fresh = mark_batch(L, id, id < a.corpus_rows, t);
        const uint64_t b = __ballot(fresh);
        if (fresh) L.ids[lanes_below(b)] = id;
        if (t == 0) L.nf = (uint32_t)__popcll(b);
    };
    if (wave == 0) {  // seeds, staged like a neighbour batch
        const uint32_t ne = a.n_entries < GS_LANES ? a.n_entries : GS_LANES;
        stage(t < ne ? a.entries[t] : GS_EMPTY);
    }
    // node's neighbours, one per lane
    auto links = [&](uint32_t node) -> uint32_t {
        return (t < a.K && node < a.graph_rows) ? a.graph[(uint64_t)node * a.K + t] : GS_EMPTY;
    };
    // the node in beam slot `slot`, marked expanded when `take` is set
    auto node_at = [&](uint32_t slot, bool take) -> uint32_t {
        uint32_t node = 0;
#pragma unroll
        for (uint32_t m = 0; m < GS_SLOTS; ++m)
            if (slot == t + GS_LANES * m) {
                if (take) ce[m] = 1u;
                node = ci[m];
            }
        return rdlane(node, slot & (GS_LANES - 1));
    };
    for (uint32_t iter = 0;; ++iter) {
        __syncthreads();
        const uint32_t nf = L.nf;
        if (nf == GS_EMPTY) break;
        // the node expanded next unless one of this batch is closer: its links
        // come in while the batch is scored
        uint32_t guess = GS_EMPTY, glinks = GS_EMPTY;
        if (wave == 0) {
            float best;
            uint32_t slot;
            beam_arg<false>(cd, ce, efA, t, best, slot);
            if (best < GS_INF) {
                guess = node_at(slot, false);
                glinks = links(guess);
            }
        }
        row_dists<L2>(L, a.corpus, qv, dim, nf);
        if (wave != 0) continue;
        fold(L, cd, ci, ce, efA, nf, t);
        float best = GS_INF;
        uint32_t slot = 0;
        if (iter < a.iter_cap) beam_arg<false>(cd, ce, efA, t, best, slot);
        if (best >= GS_INF) {
            if (t == 0) L.nf = GS_EMPTY;
            continue;
        }
        const uint32_t node = node_at(slot, true);
        stage(node == guess ? glinks : links(node));
    }
    // the raw beam (parity export) and the searcher's hits
    if (wave == 0) {
#pragma unroll
        for (uint32_t m = 0; m < GS_SLOTS; ++m) {
            L.hd[t + GS_LANES * m] = cd[m];
            L.hi[t + GS_LANES * m] = ci[m];
        }
    }
    __syncthreads();
    static_assert(GS_WG >= GRAPH_EF_CAP, "one beam slot per thread");
    const bool slot_ok = tid < GRAPH_EF_CAP;
    const uint32_t s = slot_ok ? tid : 0, my = L.hi[s];
    const float sc = -L.hd[s];
    if (a.beam_dist && slot_ok) {
        a.beam_dist[(uint64_t)q * GRAPH_EF_CAP + s] = L.hd[s];
        a.beam_id[(uint64_t)q * GRAPH_EF_CAP + s] = my;
    }
    if (!a.out_rows) return;
    // live slot: below efA, not empty, its id's first slot (flags in the
    // visited table's space, no longer needed)
    bool lv = slot_ok && s < efA && my != GS_EMPTY;
    for (uint32_t s2 = 0; s2 < efA; ++s2) lv = lv && !(s2 < s && L.hi[s2] == my);
    if (slot_ok) L.vis[s] = lv ? 1u : 0u;
    const int nlive = __syncthreads_count(lv);
    // rank = live slots with a higher score, or the same score at a lower slot
    if (lv) {
        uint32_t r = 0;
        for (uint32_t s2 = 0; s2 < efA; ++s2) {
            const float o = -L.hd[s2];
            r += (L.vis[s2] && s2 != s && (o > sc || (o == sc && s2 < s))) ? 1u : 0u;
        }
        if (r < a.k) {
            a.out_rows[(uint64_t)q * a.out_stride + r] = my;
            a.out_scores[(uint64_t)q * a.out_stride + r] = sc;
        }
    }
    const uint32_t ko = (uint32_t)nlive < a.k ? (uint32_t)nlive : a.k;
    for (uint32_t r = ko + tid; r < a.out_stride; r += GS_WG) {  // (no hit: zeros)
        a.out_rows[(uint64_t)q * a.out_stride + r] = 0u;
        a.out_scores[(uint64_t)q * a.out_stride + r] = 0.0f;
    }
    if (tid == 0) a.out_n[q] = ko;
}

}  // namespace

hipError_t launch_graph_beam(const GraphArgs &a, uint32_t nq, bool l2, hipStream_t s) {
    if (nq == 0) return hipSuccess;
    if (a.K == 0 || a.K > GS_LANES || a.efA == 0 || a.efA > GRAPH_EF_CAP || a.k > GRAPH_EF_CAP || a.dim == 0 ||
        (size_t)a.dim * 4 > 64 * 1024)
        return hipErrorInvalidValue;
    const size_t lds = (size_t)((a.dim + GS_CHUNK - 1) / GS_CHUNK * GS_CHUNK) * 4;
    if (l2)
        hipLaunchKernelGGL(graph_beam<true>, dim3(nq), dim3(GS_WG), lds, s, a);
    else
        hipLaunchKernelGGL(graph_beam<false>, dim3(nq), dim3(GS_WG), lds, s, a);
    return hipGetLastError();
}

}  // namespace bvk
