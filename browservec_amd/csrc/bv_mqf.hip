// fp32 query batches on the matrix cores: a bf16 prefilter of the rows as
// they are stored, with proven bounds.
//
// mqf_scan multiplies bf16 roundings of the rows (made on the way from LDS to
// the matrix cores; the index keeps no second copy) with bf16 queries held in
// registers, accumulates in f32, and turns each sum s into bounds of the
// single-query scan's score:
//     s - E <= score <= s + E,   E = alpha |x| + beta (+ gamma |x|^2 under l2)
// with, by Cauchy-Schwarz on the rounding errors x - bf16(x) and q - bf16(q),
//     |x.q - bf16(x).bf16(q)| <= (rx + rq + rx rq) |x| |q|
// where rq = |q - bf16(q)| / |q| of the query and rx is the largest such ratio
// of any row (kept by row_sqnorms at append; both about 0.0017 where the worst
// case of one element is 0.0039), plus the f32 rounding of both sums.  What the
// bounds let through is scored by the single-query arithmetic, so batches
// return exactly what single queries return; passes, buckets, selects and
// fallback are those of the int8 level-one batch (bv_mq.hip).
//
// Tiles of 32 rows stream through LDS as 16 KB chunks of 128 dimensions, five
// in flight, loaded straight to LDS.  A chunk that has landed is turned into a
// bf16 tile by all waves while they multiply the one before, and every wave
// multiplies the whole tile with its own 32 queries: a row is read from HBM
// and converted once per 256 queries (128 above 768 dimensions, where the
// queries take a wave's whole register file of 512).  Pieces of 16 bytes are
// stored at piece ^ row, which spreads the rows of a matrix operand over the
// banks.
// 1M x 768, 256 queries: the pass over seven eighths of the rows takes 555 us
// (4.8 TB/s; 3.07 GB cost 430 us a pass as a plain stream), 759 us the call;
// the exact fp32 products it replaces (v_mfma_f32_32x32x2f32, every row once
// per 32 queries) took 3,401 us.  Up to 64 queries the stream bounds it (674
// us a call); at 256 the matrix cores are busy a quarter of the time and the
// VALU and LDS less: the barrier per chunk is what is left.  Each wave
// converting for itself (640 us), reading further ahead at the price of a
// spill (657) and 64 queries per wave of one wave per SIMD (the compiler
// moves the sums between register files) were slower.
#include "bv_kernels.h"
#include "bv_device.h"
#include "bv_mfma.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bvk {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v8f __attribute__((ext_vector_type(8)));

constexpr uint32_t MQF_ROWS = 32;
constexpr uint32_t MQF_DIMS = 128;                      // dimensions per chunk
constexpr uint32_t MQF_CHUNK = MQF_ROWS * MQF_DIMS * 4; // bytes
constexpr uint32_t MQF_TILE = MQF_CHUNK / 2;            // the same as bf16
constexpr uint32_t MQF_STAGE = 120;                     // entries per wave per staging buffer

// The next float below x.
__device__ __forceinline__ float mqx_below(float x) {
    if (x != x) return x;  // (keeps every row)
    const uint32_t b = __float_as_uint(x);
    if ((b & 0x7fffffffu) == 0) return __uint_as_float(0x80000001u);
    if (b == 0xff800000u) return x;
    return __uint_as_float((b & 0x80000000u) ? b + 1 : b - 1);
}

struct MqfStage {
    uint64_t lk[2][8][MQF_STAGE];  // lower-bound keys, in lane order
    uint32_t uo[2][8][MQF_STAGE];  // order words of the upper bounds
    uint16_t lo[2][8][64];         // first entry of each lane
    uint16_t ln[2][8][64];         // entries of each lane
};

__device__ __forceinline__ float mqf_upper(float s, float e) { return fmaf(fabsf(s), 0x1p-20f, s + e); }
__device__ __forceinline__ float mqf_lower(float s, float e) { return fmaf(-fabsf(s), 0x1p-20f, s - e); }

// |x| from |x|^2, rounded up: no smaller than 2^-60 (below, f32 squares lose
// digits), and infinite (no bound: the row is kept) where a product with a
// query or a sum could leave the range of f32, or the square is not a number.
__device__ __forceinline__ float mqf_norm(float x2) {
    const float xn = x2 < 0x1p-120f ? 0x1p-60f : __builtin_sqrtf(x2) * (1.0f + 0x1p-20f);
    return xn < 0x1p60f ? xn : __builtin_inff();
}

// Staged entries of buffer fb into this workgroup's bucket of each query: lane
// l of flushing wave f owns query f * 64 + l of the block (its entries were
// staged by wave (f * 64 + l) / 32, lanes c and c + 32), its bucket length in
// a register.
template <int QB>
__device__ __forceinline__ void mqf_flush(const MqfArgs &a, uint32_t qb, uint32_t wg, const MqfStage &st, int fb, int f,
                                          int lane, uint32_t &len, bool &ovf) {
    asm volatile("" : "+v"(lane));  // (addresses are formed per call, not kept across the tile loop)
    const uint32_t ql = (uint32_t)f * 64 + lane, w = ql / 32, c = ql % 32;
    if (qb * QB + ql >= a.nq) return;
    const uint64_t bucket = ((uint64_t)(qb * QB + ql) * a.nwg + wg) * a.capw;
    const uint32_t off0 = st.lo[fb][w][c], n0 = st.ln[fb][w][c];
    const uint32_t off1 = st.lo[fb][w][c + 32], n1 = st.ln[fb][w][c + 32];
    for (uint32_t j = 0; j < n0 + n1; ++j) {
        const uint32_t i = j < n0 ? off0 + j : off1 + (j - n0);
        if (i >= MQF_STAGE) continue;  // (in the query's spill list)
        if (len < a.capw) {
            a.cand[bucket + len] = st.lk[fb][w][i];
            a.up_out[bucket + len] = st.uo[fb][w][i];
        } else {
            ovf = true;
        }
        ++len;
    }
}

// CH: chunks per row.  WAVES of 32 queries each; the first half issue the
// loads, the second half move staged entries to the buckets.
template <int CH, int WAVES, bool THR>
__global__ __launch_bounds__(WAVES * 64) void mqf_scan(MqfArgs a) {
    constexpr int QB = WAVES * 32, LOADERS = WAVES / 2;
    constexpr int R = 6;                                         // ring of chunks
    constexpr int PW = 16 / LOADERS;                             // loads per loader wave and chunk
    constexpr int AHEAD = 2;                                     // steps of a chunk read ahead
    // steps whose query operands stay in registers; at six chunks the last
    // one's is read from LDS (one too many for the 256 of two waves per SIMD,
    // and a spill inside the loop would wait for the chunks in flight)
    constexpr int QREG = CH == 6 ? CH * 8 - 1 : CH * 8;
    static_assert((R - 1) * PW <= 63, "the load counter holds 63");
    __shared__ __align__(1024) unsigned char ring[R * MQF_CHUNK];
    __shared__ __align__(1024) unsigned char tile[2 * MQF_TILE]; // chunks as bf16
    __shared__ __align__(16) float rs[2][MQF_ROWS];              // squared row norms, by tile parity
    __shared__ __align__(16) float rn[2][MQF_ROWS];              // their roots, rounded up
    __shared__ __align__(16) MqfQuery sq[QB];                    // the queries' constants and bounds
    __shared__ float stau[QB];
    __shared__ v8bf qlast[QREG < CH * 8 ? WAVES * 64 : 1];
    __shared__ MqfStage st;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, c = lane & 31;
    // workgroups b, b + 8, .. share an XCD: the query blocks of one row stream
    // are placed on one, and read the rows through its L2
    const uint32_t slot = blockIdx.x >> 3, xcd = blockIdx.x & 7u;
    const uint32_t qb = slot % a.qblocks, wg = (slot / a.qblocks) * 8 + xcd;
    const uint64_t ntiles = (a.n + MQF_ROWS - 1) / MQF_ROWS;
    const bool loader = wave < LOADERS;
    for (uint32_t i = threadIdx.x; i < 2 * 8 * 64; i += WAVES * 64) st.ln[i / 512][(i / 64) % 8][i % 64] = 0;
    uint32_t blen = 0;
    bool bovf = false;
    const uint32_t mine = wg < ntiles ? (uint32_t)((ntiles - wg + a.nwg - 1) / a.nwg) : 0;  // tiles wg, wg + nwg, ..
    const uint32_t total = mine * CH;

    // this wave's queries as B operands: lane l holds, at step st, piece
    // 2 st + l / 32 of query l % 32 (pieces as in the converted rows)
    const uint32_t q0 = qb * QB + (uint32_t)wave * 32;
    const bool live = q0 < a.nq;
    v8bf qreg[QREG];
    {
        const v8bf *src = (const v8bf *)(a.qbf + (uint64_t)(q0 + c < a.nq ? q0 + c : a.nq - 1) * a.qstride) + h;
#pragma unroll
        for (int s = 0; s < QREG; ++s) qreg[s] = src[2 * s];
        if constexpr (QREG < CH * 8) qlast[threadIdx.x] = src[2 * QREG];  // (read by its own lane alone)
    }
    // (held from here on: a wait for these loads inside the loop would also
    // wait for the chunks in flight)
#pragma unroll
    for (int s = 0; s < QREG; ++s) asm volatile("" : "+v"(qreg[s]));
    for (uint32_t i = threadIdx.x; i < QB; i += WAVES * 64) {
        const uint32_t qi = qb * QB + i < a.nq ? qb * QB + i : a.nq - 1;
        sq[i] = a.qk[qi];
        const uint64_t tau = THR ? a.tau[qi] : 0ull;
        stau[i] = tau ? f32_from_ord((uint32_t)(tau >> 32)) : -__builtin_inff();
    }

    const uint32_t ring0 = lds_addr(ring);
    // chunk g of this workgroup's stream into its ring slot, by the loader
    // waves: a scalar address per load, and 32 bits per lane on top of it
    // (recomputed, not kept: the registers beside the queries are few)
    const uint64_t stride = a.row_step * a.dim * 4;
    auto load_chunk = [&](uint32_t g) {
        const uint32_t t = g / CH, ch = g - t * CH;
        uint32_t lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const uint64_t row0 = (wg + (uint64_t)t * a.nwg) * MQF_ROWS;
        const bool whole = row0 + MQF_ROWS <= a.n;
        const char *base = (const char *)a.rows + row0 * stride + ch * MQF_DIMS * 4;
        const uint32_t dst = ring0 + g % R * MQF_CHUNK;
        // past the row's end a lane loads the row's last piece: it meets zeros
        // of the query, as do the up to three elements of the next row (or the
        // buffer's padding) in the last piece of a row whose length is no
        // multiple of four (a piece needs the alignment of a dword only; if
        // they are not finite the row has no bounds, and is kept)
        const uint32_t last = ((a.dim - 1) / 4 * 4 - ch * MQF_DIMS) * 4;
#pragma unroll
        for (int j = 0; j < PW; ++j) {
            const uint32_t r0 = 2 * ((uint32_t)wave * PW + j), hi = lane >> 5;  // two rows of 32 pieces
            uint32_t e = ((lane & 31) ^ hi ^ r0) * 16;
            e = e < last ? e : last;
            const char *src = base + r0 * stride;
            uint32_t off = hi * (uint32_t)stride + e;
            if (!whole) {  // rows past the end load the last row; their results are dropped
                src = (const char *)a.rows + ch * MQF_DIMS * 4 + (row0 + r0 < a.n ? row0 + r0 : a.n - 1) * stride;
                if (row0 + r0 + hi >= a.n) off = e;
            }
            lds_dma16_nt(src, off, dst + r0 * 512);
        }
    };
    auto row_norm = [&](uint32_t k) -> float {  // (lanes 0..31 of the first flushing wave)
        uint64_t li = (wg + (uint64_t)k * a.nwg) * MQF_ROWS + (uint64_t)(lane & 31);
        if (li >= a.n) li = a.n - 1;
        return a.rsq[li * a.row_step];
    };
    const bool norms = wave == LOADERS;
    float nv = norms && mine > 0 ? row_norm(0) : 0.0f;
    // waits until chunk g has landed when the chunks up to g + ahead have been
    // issued (the load counter drains in order)
    auto landed = [&](uint32_t g, uint32_t ahead) {
        uint32_t after = total - 1 - g;
        after = after < ahead ? after : ahead;
        if (after >= 5) __builtin_amdgcn_s_waitcnt(vmcnt_imm(5 * PW));
        else if (after == 4) __builtin_amdgcn_s_waitcnt(vmcnt_imm(4 * PW));
        else if (after == 3) __builtin_amdgcn_s_waitcnt(vmcnt_imm(3 * PW));
        else if (after == 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * PW));
        else if (after == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(PW));
        else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    };
    // the workgroup's chunk g to bf16: thread t takes 16-byte piece j = t % 16
    // of row t / 16, which holds fp32 pieces j and j + 16 of the chunk
    constexpr int CV = 512 / (WAVES * 64);
    auto convert_read = [&](uint32_t g, float4 (&cv)[CV][2]) {
        uint32_t t = threadIdx.x;
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int i = 0; i < CV; ++i) {
            const uint32_t r = t / 16 + i * (32 / CV);
            const unsigned char *src = ring + g % R * MQF_CHUNK + r * 512 + ((t % 16 ^ r) << 4);
            cv[i][0] = *(const float4 *)src;
            cv[i][1] = *(const float4 *)(ring + g % R * MQF_CHUNK + r * 512 + (((t % 16 + 16) ^ r) << 4));
        }
    };
    auto convert_write = [&](uint32_t g, const float4 (&cv)[CV][2]) {
        uint32_t t = threadIdx.x;
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int i = 0; i < CV; ++i) {
            const uint32_t r = t / 16 + i * (32 / CV);
            const v8f v = {cv[i][0].x, cv[i][0].y, cv[i][0].z, cv[i][0].w, cv[i][1].x, cv[i][1].y, cv[i][1].z, cv[i][1].w};
            *(v8bf *)(tile + (g & 1) * MQF_TILE + r * 256 + ((t % 16 ^ r % 16) << 4)) = __builtin_convertvector(v, v8bf);
        }
    };
    if (mine) {
        if (loader) {
            for (uint32_t g = 0; g < (uint32_t)R && g < total; ++g) load_chunk(g);
            landed(0, R - 1);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        float4 cv[CV][2];
        convert_read(0, cv);
        convert_write(0, cv);
    }

    // lane l reads row c's piece 2 s + h of step s, at piece ^ (c % 16)
    const uint32_t abase = (uint32_t)c * 256 + (((uint32_t)h ^ (uint32_t)(c & 15)) << 4);
    uint32_t g = 0;
    for (uint32_t k = 0; k < mine; ++k) {
        v16f acc = v16f{};
#pragma unroll
        for (int ch = 0; ch < CH; ++ch, ++g) {
            if (loader && g + 1 < total) landed(g + 1, R - 2);
            if (ch == 0 && norms) {
                if (lane < 32) {
                    rs[k & 1][lane] = nv;
                    rn[k & 1][lane] = mqf_norm(nv);
                }
                if (k + 1 < mine) nv = row_norm(k + 1);
            }
            // chunk g is in tile g % 2 and chunk g + 1 in its slot; every wave
            // is done with tile (g + 1) % 2 and with the slot of chunk g,
            // which chunk g + R takes
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (loader) {
                if (g + R < total) load_chunk(g + R);
            } else if (THR && ch == 0 && k > 0) {
                mqf_flush<QB>(a, qb, wg, st, (int)((k - 1) & 1), wave - LOADERS, lane, blen, bovf);
            }
            float4 cv[CV][2];
            convert_read(g + 1, cv);  // (past the last chunk: an old slot into a tile that nothing reads)
            if (!live) {
                convert_write(g + 1, cv);
            } else {
                const unsigned char *base = tile + (g & 1) * MQF_TILE;
                uint32_t ab = abase;
                asm volatile("" : "+v"(ab));  // (the addresses of the pieces are formed here, not kept)
                // (the barriers keep the compiler from reading further ahead
                // than the registers beside the queries hold)
                v8bf x[AHEAD + 1];
                auto read = [&](int s) { x[s % (AHEAD + 1)] = *(const v8bf *)(base + (ab ^ (uint32_t)(s * 32))); };
#pragma unroll
                for (int s = 0; s < AHEAD; ++s) read(s);
                convert_write(g + 1, cv);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    if (s + AHEAD < 8) read(s + AHEAD);
                    v8bf qs;
                    if constexpr (QREG < CH * 8) qs = ch * 8 + s < QREG ? qreg[ch * 8 + s < QREG ? ch * 8 + s : 0] : qlast[threadIdx.x];
                    else qs = qreg[ch * 8 + s];
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[s % (AHEAD + 1)], qs, acc, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if (!live) continue;
        int h = lane >> 5, c = lane & 31;
        asm volatile("" : "+v"(h), "+v"(c));  // (what follows from them is formed here)
        const uint32_t qlocal = (uint32_t)wave * 32 + c, q = qb * QB + qlocal;
        auto row_of = [&](int r) { return 8 * (r >> 2) + 4 * h + (r & 3); };
        // bounds of the tile's 32 rows for this lane's query: register r holds
        // row 8 (r / 4) + 4 h + r % 4
        const uint64_t t0 = (wg + (uint64_t)k * a.nwg) * MQF_ROWS;
        const MqfQuery qk = sq[qlocal];
        float ev[16];
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {  // the lane's rows come in runs of four
            const float4 n4 = *(const float4 *)&rn[k & 1][8 * g4 + 4 * h];
            const float nn[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) ev[4 * g4 + j] = fmaf(nn[j], qk.alpha, qk.beta);
            if (a.l2) {
                const float4 s4 = *(const float4 *)&rs[k & 1][8 * g4 + 4 * h];
                const float ss[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    ev[4 * g4 + j] = fmaf(nn[j] * nn[j], qk.gamma, ev[4 * g4 + j]);
                    acc[4 * g4 + j] = 2.0f * acc[4 * g4 + j] - ss[j] - qk.qsq;
                }
            }
        }
        if constexpr (!THR) {
            if (q < a.nq) {
                uint64_t *out = a.cand + (uint64_t)q * a.cap;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint64_t li = t0 + row_of(r);
                    const float lo = mqf_lower(acc[r], ev[r]);
                    if (li < a.n)
                        out[li] = make_key(lo == lo ? ord_f32(lo) : 0u, (uint32_t)(a.row_base + li * a.row_step));
                }
            }
        } else {
            const int sb = (int)(k & 1);
            const float tau_score = stau[qlocal];
            // rows that can reach the query's bound (NaN: they can): first
            // whether any of the wave's does, then bit r of each lane
            uint64_t any = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) any |= __ballot(!(mqf_upper(acc[r], ev[r]) < tau_score));
            st.ln[sb][wave][lane] = 0;
            if (!any) continue;
            uint32_t p = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) p |= (!(mqf_upper(acc[r], ev[r]) < tau_score) ? 1u : 0u) << r;
            if (t0 + MQF_ROWS > a.n) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (t0 + row_of(r) >= a.n) p &= ~(1u << r);
            }
            if (q >= a.nq) p = 0;
            const uint32_t cnt = __popc(p), incl = wave_incl_scan(cnt);
            st.lo[sb][wave][lane] = (uint16_t)(incl - cnt);
            st.ln[sb][wave][lane] = (uint16_t)cnt;
            if (__builtin_amdgcn_readlane((int)incl, 63)) {
                uint32_t pos = incl - cnt, m = p;
                auto entry = [&](uint32_t bit, uint64_t &lk, uint32_t &uo) {
                    float s = 0.0f, e = 0.0f;
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if ((uint32_t)r == bit) s = acc[r], e = ev[r];
                    const float lo = mqf_lower(s, e), up = mqf_upper(s, e);
                    const uint32_t row = (uint32_t)(a.row_base + (t0 + (uint32_t)row_of((int)bit)) * a.row_step);
                    lk = make_key(lo == lo ? ord_f32(lo) : 0u, row);
                    uo = up == up ? ord_f32(up) : 0xffffffffu;
                };
                for (; m && pos < MQF_STAGE; m &= m - 1, ++pos) entry(__builtin_ctz(m), st.lk[sb][wave][pos], st.uo[sb][wave][pos]);
                // what the staging buffer does not hold (whole tiles pass where
                // a topic's rows lie next to each other and its queries too)
                // goes to the query's spill list, behind the buckets
                if (__builtin_expect(__ballot(m != 0) != 0, 0)) {
                    const uint64_t nb = (uint64_t)a.nq * a.nwg;
                    uint64_t at = 0;
                    if (m) at = atomicAdd(&a.cnt[nb + q], (uint32_t)__popc(m));
                    for (; m; m &= m - 1, ++at) {
                        if (at >= a.cap) break;  // (a count of cap or more tells mq1_compact)
                        const uint64_t i = nb * a.capw + (uint64_t)q * a.cap + at;
                        entry(__builtin_ctz(m), a.cand[i], a.up_out[i]);
                    }
                    // (the query is run again whatever else is kept of it: from
                    // here on nothing.  Where every row passes for 64 queries,
                    // 1M x 768, a call took 4.4 ms with all of them spilled)
                    if (at >= a.cap) stau[qlocal] = __builtin_inff();
                }
            }
        }
    }
    if constexpr (THR) {
        __syncthreads();
        if (!loader) {
            if (mine) mqf_flush<QB>(a, qb, wg, st, (int)((mine - 1) & 1), wave - LOADERS, lane, blen, bovf);
            const uint32_t ql = (uint32_t)(wave - LOADERS) * 64 + lane, qq = qb * QB + ql;
            if (qq < a.nq) a.cnt[(uint64_t)qq * a.nwg + wg] = bovf ? 0xffffffffu : blen;
        }
    }
}

// One wave per query: its bf16 rounding, zero-padded to whole chunks, and the
// constants of its bounds.  ratio: the largest |x - bf16(x)| / |x| of a row.
__global__ __launch_bounds__(64) void mqf_prep(const float *q, uint32_t dim, const uint32_t *ratio_bits, int l2,
                                               unsigned char *qbf, uint64_t qstride, MqfQuery *qk, uint32_t *cnt,
                                               uint32_t cnt_value, uint32_t *spill_n) {
    const int lane = threadIdx.x;
    const float *x = q + (uint64_t)blockIdx.x * dim;
    __bf16 *out = (__bf16 *)(qbf + (uint64_t)blockIdx.x * qstride);
    double s = 0.0, res = 0.0;
    for (uint32_t i = lane; i < qstride / 2; i += 64) {
        // (piece j of a chunk holds its elements 4 j .. + 3 and 64 + 4 j .. + 3)
        const uint32_t j = i % MQF_DIMS / 8, e = i % 8, d0 = i / MQF_DIMS * MQF_DIMS + 4 * j + (e < 4 ? e : e + 60);
        const float v = d0 < dim ? x[d0] : 0.0f;
        const __bf16 b = (__bf16)v;
        out[i] = b;
        const double d = (double)v - (double)(float)b;
        s = fma((double)v, (double)v, s);
        res = fma(d, d, res);
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        s += __shfl_xor(s, o);
        res += __shfl_xor(res, o);
    }
    if (lane != 0) return;
    const double u = 0x1p-24, up = 1.0 + 0x1p-10;
    const double qn = sqrt(s) * (1.0 + 0x1p-20), qr = sqrt(res) * (1.0 + 0x1p-20);
    const double rx = (double)__uint_as_float(*ratio_bits);
    // dot: the roundings (|x| rx |q| + |x| |q - bf16 q| + their product), the
    // f32 sums of both sides, and what flushed subnormals can take away
    const double tiny = dim * 0x1p-126;
    const double dot = rx * qn + qr + rx * qr + 4.0 * (dim + 4) * u * qn + tiny;
    MqfQuery k;
    if (l2) {  // twice the dot's, and 4 (dim + 4) u (|x| + |q|)^2 for the sums and norms
        const double r = 4.0 * (dim + 4) * u;
        k.alpha = (float)((2.0 * dot + 2.0 * r * qn) * up);
        k.beta = (float)((r * qn * qn + 2.0 * tiny * (1.0 + qn)) * up);
        k.gamma = (float)(r * up);
    } else {
        k.alpha = (float)(dot * up);
        k.beta = (float)(tiny * (1.0 + qn) * up);
        k.gamma = 0.0f;
    }
    if (!(qn < 0x1p60)) k.alpha = __builtin_inff();  // (products or sums could leave the range of f32)
    k.qsq = (float)s;
    qk[blockIdx.x] = k;
    cnt[blockIdx.x] = cnt_value;
    spill_n[blockIdx.x] = 0;
}

// ------------------------------------------------------- fp32 products ----
// The same prefilter with fp32 products (v_mfma_f32_32x32x2f32), for queries
// whose kept rows overflowed under the bf16 bounds: where the rows have a
// large part in common (a mean ten times the spread), 2 x 0.0035 |x| |q| keeps
// every row, and the rounding of the f32 sums, which is all that separates
// these scores from the single-query scan's, still tells them apart.
// 1M x 768, 256 queries: 3.4 ms, against 34 for slot scans of the rows and 125
// for one fused scan per query.
//
// The block's 32 queries stay in LDS, each wave streams 64 rows.  Lane l =
// 32h + c supplies, over the four matrix steps of chunk t, elements 8t + 4h ..
// 8t + 4h + 3 of row c (A) and of query c (B), one 16-byte load each, so both
// operands pair the same elements.  A score differs from the single-query
// scan's by at most E = slack / 2 (mqx_qconst).
//
// Passes: dense (tau null: every key of logical row i at cand[q][i]), and the
// ids of the rows whose score reaches tau's score minus slack[q].  That keeps
// every row the exact scan can rank: a row in the exact top-kk has a
// single-query score >= the kk-th best single-query score >= tau's score - E,
// hence a score here >= tau's score - 2E.
template <int CHUNKS>
__global__ __launch_bounds__(MQ_WAVES * 64) void mqx_scan(MqxArgs a) {
    constexpr int G = CHUNKS < 4 ? CHUNKS : 4;
    __shared__ float4 qlds[CHUNKS][64];
    __shared__ float qts[MQ_QB];
    __shared__ float qn2[MQ_QB];
    __shared__ float rn2[MQ_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = lane >> 5, c = lane & 31;
    const uint32_t b = blockIdx.x, xcd = b & 7u, slot = b >> 3;
    const uint32_t qb = slot % a.qblocks, grp = slot / a.qblocks;
    const uint64_t tstride = 8ull * a.groups;
    uint64_t tile = xcd + 8ull * grp;
    if (tile * MQ_ROWS >= a.n) return;
    {
        uint32_t q = qb * MQ_QB + c;
        if (q >= a.nq) q = a.nq - 1;
        const float *src = a.q + (uint64_t)q * a.dim;
        for (int t = wave; t < CHUNKS; t += MQ_WAVES)
            __builtin_amdgcn_global_load_lds((glb_void *)(src + 8 * t + 4 * h), (lds_void *)&qlds[t][0], 16, 0, 0);
    }
    if (threadIdx.x < MQ_QB) {
        uint32_t q = qb * MQ_QB + threadIdx.x;
        if (q >= a.nq) q = a.nq - 1;
        const uint64_t t = a.tau ? a.tau[q] : 0ull;
        // tau's score minus the slack, rounded down
        qts[threadIdx.x] = t ? mqx_below((float)((double)f32_from_ord((uint32_t)(t >> 32)) - (double)a.slack[q]))
                             : -__builtin_inff();
        qn2[threadIdx.x] = a.l2 ? a.qsq[q] : 0.0f;
    }
    auto row_sq = [&](uint64_t t) {
        uint64_t li = t * MQ_ROWS + (uint64_t)wave * 64 + lane;
        if (li >= a.n) li = a.n - 1;
        return a.rsq[li * a.row_step];
    };
    float rsq_next = a.l2 ? row_sq(tile) : 0.0f;
    auto row_ptrs = [&](uint64_t t, const float4 *(&ap)[2]) {
        const uint64_t w0 = t * MQ_ROWS + (uint64_t)wave * 64;
#pragma unroll
        for (int fr = 0; fr < 2; ++fr) {
            uint64_t li = w0 + fr * 32 + c;
            if (li >= a.n) li = a.n - 1;  // rows past the end load a valid row; their results are dropped
            ap[fr] = (const float4 *)(a.rows + li * a.row_step * a.dim + 4 * h);
        }
    };
    const float4 *ap[2];
    row_ptrs(tile, ap);
    float4 ring[2][G][2];
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
        for (int fr = 0; fr < 2; ++fr) ring[0][j][fr] = ap[fr][2 * j];
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    const uint32_t q = qb * MQ_QB + c;
    const bool qok = q < a.nq;
    const uint32_t qq = qok ? q : a.nq - 1;
    for (;;) {
        const uint64_t ntile = tile + tstride;
        const bool more = ntile * MQ_ROWS < a.n;
        const float4 *np[2];
        row_ptrs(more ? ntile : tile, np);
        v16f acc[2] = {v16f{}, v16f{}};
#pragma unroll
        for (int t = 0; t < CHUNKS; ++t) {
            const int gp = (t / G) & 1, j = t % G;
            if (j == 0) {
                const int nt = t + G;
#pragma unroll
                for (int jj = 0; jj < G; ++jj)
#pragma unroll
                    for (int fr = 0; fr < 2; ++fr) {
                        if (nt < CHUNKS) ring[gp ^ 1][jj][fr] = ap[fr][2 * (nt + jj)];
                        else if (more) ring[gp ^ 1][jj][fr] = np[fr][2 * (nt - CHUNKS + jj)];
                    }
            }
            const float4 B = qlds[t][lane];
            const float bv[4] = {B.x, B.y, B.z, B.w};
#pragma unroll
            for (int fr = 0; fr < 2; ++fr) {
                const float4 A = ring[gp][j][fr];
                const float av[4] = {A.x, A.y, A.z, A.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[fr] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[e], bv[e], acc[fr], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr ((CHUNKS / G) & 1) {
#pragma unroll
            for (int j = 0; j < G; ++j)
#pragma unroll
                for (int fr = 0; fr < 2; ++fr) ring[0][j][fr] = ring[1][j][fr];
        }
        // l2: the score from the dot and the squared norms (this wave's 64
        // rows' norms through wave-private LDS)
        if (a.l2) {
            rn2[wave][lane] = rsq_next;
            if (more) rsq_next = row_sq(ntile);
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            const float qs2 = qn2[c];
#pragma unroll
            for (int fr = 0; fr < 2; ++fr)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float x2 = rn2[wave][fr * 32 + 8 * (r >> 2) + 4 * h + (r & 3)];
                    acc[fr][r] = 2.0f * acc[fr][r] - x2 - qs2;
                }
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
        const uint64_t w0 = tile * MQ_ROWS + (uint64_t)wave * 64;
        const bool full = w0 + 64 <= a.n;
        if (!a.tau) {
            uint64_t *out = a.cand + (uint64_t)qq * a.cap;
#pragma unroll
            for (int fr = 0; fr < 2; ++fr)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint64_t li = w0 + fr * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (qok && (full || li < a.n)) out[li] = make_key(ord_f32(acc[fr][r]), (uint32_t)(li * a.row_step));
                }
        } else {
            const float ts = qts[c];
            uint32_t pass = 0;
#pragma unroll
            for (int fr = 0; fr < 2; ++fr)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint64_t li = w0 + fr * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                    // a NaN score passes: the exact scan ranks it as it ranks any key
                    if (qok && (full || li < a.n) && !(acc[fr][r] < ts)) pass |= 1u << (fr * 16 + r);
                }
            if (__ballot(pass != 0)) {
                const uint32_t mine = __popc(pass);
                const uint32_t other = __shfl_xor(mine, 32);
                uint32_t base = 0;
                if (h == 0 && mine + other) base = atomicAdd(&a.cnt[qq], mine + other);
                base = __shfl(base, c);
                if (pass) {
                    uint32_t *ro = a.rows_out + (uint64_t)qq * a.cap;
                    uint64_t pos = (uint64_t)base + (h ? other : 0u);
#pragma unroll
                    for (int fr = 0; fr < 2; ++fr)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            if (pass & (1u << (fr * 16 + r))) {
                                const uint64_t li = w0 + fr * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                                if (pos < a.cap) ro[pos] = (uint32_t)(li * a.row_step);
                                ++pos;
                            }
                }
            }
        }
        if (!more) break;
        ap[0] = np[0];
        ap[1] = np[1];
        tile = ntile;
    }
}

// One wave per query: |q|^2 and the slack 2E.  u = 2^-24: E is 3 (dim + 2) u
// |x|max |q| for dot products, 4 (dim + 4) u (|x|max + |q|)^2 under l2, and
// room for the subnormal products a matrix core may flush.
__global__ __launch_bounds__(64) void mqx_qconst(const float *q, uint32_t dim, const uint32_t *max_bits, int l2,
                                                 float *qsq, float *slack) {
    const int lane = threadIdx.x;
    const float *x = q + (uint64_t)blockIdx.x * dim;
    double s = 0.0;
    for (uint32_t i = lane; i < dim; i += 64) s = fma((double)x[i], (double)x[i], s);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
    if (lane == 0) {
        const double u = 0x1p-24;
        const double xn = sqrt((double)__uint_as_float(*max_bits)) * (1.0 + 0x1p-20);
        const double qn = sqrt(s) * (1.0 + 0x1p-20);
        const double e = l2 ? 4.0 * (dim + 4) * u * (xn + qn) * (xn + qn) : 3.0 * (dim + 2) * u * xn * qn;
        qsq[blockIdx.x] = (float)s;
        slack[blockIdx.x] = (float)((2.0 * e + dim * 0x1p-126) * (1.0 + 0x1p-10));
    }
}

// One wave per row: f64 sum of squares rounded to f32, and over the rows the
// largest ratio |x - bf16(x)| / |x| (float bits, rounded up, at most 2^-8: a
// larger ratio comes from subnormal elements, which the bounds' absolute terms
// cover) in max_bits[0] and the largest sum (rounded up) in max_bits[1].
// Rows of zeros have none, and rows out of range have no bounds at all
// (mqf_norm).
// 1M x 768: 0.59 ms (5.2 TB/s); with an atomic per wave instead of one per
// workgroup of many rows 3.0 ms.
__global__ __launch_bounds__(256) void row_sqnorms(const float *rows, uint64_t n, uint32_t dim, float *rsq,
                                                   uint32_t *max_bits) {
    const int lane = threadIdx.x & 63;
    const uint64_t nw = (uint64_t)gridDim.x * 4;
    __shared__ uint32_t wmx[4], wsq[4];
    double mx = 0.0;  // largest squared ratio
    uint32_t sq = 0;  // largest sum's bits (the next float up: it may have been rounded down)
    for (uint64_t r = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < n; r += nw) {
        const float *x = rows + r * dim;
        double s = 0.0, res = 0.0;
        for (uint32_t i0 = 0; i0 < dim; i0 += 256) {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t i = i0 + 64 * j + lane;
                v[j] = i < dim ? x[i] : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float d = v[j] - (float)(__bf16)v[j];  // (exact)
                s = fma((double)v[j], (double)v[j], s);
                res = fma((double)d, (double)d, res);
            }
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            s += __shfl_xor(s, o);
            res += __shfl_xor(res, o);
        }
        if (lane == 0) {
            rsq[r] = (float)s;
            const uint32_t b = __float_as_uint((float)s);
            sq = max(sq, b < 0x7f800000u ? b + 1 : b);  // (inf and NaN stay)
            const double ratio = s > 0.0 && s < 0x1p122 ? res / s : 0.0;
            mx = ratio > mx ? ratio : mx;
        }
    }
    if (lane == 0) {
        const double ratio = sqrt(mx) * (1.0 + 0x1p-20);
        wsq[threadIdx.x >> 6] = sq;
        wmx[threadIdx.x >> 6] = __float_as_uint(ratio < 0x1p-8 ? (float)ratio : 0x1p-8f);
    }
    __syncthreads();
    if (threadIdx.x == 0) {  // (per workgroup: atomics serialize)
        uint32_t b = wmx[0], m = wsq[0];
        for (int i = 1; i < 4; ++i) {
            b = wmx[i] > b ? wmx[i] : b;
            m = wsq[i] > m ? wsq[i] : m;
        }
        // (the maxima only rise: what a plain read already passes need not be
        // raised, and few workgroups hold a new maximum)
        if (b > __hip_atomic_load(max_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(max_bits, b);
        if (m > __hip_atomic_load(max_bits + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(max_bits + 1, m);
    }
}

}  // namespace

hipError_t launch_row_sqnorms(const float *rows, uint64_t n, uint32_t dim, float *rsq, uint32_t *max_bits,
                              hipStream_t s) {
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n + 3) / 4;
    if (blocks > 2048) blocks = 2048;  // eight workgroups per CU
    hipLaunchKernelGGL(row_sqnorms, dim3((uint32_t)blocks), dim3(256), 0, s, rows, n, dim, rsq, max_bits);
    return hipGetLastError();
}

bool mqf_supported(uint32_t dim) { return dim >= 4 && dim <= 1024; }
uint32_t mqf_block(uint32_t dim) { return dim <= 768 ? 256u : 128u; }
uint64_t mqf_qstride(uint32_t dim) { return (uint64_t)((dim + MQF_DIMS - 1) / MQF_DIMS) * MQF_DIMS * 2; }

hipError_t launch_mqf_prep(const float *q, uint32_t nq, uint32_t dim, const uint32_t *ratio_bits, bool l2,
                           unsigned char *qbf, MqfQuery *qk, uint32_t *cnt, uint32_t cnt_value, uint32_t *spill_n,
                           hipStream_t s) {
    if (nq == 0) return hipSuccess;
    if (!mqf_supported(dim)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(mqf_prep, dim3(nq), dim3(64), 0, s, q, dim, ratio_bits, l2 ? 1 : 0, qbf, mqf_qstride(dim), qk,
                       cnt, cnt_value, spill_n);
    return hipGetLastError();
}

template <int CH, int WAVES> static hipError_t mqf_go(const MqfArgs &a, hipStream_t s) {
    const uint64_t blocks = (uint64_t)a.nwg * a.qblocks;
    if (blocks == 0 || blocks > 0x7fffffffull || a.nwg % 8 != 0 || (uint64_t)a.qblocks * WAVES * 32 < a.nq)
        return hipErrorInvalidValue;
    const dim3 g((uint32_t)blocks), wg(WAVES * 64);
    if (a.tau) hipLaunchKernelGGL((mqf_scan<CH, WAVES, true>), g, wg, 0, s, a);
    else hipLaunchKernelGGL((mqf_scan<CH, WAVES, false>), g, wg, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_mqf_scan(const MqfArgs &a, hipStream_t s) {
    if (a.n == 0 || a.nq == 0) return hipSuccess;
    if (a.n > (1ull << 32) || !mqf_supported(a.dim) || !a.cand || !a.rsq || a.qstride != mqf_qstride(a.dim) ||
        (a.tau && (!a.up_out || !a.cnt || a.capw == 0)))
        return hipErrorInvalidValue;
    switch ((a.dim + MQF_DIMS - 1) / MQF_DIMS) {
    case 1: return mqf_go<1, 8>(a, s);
    case 2: return mqf_go<2, 8>(a, s);
    case 3: return mqf_go<3, 8>(a, s);
    case 4: return mqf_go<4, 8>(a, s);
    case 5: return mqf_go<5, 8>(a, s);
    case 6: return mqf_go<6, 8>(a, s);
    case 7: return mqf_go<7, 4>(a, s);
    case 8: return mqf_go<8, 4>(a, s);
    default: return hipErrorInvalidValue;
    }
}

bool mqx_supported(uint32_t dim) {
    switch (dim) {
    case 32: case 64: case 96: case 128: case 192: case 256: case 384: case 512: case 768: case 1024: return true;
    default: return false;
    }
}

hipError_t launch_mqx_qconst(const float *q, uint32_t nq, uint32_t dim, const uint32_t *max_bits, bool l2, float *qsq,
                             float *slack, hipStream_t s) {
    if (nq == 0) return hipSuccess;
    hipLaunchKernelGGL(mqx_qconst, dim3(nq), dim3(64), 0, s, q, dim, max_bits, l2 ? 1 : 0, qsq, slack);
    return hipGetLastError();
}

hipError_t launch_mqx_scan(const MqxArgs &a, hipStream_t s) {
    if (a.n == 0 || a.nq == 0) return hipSuccess;
    if (!mqx_supported(a.dim) || a.qblocks == 0 || a.groups == 0 || (uint64_t)a.qblocks * MQ_QB < a.nq || !a.rsq ||
        !a.qsq || (a.tau ? !a.rows_out || !a.cnt || !a.slack : !a.cand || a.cap < a.n))
        return hipErrorInvalidValue;
    const uint64_t blocks = 8ull * a.groups * a.qblocks;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    const dim3 g((uint32_t)blocks), wg(MQ_WAVES * 64);
    switch (a.dim) {
    case 32: hipLaunchKernelGGL(mqx_scan<4>, g, wg, 0, s, a); break;
    case 64: hipLaunchKernelGGL(mqx_scan<8>, g, wg, 0, s, a); break;
    case 96: hipLaunchKernelGGL(mqx_scan<12>, g, wg, 0, s, a); break;
    case 128: hipLaunchKernelGGL(mqx_scan<16>, g, wg, 0, s, a); break;
    case 192: hipLaunchKernelGGL(mqx_scan<24>, g, wg, 0, s, a); break;
    case 256: hipLaunchKernelGGL(mqx_scan<32>, g, wg, 0, s, a); break;
    case 384: hipLaunchKernelGGL(mqx_scan<48>, g, wg, 0, s, a); break;
    case 512: hipLaunchKernelGGL(mqx_scan<64>, g, wg, 0, s, a); break;
    case 768: hipLaunchKernelGGL(mqx_scan<96>, g, wg, 0, s, a); break;
    case 1024: hipLaunchKernelGGL(mqx_scan<128>, g, wg, 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace bvk
