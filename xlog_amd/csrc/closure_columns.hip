// Linear closure over a dense domain, a block of target columns at a time.
//
// The program  H(X,Z) :- E(X,Z).  H(X,Z) :- F(X,Y), H(Y,Z)  never mixes the
// columns of H's bit matrix: bit (x, z) of the next layer depends on bits
// (y, z) of this one.  So a workgroup takes 32 target columns (one u32 per
// row), keeps that slice of H for every row in LDS, and runs all iterations of
// the fixpoint there:
//   new[x] = (OR over y in F[x] of H[y]) & ~H[x],   H[x] |= new[x]
// with the new words held in registers until every row has been read (the
// layers are those of the semi-naive loop: H grows by whole layers, so the OR
// over H adds nothing to the OR over the last layer that H does not hold).
// Nothing but F's adjacency is read from memory while it iterates, and the
// matrix is written once, at the end; per iteration each workgroup adds its
// count of new bits to the iteration's total.  The row-gather product of
// chain_bitmap.hip reads and writes three matrices per iteration instead
// (32,768 vertices, 98,304 edges: 24 launches of 82 us = 1.96 ms; this takes
// 0.66 ms and 0.05 for the transposition, 2,000 vertices 0.41 -> 0.22 ms whole).
//
// What bounds it is LDS and latency: a pull iteration reads one random 4-byte
// word per edge.  Rows are renumbered by descending out-degree and stored in
// slices of 64 (one wave wide, four ids per lane and load, padded to the
// slice's largest degree), so the lanes of a wave have equally many edges to
// read; a slice whose largest row is far above its average (hubs) is read a
// row at a time by the whole wave instead.  An iteration that starts from few
// changed rows (the first ones, and the tail) pushes instead: the changed rows
// and their new bits are in a queue, and each goes to the rows that have an
// edge to it.
#include "internal.hpp"

#include <algorithm>

namespace xh {

namespace {

constexpr int CL_TB = 1024, CL_WAVES = CL_TB / WAVE;
// rows per thread of the largest instance: CL_MAX_RPT * 1024 four-byte slots
// and the zero slot are 152 KB of the 160 KB of LDS
constexpr int CL_MAX_RPT = 38;
constexpr uint32_t CL_HEAVY = 1u << 31;  // slice read a row at a time
constexpr uint32_t CL_QUAD = 4;          // ids per lane and load: a slice's depth counts quads
constexpr int CL_DEG_BINS = 1024;

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o, WAVE));
    return v;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += (uint32_t)__shfl_xor((int)v, o, WAVE);
    return v;
}
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v |= (uint32_t)__shfl_xor((int)v, o, WAVE);
    return v;
}

// the bin of a row's degree: large degrees first
__device__ __forceinline__ uint32_t bin_of(const uint64_t *__restrict__ row_ptr, uint32_t x) {
    const uint64_t deg = row_ptr[x + 1] - row_ptr[x];
    return (uint32_t)CL_DEG_BINS - 1 - (uint32_t)min(deg, (uint64_t)CL_DEG_BINS - 1);
}

// Position of each lane's row among the rows of its degree bin: one atomic
// per distinct bin of the wave (most rows share a few bins).
__device__ __forceinline__ uint32_t bin_take(uint32_t *bins, uint32_t bin, bool valid, int lane) {
    uint32_t pos = 0;
    uint64_t todo = __ballot(valid);
    while (todo) {
        const int l = __ffsll((unsigned long long)todo) - 1;
        const uint32_t b = (uint32_t)__shfl((int)bin, l, WAVE);
        const uint64_t m = __ballot(valid && bin == b);
        uint32_t base = 0;
        if (lane == l) base = atomicAdd(&bins[b], (uint32_t)__popcll(m));
        base = (uint32_t)__shfl((int)base, l, WAVE);
        if (valid && bin == b) pos = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        todo &= ~m;
    }
    return pos;
}

// Rows per out-degree bin.
__global__ __launch_bounds__(256) void k_cl_bins(const uint64_t *__restrict__ row_ptr, uint32_t domain,
                                                 uint32_t *bins) {
    __shared__ uint32_t s_bin[CL_DEG_BINS];
    const int lane = threadIdx.x & (WAVE - 1);
    for (int i = threadIdx.x; i < CL_DEG_BINS; i += 256) s_bin[i] = 0;
    __syncthreads();
    const uint32_t t = blockIdx.x * 256 + threadIdx.x, stride = gridDim.x * 256;
    for (uint32_t b = t - lane; b < domain; b += stride) {
        const uint32_t x = b + lane;
        const bool valid = x < domain;
        bin_take(s_bin, valid ? bin_of(row_ptr, x) : 0u, valid, lane);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < CL_DEG_BINS; i += 256)
        if (s_bin[i]) atomicAdd(&bins[i], s_bin[i]);
}

// Edges per target (in_deg, by internal row) and each edge's rank among its
// target's (any order), and the same of the seed pairs when they are not the
// edges.  One atomic per edge, which also spares the lists' fill its own, or one
// for the edges of a wave to a hub target: hubs' atomics wait for each other
// (30,000 vertices, 90,000 edges, 55 % of them to one target: the closure 858 us
// with an atomic each, 719 so, by row gathers 673).
__device__ __forceinline__ uint32_t take_rank(uint32_t *count, uint32_t z, bool valid, int lane) {
    constexpr int TRIES = 4, MANY = 8;  // targets looked at, edges of the wave that make one a hub
    uint32_t rank = 0;
    uint64_t todo = __ballot(valid);
    for (int r = 0; r < TRIES && todo; ++r) {
        const uint32_t hub = (uint32_t)__builtin_amdgcn_readlane((int)z, __ffsll((unsigned long long)todo) - 1);
        const uint64_t m = __ballot(valid && z == hub);
        todo &= ~m;
        if (__popcll(m) < MANY) continue;  // wave-uniform
        uint32_t base = 0;
        const int first = __ffsll((unsigned long long)m) - 1;
        if (lane == first) base = atomicAdd(&count[hub], (uint32_t)__popcll(m));
        base = (uint32_t)__builtin_amdgcn_readlane((int)base, first);
        if ((m >> lane) & 1ull) {
            rank = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            valid = false;
        }
    }
    if (valid) rank = atomicAdd(&count[z], 1u);
    return rank;
}
__global__ __launch_bounds__(256) void k_cl_in_degrees(const uint32_t *__restrict__ adj, uint64_t m,
                                                       const uint64_t *__restrict__ seed, uint64_t n_seed,
                                                       const uint16_t *__restrict__ inv, uint32_t *in_deg,
                                                       uint32_t *seed_deg, uint32_t *__restrict__ rank,
                                                       uint32_t *__restrict__ seed_rank) {
    const int lane = threadIdx.x & (WAVE - 1);
    const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x, stride = (uint64_t)gridDim.x * 256;
    for (uint64_t b = t - lane; b < m; b += stride) {
        const uint64_t e = b + lane;
        const uint32_t r = take_rank(in_deg, e < m ? inv[adj[e]] : 0u, e < m, lane);
        if (e < m) rank[e] = r;
    }
    if (!seed) return;
    for (uint64_t b = t - lane; b < n_seed; b += stride) {
        const uint64_t e = b + lane;
        const uint32_t r = take_rank(seed_deg, e < n_seed ? inv[(uint32_t)seed[e]] : 0u, e < n_seed, lane);
        if (e < n_seed) seed_rank[e] = r;
    }
}

// Rows in descending order of degree (perm: internal row -> vertex, inv: its
// inverse; the order inside a bin is any).
__global__ __launch_bounds__(CL_TB) void k_cl_place(const uint64_t *__restrict__ row_ptr, uint32_t domain,
                                                    const uint32_t *__restrict__ bins, uint32_t *cursor,
                                                    uint32_t *__restrict__ perm, uint16_t *__restrict__ inv) {
    __shared__ uint32_t s_bin[CL_DEG_BINS], s_own[CL_DEG_BINS];
    __shared__ uint32_t s_part[CL_WAVES];
    static_assert(CL_DEG_BINS == CL_TB, "one bin per thread");
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid >> 6;
    const uint32_t v = bins[tid];
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)inc, o, WAVE);
        if (lane >= o) inc += t;
    }
    if (lane == WAVE - 1) s_part[wave] = inc;
    __syncthreads();
    uint32_t pre = 0;
    for (int w = 0; w < wave; ++w) pre += s_part[w];
    s_own[tid] = 0;
    __syncthreads();
    // the block's rows are placed in its own bins first, then each bin takes its place with one global atomic
    const uint32_t x = blockIdx.x * CL_TB + tid;
    const bool valid = x < domain;
    const uint32_t bin = valid ? bin_of(row_ptr, x) : 0u;
    const uint32_t own = bin_take(s_own, bin, valid, lane);
    __syncthreads();
    s_bin[tid] = pre + inc - v + (s_own[tid] ? atomicAdd(&cursor[tid], s_own[tid]) : 0u);
    __syncthreads();
    const uint32_t pos = s_bin[bin] + own;
    if (valid) {
        perm[pos] = x;
        inv[x] = (uint16_t)pos;
    }
}

// A wave per slice: its depth in quads (CL_HEAVY when reading its rows one by
// one is cheaper), its place in sell (any order) and its entries (internal row
// ids; `zero`, the slot that stays 0, past a row's edges).  Then the internal
// ids of all edges in CSR order (heavy slices), and, grouped by target, the
// internal sources of every edge and seed pair.
struct ClFill {
    const uint64_t *row_ptr;
    const uint32_t *adj;
    uint64_t m;
    uint32_t domain, slices, zero;
    const uint32_t *perm;
    const uint16_t *inv;
    uint32_t *slice_off, *slice_m, *sell_next;
    uint64_t *sell;
    uint16_t *col;
    const uint64_t *edge;      // the pairs of the CSR, in its order
    const uint32_t *in_ptr;
    const uint32_t *rank;
    uint16_t *in_src;
    const uint64_t *seed;      // null: the seed pairs are the edges
    uint64_t n_seed;
    const uint32_t *seed_ptr;
    const uint32_t *seed_rank;
    uint16_t *seed_src;
};
__global__ __launch_bounds__(256) void k_cl_fill(ClFill a) {
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    const uint32_t gwave = (blockIdx.x * 256 + threadIdx.x) >> 6, nwaves = gridDim.x * (256 / WAVE);
    for (uint32_t s = gwave; s < a.slices; s += nwaves) {
        const uint32_t i = s * WAVE + lane;
        uint64_t st = 0;
        uint32_t d = 0;
        if (i < a.domain) {
            const uint32_t x = a.perm[i];
            st = a.row_ptr[x];
            d = (uint32_t)(a.row_ptr[x + 1] - st);
        }
        const uint32_t deepest = wave_max(d), steps = wave_sum((d + WAVE - 1) / WAVE);
        // LDS reads of the wave: `deepest` column-major; row by row one per 64
        // edges and a reduction worth about eight more for each of the 64 rows
        const bool heavy = deepest > steps + 8 * WAVE;
        const uint32_t quads = heavy ? 0u : (deepest + CL_QUAD - 1) / CL_QUAD;
        uint32_t off = 0;
        if (lane == 0 && quads) off = atomicAdd(a.sell_next, quads * WAVE);
        off = (uint32_t)__shfl((int)off, 0, WAVE);
        if (lane == 0) {
            a.slice_m[s] = heavy ? CL_HEAVY : quads;
            a.slice_off[s] = off;
        }
        for (uint32_t k = 0; k < quads; ++k) {
            uint64_t w = 0;
#pragma unroll
            for (uint32_t q = 0; q < CL_QUAD; ++q) {
                const uint32_t e = k * CL_QUAD + q;
                w |= (uint64_t)(e < d ? a.inv[a.adj[st + e]] : (uint16_t)a.zero) << (16 * q);
            }
            a.sell[(uint64_t)off + k * WAVE + lane] = w;
        }
    }
    const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x, stride = (uint64_t)gridDim.x * 256;
    for (uint64_t e = t; e < a.m; e += stride) {
        const uint64_t p = a.edge[e];
        const uint16_t z = a.inv[(uint32_t)p];
        a.col[e] = z;
        a.in_src[a.in_ptr[z] + a.rank[e]] = a.inv[p >> 32];
    }
    if (a.seed)
        for (uint64_t e = t; e < a.n_seed; e += stride) {
            const uint64_t p = a.seed[e];
            const uint16_t z = a.inv[(uint32_t)p];
            a.seed_src[a.seed_ptr[z] + a.seed_rank[e]] = a.inv[p >> 32];
        }
}

struct ClArgs {
    const uint64_t *sell;
    const uint16_t *col;
    const uint32_t *slice_off, *slice_m;
    const uint64_t *row_ptr;
    const uint32_t *perm;
    const uint16_t *inv;
    const uint32_t *in_ptr;       // by internal row: where its sources start in in_src (in_ptr[domain]: their number)
    const uint16_t *in_src;
    const uint32_t *seed_ptr;     // the same of the seed pairs
    const uint16_t *seed_src;
    uint32_t domain, slices;
    uint64_t max_iter;
    unsigned long long *counts;   // [0]: largest number of non-empty layers, [1 + i]: new bits of iteration i
    uint32_t *S;                  // cols x domain, rows in internal order
};

// The OR over the edges of each of a slice's rows (the lanes' own results): the
// wave reads one row at a time, a lane per edge.
__device__ __forceinline__ uint32_t heavy_slice(const ClArgs &a, const uint32_t *s_r, uint32_t row0, uint32_t lane) {
    uint64_t st = 0;
    uint32_t d = 0, acc = 0;
    if (row0 + lane < a.domain) {
        const uint32_t x = a.perm[row0 + lane];
        st = a.row_ptr[x];
        d = (uint32_t)(a.row_ptr[x + 1] - st);
    }
    for (int r = 0; r < WAVE; ++r) {
        const uint64_t rs = (uint64_t)__shfl((unsigned long long)st, r, WAVE);
        const uint32_t rd = (uint32_t)__shfl((int)d, r, WAVE);
        uint32_t v = 0;
        for (uint32_t e = lane; e < rd; e += WAVE) v |= s_r[a.col[rs + e]];
        v = wave_or(v);
        if (lane == (uint32_t)r) acc = v;
    }
    return acc;
}

// One block of 32 columns to its fixpoint.  Thread t owns internal rows
// t, t + 1024, ... (RPT of them), so slice i * 16 + wave belongs to one wave.
template <int RPT>
__global__ __launch_bounds__(CL_TB) void k_cl_columns(ClArgs a) {
    constexpr uint32_t ROWS = RPT * CL_TB;
    constexpr int GRP = RPT < 4 ? RPT : (RPT % 4 == 0 ? 4 : 2);  // slices whose loads are in flight together
    constexpr int QT = RPT >= 4 ? (RPT <= 32 ? 4 : 1) : 0;       // queue entries per thread (0: pulls only)
    constexpr uint32_t QCAP = QT * CL_TB;
    static_assert(RPT % GRP == 0, "whole groups");
    __shared__ uint32_t s_r[ROWS + 1];
    __shared__ uint32_t s_cnt[3], s_qn[3];
    __shared__ uint32_t s_qbits[QCAP ? QCAP : 1];
    __shared__ uint16_t s_qrow[QCAP ? QCAP : 1];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t cw = blockIdx.x;
#pragma unroll
    for (int i = 0; i < RPT; ++i) s_r[i * CL_TB + tid] = 0;
    if (tid == 0) {
        s_r[ROWS] = 0;
        s_cnt[0] = s_cnt[1] = s_cnt[2] = 0;
        s_qn[0] = s_qn[1] = s_qn[2] = 0;
    }
    // lane i keeps slice i's depth and offset (RPT <= 64)
    uint32_t my_m = 0, my_off = 0;
    if (lane < RPT && (uint32_t)(lane * CL_WAVES + wave) < a.slices) {
        my_m = a.slice_m[lane * CL_WAVES + wave];
        my_off = a.slice_off[lane * CL_WAVES + wave];
    }
    __syncthreads();
    // the seed: every source of each of the block's targets (two targets a wave)
    {
        const uint32_t z = cw * 32 + wave * 2 + (lane >> 5);
        if (z < a.domain) {
            const uint32_t y = a.inv[z], b = a.seed_ptr[y], e1 = a.seed_ptr[y + 1], bit = 1u << (z & 31u);
            for (uint32_t e = b + (lane & 31); e < e1; e += 32) {
                const uint32_t x = a.seed_src[e];
                atomicOr(&s_r[x], bit);
                const uint32_t pos = atomicAdd(&s_qn[0], 1u);
                if (pos < QCAP) {
                    s_qrow[pos] = (uint16_t)x;
                    s_qbits[pos] = bit;
                }
            }
        }
    }
    __syncthreads();
    uint64_t it = 0;
    for (; it < a.max_iter; ++it) {
        const uint32_t slot = (uint32_t)(it % 3), next = (uint32_t)((it + 1) % 3), after = (uint32_t)((it + 2) % 3);
        const uint32_t qn = s_qn[slot];  // changed (row, bits) entries, or more than the queue holds
        uint32_t cnt = 0;
        if (QT > 0 && qn <= QCAP) {
            if (qn == 0) break;  // block-uniform: nothing changed
            uint32_t d[QT ? QT : 1], b[QT ? QT : 1], n[QT ? QT : 1];
#pragma unroll
            for (int k = 0; k < QT; ++k) {
                const uint32_t e = (uint32_t)(k * CL_TB + tid), y = e < qn ? s_qrow[e] : 0u;
                d[k] = e < qn ? s_qbits[e] : 0u;
                b[k] = a.in_ptr[y];
                n[k] = e < qn ? a.in_ptr[y + 1] - b[k] : 0u;
            }
            __syncthreads();  // the queue has been read
            if (tid == 0) s_cnt[after] = s_qn[after] = 0;  // of the iteration before: every thread is past reading it
            // bits t of a changed row go to each of four rows x; the ones a row did not hold are its new bits
            auto push4 = [&](const uint32_t *x, const bool *live, uint32_t bits) {
                uint32_t t[4], total = 0, before = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) t[q] = live[q] ? bits & ~s_r[x[q]] : 0u;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (t[q]) t[q] &= ~atomicOr(&s_r[x[q]], t[q]);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint64_t bal = __ballot(t[q] != 0);
                    cnt += (uint32_t)__popc(t[q]);
                    before += __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
                    total += (uint32_t)__popcll(bal);
                }
                if (!total) return;
                uint32_t pos = 0;
                if (lane == 0) pos = atomicAdd(&s_qn[next], total);
                pos = (uint32_t)__builtin_amdgcn_readfirstlane((int)pos) + before;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (t[q]) {
                        if (pos < QCAP) {
                            s_qrow[pos] = (uint16_t)x[q];
                            s_qbits[pos] = t[q];
                        }
                        ++pos;
                    }
            };
#pragma unroll
            for (int k = 0; k < QT; ++k) {
                if ((uint32_t)(k * CL_TB + wave * WAVE) >= qn) break;  // wave-uniform: no entries
                // up to 16 sources by the entry's own lane, the rest by the whole wave
                const uint32_t own = min(n[k], 16u);
                for (uint32_t e = 0; __ballot(e < own) != 0; e += 4) {
                    uint32_t x[4];
                    bool live[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        live[q] = e + q < own;
                        x[q] = live[q] ? a.in_src[b[k] + e + q] : 0u;
                    }
                    push4(x, live, d[k]);
                }
                for (uint64_t todo = __ballot(n[k] > 16); todo; todo &= todo - 1) {
                    const int l = __ffsll((unsigned long long)todo) - 1;
                    const uint32_t rb = (uint32_t)__builtin_amdgcn_readlane((int)b[k], l);
                    const uint32_t rn = (uint32_t)__builtin_amdgcn_readlane((int)n[k], l);
                    const uint32_t rd = (uint32_t)__builtin_amdgcn_readlane((int)d[k], l);
                    for (uint32_t e0 = 16; e0 < rn; e0 += 4 * WAVE) {
                        uint32_t x[4];
                        bool live[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            live[q] = e0 + q * WAVE + lane < rn;
                            x[q] = live[q] ? a.in_src[rb + e0 + q * WAVE + lane] : 0u;
                        }
                        push4(x, live, rd);
                    }
                }
            }
            cnt = wave_sum(cnt);
            if (lane == 0 && cnt) atomicAdd(&s_cnt[slot], cnt);
            __syncthreads();
            const uint32_t total = s_cnt[slot];
            if (total == 0) break;  // block-uniform
            if (tid == 0) atomicAdd(&a.counts[1 + it], (unsigned long long)total);
            continue;
        }
        uint32_t nw[RPT];
        uint32_t changed = 0;  // rows of the wave with new bits
        uint32_t ln = (uint32_t)lane;
        // (keeps the slices' addresses from being hoisted out of the iterations into registers that are not there)
        asm volatile("" : "+v"(my_m), "+v"(my_off), "+v"(ln));
        constexpr uint64_t NONE = ROWS * 0x0001000100010001ull;  // four times the slot that stays 0
        // quad k of slice i, its last one past its end (an OR takes it twice), NONE for an empty or heavy slice
        auto load_quad = [&](int i, uint32_t k) -> uint64_t {
            const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)my_m, i) & ~CL_HEAVY;
            const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)my_off, i) + ln;
            const uint64_t v = a.sell[p + (m ? min(k, m - 1) : 0u) * WAVE];
            return m ? v : NONE;
        };
        auto read_quad = [&](uint64_t w) {
            return s_r[w & 0xFFFFu] | s_r[(w >> 16) & 0xFFFFu] | s_r[(w >> 32) & 0xFFFFu] | s_r[w >> 48];
        };
        uint64_t w[GRP], wn[GRP];
#pragma unroll
        for (int j = 0; j < GRP; ++j) w[j] = load_quad(j, 0);
#pragma unroll
        for (int i0 = 0; i0 < RPT; i0 += GRP) {
            // the next group's first ids load under this group's reads
            if (i0 + GRP < RPT)
#pragma unroll
                for (int j = 0; j < GRP; ++j) wn[j] = load_quad(i0 + GRP + j, 0);
            uint32_t acc[GRP], depth = 0;
#pragma unroll
            for (int j = 0; j < GRP; ++j) acc[j] = read_quad(w[j]);
#pragma unroll
            for (int j = 0; j < GRP; ++j) depth = max(depth, (uint32_t)__builtin_amdgcn_readlane((int)my_m, i0 + j));
            if (depth > 1) {  // wave-uniform
                for (uint32_t k = 1; k < (depth & ~CL_HEAVY); ++k) {
                    uint64_t more[GRP];
#pragma unroll
                    for (int j = 0; j < GRP; ++j) more[j] = load_quad(i0 + j, k);
#pragma unroll
                    for (int j = 0; j < GRP; ++j) acc[j] |= read_quad(more[j]);
                }
                if (depth & CL_HEAVY) {  // the wave reads a heavy slice's rows one by one
#pragma unroll
                    for (int j = 0; j < GRP; ++j) {
                        const uint32_t mj = (uint32_t)__builtin_amdgcn_readlane((int)my_m, i0 + j);
                        if (mj & CL_HEAVY)
                            acc[j] = heavy_slice(a, s_r, (uint32_t)((i0 + j) * CL_WAVES + wave) * WAVE, ln);
                        // (its group's light slices, past the depth that CL_HEAVY hides)
                        for (uint32_t k = 1; !(mj & CL_HEAVY) && k < mj; ++k) acc[j] |= read_quad(load_quad(i0 + j, k));
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < GRP; ++j) {
                const uint32_t v = acc[j] & ~s_r[(i0 + j) * CL_TB + tid];
                nw[i0 + j] = v;
                cnt += (uint32_t)__popc(v);
                changed += (uint32_t)__popcll(__ballot(v != 0));
            }
#pragma unroll
            for (int j = 0; j < GRP; ++j) w[j] = wn[j];
        }
        cnt = wave_sum(cnt);
        uint32_t pos = 0;
        if (lane == 0 && changed) {
            atomicAdd(&s_cnt[slot], cnt);
            pos = atomicAdd(&s_qn[next], changed);
        }
        __syncthreads();  // every row has been read
        if (tid == 0) s_cnt[after] = s_qn[after] = 0;  // of the iteration before: every thread is past reading it
        const uint32_t total = s_cnt[slot];
        if (total == 0) break;  // block-uniform
        if (tid == 0) atomicAdd(&a.counts[1 + it], (unsigned long long)total);
        const bool queue = QT > 0 && s_qn[next] <= QCAP;  // block-uniform
        pos = (uint32_t)__builtin_amdgcn_readfirstlane((int)pos);
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            if (nw[i]) s_r[i * CL_TB + tid] |= nw[i];
            if (queue) {
                const uint64_t bal = __ballot(nw[i] != 0);
                if (nw[i]) {
                    const uint32_t at = pos + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
                    s_qrow[at] = (uint16_t)(i * CL_TB + tid);
                    s_qbits[at] = nw[i];
                }
                pos += (uint32_t)__popcll(bal);
            }
        }
        __syncthreads();
    }
    if (tid == 0) atomicMax(&a.counts[0], (unsigned long long)it);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const uint32_t row = i * CL_TB + tid;
        if (row < a.domain) a.S[(uint64_t)cw * a.domain + row] = s_r[row];
    }
}

// The columns' slices (cols x domain, internal row order) as a bit matrix
// (row perm[i], cols words a row) with its row counts.  A block takes TR_ROWS
// rows: 64 columns of them at a time go through LDS, so that both sides move
// whole lines (the columns' blocks writing the matrix themselves, four bytes of
// a line at a time, took a fifth of their time).
constexpr int TR_ROWS = 32, TR_COLS = 64;
__global__ __launch_bounds__(256) void k_cl_transpose(const uint32_t *__restrict__ S, uint32_t domain, uint32_t cols,
                                                      const uint32_t *__restrict__ perm, uint32_t *__restrict__ R,
                                                      uint64_t *__restrict__ row_count) {
    __shared__ uint32_t t[TR_COLS][TR_ROWS + 1];
    constexpr int RPW = TR_ROWS / 4, LD = TR_ROWS * TR_COLS / 256;  // rows per wave, loads per thread
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid >> 6;
    const uint32_t row0 = blockIdx.x * TR_ROWS, r = tid % TR_ROWS, c = tid / TR_ROWS;
    const uint32_t src = min(row0 + r, domain - 1);
    uint32_t to[RPW], ones[RPW];
#pragma unroll
    for (int k = 0; k < RPW; ++k) {
        to[k] = perm[min(row0 + wave * RPW + k, domain - 1)];
        ones[k] = 0;
    }
    for (uint32_t c0 = 0; c0 < cols; c0 += TR_COLS) {
        uint32_t v[LD];
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const uint32_t cc = c0 + c + q * (256 / TR_ROWS);
            v[q] = cc < cols ? S[(uint64_t)cc * domain + src] : 0u;
        }
        __syncthreads();  // the tile before has been written
#pragma unroll
        for (int q = 0; q < LD; ++q) t[c + q * (256 / TR_ROWS)][r] = v[q];
        __syncthreads();
        if (c0 + lane < cols) {
#pragma unroll
            for (int k = 0; k < RPW; ++k) {
                const uint32_t w = t[lane][wave * RPW + k];
                ones[k] += (uint32_t)__popc(w);
                if (row0 + wave * RPW + k < domain) R[(uint64_t)to[k] * cols + c0 + lane] = w;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < RPW; ++k) {
        const uint32_t n = wave_sum(ones[k]);
        if (lane == 0 && row0 + wave * RPW + k < domain) row_count[to[k]] = n;
    }
}

}  // namespace

// A slice of every row has to fit LDS, and the edges an XCD's L2 (every
// workgroup reads them each iteration).  With many edges a row the fixpoint has
// few iterations and the lists' preparation is the larger part: 50 a row took
// 0.59 ms here against 0.55 by row gathers at 8,000 vertices, but 1.27 against
// 1.48 at 16,000 and 3.8 against 5.5 at 32,000 (3 a row: 0.43 / 0.85, 0.78 /
// 1.16 and 2.4 / 3.7 ms); 500 a row (1,000 x 1,000 complete bipartite) 0.64 / 0.33.
bool closure_columns_fits(uint32_t domain, uint64_t edges, uint64_t seeds) {
    const uint64_t per_row = domain >= 12288 ? 64 : 32;
    return domain <= (uint32_t)CL_MAX_RPT * CL_TB &&
           edges <= std::min<uint64_t>(per_row * domain, CLOSURE_COLUMNS_EDGES) && seeds <= CLOSURE_COLUMNS_EDGES;
}

uint64_t closure_columns(Ctx *ctx, const uint64_t *edge, uint64_t m, const uint64_t *row_ptr, const uint32_t *adj,
                         const uint64_t *seed, uint64_t n_seed, uint32_t domain, uint64_t words, uint64_t max_iter,
                         uint64_t *R, uint64_t *row_counts, std::vector<uint64_t> &layers) {
    XH_REQUIRE(domain >= 1 && closure_columns_fits(domain, m, n_seed), XLOG_HIP_INVALID_ARG,
               "closure columns: domain or relations too large");
    const uint32_t slices = (domain + WAVE - 1) / WAVE;
    const uint32_t rpt = (domain + CL_TB - 1) / CL_TB;
    static constexpr uint32_t kRpt[] = {1, 2, 4, 8, 16, 24, 32, (uint32_t)CL_MAX_RPT};
    uint32_t inst = 0;
    while (kRpt[inst] < rpt) ++inst;
    const uint64_t cap = std::min<uint64_t>(max_iter, (uint64_t)domain + 1);
    const bool own_seed = seed != edge || n_seed != m;
    // a light slice is at most (sum of ceil(degree / 64) over its rows) + 8 * 64 edges deep, then rounded up to a quad
    const uint64_t sell_n = (m + (uint64_t)slices * WAVE * (WAVE + 8 * WAVE + CL_QUAD)) / CL_QUAD;
    // zeroed: [counts: 1 + cap][bins][cursors][sell_next][in_ptr: domain + 1][seed_ptr: domain + 1]
    const uint64_t d1 = (uint64_t)domain + 1, n32 = 2 * CL_DEG_BINS + 2 + (own_seed ? 2 : 1) * d1;
    Buf<uint64_t> z(ctx, 1 + cap + (n32 + 1) / 2);
    unsigned long long *counts = reinterpret_cast<unsigned long long *>(z.p);
    uint32_t *bins = reinterpret_cast<uint32_t *>(z.p + 1 + cap), *cursor = bins + CL_DEG_BINS;
    uint32_t *sell_next = cursor + CL_DEG_BINS, *in_ptr = sell_next + 2;
    uint32_t *seed_ptr = own_seed ? in_ptr + d1 : in_ptr;
    Buf<uint32_t> perm(ctx, domain), slice(ctx, 2 * (uint64_t)slices), S(ctx, 2 * words * (uint64_t)domain),
        rank(ctx, m ? m : 1), seed_rank(ctx, own_seed ? n_seed : 0);
    Buf<uint16_t> inv(ctx, domain), col(ctx, m ? m : 1), in_src(ctx, m ? m : 1), own_src(ctx, own_seed ? n_seed : 0);
    uint16_t *seed_src = own_seed ? own_src.p : in_src.p;
    Buf<uint64_t> sell(ctx, sell_n);
    Buf<unsigned long long> sum(ctx, 1);
    fill_u64(ctx, z.p, 0ull, z.n);
    const uint64_t work = std::max<uint64_t>(std::max(m, n_seed), (uint64_t)slices * WAVE);
    hipLaunchKernelGGL(k_cl_bins, dim3(grid_for(domain, 256, 128)), dim3(256), 0, ctx->stream, row_ptr, domain, bins);
    hipLaunchKernelGGL(k_cl_place, dim3((domain + CL_TB - 1) / CL_TB), dim3(CL_TB), 0, ctx->stream, row_ptr, domain,
                       bins, cursor, perm.p, inv.p);
    hipLaunchKernelGGL(k_cl_in_degrees, dim3(grid_for(std::max(m, n_seed), 256, 1024)), dim3(256), 0, ctx->stream, adj,
                       m, own_seed ? seed : nullptr, n_seed, inv.p, in_ptr, seed_ptr, rank.p, seed_rank.p);
    XH_CHECK_HIP(hipGetLastError());
    scan_u32_inplace(ctx, in_ptr, d1, sum.p);
    if (own_seed) scan_u32_inplace(ctx, seed_ptr, d1, sum.p);
    const ClFill fa{row_ptr, adj, m, domain, slices, kRpt[inst] * CL_TB, perm.p, inv.p, slice.p, slice.p + slices,
                    sell_next, sell.p, col.p, edge, in_ptr, rank.p, in_src.p, own_seed ? seed : nullptr, n_seed,
                    seed_ptr, seed_rank.p, seed_src};
    hipLaunchKernelGGL(k_cl_fill, dim3(grid_for(work, 256, 1024)), dim3(256), 0, ctx->stream, fa);
    XH_CHECK_HIP(hipGetLastError());
    const ClArgs a{sell.p, col.p, slice.p, slice.p + slices, row_ptr, perm.p, inv.p, in_ptr, in_src.p, seed_ptr,
                   seed_src, domain, slices, max_iter, counts, S.p};
    const dim3 grid((unsigned)(2 * words));
    {
        // the matrix written; everything else is read from caches
        Prof prof(ctx, XLOG_HIP_KERNEL_CHAIN_PRODUCT, 8.0 * (double)domain * (double)words + 2.0 * (double)m);
        switch (kRpt[inst]) {
            case 1: hipLaunchKernelGGL(k_cl_columns<1>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
            case 2: hipLaunchKernelGGL(k_cl_columns<2>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
            case 4: hipLaunchKernelGGL(k_cl_columns<4>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
            case 8: hipLaunchKernelGGL(k_cl_columns<8>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
            case 16: hipLaunchKernelGGL(k_cl_columns<16>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
            case 24: hipLaunchKernelGGL(k_cl_columns<24>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
            case 32: hipLaunchKernelGGL(k_cl_columns<32>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
            default: hipLaunchKernelGGL(k_cl_columns<CL_MAX_RPT>, grid, dim3(CL_TB), 0, ctx->stream, a); break;
        }
        XH_CHECK_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_cl_transpose, dim3((domain + TR_ROWS - 1) / TR_ROWS), dim3(256), 0, ctx->stream, S.p, domain,
                       (uint32_t)(2 * words), perm.p, reinterpret_cast<uint32_t *>(R), row_counts);
    XH_CHECK_HIP(hipGetLastError());
    const uint64_t head = std::min<uint64_t>(cap + 1, 256);
    ctx->read_scalars(counts, head);
    const uint64_t n = ctx->host_scalars[0];
    layers.assign(n, 0);
    for (uint64_t i = 0; i < n && i + 1 < head; ++i) layers[i] = ctx->host_scalars[1 + i];
    if (n + 1 > head) {
        XH_CHECK_HIP(hipMemcpyAsync(layers.data() + (head - 1), counts + head, (n + 1 - head) * sizeof(uint64_t),
                                    hipMemcpyDeviceToHost, ctx->stream));
        ctx->sync();
    }
    return n;
}

}  // namespace xh
