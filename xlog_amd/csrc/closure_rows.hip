// Linear closure over ids of any range, a few source rows at a time.
//
// The program  H(X,Z) :- E(X,Z).  H(X,Z) :- H(X,Y), E(Y,Z)  (or E(X,Y), H(Y,Z))
// never mixes the sources of H: what a source reaches is a breadth-first walk
// of E from it, and the layers of the walk are the iterations of the
// semi-naive loop.  So a wave takes CR_EDGES consecutive rows of E, walks from
// the sources that begin there with the pairs reached in an LDS set, sorts
// them there (every pair counts the smaller ones: there are few) and writes
// them out; a last pass closes the gaps between the waves' regions.  Nothing
// that grows with H is probed in memory and nothing of it is sorted there,
// which is where the hash-set loop spends its time (2^20 vertices, 943,718
// edges, 9.4 * 10^6 pairs, ids over 32 bits: 80 insert launches, two rehashes
// and 8 passes of a sort, 4.24 ms whole; this takes 1.10 ms, 0.65 of them the
// walks and 0.15 those of the listed sources).
//
// What bounds it is latency and the instructions of passes that few lanes take
// part in: a layer is one dependent read of E's records (8 bytes: target, and
// where the target's own run starts and how long it is) and a few LDS
// accesses, for as many edges as the batch's sources have in that layer.  So a
// lane takes one edge (four edges a lane, the batch half as large: 1.76 ms),
// one wave is a workgroup with a set of 1,024 pairs, 15 of them on a CU, and a
// batch is the largest that seldom outgrows it (32 edges: more sources listed,
// the call 1.18 ms; 16: 1.17; 14 with sets of 512: 1.74).  The sources of a
// batch that does not fit are listed and walked one by one with larger sets;
// when they are many the attempt ends early and the caller goes on with its loop
// over hash sets.  A few that outgrow the largest set are handed back instead:
// the caller's loop then runs from their edges alone (when one of them ended the
// attempt, a source with 10,000 edges among 2^19 others cost 1,523 us
// where the loop alone took 1,300; so 688).
#include "internal.hpp"
#include "host.hpp"

#include <algorithm>

namespace xh {

namespace {

constexpr int CR_EDGES = 24;  // rows of E whose sources one wave walks together: about 16 sources at 1.5 rows each
constexpr int CR_ROWS = 32;
constexpr uint32_t CR_CAP1 = 896, CR_CAP2 = 1792, CR_CAP3 = 7168;  // pairs: 7/8 of the tiers' sets
// Sources listed up to batch b: at most CR_LISTED and one a batch (one batch in 16 or so) of b, or of CR_AT_ONCE where
// that is more.  At 0.9 edges a vertex 1 % of the batches are listed; at 0.95 a fifth would be, and the tiers after the
// first are then no faster than the hash loop (2^20 vertices and as many edges: 18 ms in the second tier before it gave
// up, of a call of 83 ms without it).  CR_AT_ONCE is about as many batches as run at a time: one of the first may fail
// when many have begun, and with CR_LISTED + b alone it could end an attempt that lists 2,000 sources in all (2^20
// vertices at 0.9 edges: 1.1 or 5.2 ms, as it happened).
constexpr uint32_t CR_LISTED = 512, CR_AT_ONCE = 4096;
constexpr int CR_LAYERS = 4096;                                    // layers of the largest tier
constexpr int CR_BINS = 32;                                        // copies of the layer counters
constexpr uint64_t CR_EMPTY = ~0ull;                               // no pair is: its row is below CR_ROWS

struct CrArgs {
    const uint64_t *edge;  // m sorted unique packed pairs
    uint64_t m;
    uint64_t *rec;  // per edge: target << 32 | first edge of the target's run << 8 | min(its length, 255)
    const unsigned long long *table;  // run index over the first column
    uint64_t mask;
    int bits;
    uint64_t *scratch;
    uint32_t *cnt, *pos;  // per edge that begins a source: pairs, their place in scratch (cnt 0 at the others)
    unsigned long long *layers;  // [CR_LAYERS][CR_BINS]
    unsigned long long *next;    // [CR_BINS] edges that follow an edge, over all edges
    // give up; sources listed for tier 2, for tier 3, handed back; pairs of tiers 2 and 3 in scratch
    uint32_t *ctl;
    uint32_t *list[3];
    uint32_t list_cap[3];
    uint32_t region, region_n;  // of scratch, for the listed sources
};

// the attempt's end: any block of a launch may raise it while others of the same launch are still starting
__device__ __forceinline__ void cr_give_up(const CrArgs &a) {
    __hip_atomic_store(a.ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t cr_gave_up(const CrArgs &a) {
    return __hip_atomic_load(a.ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t cr_run(const CrArgs &a, uint32_t key, uint32_t *start) {
    uint64_t h = (uint64_t)(((uint64_t)key * 0x9E3779B97F4A7C15ull) >> (64 - a.bits));
    for (;;) {
        const u64x2 s = *reinterpret_cast<const u64x2 *>(a.table + 2 * h);
        if (s.x == 0ull) return 0;
        if ((uint32_t)(s.x >> 32) == key) {
            *start = (uint32_t)s.y;
            return (uint32_t)s.x;
        }
        h = (h + 1) & a.mask;
    }
}

__global__ __launch_bounds__(256) void k_cr_records(CrArgs a) {
    const uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    uint32_t len = 0;
    if (e == 0) a.cnt[a.m] = 0;  // the scan's last
    if (e < a.m) {
        const uint32_t to = (uint32_t)a.edge[e];
        uint32_t start = 0;
        len = cr_run(a, to, &start);
        a.rec[e] = ((uint64_t)to << 32) | ((uint64_t)start << 8) | min(len, 255u);
    }
    unsigned long long sum = len;
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, WAVE);
    __shared__ unsigned long long s_sum[4];
    if ((threadIdx.x & (WAVE - 1)) == 0) s_sum[threadIdx.x / WAVE] = sum;
    __syncthreads();
    sum = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
    if (threadIdx.x == 0 && sum) atomicAdd(a.next + (blockIdx.x % CR_BINS), sum);
}

// The edges that follow an edge, on average: near one a walk hardly ends, above it most sources reach most of the
// graph.  From 15/16 the attempt ends here (at 0.95 the walks would take as long as the hash loop, and finding it
// out by the lists took 0.6 ms of 7.3 at 2^20 vertices, 0.36 of 1.8 at 20,000).
__global__ __launch_bounds__(WAVE) void k_cr_gate(CrArgs a) {
    unsigned long long next = threadIdx.x < CR_BINS ? a.next[threadIdx.x] : 0ull;
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) next += __shfl_xor(next, o, WAVE);
    if (threadIdx.x == 0 && 16 * next >= 15 * a.m) cr_give_up(a);
}

template <int SLOTS, int FR, int LV>
struct CrLds {
    // row << 32 | target; at the end the targets alone, a segment per row
    alignas(16) unsigned long long set[SLOTS];
    uint32_t fr[2][FR];  // the edges to follow: edge << 5 | row
    uint32_t nf[2], total, fail, item;
    uint32_t row_n[CR_ROWS], src[CR_ROWS];
    uint32_t row_at[CR_ROWS + 1], row_out[CR_ROWS];  // a row's segment (of whole quads) and place in the result
    uint32_t lev[LV];
};

// a run's edges to follow (all or, when they do not fit, none)
template <int FR, class L>
__device__ __forceinline__ void cr_push(L &l, int f, uint32_t row, uint32_t start, uint32_t len) {
    uint32_t p = FR;
    if (len <= (uint32_t)FR) p = atomicAdd(&l.nf[f], len);
    if (p + len > (uint32_t)FR) {
        l.fail = 1;
        return;
    }
    for (uint32_t q = 0; q < len; ++q) l.fr[f][p + q] = ((start + q) << 5) | row;
}

// an empty walk (the caller pushes its first edges after the barrier)
template <int T, int SLOTS, class L>
__device__ __forceinline__ void cr_reset(L &l) {
    __syncthreads();
    for (int i = threadIdx.x; i < SLOTS; i += T) l.set[i] = CR_EMPTY;
    if (threadIdx.x < CR_ROWS) l.row_n[threadIdx.x] = 0;
    if (threadIdx.x == 0) l.nf[0] = l.nf[1] = l.total = l.fail = 0;
    __syncthreads();
}

// Walks layer by layer from the edges pushed; the number of layers expanded,
// or -1 when the walk does not fit.
template <int T, int SLOTS, int FR, int LV, class L>
__device__ int cr_walk(L &l, const CrArgs &a, uint32_t cap) {
    const int t = threadIdx.x;
    int cur = 0;
    uint32_t prev = 0;
    for (int lv = 0;; ++lv) {
        __syncthreads();
        const uint32_t nf = l.nf[cur], fail = l.fail, total = l.total;
        __syncthreads();
        if (fail || total > cap) return -1;
        if (t == 0) {
            if (lv) l.lev[lv - 1] = total - prev;
            l.nf[cur] = 0;
        }
        prev = total;
        if (nf == 0) return lv;
        if (lv == LV) return -1;
        for (uint32_t base = 0; base < nf; base += T) {
            bool novel = false;
            if (base + t < nf) {
                const uint32_t f = l.fr[cur][base + t], row = f & (CR_ROWS - 1);
                const uint64_t r = a.rec[f >> 5];
                const uint32_t to = (uint32_t)(r >> 32);
                const unsigned long long key = ((unsigned long long)row << 32) | to;
                uint32_t h = ((to ^ (row << 20)) * 0x9E3779B1u) >> (32 - __builtin_ctz(SLOTS));
                bool found = false;
                for (int p = 0; p < SLOTS && !found; ++p) {  // ends: a full table is a walk that does not fit
                    unsigned long long c = l.set[h];
                    if (c == CR_EMPTY) {
                        c = atomicCAS(&l.set[h], (unsigned long long)CR_EMPTY, key);
                        novel = c == CR_EMPTY;
                    }
                    found = novel || c == key;
                    h = (h + 1) & (SLOTS - 1);
                }
                if (!found) l.fail = 1;
                uint32_t len = (uint32_t)r & 255u, first = (uint32_t)(r >> 8) & 0xFFFFFFu;
                if (novel && len) {
                    if (len == 255u) len = cr_run(a, to, &first);
                    cr_push<FR>(l, cur ^ 1, row, first, len);
                }
            }
            const uint32_t c = (uint32_t)__popcll(__ballot(novel));
            if ((t & (WAVE - 1)) == 0 && c) atomicAdd(&l.total, c);
        }
        cur ^= 1;
    }
}

// The walk's pairs in order to out[0, total): the targets row by row (the rows
// ascend), and in a row each counts the smaller ones, four per LDS read.
template <int T, int SLOTS, class L>
__device__ void cr_write(L &l, uint64_t *__restrict__ out) {
    constexpr int R = SLOTS / T;
    const int t = threadIdx.x;
    unsigned long long k[R];
    uint32_t at[R];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < R; ++q) k[q] = l.set[q * T + t];
#pragma unroll
    for (int q = 0; q < R; ++q) at[q] = k[q] != CR_EMPTY ? atomicAdd(&l.row_n[k[q] >> 32], 1u) : 0u;
    __syncthreads();
    if (t < WAVE) {
        const uint32_t c = t < CR_ROWS ? l.row_n[t] : 0u, c4 = (c + 3) & ~3u;
        uint32_t quads = c4, rows = c;
#pragma unroll
        for (int o = 1; o < CR_ROWS; o <<= 1) {
            const uint32_t u = __shfl_up(quads, o, WAVE), v = __shfl_up(rows, o, WAVE);
            if (t >= o) {
                quads += u;
                rows += v;
            }
        }
        if (t < CR_ROWS) {
            l.row_at[t + 1] = quads;
            l.row_out[t] = rows - c;
        }
        if (t == 0) l.row_at[0] = 0;
    }
    __syncthreads();
    uint32_t *seg = reinterpret_cast<uint32_t *>(l.set);
#pragma unroll
    for (int q = 0; q < R; ++q)
        if (k[q] != CR_EMPTY) seg[l.row_at[k[q] >> 32] + at[q]] = (uint32_t)k[q];
    if (t < CR_ROWS)  // (all ones is smaller than no target)
        for (uint32_t i = l.row_at[t] + l.row_n[t]; i < l.row_at[t + 1]; ++i) seg[i] = ~0u;
    __syncthreads();
    const uint32_t n = l.row_at[CR_ROWS];
    for (uint32_t i = t; i < n; i += T) {
        int r = 0;  // the last row that begins at or before i and is not empty
#pragma unroll
        for (int s = CR_ROWS / 2; s > 0; s >>= 1)
            if (l.row_at[r + s] <= i) r += s;
        const uint32_t lo = l.row_at[r];
        if (i - lo >= l.row_n[r]) continue;
        const uint32_t to = seg[i], hi = l.row_at[r + 1];
        uint32_t rank = 0;
#pragma unroll 4
        for (uint32_t j = lo; j < hi; j += 4) {
            const uint4 v = *reinterpret_cast<const uint4 *>(seg + j);
            rank += (v.x < to ? 1u : 0u) + (v.y < to ? 1u : 0u) + (v.z < to ? 1u : 0u) + (v.w < to ? 1u : 0u);
        }
        out[l.row_out[r] + rank] = ((uint64_t)l.src[r] << 32) | to;
    }
}

constexpr int CR_SLOTS1 = 1024, CR_FR1 = 256, CR_LV1 = 128;
__global__ __launch_bounds__(WAVE) void k_cr_walk(CrArgs a) {
    __shared__ CrLds<CR_SLOTS1, CR_FR1, CR_LV1> l;
    const int lane = threadIdx.x;
    const uint64_t b = blockIdx.x, e = b * CR_EDGES + lane;
    // the sources that begin in the batch's edges, the last one's run as far as the lanes see it
    const bool mine = lane < CR_EDGES && e < a.m;
    const uint32_t src = e < a.m ? (uint32_t)(a.edge[e] >> 32) : 0u;
    const bool head = mine && (e == 0 || (uint32_t)(a.edge[e - 1] >> 32) != src);
    if (cr_gave_up(a)) return;  // (the workgroup is one wave, whose lanes read one word in one load)
    const uint64_t heads = __ballot(head);
    const int row = __popcll(heads & ((2ull << min(lane, CR_EDGES - 1)) - 1ull)) - 1;  // -1: an earlier batch's
    const uint32_t last_src = __shfl(src, CR_EDGES - 1, WAVE);
    const bool walks = row >= 0 && e < a.m && (lane < CR_EDGES || src == last_src);
    cr_reset<WAVE, CR_SLOTS1>(l);
    if (head) l.src[row] = src;
    if (walks) cr_push<CR_FR1>(l, 0, row, (uint32_t)e, 1);
    if (walks && lane == WAVE - 1) {  // what lies past the lanes
        uint32_t start = 0;
        const uint32_t len = cr_run(a, src, &start);
        cr_push<CR_FR1>(l, 0, row, (uint32_t)e + 1, len - ((uint32_t)e + 1 - start));
    }
    const int nl = cr_walk<WAVE, CR_SLOTS1, CR_FR1, CR_LV1>(l, a, CR_CAP1);
    __syncthreads();
    if (nl >= 0) {
        for (int q = lane; q < nl; q += WAVE)
            if (l.lev[q]) atomicAdd(&a.layers[q * CR_BINS + b % CR_BINS], (unsigned long long)l.lev[q]);
        cr_write<WAVE, CR_SLOTS1>(l, a.scratch + b * CR_CAP1);
        if (mine) {
            a.cnt[e] = head ? l.row_n[row] : 0u;
            a.pos[e] = (uint32_t)(b * CR_CAP1) + (head ? l.row_out[row] : 0u);
        }
        return;
    }
    // together they do not fit: each goes on the list
    if (mine && !head) a.cnt[e] = 0;
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(&a.ctl[1], (uint32_t)__popcll(heads));
    at = __shfl(at, 0, WAVE) + (uint32_t)row;
    if (!head) return;
    // batches begin about in order, so a graph whose sources reach too much ends the attempt in its first batches
    if (at < min(CR_LISTED + max((uint32_t)b, CR_AT_ONCE), a.list_cap[0]))
        a.list[0][at] = (uint32_t)e;
    else
        cr_give_up(a);
}

// the listed sources, one at a time; those that do not fit go to the next list
template <int T, int SLOTS, int FR, int LV, int TIER>
__global__ __launch_bounds__(T) void k_cr_walk_one(CrArgs a, uint32_t cap) {
    __shared__ CrLds<SLOTS, FR, LV> l;
    // One thread reads whether the attempt has ended: blocks of this launch raise it, too, and waves that read it each
    // for themselves could part, some leaving before the barriers that reset what the others go on to use.
    if (threadIdx.x == 0) l.item = cr_gave_up(a);
    __syncthreads();
    if (l.item) return;
    const uint32_t n = min(a.ctl[TIER], a.list_cap[TIER - 1]);
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        cr_reset<T, SLOTS>(l);
        if (threadIdx.x == 0) {
            if (cr_gave_up(a)) l.fail = 1;
            const uint32_t src = (uint32_t)(a.edge[a.list[TIER - 1][i]] >> 32);
            uint32_t start = 0;
            const uint32_t len = cr_run(a, src, &start);
            l.src[0] = src;
            cr_push<FR>(l, 0, 0, start, len);
        }
        const int nl = cr_walk<T, SLOTS, FR, LV>(l, a, cap);
        __syncthreads();
        const uint32_t e = a.list[TIER - 1][i];
        auto pass_on = [&](int to) {  // to list `to`, where the source has no pairs of its own yet
            const uint32_t j = atomicAdd(&a.ctl[1 + to], 1u);
            if (j < a.list_cap[to]) {
                a.list[to][j] = e;
                a.cnt[e] = 0;
            } else {
                cr_give_up(a);
            }
        };
        if (nl < 0) {
            if (threadIdx.x == 0) pass_on(TIER);
            continue;
        }
        const uint32_t total = l.total;
        if (threadIdx.x == 0) {
            const uint32_t p = atomicAdd(&a.ctl[4], total);
            const bool fits = p <= a.region_n && total <= a.region_n - p;
            l.item = fits ? p : ~0u;
            if (fits) {
                a.cnt[e] = total;
                a.pos[e] = a.region + p;
            } else {
                pass_on(2);
            }
        }
        __syncthreads();
        const uint32_t p = l.item;
        if (p == ~0u) continue;
        for (int q = threadIdx.x; q < nl; q += T)
            if (l.lev[q]) atomicAdd(&a.layers[q * CR_BINS + blockIdx.x % CR_BINS], (unsigned long long)l.lev[q]);
        cr_write<T, SLOTS>(l, a.scratch + a.region + p);
    }
}

// a.list[2]'s sources as flags of their edges
__global__ __launch_bounds__(256) void k_cr_rest(CrArgs a, uint32_t n, uint8_t *__restrict__ flags) {
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        uint32_t start = 0;
        const uint32_t len = cr_run(a, (uint32_t)(a.edge[a.list[2][i]] >> 32), &start);
        for (uint32_t q = threadIdx.x; q < len; q += 256) flags[start + q] = 1;
    }
}

// result: [0] gave up, [1] pairs, [2 + k] sources on list k, [5 + k] pairs of layer k
constexpr int CR_HEAD = 5;
__global__ __launch_bounds__(256) void k_cr_result(CrArgs a, const unsigned long long *total, uint64_t *result) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k == 0) {
        result[0] = a.ctl[0];
        result[1] = *total;
        for (int q = 0; q < 3; ++q) result[2 + q] = a.ctl[1 + q];
    }
    if (k >= CR_LAYERS) return;
    unsigned long long s = 0;
    for (int b = 0; b < CR_BINS; ++b) s += a.layers[k * CR_BINS + b];
    result[CR_HEAD + k] = s;
}

// Closes the gaps: a wave per 64 edges, whose sources' pairs are one span of
// the result (off: m + 1 offsets), written in order.
__global__ __launch_bounds__(256) void k_cr_gather(const uint64_t *__restrict__ scratch,
                                                   const uint32_t *__restrict__ off, const uint32_t *__restrict__ pos,
                                                   uint64_t m, uint64_t *__restrict__ out) {
    __shared__ uint32_t s_off[4][WAVE + 1], s_pos[4][WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x >> 6;
    const uint64_t e0 = ((uint64_t)blockIdx.x * 4 + wave) * WAVE;
    const uint64_t e = min(e0 + lane, m);
    s_off[wave][lane] = off[e];
    if (lane == 0) s_off[wave][WAVE] = off[min(e0 + WAVE, m)];
    s_pos[wave][lane] = e < m ? pos[e] : 0u;
    __syncthreads();
    const uint32_t lo = s_off[wave][0], hi = s_off[wave][WAVE];
    for (uint32_t o = lo + lane; o < hi; o += WAVE) {
        int r = 0;  // the last edge whose offset is at most o: the one that has it
#pragma unroll
        for (int s = WAVE / 2; s > 0; s >>= 1)
            if (s_off[wave][r + s] <= o) r += s;
        out[o] = scratch[(uint64_t)s_pos[wave][r] + (o - s_off[wave][r])];
    }
}

}  // namespace

// device bytes closure_rows takes besides the result
static uint64_t closure_rows_bytes(uint64_t m) {
    return ((m + CR_EDGES - 1) / CR_EDGES * CR_CAP1 + 16 * m + (1ull << 20)) * 8 + 102 * m + (1ull << 21);
}

bool closure_rows_takes(Ctx *ctx, uint64_t m) {
    return m >= 1 && m <= (1ull << 24) && closure_rows_bytes(m) <= device_room(ctx) / 4;
}

uint64_t *closure_rows(Ctx *ctx, const uint64_t *edge, uint64_t m, uint64_t max_iter, uint64_t *n,
                       std::vector<uint64_t> &layers, Buf<uint64_t> &rest, uint64_t *rest_n) {
    XH_REQUIRE(m >= 1 && m <= (1ull << 24), XLOG_HIP_INVALID_ARG, "closure rows: relation too large");
    // the runs of E and their table, sized for m runs: no read-back
    RunIndex ix;
    RunScratch rs;
    Buf<uint64_t> runs(ctx, 2);
    fill_u64(ctx, runs.p + 1, m, 1);
    build_run_index_async(ctx, edge, m, nullptr, rs, runs.p);
    uint64_t slots = 1024;
    while (slots < 2 * m) slots <<= 1;
    ix.table = Buf<unsigned long long>(ctx, 2 * slots);
    ix.table_mask = slots - 1;
    run_index_insert_dev(ctx, rs.run_key.p, rs.run_start.p, runs.p, m, runs.p + 1, ix, nullptr);
    const uint64_t nb = (m + CR_EDGES - 1) / CR_EDGES;
    const uint64_t region = nb * CR_CAP1, region_n = 16 * m + (1ull << 20);  // both below 2^32
    const uint64_t cap2 = CR_LISTED + nb, cap3 = m / 4096 + 64;
    Buf<uint64_t> rec(ctx, m), scratch(ctx, region + region_n), result(ctx, CR_HEAD + CR_LAYERS);
    Buf<uint32_t> off(ctx, m + 1), pos(ctx, m), list(ctx, cap2 + 2 * cap3);
    Buf<uint64_t> z(ctx, (uint64_t)(CR_LAYERS + 1) * CR_BINS + 4);  // zeroed: layers, next, ctl, the scan's total
    fill_u64(ctx, z.p, 0ull, z.n);
    CrArgs a;
    a.edge = edge;
    a.m = m;
    a.rec = rec.p;
    a.table = ix.table.p;
    a.mask = ix.table_mask;
    a.bits = __builtin_ctzll(ix.table_mask + 1);
    a.scratch = scratch.p;
    a.cnt = off.p;
    a.pos = pos.p;
    a.layers = reinterpret_cast<unsigned long long *>(z.p);
    a.next = a.layers + (uint64_t)CR_LAYERS * CR_BINS;
    a.ctl = reinterpret_cast<uint32_t *>(a.next + CR_BINS);
    a.list[0] = list.p;
    a.list[1] = list.p + cap2;
    a.list[2] = list.p + cap2 + cap3;
    a.list_cap[0] = (uint32_t)cap2;
    a.list_cap[1] = a.list_cap[2] = (uint32_t)cap3;
    a.region = (uint32_t)region;
    a.region_n = (uint32_t)region_n;
    unsigned long long *total = a.next + CR_BINS + 3;
    const unsigned cus = (unsigned)ctx->num_cus;
    hipLaunchKernelGGL(k_cr_records, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, ctx->stream, a);
    hipLaunchKernelGGL(k_cr_gate, dim3(1), dim3(WAVE), 0, ctx->stream, a);
    {
        Prof prof(ctx, XLOG_HIP_KERNEL_HASH_INSERT, 16.0 * (double)m);  // the edges and their records, read once
        hipLaunchKernelGGL(k_cr_walk, dim3((unsigned)nb), dim3(WAVE), 0, ctx->stream, a);
        XH_CHECK_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL((k_cr_walk_one<WAVE, 2048, 512, 512, 1>), dim3((unsigned)std::min<uint64_t>(cap2, 7 * cus)),
                       dim3(WAVE), 0, ctx->stream, a, CR_CAP2);
    hipLaunchKernelGGL((k_cr_walk_one<512, 8192, 2048, CR_LAYERS, 2>), dim3((unsigned)std::min<uint64_t>(cap3, cus)),
                       dim3(512), 0, ctx->stream, a, CR_CAP3);
    XH_CHECK_HIP(hipGetLastError());
    scan_u32_inplace(ctx, off.p, m + 1, total);
    hipLaunchKernelGGL(k_cr_result, dim3(CR_LAYERS / 256), dim3(256), 0, ctx->stream, a, total, result.p);
    XH_CHECK_HIP(hipGetLastError());
    const uint64_t first = 128;
    ctx->read_scalars(result.p, first);
    const uint64_t *h = ctx->host_scalars;
    if (trace_on())
        fprintf(stderr,
                "[xlog_hip] closure walks: %llu sources listed, %llu for the largest sets, %llu handed back%s\n",
                (unsigned long long)h[2], (unsigned long long)h[3], (unsigned long long)h[4], h[0] ? ": gave up" : "");
    const uint64_t pairs = h[1], n_rest = h[4];
    if (h[0] || pairs == 0) return nullptr;
    layers.assign(h + CR_HEAD, h + first);
    if (layers.back()) {
        layers.resize(CR_LAYERS);
        XH_CHECK_HIP(hipMemcpyAsync(layers.data(), result.p + CR_HEAD, CR_LAYERS * sizeof(uint64_t),
                                    hipMemcpyDeviceToHost, ctx->stream));
        XH_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    }
    while (!layers.empty() && !layers.back()) layers.pop_back();
    if (layers.size() > max_iter) return nullptr;  // the loop reports the limit
    Owned out(ctx, alloc_keys(ctx, pairs));
    hipLaunchKernelGGL(k_cr_gather, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, ctx->stream, scratch.p, off.p,
                       pos.p, m, out.p);
    XH_CHECK_HIP(hipGetLastError());
    *n = pairs;
    *rest_n = 0;
    if (n_rest) {
        Buf<uint8_t> flags(ctx, m + 3);
        Buf<uint64_t> cnt(ctx, 1);
        rest = Buf<uint64_t>(ctx, m);
        fill_u32(ctx, reinterpret_cast<uint32_t *>(flags.p), 0u, (m + 3) / 4);
        hipLaunchKernelGGL(k_cr_rest, dim3((unsigned)std::min<uint64_t>(n_rest, 8 * cus)), dim3(256), 0, ctx->stream, a,
                           (uint32_t)n_rest, flags.p);
        XH_CHECK_HIP(hipGetLastError());
        select_flags(ctx, edge, flags.p, m, rest.p, cnt.p);
        ctx->read_scalars(cnt.p, 1);
        *rest_n = ctx->host_scalars[0];
    }
    return out.release();
}

}  // namespace xh
