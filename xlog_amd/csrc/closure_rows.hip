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
// and 8 passes of a sort, 4.24 ms).
//
// What bounds it is latency: a layer is one dependent read of E's records (8
// bytes: target, and where the target's own run starts and how long it is) and
// a few LDS accesses.  Hence one wave per workgroup, with a set small enough
// for 24 of them on a CU.  Sources that reach more are listed and walked
// by larger workgroups with larger sets; when they are many, or one of them
// outgrows the largest set, the call gives up early and the caller goes on with
// its loop over hash sets.
#include "internal.hpp"
#include "host.hpp"

#include <algorithm>

namespace xh {

namespace {

constexpr int CR_EDGES = 12;  // rows of E whose sources one wave walks together: about 8 sources at 1.5 rows each
constexpr int CR_ROWS = 16;
constexpr uint32_t CR_CAP1 = 448, CR_CAP2 = 1792, CR_CAP3 = 7168;  // pairs: 7/8 of the tiers' sets
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
    uint32_t *ctl;               // give up, sources listed for tier 2, for tier 3, pairs of both in scratch
    uint32_t *list[2];
    uint32_t list_cap[2];
    uint32_t region, region_n;  // of scratch, for the listed sources
};

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
    if (e >= a.m) return;
    const uint32_t to = (uint32_t)a.edge[e];
    uint32_t start = 0;
    const uint32_t len = cr_run(a, to, &start);
    a.rec[e] = ((uint64_t)to << 32) | ((uint64_t)start << 8) | min(len, 255u);
}

template <int SLOTS, int FR, int LV>
struct CrLds {
    unsigned long long set[SLOTS];  // row << 32 | target; compacted in place at the end
    uint32_t fr[2][FR];             // up to four edges each: first edge << 6 | (edges - 1) << 4 | row
    uint32_t nf[2], total, fail, packed, item;
    uint32_t row_n[CR_ROWS], src[CR_ROWS];
    uint32_t lev[LV];
};

template <int FR, class L>
__device__ __forceinline__ void cr_push(L &l, int f, uint32_t row, uint32_t start, uint32_t len) {
    const uint32_t np = (len + 3) / 4;
    if (np > (uint32_t)FR) {
        l.fail = 1;
        return;
    }
    const uint32_t p = atomicAdd(&l.nf[f], np);
    if (p + np > (uint32_t)FR) {
        l.fail = 1;
        return;
    }
    for (uint32_t q = 0; q < np; ++q)
        l.fr[f][p + q] = ((start + 4 * q) << 6) | ((min(len - 4 * q, 4u) - 1) << 4) | row;
}

// an empty walk (the caller pushes its first edges after the barrier)
template <int T, int SLOTS, class L>
__device__ __forceinline__ void cr_reset(L &l) {
    __syncthreads();
    for (int i = threadIdx.x; i < SLOTS; i += T) l.set[i] = CR_EMPTY;
    if (threadIdx.x < CR_ROWS) l.row_n[threadIdx.x] = 0;
    if (threadIdx.x == 0) l.nf[0] = l.nf[1] = l.total = l.fail = l.packed = 0;
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
        for (uint32_t i = t; i < nf; i += T) {
            const uint32_t f = l.fr[cur][i], start = f >> 6, n = ((f >> 4) & 3) + 1, row = f & 15;
            uint64_t r[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) r[u] = u < n ? a.rec[start + u] : 0ull;
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                if (u >= n) continue;
                const uint32_t to = (uint32_t)(r[u] >> 32);
                const unsigned long long key = ((unsigned long long)row << 32) | to;
                uint32_t h = ((to ^ (row << 20)) * 0x9E3779B1u) >> (32 - __builtin_ctz(SLOTS));
                bool novel = false, found = false;
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
                if (!novel) continue;
                atomicAdd(&l.total, 1u);
                atomicAdd(&l.row_n[row], 1u);
                uint32_t len = (uint32_t)r[u] & 255u, first = (uint32_t)(r[u] >> 8) & 0xFFFFFFu;
                if (len == 255u) len = cr_run(a, to, &first);
                if (len) cr_push<FR>(l, cur ^ 1, row, first, len);
            }
        }
        cur ^= 1;
    }
}

// The walk's pairs in order to out[0, n).
template <int T, int SLOTS, class L>
__device__ void cr_write(L &l, uint32_t n, uint64_t *__restrict__ out) {
    constexpr int R = SLOTS / T;
    const int t = threadIdx.x, lane = t & (WAVE - 1);
    unsigned long long k[R];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < R; ++q) k[q] = l.set[q * T + t];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const bool v = k[q] != CR_EMPTY;
        const uint64_t m = __ballot(v);
        uint32_t base = 0;
        if (lane == 0 && m) base = atomicAdd(&l.packed, (uint32_t)__popcll(m));
        base = __shfl(base, 0, WAVE);
        if (v) l.set[base + __popcll(m & ((1ull << lane) - 1ull))] = k[q];
    }
    __syncthreads();
    for (uint32_t i = t; i < n; i += T) {
        const unsigned long long key = l.set[i];
        uint32_t rank = 0;
#pragma unroll 8
        for (uint32_t j = 0; j < n; ++j) rank += l.set[j] < key ? 1u : 0u;
        out[rank] = ((uint64_t)l.src[key >> 32] << 32) | (uint32_t)key;
    }
}

constexpr int CR_SLOTS1 = 512, CR_FR1 = 256, CR_LV1 = 64;
__global__ __launch_bounds__(WAVE) void k_cr_walk(CrArgs a) {
    __shared__ CrLds<CR_SLOTS1, CR_FR1, CR_LV1> l;
    __shared__ uint32_t hist[CR_LV1];
    const int lane = threadIdx.x;
    hist[lane] = 0;
    const uint64_t nb = (a.m + CR_EDGES - 1) / CR_EDGES;
    for (uint64_t b = blockIdx.x; b < nb; b += gridDim.x) {
        const uint64_t e = b * CR_EDGES + lane;
        const bool mine = lane < CR_EDGES && e < a.m;
        const uint32_t src = mine ? (uint32_t)(a.edge[e] >> 32) : 0u;
        const bool head = mine && (e == 0 || (uint32_t)(a.edge[e - 1] >> 32) != src);
        if (__hip_atomic_load(a.ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
        const uint64_t heads = __ballot(head);
        const int rows = __popcll(heads);
        const uint32_t row = __popcll(heads & ((1ull << lane) - 1ull));
        uint32_t start = 0, len = 0;
        if (head) len = cr_run(a, src, &start);
        cr_reset<WAVE, CR_SLOTS1>(l);
        if (head) {
            l.src[row] = src;
            cr_push<CR_FR1>(l, 0, row, start, len);
        }
        const int nl = cr_walk<WAVE, CR_SLOTS1, CR_FR1, CR_LV1>(l, a, CR_CAP1);
        __syncthreads();
        if (nl >= 0) {
            uint32_t before = 0;
            for (uint32_t r = 0; head && r < row; ++r) before += l.row_n[r];
            if (mine) {
                a.cnt[e] = head ? l.row_n[row] : 0u;
                a.pos[e] = (uint32_t)(b * CR_CAP1) + before;
            }
            if (lane < nl) hist[lane] += l.lev[lane];
            cr_write<WAVE, CR_SLOTS1>(l, l.total, a.scratch + b * CR_CAP1);
            continue;
        }
        // together they do not fit: one source at a time, and those that do not fit alone are listed
        if (mine && !head) a.cnt[e] = 0;
        uint32_t used = 0;
        for (int r = 0; r < rows; ++r) {
            cr_reset<WAVE, CR_SLOTS1>(l);
            const bool it = head && row == (uint32_t)r;
            if (it) cr_push<CR_FR1>(l, 0, row, start, len);
            const int n1 = cr_walk<WAVE, CR_SLOTS1, CR_FR1, CR_LV1>(l, a, CR_CAP1 - used);
            __syncthreads();
            if (n1 < 0) {
                if (it) {
                    const uint32_t i = atomicAdd(&a.ctl[1], 1u);
                    if (i < a.list_cap[0])
                        a.list[0][i] = (uint32_t)e;
                    else
                        a.ctl[0] = 1u;
                }
                continue;
            }
            const uint32_t n = l.total;
            if (it) {
                a.cnt[e] = n;
                a.pos[e] = (uint32_t)(b * CR_CAP1) + used;
            }
            if (lane < n1) hist[lane] += l.lev[lane];
            cr_write<WAVE, CR_SLOTS1>(l, n, a.scratch + b * CR_CAP1 + used);
            used += n;
        }
    }
    if (hist[lane]) atomicAdd(&a.layers[lane * CR_BINS + blockIdx.x % CR_BINS], (unsigned long long)hist[lane]);
}

// the listed sources, one at a time; those that do not fit go to the next
// list, or end the attempt
template <int T, int SLOTS, int FR, int LV, int TIER>
__global__ __launch_bounds__(T) void k_cr_walk_one(CrArgs a, uint32_t cap) {
    __shared__ CrLds<SLOTS, FR, LV> l;
    const uint32_t n = min(a.ctl[TIER], a.list_cap[TIER - 1]);
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        cr_reset<T, SLOTS>(l);
        if (threadIdx.x == 0) {
            if (__hip_atomic_load(a.ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) l.fail = 1;
            const uint32_t src = (uint32_t)(a.edge[a.list[TIER - 1][i]] >> 32);
            uint32_t start = 0;
            const uint32_t len = cr_run(a, src, &start);
            l.src[0] = src;
            cr_push<FR>(l, 0, 0, start, len);
        }
        const int nl = cr_walk<T, SLOTS, FR, LV>(l, a, cap);
        __syncthreads();
        const uint32_t e = a.list[TIER - 1][i];
        if (nl < 0) {
            if (threadIdx.x == 0) {
                const uint32_t j = TIER == 1 ? atomicAdd(&a.ctl[2], 1u) : ~0u;
                if (TIER == 1 && j < a.list_cap[1])
                    a.list[1][j] = e;
                else
                    a.ctl[0] = 1u;
            }
            continue;
        }
        const uint32_t total = l.total;
        if (threadIdx.x == 0) {
            const uint32_t p = atomicAdd(&a.ctl[3], total);
            const bool fits = p <= a.region_n && total <= a.region_n - p;
            l.item = fits ? p : ~0u;
            if (fits) {
                a.cnt[e] = total;
                a.pos[e] = a.region + p;
            } else {
                a.ctl[0] = 1u;
            }
        }
        __syncthreads();
        const uint32_t p = l.item;
        if (p == ~0u) continue;
        for (int q = threadIdx.x; q < nl; q += T)
            if (l.lev[q]) atomicAdd(&a.layers[q * CR_BINS + blockIdx.x % CR_BINS], (unsigned long long)l.lev[q]);
        cr_write<T, SLOTS>(l, total, a.scratch + a.region + p);
    }
}

// result: [0] gave up, [1] pairs, [2 + k] pairs of layer k
__global__ __launch_bounds__(256) void k_cr_result(CrArgs a, const unsigned long long *total, uint64_t *result) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k == 0) {
        result[0] = a.ctl[0];
        result[1] = *total;
    }
    if (k >= CR_LAYERS) return;
    unsigned long long s = 0;
    for (int b = 0; b < CR_BINS; ++b) s += a.layers[k * CR_BINS + b];
    result[2 + k] = s;
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
    return ((m + CR_EDGES - 1) / CR_EDGES * CR_CAP1 + 16 * m + 65536) * 8 + 17 * m + (1ull << 21);
}

bool closure_rows_takes(Ctx *ctx, uint64_t m) {
    return m >= 1 && m <= (1ull << 24) && closure_rows_bytes(m) <= device_room(ctx) / 4;
}

uint64_t *closure_rows(Ctx *ctx, const uint64_t *edge, uint64_t m, const RunIndex &ix, uint64_t max_iter, uint64_t *n,
                       std::vector<uint64_t> &layers) {
    XH_REQUIRE(m >= 1 && m <= (1ull << 24) && !ix.direct && ix.table_mask, XLOG_HIP_INVALID_ARG,
               "closure rows: relation too large");
    const uint64_t nb = (m + CR_EDGES - 1) / CR_EDGES;
    const uint64_t region = nb * CR_CAP1, region_n = 16 * m + 65536;  // both below 2^32
    const uint64_t cap2 = m / 32 + 64, cap3 = m / 512 + 64;
    Buf<uint64_t> rec(ctx, m), scratch(ctx, region + region_n), result(ctx, 2 + CR_LAYERS);
    Buf<uint32_t> off(ctx, m + 1), pos(ctx, m), list(ctx, cap2 + cap3);
    Buf<uint64_t> z(ctx, (uint64_t)CR_LAYERS * CR_BINS + 3);  // zeroed: layers, ctl, the scan's total
    fill_u64(ctx, z.p, 0ull, z.n);
    fill_u32(ctx, off.p + m, 0u, 1);
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
    a.ctl = reinterpret_cast<uint32_t *>(z.p + (uint64_t)CR_LAYERS * CR_BINS);
    a.list[0] = list.p;
    a.list[1] = list.p + cap2;
    a.list_cap[0] = (uint32_t)cap2;
    a.list_cap[1] = (uint32_t)cap3;
    a.region = (uint32_t)region;
    a.region_n = (uint32_t)region_n;
    unsigned long long *total = reinterpret_cast<unsigned long long *>(z.p + (uint64_t)CR_LAYERS * CR_BINS + 2);
    const unsigned cus = (unsigned)ctx->num_cus;
    hipLaunchKernelGGL(k_cr_records, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, ctx->stream, a);
    {
        Prof prof(ctx, XLOG_HIP_KERNEL_HASH_INSERT, 16.0 * (double)m);  // the edges and their records, read once
        hipLaunchKernelGGL(k_cr_walk, dim3((unsigned)std::min<uint64_t>(nb, 24 * cus)), dim3(WAVE), 0, ctx->stream, a);
        XH_CHECK_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL((k_cr_walk_one<128, 2048, 512, 512, 1>), dim3((unsigned)std::min<uint64_t>(cap2, 6 * cus)),
                       dim3(128), 0, ctx->stream, a, CR_CAP2);
    hipLaunchKernelGGL((k_cr_walk_one<512, 8192, 2048, CR_LAYERS, 2>), dim3((unsigned)std::min<uint64_t>(cap3, cus)),
                       dim3(512), 0, ctx->stream, a, CR_CAP3);
    XH_CHECK_HIP(hipGetLastError());
    scan_u32_inplace(ctx, off.p, m + 1, total);
    hipLaunchKernelGGL(k_cr_result, dim3(CR_LAYERS / 256), dim3(256), 0, ctx->stream, a, total, result.p);
    XH_CHECK_HIP(hipGetLastError());
    const uint64_t first = 128;
    ctx->read_scalars(result.p, first);
    if (ctx->host_scalars[0]) return nullptr;
    const uint64_t pairs = ctx->host_scalars[1];
    layers.assign(ctx->host_scalars + 2, ctx->host_scalars + first);
    if (layers.back()) {
        layers.resize(CR_LAYERS);
        XH_CHECK_HIP(hipMemcpyAsync(layers.data(), result.p + 2, CR_LAYERS * sizeof(uint64_t), hipMemcpyDeviceToHost,
                                    ctx->stream));
        XH_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    }
    while (!layers.empty() && !layers.back()) layers.pop_back();
    if (layers.size() > max_iter) return nullptr;  // the loop reports the limit
    Owned out(ctx, alloc_keys(ctx, pairs));
    hipLaunchKernelGGL(k_cr_gather, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, ctx->stream, scratch.p, off.p,
                       pos.p, m, out.p);
    XH_CHECK_HIP(hipGetLastError());
    *n = pairs;
    return out.release();
}

}  // namespace xh
