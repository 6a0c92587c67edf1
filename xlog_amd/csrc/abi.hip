// C ABI of libxlog_hip: context, relation handles and operators.  Host code;
// the semi-naive fixpoint driver is in fixpoint.hip, the kernels in sort.hip,
// select.hip, join.hip, tc_bitmap.hip, chain_bitmap.hip and hash_set.hip.
#include "host.hpp"

#include <algorithm>
#include <cmath>
#include <array>
#include <chrono>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fcntl.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <unistd.h>
#include <memory>

namespace xh {

// ---------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------
static thread_local std::string g_last_error;
void set_error(const std::string &msg) { g_last_error = msg; }

template <class F>
static xlog_hip_status guarded(F &&f) {
    try {
        f();
        g_last_error.clear();
        return XLOG_HIP_OK;
    } catch (const Error &e) {
        g_last_error = e.msg;
        return e.code;
    } catch (const std::bad_alloc &) {
        g_last_error = "host allocation failed";
        return XLOG_HIP_OOM;
    } catch (const std::exception &e) {
        g_last_error = e.what();
        return XLOG_HIP_DEVICE_ERROR;
    }
}

// ---------------------------------------------------------------------------
// pool
// ---------------------------------------------------------------------------
size_t Pool::round_up(size_t b) {
    if (b < 256) return 256;
    // four size classes per power of two
    int lg = 63 - __builtin_clzll(b);
    size_t q = (lg >= 2) ? (size_t)1 << (lg - 2) : 1;
    return (b + q - 1) / q * q;
}
void *Pool::alloc(size_t bytes) {
    size_t sz = round_up(bytes);
    // the budget bounds the live bytes, as the reference's GpuMemoryManager
    // (crates/xlog-cuda/src/memory.rs:756-770; MemoryBudget::with_limit aborts on exceed)
    if (budget_ && in_use_ + sz > budget_)
        throw Error{XLOG_HIP_OOM, "GPU memory budget exceeded: requested " + std::to_string(sz) + " bytes with " +
                                      std::to_string(in_use_) + " in use, budget " + std::to_string(budget_)};
    auto it = free_.find(sz);
    void *p = nullptr;
    if (it != free_.end()) {
        p = it->second;
        free_.erase(it);
        cached_ -= sz;
    } else {
        if (budget_ && in_use_ + cached_ + sz > budget_) trim();  // the footprint stays within the budget
        hipError_t e = hipMalloc(&p, sz);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            trim();
            e = hipMalloc(&p, sz);
            if (e != hipSuccess) {
                (void)hipGetLastError();
                throw Error{XLOG_HIP_OOM, "device allocation of " + std::to_string(sz) + " bytes failed"};
            }
        }
    }
    live_[p] = sz;
    in_use_ += sz;
    if (in_use_ > peak_) peak_ = in_use_;
    return p;
}
void Pool::free(void *p) {
    if (!p) return;
    auto it = live_.find(p);
    if (it == live_.end()) return;
    size_t sz = it->second;
    live_.erase(it);
    in_use_ -= sz;
    free_.emplace(sz, p);
    cached_ += sz;
}
void Pool::trim() {
    (void)hipDeviceSynchronize();
    for (auto &kv : free_) (void)hipFree(kv.second);
    free_.clear();
    cached_ = 0;
}
Pool::~Pool() {
    (void)hipDeviceSynchronize();
    for (auto &kv : free_) (void)hipFree(kv.second);
    for (auto &kv : live_) (void)hipFree(kv.first);
}

namespace {
__global__ __launch_bounds__(256) void k_read_back(const uint64_t *__restrict__ src, uint32_t n, uint64_t *dst,
                                                   const uint64_t *__restrict__ also, uint64_t *seq, uint64_t v) {
    if (also && threadIdx.x == 0) dst[n] = *also;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) dst[i] = src[i];
    __threadfence_system();  // the words reach the host before the number does
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(seq, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace
void Ctx::post_read(const void *dev, size_t count_u64, const uint64_t *also) {
    XH_REQUIRE(count_u64 + (also ? 1 : 0) <= HOST_STAGE_U64, XLOG_HIP_INVALID_ARG,
               "read-back: more than the pinned staging holds");
    hipLaunchKernelGGL(k_read_back, dim3(1), dim3(count_u64 > 64 ? 256 : 64), 0, stream,
                       static_cast<const uint64_t *>(dev), (uint32_t)count_u64, host_scalars, also, host_seq,
                       ++read_seq);
    XH_CHECK_HIP(hipGetLastError());
}
void Ctx::wait_read() {
    ++host_waits;
    for (uint64_t spins = 1; __atomic_load_n(host_seq, __ATOMIC_ACQUIRE) != read_seq; ++spins) {
        __builtin_ia32_pause();
        if (spins % 4096) continue;
        // (now and then: a device error, or a stream that is done and has not stored the number)
        const hipError_t e = hipStreamQuery(stream);
        if (e == hipErrorNotReady) continue;
        XH_CHECK_HIP(e);
        XH_CHECK_HIP(hipStreamSynchronize(stream));
        XH_REQUIRE(__atomic_load_n(host_seq, __ATOMIC_ACQUIRE) == read_seq, XLOG_HIP_DEVICE_ERROR,
                   "read-back did not arrive");
    }
}

// ---------------------------------------------------------------------------
// small kernels used only by the host layer
// ---------------------------------------------------------------------------
namespace {

__global__ void k_widen(const uint32_t *__restrict__ c0, uint64_t n, uint64_t *__restrict__ out) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = c0[i];
}

// device view of a relation's words (or of any packed word arrays)
struct RelView {
    const uint64_t *w[MAX_WORDS];
    int arity;
};
struct RelOut {
    uint64_t *w[MAX_WORDS];
};
// value of column c (0..arity-1) of row i
__device__ __forceinline__ uint32_t col_value(const RelView &v, int c, uint64_t i) {
    if (v.arity == 1) return (uint32_t)v.w[0][i];
    const uint64_t x = v.w[c >> 1][i];
    return (c & 1) ? (uint32_t)x : (uint32_t)(x >> 32);
}
// Row i of a relation of the given arity from value(c), the value of its
// column c (called with uniform c: an array of a row's values, indexed by a
// run-time arity, would live in scratch memory: 4.2e6 rows joined into 6 columns
// took 275 us through one, 84 without).
template <class V>
__device__ __forceinline__ void put_row(const RelOut &o, int arity, uint64_t i, V value) {
    if (arity == 1) {
        o.w[0][i] = value(0);
        return;
    }
    for (int k = 0; 2 * k < arity; ++k)
        o.w[k][i] = ((uint64_t)value(2 * k) << 32) | (2 * k + 1 < arity ? value(2 * k + 1) : 0u);
}

struct ProjSpec {
    int in_arity, out_arity;
    int cols[MAX_ARITY];
};
__global__ void k_project(RelView in, uint64_t n, ProjSpec s, RelOut out) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        put_row(out, s.out_arity, i, [&](int c) { return col_value(in, s.cols[c], i); });
}

// OR of the words of a relation's rows (the bits its columns use), a word array
// per blockIdx.y
__global__ __launch_bounds__(256) void k_key_bits(RelView in, uint64_t n, unsigned long long *used) {
    constexpr int LD = 8;
    const uint64_t *w = in.w[blockIdx.y];
    const uint64_t stride = (uint64_t)gridDim.x * 256 * LD;
    uint64_t v = 0;
    for (uint64_t b = (uint64_t)blockIdx.x * 256 * LD + threadIdx.x; b < n; b += stride) {
        uint64_t x[LD];
#pragma unroll
        for (int q = 0; q < LD; ++q) x[q] = b + q * 256 < n ? w[b + q * 256] : 0ull;
#pragma unroll
        for (int q = 0; q < LD; ++q) v |= x[q];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, WAVE);
    __shared__ uint64_t s_v[4];
    if ((threadIdx.x & (WAVE - 1)) == 0) s_v[threadIdx.x >> 6] = v;
    __syncthreads();
    // (bits that another block has set already need no atomic)
    v = s_v[0] | s_v[1] | s_v[2] | s_v[3];
    if (threadIdx.x == 0 && (v & ~__hip_atomic_load(&used[blockIdx.y], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
        atomicOr(&used[blockIdx.y], (unsigned long long)v);
}
// group-start flags over sorted rows for the given key columns
__global__ void k_group_flags(RelView in, ProjSpec keys, uint64_t n, uint8_t *__restrict__ flags) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        bool f = (i == 0);
        if (!f)
            for (int j = 0; j < keys.out_arity; ++j)
                if (col_value(in, keys.cols[j], i) != col_value(in, keys.cols[j], i - 1)) f = true;
        flags[i] = f;
    }
}
__global__ void k_col_unsorted(RelView in, int c, uint64_t n, uint32_t *flag) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i + 1 < n; i += stride)
        if (col_value(in, c, i) > col_value(in, c, i + 1)) *flag = 1u;
}
// The largest word of n packed rows into *mx (atomicMax: *mx starts at 0 or
// at an earlier maximum).  One atomic per block; launched with at most
// 1024 blocks of 256 threads (MAX_LAUNCH_1D), so the atomics on the one
// address stay few.
__global__ __launch_bounds__(256) void k_max_u32_of_packed(const uint64_t *__restrict__ k, uint64_t n,
                                                           unsigned int *mx) {
    __shared__ unsigned int s_m[4];
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    unsigned int m = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        uint64_t x = k[i];
        unsigned a = (unsigned)(x >> 32), b = (unsigned)x;
        m = max(m, max(a, b));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
    if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(mx, max(max(s_m[0], s_m[1]), max(s_m[2], s_m[3])));
}
__global__ void k_u64_to_u32(const uint64_t *__restrict__ in, uint64_t n, uint32_t *__restrict__ out) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = (uint32_t)in[i];
}

}  // namespace

// defined in join.hip / tc_bitmap.hip
uint64_t join_probe_general(Ctx *ctx, const uint64_t *probe, uint64_t n, int pcol, const RunIndex &ix,
                            const uint32_t *payload, int out_arity, const int oc[4], uint64_t **out0,
                            uint64_t **out1);
void join_match_flags(Ctx *ctx, const uint64_t *probe, uint64_t n, int pcol, const RunIndex &ix, int want,
                      uint8_t *flags);
// the set of the key words pcol of n packed rows; a flag per row: its key is in the set (want 1) or not (0)
void key_set_build(Ctx *ctx, const uint64_t *rows, uint64_t n, int pcol, Buf<unsigned long long> &set);
void key_set_flags(Ctx *ctx, const uint64_t *rows, uint64_t n, int pcol, const Buf<unsigned long long> &set, int want,
                   uint8_t *flags);

#define LAUNCH_1D(kern, n, ...)                                                                             \
    do {                                                                                                    \
        if ((n) > 0) {                                                                                      \
            hipLaunchKernelGGL(kern, dim3(grid_for((n), 256, 16384)), dim3(256), 0, ctx->stream, __VA_ARGS__); \
            XH_CHECK_HIP(hipGetLastError());                                                                \
        }                                                                                                   \
    } while (0)
// LAUNCH_1D with at most 1024 blocks (grid-stride reductions into one word)
#define MAX_LAUNCH_1D(kern, n, ...)                                                                         \
    do {                                                                                                    \
        if ((n) > 0) {                                                                                      \
            hipLaunchKernelGGL(kern, dim3(grid_for((n), 256, 1024)), dim3(256), 0, ctx->stream, __VA_ARGS__);  \
            XH_CHECK_HIP(hipGetLastError());                                                                \
        }                                                                                                   \
    } while (0)

// ---------------------------------------------------------------------------
// relations
// ---------------------------------------------------------------------------
xlog_hip_rel *rel_new(Ctx *ctx, uint32_t arity, uint64_t cap) {
    XH_REQUIRE(arity >= 1 && arity <= MAX_ARITY, XLOG_HIP_INVALID_ARG, "relation arity must be 1..8");
    std::unique_ptr<xlog_hip_rel> r(new xlog_hip_rel());
    r->ctx = ctx;
    r->arity = arity;
    r->cap = cap;
    if (cap) {
        try {
            for (int k = 0; k < r->nwords(); ++k) r->w[k] = static_cast<uint64_t *>(ctx->alloc(cap * sizeof(uint64_t)));
        } catch (...) {
            for (int k = 0; k < MAX_WORDS; ++k) ctx->free(r->w[k]);
            throw;
        }
    }
    return r.release();
}
void rel_free(xlog_hip_rel *r) {
    if (!r) return;
    if (r->ctx)
        for (int k = 0; k < MAX_WORDS; ++k) r->ctx->free(r->w[k]);
    delete r;
}
static RelView view_of(const xlog_hip_rel *r) {
    RelView v{{r->w[0], r->w[1], r->w[2], r->w[3]}, (int)r->arity};
    return v;
}
static RelOut out_of(xlog_hip_rel *r) {
    RelOut o{{r->w[0], r->w[1], r->w[2], r->w[3]}};
    return o;
}
// (a, b) words -> (word h0, word h1) words of n packed pairs (h in {0, 1}: the
// high or the low word of the input)
void project_pairs(Ctx *ctx, const uint64_t *in, uint64_t n, int h0, int h1, uint64_t *out) {
    ProjSpec s{2, 2, {h0, h1, 0, 0, 0, 0, 0, 0}};
    RelView v{{in, nullptr, nullptr, nullptr}, 2};
    RelOut o{{out, nullptr, nullptr, nullptr}};
    LAUNCH_1D(k_project, n, v, n, s, o);
}
void max_u32_of_packed(Ctx *ctx, const uint64_t *k, uint64_t n, unsigned int *mx) {
    MAX_LAUNCH_1D(k_max_u32_of_packed, n, k, n, mx);
}
// adopt device buffers (ownership moves to the relation)
xlog_hip_rel *rel_adopt(Ctx *ctx, uint32_t arity, uint64_t rows, uint64_t *w0, uint64_t *w1, uint32_t flags) {
    xlog_hip_rel *r = new xlog_hip_rel();
    r->ctx = ctx;
    r->arity = arity;
    r->rows = rows;
    r->cap = rows;
    r->w[0] = w0;
    r->w[1] = w1;
    r->flags = flags;
    return r;
}
// packs device-resident u32 columns (arity 1..8) into the words of r
static void pack_device_columns(Ctx *ctx, const uint32_t *const *cols, uint32_t arity, uint64_t rows, xlog_hip_rel *r) {
    if (!rows) return;
    if (arity == 1) {
        LAUNCH_1D(k_widen, rows, cols[0], rows, r->w[0]);
        return;
    }
    for (int k = 0; k < words_for(arity); ++k)
        pack_columns(ctx, cols[2 * k], 2u * k + 1 < arity ? cols[2 * k + 1] : nullptr, rows, r->w[k]);
}
// adopt all words (ownership moves to the relation)
static xlog_hip_rel *rel_adopt_words(Ctx *ctx, uint32_t arity, uint64_t rows, uint64_t *const *w, uint32_t flags) {
    xlog_hip_rel *r = rel_adopt(ctx, arity, rows, w[0], w[1], flags);
    r->w[2] = w[2];
    r->w[3] = w[3];
    return r;
}
void copy_d2d(Ctx *ctx, uint64_t *dst, const uint64_t *src, uint64_t n) {
    if (n) XH_CHECK_HIP(hipMemcpyAsync(dst, src, n * sizeof(uint64_t), hipMemcpyDeviceToDevice, ctx->stream));
}
static xlog_hip_rel *rel_clone(Ctx *ctx, const xlog_hip_rel *in) {
    xlog_hip_rel *r = rel_new(ctx, in->arity, in->rows);
    r->rows = in->rows;
    r->flags = in->flags;
    for (int k = 0; k < in->nwords(); ++k) copy_d2d(ctx, r->w[k], in->w[k], in->rows);
    return r;
}

uint64_t read_count(Ctx *ctx, const uint64_t *d) {
    ctx->read_scalars(d, 1);
    return ctx->host_scalars[0];
}

uint64_t *alloc_keys(Ctx *ctx, uint64_t n) {
    return static_cast<uint64_t *>(ctx->alloc((n ? n : 1) * sizeof(uint64_t)));
}

std::vector<Bags> bags_per_pred(Ctx *ctx, uint32_t n) {
    std::vector<Bags> r;
    r.reserve(n);
    for (uint32_t i = 0; i < n; ++i) r.emplace_back(ctx);
    return r;
}

// ---------------------------------------------------------------------------
// sorting helpers
// ---------------------------------------------------------------------------

// Sort a u64 key array of any length; the result is returned in a buffer
// owned by the caller (either `keys` itself or a new one).  With keys_owned
// the call consumes `keys`: it is either returned or freed.
// digit_lo / digit_hi restrict the sort to 8-bit digits [lo, hi) (4..8 = by
// the high word only, stable otherwise).
uint64_t *sort_keys(Ctx *ctx, uint64_t *keys, uint64_t n, bool keys_owned, int digit_lo, int digit_hi,
                    uint32_t known_digits, bool *whole, int in_order) {
    if (whole) *whole = false;
    // a consumed input is freed if an error unwinds from here
    Owned in_guard(ctx, keys_owned ? keys : nullptr);
    if (n < 2) {
        if (keys_owned || n == 0) return in_guard.release();
        uint64_t *c = static_cast<uint64_t *>(ctx->alloc(n * sizeof(uint64_t)));
        copy_d2d(ctx, c, keys, n);
        return c;
    }
    const uint64_t CHUNK = 1ull << 29;
    if (n < (1ull << 30)) {
        Owned ga(ctx, keys_owned ? in_guard.release() : alloc_keys(ctx, n));
        Owned gb(ctx, alloc_keys(ctx, n));
        uint64_t *a = ga.p, *b = gb.p;
        // without keys_owned the first pass reads the caller's keys; both ping-pong buffers are ours
        radix_sort_u64(ctx, &a, &b, n, digit_lo, digit_hi, keys_owned ? nullptr : keys, known_digits,
                       nullptr, whole, in_order);
        ga.release();
        gb.release();
        ctx->free(b);
        return a;
    }
    XH_REQUIRE(digit_lo == 0 && digit_hi == 8, XLOG_HIP_UNSUPPORTED, "partial-key sort above 2^30 keys");
    // chunked: sort pieces of 2^29 then merge pairwise
    Owned ga(ctx, keys_owned ? in_guard.release() : alloc_keys(ctx, n));
    uint64_t *a = ga.p;
    if (!keys_owned) copy_d2d(ctx, a, keys, n);
    Owned gb(ctx, alloc_keys(ctx, n));
    uint64_t *b = gb.p;
    std::vector<std::pair<uint64_t, uint64_t>> runs;
    for (uint64_t s = 0; s < n; s += CHUNK) {
        uint64_t len = std::min(CHUNK, n - s);
        uint64_t *ka = a + s, *kb = b + s;
        radix_sort_u64(ctx, &ka, &kb, len, 0, 8, nullptr, known_digits);
        if (ka != a + s) copy_d2d(ctx, a + s, ka, len);
        runs.push_back({s, len});
    }
    uint64_t *src = a, *dst = b;
    while (runs.size() > 1) {
        std::vector<std::pair<uint64_t, uint64_t>> next;
        for (size_t i = 0; i < runs.size(); i += 2) {
            if (i + 1 < runs.size()) {
                merge_sorted(ctx, src + runs[i].first, runs[i].second, src + runs[i + 1].first, runs[i + 1].second,
                             dst + runs[i].first);
                next.push_back({runs[i].first, runs[i].second + runs[i + 1].second});
            } else {
                copy_d2d(ctx, dst + runs[i].first, src + runs[i].first, runs[i].second);
                next.push_back(runs[i]);
            }
        }
        runs.swap(next);
        std::swap(src, dst);
    }
    ga.release();
    gb.release();
    ctx->free(dst);
    return src;
}

// sorted (any) keys -> unique keys in a new buffer; returns count
static uint64_t unique_keys(Ctx *ctx, const uint64_t *sorted, uint64_t n, uint64_t **out) {
    Owned o(ctx, alloc_keys(ctx, n));
    Buf<uint64_t> cnt(ctx, 1);
    select_unique(ctx, sorted, n, o.p, cnt.p);
    const uint64_t c = read_count(ctx, cnt.p);
    *out = o.release();
    return c;
}

// Sorted unique copy of n keys (the caller's buffer is left as it is): returns
// the count, *out is a new buffer.  A large input whose high word splits it
// into short runs gets its unique keys from the fused short-run pass.
// known_digits: the digits the keys may vary in (0: unknown, the histograms decide)
void sort_unique_keys_async(Ctx *ctx, const uint64_t *keys, uint64_t n, uint64_t **out, uint64_t *d_count,
                            uint32_t known_digits) {
    if (n && n <= BLOCK_SORT_KEYS) {
        Owned o(ctx, alloc_keys(ctx, n));
        if (block_sort_unique(ctx, keys, n, o.p, d_count)) {
            *out = o.release();
            return;
        }
    }
    if (n >= 2 && n < (1ull << 30)) {
        Owned ga(ctx, alloc_keys(ctx, n)), gb(ctx, alloc_keys(ctx, n));
        uint64_t *a = ga.p, *b = gb.p;
        SortUnique uq;
        radix_sort_u64(ctx, &a, &b, n, 0, 8, keys, known_digits, &uq);
        ga.release();
        gb.release();
        Owned sorted(ctx, a), other(ctx, b);
        if (uq.done) {
            fill_u64(ctx, d_count, uq.count, 1);
            *out = sorted.release();
            return;
        }
        select_unique(ctx, a, n, b, d_count);
        *out = other.release();
        return;
    }
    uint64_t *s = sort_keys(ctx, const_cast<uint64_t *>(keys), n, false, 0, 8, known_digits);
    Owned gs(ctx, s != keys ? s : nullptr);
    Owned o(ctx, alloc_keys(ctx, n));
    select_unique(ctx, s, n, o.p, d_count);
    *out = o.release();
}
// The same by buckets: *d_count is ~0, and *out incomplete, when a bucket is too long for the route
bool bucket_unique_keys_async(Ctx *ctx, const uint64_t *keys, uint64_t n, uint64_t **out, uint64_t *d_count) {
    if (!bucket_sort_takes(n)) return false;
    Owned o(ctx, alloc_keys(ctx, n));
    Buf<uint64_t> st;
    if (!bucket_sort(ctx, keys, n, o.p, d_count, st)) return false;
    *out = o.release();
    return true;
}
// The same with the count read back (returned).
static uint64_t sort_unique_keys(Ctx *ctx, const uint64_t *keys, uint64_t n, uint64_t **out) {
    Buf<uint64_t> cnt(ctx, 1);
    if (bucket_unique_keys_async(ctx, keys, n, out, cnt.p)) {
        Owned o(ctx, *out);
        const uint64_t c = read_count(ctx, cnt.p);
        if (c != ~0ull) {
            o.release();
            return c;
        }
    }
    sort_unique_keys_async(ctx, keys, n, out, cnt.p);
    return read_count(ctx, cnt.p);
}

// Canonical (sorted, unique) copy of the packed keys of an arity<=2 relation
// or the relation's own buffer when it is already canonical (borrowed = true).
static void canonical_keys(Ctx *ctx, const xlog_hip_rel *r, Canon &c) {
    c.ctx = ctx;
    if (r->flags & REL_CANONICAL) {
        c.k = r->w[0];
        c.n = r->rows;
        return;
    }
    uint64_t *u;
    c.n = sort_unique_keys(ctx, r->w[0], r->rows, &u);
    c.owned = u;
    c.k = u;
}

// ---------------------------------------------------------------------------
// Stable sort of rows by key columns.  The columns' used bits, side by side and
// most significant first, are one number; its leading bits (as many as the row's
// number leaves in 64) and the row's number make a u64 key per row, and the u64
// sorts order those: one sort whatever the columns, all keys different, rows of
// equal prefix in input order.  Then one pass fetches the rows in that order
// (from a copy that holds a row's words together: one line a row, where word
// arrays cost one each), orders each run of equal prefix by the rest of the key
// when the prefix does not hold all of it, and writes rows and group flags.
// Runs of more than RUN_MAX rows it leaves out.  Their rows alone are sorted
// again, by (run, the key's next bits, row's number), and so on.  Where that
// would go on for long (most rows, runs that each bit splits little), the whole
// key is taken in pieces from its low end instead, one stable sort of (piece,
// row's number) each, by the piece's digits.
// (Dedup of 10^7 rows of four columns, 86 bits: four key + payload sorts with
// their gathers 2.3 ms, one prefix sort and this pass, 0.24 of it, 0.73.  Four
// hashed columns, 128 bits: 2.60 / 0.72 ms; the first with a value that a tenth
// of the rows have 2.60 / 1.47, with 100 values in all 2.59 / 2.02.  What gains
// nothing are hashed columns of a few values each, where 40 bits of the key tell
// as little as 10: 20 values in each 2.47 / 2.80, 10^6 rows 0.54 / 0.82.)
// ---------------------------------------------------------------------------
struct KeyBits {
    int n = 0, total = 0;
    int col[MAX_ARITY] = {0}, len[MAX_ARITY] = {0};  // distinct columns, bits they use
    bool known = true;                               // (or may use)
};
// bits [lo, lo + bits) of the number, at the top of 64; the row's number in row_bits from row_shift up
struct KeyPiece {
    int n = 0, bits = 0;
    int col[MAX_ARITY] = {0}, rs[MAX_ARITY] = {0}, ls[MAX_ARITY] = {0};
    uint32_t mask[MAX_ARITY] = {0};
    int row_bits = 0, row_shift = 0;
};
namespace {
// with aos: the row's W words together; with prev: of the rows that those words number (from prev_shift up); with
// group: the group's number (group[i + 1] - 1) above the piece
template <int W>
__global__ __launch_bounds__(256) void k_key_pieces(RelView in, KeyPiece kp, uint64_t n, uint64_t *__restrict__ out,
                                                    uint64_t *__restrict__ aos, const uint64_t *__restrict__ prev,
                                                    int prev_shift, const uint32_t *__restrict__ group,
                                                    int group_bits) {
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
        const uint64_t r = prev ? (prev[i] >> prev_shift) & ((1ull << kp.row_bits) - 1) : i;
        uint64_t w = r << kp.row_shift;
        for (int t = 0; t < kp.n; ++t)
            w |= (uint64_t)((col_value(in, kp.col[t], r) >> kp.rs[t]) & kp.mask[t]) << kp.ls[t];
        if (group) w |= (uint64_t)(group[i + 1] - 1) << (64 - group_bits);
        out[i] = w;
        if (aos) {
#pragma unroll
            for (int q = 0; q < W; ++q) aos[i * W + q] = in.w[q][r];
        }
    }
}
constexpr int ROWS_TB = 512, ROWS_TILE = 1024, RUN_MAX = 64;
// -1, 0, 1: the key columns of row a against those of row b
template <int W>
__device__ __forceinline__ int compare_rows(const uint64_t *a, const uint64_t *b, const KeyBits &kb, bool one) {
    for (int t = 0; t < kb.n; ++t) {
        const int c = kb.col[t], sh = one || (c & 1) ? 0 : 32;
        const uint32_t x = (uint32_t)(a[c >> 1] >> sh), y = (uint32_t)(b[c >> 1] >> sh);
        if (x != y) return x < y ? -1 : 1;
    }
    return 0;
}
// A tile takes the runs of equal prefix that start in it (ties: they are ordered
// by the whole key, and long ones left out; otherwise the order is final and a
// run is only a group).  With pos, row i of the order goes to place pos[i].
template <int W>
__global__ __launch_bounds__(ROWS_TB) void k_sorted_rows(const uint64_t *__restrict__ sorted, KeyPiece kp, uint64_t n,
                                                         const uint64_t *__restrict__ aos, KeyBits kb, int arity,
                                                         int ties, RelOut out, uint8_t *__restrict__ flags, uint64_t *d_long,
                                                         const uint32_t *__restrict__ pos) {
    constexpr int SPAN = ROWS_TILE + RUN_MAX + 1;  // (one past the longest run shows its end)
    __shared__ uint64_t s_key[SPAN];
    __shared__ uint64_t s_row[SPAN * W];
    const int tid = threadIdx.x;
    const uint64_t base = (uint64_t)blockIdx.x * ROWS_TILE;
    const int len = (int)(n - base < (uint64_t)SPAN ? n - base : (uint64_t)SPAN);
    const int own = len < ROWS_TILE ? len : ROWS_TILE;
    const uint64_t rmask = (1ull << kp.row_bits) - 1;
    auto prefix = [&](uint64_t w) { return kp.bits ? w >> (64 - kp.bits) : 0ull; };
    constexpr int LD = (SPAN + ROWS_TB - 1) / ROWS_TB;
    const int want = ties ? len : own;
    uint64_t w[LD];
#pragma unroll
    for (int q = 0; q < LD; ++q) w[q] = q * ROWS_TB + tid < len ? sorted[base + q * ROWS_TB + tid] : 0ull;
    uint64_t row[LD][W];
#pragma unroll
    for (int q = 0; q < LD; ++q)
#pragma unroll
        for (int j = 0; j < W; ++j)
            row[q][j] = q * ROWS_TB + tid < want ? aos[((w[q] >> kp.row_shift) & rmask) * W + j] : 0ull;
#pragma unroll
    for (int q = 0; q < LD; ++q)
        if (q * ROWS_TB + tid < len) {
            s_key[q * ROWS_TB + tid] = prefix(w[q]);
#pragma unroll
            for (int j = 0; j < W; ++j) s_row[(q * ROWS_TB + tid) * W + j] = row[q][j];
        }
    const uint64_t before = base ? prefix(sorted[base - 1]) : 0ull;  // prefix of the row before the tile
    __syncthreads();
    if (!ties) {
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const int i = q * ROWS_TB + tid;
            if (i >= own) continue;
            const uint64_t o = pos ? pos[base + i] : base + i;
#pragma unroll
            for (int j = 0; j < W; ++j) out.w[j][o] = row[q][j];
            if (flags) flags[o] = i ? s_key[i] != s_key[i - 1] : (base == 0 || s_key[0] != before);
        }
        return;
    }
    for (int i = tid; i < len; i += ROWS_TB) {
        const uint64_t k = s_key[i];
        int a = i;
        while (a > 0 && s_key[a - 1] == k && i - a <= RUN_MAX) --a;
        if (a == 0 && base && before == k) continue;  // the run started in an earlier tile
        if (a >= ROWS_TILE) continue;                 // it starts in the next tile
        int e = i + 1;
        while (e < len && s_key[e] == k && e - a <= RUN_MAX) ++e;
        if (e - a > RUN_MAX) {
            if ((uint32_t)__ffsll((unsigned long long)__ballot(true)) - 1 == (threadIdx.x & (WAVE - 1))) *d_long = 1;
            continue;
        }
        int rank = 0, same = 0;
        for (int j = a; j < e; ++j) {
            if (j == i) continue;
            const int c = compare_rows<W>(&s_row[j * W], &s_row[i * W], kb, arity == 1);
            rank += (c < 0 || (c == 0 && j < i)) ? 1 : 0;
            same |= (c == 0 && j < i) ? 1 : 0;
        }
        const uint64_t o = pos ? pos[base + a + rank] : base + a + rank;
#pragma unroll
        for (int j = 0; j < W; ++j) out.w[j][o] = s_row[i * W + j];
        if (flags) flags[o] = !same;
    }
}
// the rows that words number (row_shift 0), and a word array in that order
__global__ void k_rows_of(const uint64_t *__restrict__ words, int row_bits, uint64_t n, uint32_t *__restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = (uint32_t)(words[i] & ((1ull << row_bits) - 1));
}
__global__ void k_take_rows(const uint64_t *__restrict__ in, const uint32_t *__restrict__ rows, uint64_t n,
                            uint64_t *__restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = in[rows[i]];
}
// in_long[i] = 1 for the sorted words whose run of equal prefix has more than RUN_MAX (in_long[n] = 0: n + 1 entries)
__global__ void k_long_runs(const uint64_t *__restrict__ sorted, KeyPiece kp, uint64_t n,
                            uint32_t *__restrict__ in_long) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const int shift = 64 - kp.bits;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i <= n; i += stride) {
        uint32_t is_long = 0;
        if (i < n) {
            const uint64_t k = sorted[i] >> shift;
            uint64_t lo = i > (uint64_t)RUN_MAX ? i - RUN_MAX : 0, hi = i;  // the run's first, as far back as matters
            while (lo < hi) {
                const uint64_t mid = (lo + hi) >> 1;
                if ((sorted[mid] >> shift) == k) hi = mid; else lo = mid + 1;
            }
            is_long = lo + RUN_MAX < n && (sorted[lo + RUN_MAX] >> shift) == k;
        }
        in_long[i] = is_long;
    }
}
// the words of long runs (in_long: scanned) with their places, and head = 1 where a run begins (m + 1 entries)
__global__ void k_long_take(const uint64_t *__restrict__ sorted, KeyPiece kp, uint64_t n,
                            const uint32_t *__restrict__ in_long, const uint32_t *__restrict__ pos,
                            uint64_t *__restrict__ out, uint32_t *__restrict__ out_pos, uint32_t *__restrict__ head) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const int shift = 64 - kp.bits;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint32_t q = in_long[i];
        if (i == 0) head[in_long[n]] = 0;
        if (in_long[i + 1] == q) continue;
        out[q] = sorted[i];
        out_pos[q] = pos ? pos[i] : (uint32_t)i;
        head[q] = i == 0 || (sorted[i] >> shift) != (sorted[i - 1] >> shift);
    }
}
}  // namespace
// The columns of a key list, most significant first, each once, and the bits
// they use over the relation (one read-back).
static KeyBits key_bits(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols) {
    KeyBits kb;
    for (int c : cols)
        if (std::find(kb.col, kb.col + kb.n, c) == kb.col + kb.n) kb.col[kb.n++] = c;
    if (kb.n == 1 && in->nwords() == 1) {  // the sort's own histograms tell as much
        kb.len[0] = kb.total = 32;
        kb.known = false;
        return kb;
    }
    Buf<unsigned long long> used(ctx, MAX_WORDS);
    fill_u64(ctx, reinterpret_cast<uint64_t *>(used.p), 0ull, MAX_WORDS);
    hipLaunchKernelGGL(k_key_bits, dim3(grid_for(in->rows, 256 * 8, 256), in->nwords()), dim3(256), 0, ctx->stream,
                       view_of(in), in->rows, used.p);
    XH_CHECK_HIP(hipGetLastError());
    ctx->read_scalars(used.p, MAX_WORDS);
    for (int t = 0; t < kb.n; ++t) {
        const uint64_t w = ctx->host_scalars[kb.col[t] >> 1];
        const uint32_t u = in->arity == 1 || (kb.col[t] & 1) ? (uint32_t)w : (uint32_t)(w >> 32);
        kb.len[t] = u ? 32 - __builtin_clz(u) : 0;
        kb.total += kb.len[t];
    }
    return kb;
}
// (above: bits that the caller puts above the piece)
static KeyPiece key_piece(const KeyBits &kb, int lo, int bits, uint64_t n, int above = 0) {
    KeyPiece kp;
    kp.bits = above + bits;
    while (kp.row_bits < 31 && (1ull << kp.row_bits) < n) ++kp.row_bits;
    kp.row_shift = 64 - kp.bits - kp.row_bits;
    int at = kb.total;  // bit above the column
    for (int t = 0; t < kb.n; ++t) {
        at -= kb.len[t];
        const int a = std::max(at, lo), b = std::min(at + kb.len[t], lo + bits);
        if (a >= b) continue;
        kp.col[kp.n] = kb.col[t];
        kp.rs[kp.n] = a - at;
        kp.mask[kp.n] = b - a == 32 ? 0xFFFFFFFFu : (1u << (b - a)) - 1u;
        kp.ls[kp.n++] = 64 - kp.bits + (a - lo);
    }
    return kp;
}
// The long runs of an order by kp's words (sorted, n of them, places pos or
// their own): their words, places and group numbers (one more than each, in
// group[1 ..]).  Returns their number.
struct LongRuns {
    Buf<uint64_t> words;
    Buf<uint32_t> pos, group;
    uint64_t n = 0, groups = 0;
};
static void long_runs(Ctx *ctx, const uint64_t *sorted, const KeyPiece &kp, uint64_t n, const uint32_t *pos,
                      LongRuns &out) {
    Buf<uint32_t> in_long(ctx, n + 1);
    Buf<unsigned long long> sum(ctx, 1);
    LAUNCH_1D(k_long_runs, n + 1, sorted, kp, n, in_long.p);
    scan_u32_inplace(ctx, in_long.p, n + 1, sum.p);
    out.n = read_count(ctx, reinterpret_cast<const uint64_t *>(sum.p));
    out.words = Buf<uint64_t>(ctx, out.n);
    out.pos = Buf<uint32_t>(ctx, out.n);
    out.group = Buf<uint32_t>(ctx, out.n + 1);
    LAUNCH_1D(k_long_take, n, sorted, kp, n, in_long.p, pos, out.words.p, out.pos.p, out.group.p);
    scan_u32_inplace(ctx, out.group.p, out.n + 1, sum.p);
    out.groups = read_count(ctx, reinterpret_cast<const uint64_t *>(sum.p));
}
typedef std::unique_ptr<xlog_hip_rel, void (*)(xlog_hip_rel *)> RelOwner;
template <int W>
static void fetch_rows(Ctx *ctx, const xlog_hip_rel *in, const KeyBits &kb, const uint64_t *w, const KeyPiece &kp,
                       uint64_t n, const uint64_t *aos, bool ties, xlog_hip_rel *out, uint8_t *flags,
                       uint64_t *d_long, const uint32_t *pos) {
    hipLaunchKernelGGL(k_sorted_rows<W>, dim3((unsigned)((n + ROWS_TILE - 1) / ROWS_TILE)), dim3(ROWS_TB), 0,
                       ctx->stream, w, kp, n, W > 1 ? aos : in->w[0], kb, (int)in->arity, ties ? 1 : 0, out_of(out),
                       flags, d_long, pos);
    XH_CHECK_HIP(hipGetLastError());
}
// By prefixes; false where pieces of the whole key are the better way on.  The
// rows to o (allocated here), their copy to aos, where one is made.
template <int W>
static bool rows_by_prefix(Ctx *ctx, const xlog_hip_rel *in, const KeyBits &kb, uint8_t *flags, RelOwner &o,
                           Buf<uint64_t> &aos) {
    const uint64_t n = in->rows;
    o.reset(rel_new(ctx, in->arity, n));
    o->rows = n;
    KeyPiece kp = key_piece(kb, 0, 0, n);
    const int room = 64 - kp.row_bits;
    int left = std::max(0, kb.total - room);  // bits of the key below the prefix
    kp = key_piece(kb, left, kb.total - left, n);
    if (W > 1) aos = Buf<uint64_t>(ctx, n * W);
    Buf<uint64_t> d_long(ctx, 1);
    Owned w(ctx, alloc_keys(ctx, n));
    LAUNCH_1D(k_key_pieces<W>, n, view_of(in), kp, n, w.p, W > 1 ? aos.p : nullptr, nullptr, 0, nullptr, 0);
    LongRuns runs;
    for (uint64_t m = n;;) {
        // (the words are all different; rows of equal prefix are in order)
        // Short prefixes take the passes of their digits (10^6 rows by a column of 200 values 127 us by buckets, 68 so;
        // of 5,000 128 / 88; of 32 bits 132 / 125, but 10^5 rows 69 / 95).
        const int digit = std::min(7, (64 - kp.bits) / 8);
        if (m > BLOCK_SORT_KEYS && !kb.known)
            w.reset(sort_keys(ctx, w.release(), m, true, digit, 8));
        else if (m > BLOCK_SORT_KEYS && (digit > 4 || (digit == 4 && m > (1ull << 18))))
            w.reset(sort_keys(ctx, w.release(), m, true, digit, 8, 0xFFu & ~((1u << digit) - 1u)));
        else
            w.reset(sort_keys(ctx, w.release(), m, true, 0, 8, 0, nullptr, digit));
        if (left) fill_u64(ctx, d_long.p, 0ull, 1);
        const uint32_t *pos = m < n ? runs.pos.p : nullptr;
        fetch_rows<W>(ctx, in, kb, w.p, kp, m, aos.p, left > 0, o.get(), flags, d_long.p, pos);
        if (!left || read_count(ctx, d_long.p) == 0) return true;
        LongRuns next;
        long_runs(ctx, w.p, kp, m, pos, next);
        int gbits = 0;
        while ((1ull << gbits) < next.groups) ++gbits;
        const int bits = std::min(left, room - gbits);
        // (how many bits would make the runs short, if the rest of the key splits them as the bits so far did)
        const double split = std::log2((double)next.groups) / (kb.total - left);
        if (bits < std::min(left, 8) || (2 * next.n > n && next.groups >= 16 &&
                                         std::log2((double)next.n / next.groups / (RUN_MAX / 2)) > split * bits))
            return false;
        const int shift = kp.row_shift;
        left -= bits;
        kp = key_piece(kb, left, bits, n, gbits);
        runs = std::move(next);
        m = runs.n;
        w.reset();
        w.reset(alloc_keys(ctx, m));
        LAUNCH_1D(k_key_pieces<W>, m, view_of(in), kp, m, w.p, nullptr, runs.words.p, shift,
                  gbits ? runs.group.p : nullptr, gbits);
    }
}
// By pieces of whole bytes, as many as the row's number leaves and of about
// equal length: two buffers of keys, then the rows and four bytes for each of
// them (o and aos when they are there already).
template <int W>
static void rows_by_pieces(Ctx *ctx, const xlog_hip_rel *in, const KeyBits &kb, uint8_t *flags, RelOwner &o,
                           const Buf<uint64_t> &aos) {
    const uint64_t n = in->rows;
    KeyPiece kp = key_piece(kb, 0, 0, n);
    const int most = (64 - kp.row_bits) & ~7, pieces = std::max(1, (kb.total + most - 1) / most),
              step = ((kb.total + pieces - 1) / pieces + 7) & ~7;
    Owned w(ctx);
    for (int p = 0; p < pieces; ++p) {
        kp = key_piece(kb, p * step, std::min(step, kb.total - p * step), n);
        kp.row_shift = 0;
        Owned next(ctx, alloc_keys(ctx, n));
        LAUNCH_1D(k_key_pieces<W>, n, view_of(in), kp, n, next.p, nullptr, p ? w.p : nullptr, 0, nullptr, 0);
        w.reset();
        const int digit = (64 - kp.bits) / 8;
        w.reset(sort_keys(ctx, next.release(), n, true, digit, 8, 0xFFu & ~((1u << digit) - 1u)));
    }
    if (o) {
        kp.bits = 0;  // (the order is final)
        fetch_rows<W>(ctx, in, kb, w.p, kp, n, aos.p, false, o.get(), nullptr, nullptr, nullptr);
    } else {
        Buf<uint32_t> order(ctx, n);
        LAUNCH_1D(k_rows_of, n, w.p, kp.row_bits, n, order.p);
        w.reset();
        o.reset(rel_new(ctx, in->arity, n));
        o->rows = n;
        for (int q = 0; q < W; ++q) LAUNCH_1D(k_take_rows, n, in->w[q], order.p, n, o->w[q]);
    }
    if (flags) {
        ProjSpec ks{(int)in->arity, kb.n, {0}};
        for (int t = 0; t < kb.n; ++t) ks.cols[t] = kb.col[t];
        LAUNCH_1D(k_group_flags, n, view_of(o.get()), ks, n, flags);
    }
}
// Rows of `in` sorted by kb's columns (stable).  With flags: 1 for the first row
// of every group of rows equal on those columns.
template <int W>
static xlog_hip_rel *sorted_rows(Ctx *ctx, const xlog_hip_rel *in, const KeyBits &kb, uint8_t *flags) {
    RelOwner o(nullptr, rel_free);
    Buf<uint64_t> aos;
    bool done = false;
    if (!fits_memory([&] { done = rows_by_prefix<W>(ctx, in, kb, flags, o, aos); })) {
        o.reset();
        aos = Buf<uint64_t>();
    }
    if (!done) rows_by_pieces<W>(ctx, in, kb, flags, o, aos);
    return o.release();
}
static xlog_hip_rel *sort_rows(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols, uint8_t *flags) {
    XH_REQUIRE(in->rows < (1ull << 30), XLOG_HIP_CAPACITY_OVERFLOW, "sort: keyed sort limited to 2^30 rows");
    const KeyBits kb = key_bits(ctx, in, cols);
    switch (in->nwords()) {
        case 1: return sorted_rows<1>(ctx, in, kb, flags);
        case 2: return sorted_rows<2>(ctx, in, kb, flags);
        case 3: return sorted_rows<3>(ctx, in, kb, flags);
        default: return sorted_rows<4>(ctx, in, kb, flags);
    }
}

static bool is_full_key(const xlog_hip_rel *in, const std::vector<int> &cols) {
    std::vector<int> uniq;
    for (int c : cols)
        if (std::find(uniq.begin(), uniq.end(), c) == uniq.end()) uniq.push_back(c);
    if (uniq.size() != in->arity) return false;
    for (size_t i = 0; i < uniq.size(); ++i)
        if (uniq[i] != (int)i) return false;
    return true;
}

static std::vector<int> check_cols(const xlog_hip_rel *in, const uint32_t *cols, uint32_t n) {
    XH_REQUIRE(n == 0 || cols, XLOG_HIP_INVALID_ARG, "key column list is NULL");
    std::vector<int> v;
    for (uint32_t i = 0; i < n; ++i) {
        XH_REQUIRE(cols[i] < in->arity, XLOG_HIP_INVALID_ARG,
                   "key column " + std::to_string(cols[i]) + " out of range for arity " + std::to_string(in->arity));
        v.push_back((int)cols[i]);
    }
    return v;
}

static xlog_hip_rel *op_sort(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols) {
    if (in->rows < 2 || cols.empty()) return rel_clone(ctx, in);
    if (in->arity <= 2 && is_full_key(in, cols)) {
        if (in->flags & REL_CANONICAL) return rel_clone(ctx, in);
        uint64_t *s = sort_keys(ctx, in->w[0], in->rows, false);
        return rel_adopt(ctx, in->arity, in->rows, s, nullptr, 0);
    }
    return sort_rows(ctx, in, cols, nullptr);
}

static xlog_hip_rel *compact_rel(Ctx *ctx, const xlog_hip_rel *in, const uint8_t *flags) {
    Buf<uint64_t> cnt(ctx, in->nwords());
    Buf<uint64_t> o[MAX_WORDS];
    for (int k = 0; k < in->nwords(); ++k) {
        o[k] = Buf<uint64_t>(ctx, in->rows ? in->rows : 1);
        select_flags(ctx, in->w[k], flags, in->rows, o[k].p, cnt.p + k);
    }
    uint64_t n = read_count(ctx, cnt.p);
    uint64_t *w[MAX_WORDS] = {o[0].release(), o[1].release(), o[2].release(), o[3].release()};
    return rel_adopt_words(ctx, in->arity, n, w, 0);
}

// the first row of every group of rows equal on cols, sorted by cols
static xlog_hip_rel *dedup_rows(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols) {
    if (in->rows < 2) return rel_clone(ctx, in);
    Buf<uint8_t> flags(ctx, in->rows);
    std::unique_ptr<xlog_hip_rel, void (*)(xlog_hip_rel *)> s(sort_rows(ctx, in, cols, flags.p), rel_free);
    return compact_rel(ctx, s.get(), flags.p);
}

static xlog_hip_rel *op_dedup_full(Ctx *ctx, const xlog_hip_rel *in) {
    if (in->flags & REL_CANONICAL) return rel_clone(ctx, in);
    if (in->arity <= 2) {
        uint64_t *u;
        const uint64_t n = sort_unique_keys(ctx, in->w[0], in->rows, &u);
        return rel_adopt(ctx, in->arity, n, u, nullptr, REL_CANONICAL);
    }
    std::vector<int> all;
    for (uint32_t c = 0; c < in->arity; ++c) all.push_back((int)c);
    xlog_hip_rel *r = dedup_rows(ctx, in, all);
    r->flags = REL_CANONICAL;
    return r;
}

static xlog_hip_rel *op_dedup(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols) {
    if (is_full_key(in, cols)) return op_dedup_full(ctx, in);
    XH_REQUIRE(!cols.empty(), XLOG_HIP_INVALID_ARG, "dedup needs at least one key column");
    xlog_hip_rel *r = dedup_rows(ctx, in, cols);
    r->flags = 0;
    return r;
}

static xlog_hip_rel *op_union_many(Ctx *ctx, const xlog_hip_rel *const *ins, uint32_t n) {
    XH_REQUIRE(n >= 1 && ins, XLOG_HIP_INVALID_ARG, "union needs at least one input");
    uint32_t arity = ins[0]->arity;
    uint64_t total = 0;
    for (uint32_t i = 0; i < n; ++i) {
        XH_REQUIRE(ins[i], XLOG_HIP_INVALID_ARG, "union input is NULL");
        XH_REQUIRE(ins[i]->arity == arity, XLOG_HIP_TYPE_MISMATCH, "union inputs have different arity");
        total += ins[i]->rows;
    }
    if (arity <= 2 && n == 2 && (ins[0]->flags & ins[1]->flags & REL_CANONICAL)) {
        // Sets that share nothing (an iteration's new rows and the relation they were checked against) are united
        // by the merge alone; the unique pass queued after it ends at once unless the merge found a shared key.
        Owned m(ctx, alloc_keys(ctx, total)), u(ctx, alloc_keys(ctx, total));
        if (total == 0) return rel_adopt(ctx, arity, 0, m.release(), nullptr, REL_CANONICAL);
        Buf<uint64_t> res(ctx, 2);
        merge_unique_sorted(ctx, ins[0]->w[0], ins[0]->rows, ins[1]->w[0], ins[1]->rows, m.p, u.p, res.p);
        ctx->read_scalars(res.p, 2);
        const bool apart = ctx->host_scalars[0] == 0;
        const uint64_t cnt = apart ? total : ctx->host_scalars[1];
        return rel_adopt(ctx, arity, cnt, apart ? m.release() : u.release(), nullptr, REL_CANONICAL);
    }
    xlog_hip_rel *cat = rel_new(ctx, arity, total);
    cat->rows = total;
    uint64_t off = 0;
    for (uint32_t i = 0; i < n; ++i) {
        for (int k = 0; k < cat->nwords(); ++k) copy_d2d(ctx, cat->w[k] + off, ins[i]->w[k], ins[i]->rows);
        off += ins[i]->rows;
    }
    xlog_hip_rel *r = op_dedup_full(ctx, cat);
    rel_free(cat);
    return r;
}

static xlog_hip_rel *op_diff(Ctx *ctx, const xlog_hip_rel *a, const xlog_hip_rel *b) {
    XH_REQUIRE(a->arity == b->arity, XLOG_HIP_TYPE_MISMATCH, "diff inputs have different arity");
    XH_REQUIRE(a->arity <= 2, XLOG_HIP_UNSUPPORTED, "diff: arity above 2 is not supported");
    Canon ca, cb;
    canonical_keys(ctx, a, ca);
    canonical_keys(ctx, b, cb);
    uint64_t *o = static_cast<uint64_t *>(ctx->alloc((ca.n ? ca.n : 1) * sizeof(uint64_t)));
    Buf<uint64_t> cnt(ctx, 1);
    if (!diff_by_merge_takes(ca.n, cb.n) || !diff_by_merge(ctx, ca.k, ca.n, cb.k, cb.n, o, cnt.p))
        select_unique_diff(ctx, ca.k, ca.n, cb.k, cb.n, o, cnt.p);
    uint64_t n = read_count(ctx, cnt.p);
    return rel_adopt(ctx, a->arity, n, o, nullptr, REL_CANONICAL);
}

// The build side of a join on a key list, folded into dense ids (see
// op_join_keys): one sorted unique u64 key array per folding step, in which
// the probe side's keys are ranked, and the run index over (id << 32) | row.
struct KeyFold {
    std::vector<Buf<uint64_t>> dict;
    std::vector<uint64_t> dict_n;
    JoinIndex J;
};
}  // namespace xh
// Reusable join index handle of the C ABI (one build, many probes): one key
// column of a relation of at most two columns is indexed directly (J, runs of
// that column's values, payload = the other column); any other key list is
// folded (F).
struct xlog_hip_join_index {
    xh::Ctx *ctx = nullptr;
    xh::JoinIndex J;
    std::unique_ptr<xh::KeyFold> F;
    uint32_t arity = 0;
    std::vector<uint32_t> keys;
    uint64_t rows = 0;
};
namespace xh {
// payload_sorted: the payload order inside a run is ascending; unique_rows
// (implies payload_sorted): duplicate (key, payload) rows are dropped, so a
// run's payloads are distinct (set-semantics callers only).
void build_join_index(Ctx *ctx, const uint64_t *keys, uint64_t n, uint32_t arity, int col, bool canonical,
                      JoinIndex &J, bool payload_sorted, bool unique_rows) {
    if (unique_rows) payload_sorted = true;
    J.n = n;
    uint64_t *sk = nullptr;
    bool own = false;
    // Runs of equal keys must be contiguous; unless payload_sorted is asked
    // for, the payload order inside a run is irrelevant and only the key word
    // (digits 4..7) is sorted.
    const int dlo = payload_sorted ? 0 : 4;
    if (arity == 1) {
        // (c0 << 32) | 0
        sk = static_cast<uint64_t *>(ctx->alloc((n ? n : 1) * sizeof(uint64_t)));
        swap_words(ctx, keys, n, sk);
        own = true;
        sk = sort_keys(ctx, sk, n, true, 4, 8);
    } else if (col == 0) {
        if (canonical) sk = const_cast<uint64_t *>(keys);
        else { sk = sort_keys(ctx, const_cast<uint64_t *>(keys), n, false, dlo, 8); own = true; }
    } else {
        sk = static_cast<uint64_t *>(ctx->alloc((n ? n : 1) * sizeof(uint64_t)));
        swap_words(ctx, keys, n, sk);
        own = true;
        sk = sort_keys(ctx, sk, n, true, dlo, 8);
    }
    if (unique_rows && n > 1 && !(canonical && col == 0 && arity == 2)) {
        uint64_t *u;
        const uint64_t un = unique_keys(ctx, sk, n, &u);
        if (own) ctx->free(sk);
        sk = u;
        own = true;
        n = un;
        J.n = un;
    }
    build_run_index(ctx, sk, n, J.ix);
    J.payload = Buf<uint32_t>(ctx, n ? n : 1);
    low_words(ctx, sk, n, J.payload.p);
    if (own) ctx->free(sk);
}

// Join step of a rule body with bounded memory.  A probe output of at most
// kChunkRows rows (default 2^30 - 1: 8 GiB of packed rows, one radix sort
// call) is emitted whole (a bag).  A larger one is emitted in tile
// ranges of at most kChunkRows rows; each range is sorted and deduplicated and
// merged into the result, which is then a sorted set.  Rule bodies only feed
// set operations (union, diff), so either form gives the same fixpoint, and
// duplicate-heavy joins (points-to hubs) no longer materialise their bag.
// XLOG_HIP_JOIN_CHUNK_ROWS overrides the chunk size (tests force multi-chunk
// folds with it, like the reference's XLOG_UNION_CHUNK_BYTES, relational.rs:36-42).
static uint64_t join_chunk_rows() {
    const char *e = getenv("XLOG_HIP_JOIN_CHUNK_ROWS");
    if (e && *e) {
        unsigned long long v = strtoull(e, nullptr, 10);
        if (v > 0) return v;
    }
    return (1ull << 30) - 1;
}
// XLOG_HIP_TRACE=1: one line on stderr per fixpoint iteration, per queue of
// iterations and per piece of a large join step (progress of long runs).
bool trace_on() {
    const char *e = getenv("XLOG_HIP_TRACE");
    return e && e[0] == '1';
}

// The emit side of a join step whose count pass has run (job.total known).
// digits: the sort's known varying digits (0: from the histograms).
uint64_t join_emit(Ctx *ctx, ProbeJob &job, const int oc[4], uint64_t **out, uint64_t max_rows, uint32_t digits) {
    const uint64_t kChunkRows = join_chunk_rows();
    const uint64_t total = job.total;
    *out = nullptr;
    if (total == 0) return 0;
    // the bag size is known before anything is materialised (the reference
    // refuses joins above its u32 row limit at the same point, relational.rs:4550-4555)
    XH_REQUIRE(max_rows == 0 || total <= max_rows, XLOG_HIP_CAPACITY_OVERFLOW,
               "Join produced " + std::to_string(total) + " rows which exceeds the row limit " +
                   std::to_string(max_rows));
    if (total <= kChunkRows) {
        uint64_t *o = static_cast<uint64_t *>(ctx->alloc(total * sizeof(uint64_t)));
        Owned go(ctx, o);
        probe_emit_range(ctx, job, 0, job.tiles, total, 2, oc, o, nullptr);
        *out = go.release();
        return total;
    }
    std::vector<uint64_t> off = probe_tile_offsets(ctx, job);
    Owned acc(ctx);
    uint64_t acc_n = 0;
    for (uint64_t t0 = 0; t0 < job.tiles;) {
        uint64_t t1 = t0 + 1;
        while (t1 < job.tiles && off[t1 + 1] - off[t0] <= kChunkRows) ++t1;
        const uint64_t m = off[t1] - off[t0];
        if (trace_on())
            fprintf(stderr, "[xlog_hip] join step of %llu rows: piece of %llu rows from tile %llu of %llu\n",
                    (unsigned long long)total, (unsigned long long)m, (unsigned long long)t0,
                    (unsigned long long)job.tiles);
        if (m) {
            uint64_t *b = static_cast<uint64_t *>(ctx->alloc(m * sizeof(uint64_t)));
            {
                Owned gb(ctx, b);
                probe_emit_range(ctx, job, t0, t1, m, 2, oc, b, nullptr);
                gb.release();
            }
            Owned srt(ctx, sort_keys(ctx, b, m, true, 0, 8, digits));  // consumes b
            uint64_t *u;
            uint64_t un = unique_keys(ctx, srt.p, m, &u);
            Owned gu(ctx, u);
            srt.reset();
            if (!acc.p) {
                acc.reset(gu.release());
                acc_n = un;
            } else {
                Owned mg(ctx, alloc_keys(ctx, acc_n + un));
                merge_sorted(ctx, acc.p, acc_n, u, un, mg.p);
                acc.reset();
                gu.reset();
                uint64_t *u2;
                uint64_t n2 = unique_keys(ctx, mg.p, acc_n + un, &u2);
                acc.reset(u2);
                acc_n = n2;
            }
        }
        t0 = t1;
    }
    *out = acc.release();
    return acc_n;
}
uint64_t join_step(Ctx *ctx, const uint64_t *probe, uint64_t n, int pcol, const JoinIndex &J, const int oc[4],
                   uint64_t **out, uint64_t max_rows, uint32_t digits) {
    ProbeJob job;
    job.probe = probe;
    job.n = n;
    job.pcol = pcol;
    job.ix = &J.ix;
    job.payload = J.payload.p;
    *out = nullptr;
    if (probe_prepare(ctx, job) == 0) return 0;
    return join_emit(ctx, job, oc, out, max_rows, digits);
}

// value-index of a relation column for the probe side: arity 1 stores c0 in
// the low word (v1), arity 2 stores c0 high (v0) and c1 low (v1)
static int probe_vidx(uint32_t arity, uint32_t c) { return arity == 1 ? 1 : (int)c; }

// The output values of a join of relations of at most two columns, as indexes
// 0..3 into (probe c0, probe c1, key, payload): left ++ right, or out_cols of
// it.  Returns the output's arity.
static int join_values(const xlog_hip_rel *l, uint32_t r_arity, uint32_t rk, const std::vector<int> *out_cols,
                       int oc[4]) {
    std::vector<int> vmap;
    for (uint32_t c = 0; c < l->arity; ++c) vmap.push_back(probe_vidx(l->arity, c));
    for (uint32_t c = 0; c < r_arity; ++c) vmap.push_back(c == rk ? 2 : 3);
    std::vector<int> sel;
    if (out_cols) {
        for (int c : *out_cols) {
            XH_REQUIRE(c >= 0 && c < (int)vmap.size(), XLOG_HIP_INVALID_ARG, "projection column out of range");
            sel.push_back(vmap[c]);
        }
    } else {
        sel = vmap;
    }
    XH_REQUIRE(!sel.empty() && sel.size() <= 4, XLOG_HIP_UNSUPPORTED, "join output arity must be 1..4");
    for (size_t i = 0; i < sel.size(); ++i) oc[i] = sel[i];
    return (int)sel.size();
}

// SEMI / ANTI: the rows of l whose key is / is not among the right side's (the
// key words pcol of l's probe rows and rcol of the right rows).  Only the keys
// matter, so they go into a hash set as they are: no sort, no runs.
static xlog_hip_rel *key_set_join(Ctx *ctx, const xlog_hip_rel *l, const uint64_t *probe, int pcol,
                                  const uint64_t *rows, uint64_t nr, int rcol, int type, bool canonical) {
    Buf<unsigned long long> set;
    key_set_build(ctx, rows, nr, rcol, set);
    Buf<uint8_t> flags(ctx, l->rows);
    key_set_flags(ctx, probe, l->rows, pcol, set, type == XLOG_HIP_JOIN_SEMI, flags.p);
    xlog_hip_rel *o = compact_rel(ctx, l, flags.p);
    if (canonical) o->flags = REL_CANONICAL;  // a subset of a sorted set is one
    return o;
}

// Join of `l` against an index built over column rk of a relation of arity
// r_arity.  max_output > 0 keeps the first max_output rows of the output
// (row order: probe-row major).
static xlog_hip_rel *op_join_indexed(Ctx *ctx, const xlog_hip_rel *l, uint32_t lk, const JoinIndex &J, uint32_t r_arity,
                                     uint32_t rk, int type, const std::vector<int> *out_cols, uint64_t max_output = 0) {
    XH_REQUIRE(lk < l->arity, XLOG_HIP_INVALID_ARG, "join key column out of range");
    XH_REQUIRE(l->arity <= 2, XLOG_HIP_UNSUPPORTED, "join: input arity above 2 is not supported");
    const int pcol = probe_vidx(l->arity, lk);
    if (type == XLOG_HIP_JOIN_SEMI || type == XLOG_HIP_JOIN_ANTI) {
        Buf<uint8_t> flags(ctx, l->rows ? l->rows : 1);
        join_match_flags(ctx, l->w[0], l->rows, pcol, J.ix, type == XLOG_HIP_JOIN_SEMI, flags.p);
        return compact_rel(ctx, l, flags.p);
    }
    XH_REQUIRE(type == XLOG_HIP_JOIN_INNER, XLOG_HIP_INVALID_ARG, "unknown join type");
    int oc[4] = {0, 0, 0, 0};
    const int out_arity = join_values(l, r_arity, rk, out_cols, oc);
    uint64_t *o0 = nullptr, *o1 = nullptr;
    uint64_t n = join_probe_general(ctx, l->w[0], l->rows, pcol, J.ix, J.payload.p, out_arity, oc, &o0, &o1);
    if (n == 0) return rel_new(ctx, (uint32_t)out_arity, 0);
    if (max_output && n > max_output) n = max_output;
    return rel_adopt(ctx, (uint32_t)out_arity, n, o0, o1, 0);
}

static xlog_hip_rel *op_join_keys(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, const std::vector<int> &lk,
                                  const std::vector<int> &rk, int type);
static xlog_hip_rel *op_project(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols);

// ---------------------------------------------------------------------------
// Equi-join on lists of key columns, inputs of any arity (reference
// hash_join_v2 with key lists, relational.rs:2926-2992, whose keys are packed
// row-major and hashed by pack_and_hash_keys, pack.cu:144-214).
//
// Instead of hashing variable-length packed key bytes, every key column is
// folded into a dense u32 id: the first step keys each row by its first one or
// two key columns as one u64, later steps by (previous id << 32) | next key
// column; the id is the key's rank among the build side's sorted unique keys
// (a left key absent from the build side gets KEY_NONE, which no build id
// equals).  The equal-id join then runs on (id << 32) | row words through the
// single-key run index and the wave-cooperative probe, which emit
// (left row << 32) | right row in left-row-major, right-row order; a gather
// writes the left ++ right columns.
// ---------------------------------------------------------------------------
namespace {
constexpr uint32_t KEY_NONE = 0xFFFFFFFFu;

// u64 key of one folding step: (hi << 32) | column c1, hi = prev[i] when given,
// else column c0; c1 < 0 keys by hi alone
__global__ void k_fold_key(RelView in, const uint32_t *__restrict__ prev, int c0, int c1, uint64_t n,
                           uint64_t *__restrict__ out) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t hi = prev ? (uint64_t)prev[i] : (uint64_t)col_value(in, c0, i);
        out[i] = c1 < 0 ? hi : ((hi << 32) | col_value(in, c1, i));
    }
}
// rank of each key among the sorted unique keys u[0..nu), KEY_NONE when absent
__global__ void k_rank_ids(const uint64_t *__restrict__ keys, uint64_t n, const uint64_t *__restrict__ u, uint64_t nu,
                           uint32_t *__restrict__ ids) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t k = keys[i];
        uint64_t lo = 0, hi = nu;
        while (lo < hi) {
            const uint64_t mid = lo + ((hi - lo) >> 1);
            if (u[mid] < k) lo = mid + 1; else hi = mid;
        }
        ids[i] = (lo < nu && u[lo] == k) ? (uint32_t)lo : KEY_NONE;
    }
}
// (id << 32) | row index
__global__ void k_id_rows(const uint32_t *__restrict__ ids, uint64_t n, uint64_t *__restrict__ out) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = ((uint64_t)ids[i] << 32) | (uint32_t)i;
}
__global__ void k_found_flags(const uint32_t *__restrict__ ids, uint64_t n, int want, uint8_t *__restrict__ flags) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        flags[i] = (ids[i] != KEY_NONE) == (want != 0);
}
// Where the columns of a join's output row come from: a column of its left row
// (the join keys, too), the payload itself, or a column of the right row that
// the payload numbers.
struct JoinMap {
    enum { LEFT, PAYLOAD, RIGHT };
    int arity = 0;
    int kind[MAX_ARITY] = {0}, col[MAX_ARITY] = {0};
};
// output row r from the pair (left row << 32) | payload
__global__ void k_join_rows(RelView L, RelView R, JoinMap m, const uint64_t *__restrict__ pairs, uint64_t n,
                            RelOut out) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += stride) {
        const uint64_t pr = pairs[r];
        put_row(out, m.arity, r, [&](int c) {
            if (m.kind[c] == JoinMap::LEFT) return col_value(L, m.col[c], pr >> 32);
            if (m.kind[c] == JoinMap::PAYLOAD) return (uint32_t)pr;
            return col_value(R, m.col[c], (uint32_t)pr);
        });
    }
}
// (column c << 32) | row index
__global__ void k_key_rows(RelView in, int c, uint64_t n, uint64_t *__restrict__ out) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = ((uint64_t)col_value(in, c, i) << 32) | (uint32_t)i;
}
}  // namespace

// left ++ right: a right key column is the left one it was matched with; the
// others come from the payload, which is column `payload_col` of the right side,
// or, when that is negative, the number of its row.
static JoinMap join_map(const xlog_hip_rel *l, uint32_t r_arity, const std::vector<int> &lk, const std::vector<int> &rk,
                        int payload_col) {
    JoinMap m;
    m.arity = (int)(l->arity + r_arity);
    for (int c = 0; c < (int)l->arity; ++c) m.col[c] = c;
    for (int c = 0; c < (int)r_arity; ++c) {
        const int o = (int)l->arity + c;
        const size_t t = std::find(rk.begin(), rk.end(), c) - rk.begin();
        m.kind[o] = t < rk.size() ? JoinMap::LEFT : (c == payload_col ? JoinMap::PAYLOAD : JoinMap::RIGHT);
        m.col[o] = t < rk.size() ? lk[t] : c;
    }
    return m;
}

// The folding steps of a key list of nk columns: step 0 keys by columns
// (c[0], c[1]) as one u64 (c[0] alone when nk == 1), step s >= 1 by
// (id of step s - 1, c[s + 1]).
static size_t fold_steps(size_t nk) { return nk >= 2 ? nk - 1 : 1; }
static void fold_cols(const std::vector<int> &c, size_t step, int *c0, int *c1) {
    if (step == 0) {
        *c0 = c[0];
        *c1 = c.size() >= 2 ? c[1] : -1;
    } else {
        *c0 = -1;
        *c1 = c[step + 1];
    }
}

// The build side's fold over its key columns rk: every step's dictionary
// (sorted unique keys) and, with runs, the run index over (id << 32) | row
// (a stable sort, so a run lists its rows in input order).
static void fold_build(Ctx *ctx, const xlog_hip_rel *r, const std::vector<int> &rk, KeyFold &F, bool runs) {
    const uint64_t nr = r->rows;
    Buf<uint32_t> rid(ctx, nr);
    Buf<uint64_t> rkey(ctx, nr);
    for (size_t st = 0; st < fold_steps(rk.size()); ++st) {
        int c0, c1;
        fold_cols(rk, st, &c0, &c1);
        LAUNCH_1D(k_fold_key, nr, view_of(r), st == 0 ? nullptr : rid.p, c0, c1, nr, rkey.p);
        uint64_t *sorted = sort_keys(ctx, rkey.p, nr, false);
        uint64_t *u = nullptr;
        uint64_t nu = 0;
        try {
            nu = unique_keys(ctx, sorted, nr, &u);
        } catch (...) {
            ctx->free(sorted);
            throw;
        }
        ctx->free(sorted);
        Buf<uint64_t> d;
        d.ctx = ctx;
        d.p = u;
        d.n = nu;
        F.dict.push_back(std::move(d));
        F.dict_n.push_back(nu);
        LAUNCH_1D(k_rank_ids, nr, rkey.p, nr, u, nu, rid.p);
    }
    if (!runs) return;
    Buf<uint64_t> rp(ctx, nr);
    LAUNCH_1D(k_id_rows, nr, rid.p, nr, rp.p);
    rid = Buf<uint32_t>();
    rkey = Buf<uint64_t>();
    build_join_index(ctx, rp.p, nr, 2, 0, false, F.J);
}

// The probe side's ids in the build side's dictionaries (KEY_NONE for a key
// no build row has: it stays KEY_NONE through later steps, since every
// dictionary key of a later step has a build id, below KEY_NONE, in its high
// word).
static void fold_probe(Ctx *ctx, const xlog_hip_rel *l, const std::vector<int> &lk, const KeyFold &F,
                       Buf<uint32_t> &lid, Buf<uint64_t> &lkey) {
    const uint64_t nl = l->rows;
    for (size_t st = 0; st < fold_steps(lk.size()); ++st) {
        int c0, c1;
        fold_cols(lk, st, &c0, &c1);
        LAUNCH_1D(k_fold_key, nl, view_of(l), st == 0 ? nullptr : lid.p, c0, c1, nl, lkey.p);
        LAUNCH_1D(k_rank_ids, nl, lkey.p, nl, F.dict[st].p, F.dict_n[st], lid.p);
    }
}

// The join of non-empty inputs against the fold of r: INNER rows left ++
// right in left-row-major, right-row order (the first max_output when set),
// SEMI / ANTI the left rows with / without a match in input order.
static xlog_hip_rel *keyed_join_probe(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r,
                                      const std::vector<int> &lk, const KeyFold &F, int type, uint64_t max_output) {
    const uint64_t nl = l->rows;
    const uint32_t arity = l->arity + r->arity;
    Buf<uint32_t> lid(ctx, nl);
    Buf<uint64_t> lkey(ctx, nl);
    fold_probe(ctx, l, lk, F, lid, lkey);
    if (type != XLOG_HIP_JOIN_INNER) {
        Buf<uint8_t> flags(ctx, nl);
        LAUNCH_1D(k_found_flags, nl, lid.p, nl, type == XLOG_HIP_JOIN_SEMI ? 1 : 0, flags.p);
        xlog_hip_rel *o = compact_rel(ctx, l, flags.p);
        if (l->flags & REL_CANONICAL) o->flags = REL_CANONICAL;  // a subset of a sorted set is one
        return o;
    }
    // (id << 32) | row on the probe side (the left keys are no longer needed)
    LAUNCH_1D(k_id_rows, nl, lid.p, nl, lkey.p);
    lid = Buf<uint32_t>();
    const int oc[4] = {1, 3, 0, 0};  // (left row << 32) | right row
    uint64_t *pairs = nullptr;
    uint64_t n = join_probe_general(ctx, lkey.p, nl, 0, F.J.ix, F.J.payload.p, 2, oc, &pairs, nullptr);
    if (n == 0) return rel_new(ctx, arity, 0);
    Buf<uint64_t> pb;
    pb.ctx = ctx;
    pb.p = pairs;
    if (max_output && n > max_output) n = max_output;
    std::unique_ptr<xlog_hip_rel, void (*)(xlog_hip_rel *)> o(rel_new(ctx, arity, n), rel_free);
    o->rows = n;
    LAUNCH_1D(k_join_rows, n, view_of(l), view_of(r), join_map(l, r->arity, {}, {}, -1), pairs, n, out_of(o.get()));
    return o.release();
}

// The join of l (any arity) against the direct index over column rk of a
// relation of r_arity <= 2 columns: probe words (key << 32) | left row, the
// right row rebuilt from the key and the payload.
static xlog_hip_rel *direct_join_wide_left(Ctx *ctx, const xlog_hip_rel *l, uint32_t lk, const JoinIndex &J,
                                           uint32_t r_arity, uint32_t rk, int type, uint64_t max_output) {
    const uint64_t nl = l->rows;
    Buf<uint64_t> probe(ctx, nl);
    LAUNCH_1D(k_key_rows, nl, view_of(l), (int)lk, nl, probe.p);
    if (type != XLOG_HIP_JOIN_INNER) {
        Buf<uint8_t> flags(ctx, nl);
        join_match_flags(ctx, probe.p, nl, 0, J.ix, type == XLOG_HIP_JOIN_SEMI, flags.p);
        xlog_hip_rel *o = compact_rel(ctx, l, flags.p);
        if (l->flags & REL_CANONICAL) o->flags = REL_CANONICAL;
        return o;
    }
    const uint32_t arity = l->arity + r_arity;
    XH_REQUIRE(arity <= MAX_ARITY, XLOG_HIP_UNSUPPORTED, "join: output arity (left ++ right) above 8");
    const int oc[4] = {1, 3, 0, 0};  // (left row << 32) | payload
    uint64_t *w = nullptr;
    uint64_t n = join_probe_general(ctx, probe.p, nl, 0, J.ix, J.payload.p, 2, oc, &w, nullptr);
    if (n == 0) return rel_new(ctx, arity, 0);
    Buf<uint64_t> wb;
    wb.ctx = ctx;
    wb.p = w;
    if (max_output && n > max_output) n = max_output;
    std::unique_ptr<xlog_hip_rel, void (*)(xlog_hip_rel *)> o(rel_new(ctx, arity, n), rel_free);
    o->rows = n;
    LAUNCH_1D(k_join_rows, n, view_of(l), view_of(l),
              join_map(l, r_arity, {(int)lk}, {(int)rk}, r_arity == 2 ? 1 - (int)rk : -1), w, n, out_of(o.get()));
    return o.release();
}

// Join keys as one u32.  A single key column is it.  Several are packed side by
// side when the bits that the build side's columns use allow it (ids of a
// domain, small attributes): then no dictionary is needed, and a probe row with
// a bit that no build row has cannot match.  The one-key run index and key set
// serve any key list this way: 2^22 rows against 2^21 on two columns took 1.20
// ms through dictionaries (two rank searches of 0.21 ms, sorts) and 0.55 so.
struct KeyPack {
    int n = 0;
    int bits = 32;     // keys are below 2^bits
    bool mix = false;  // packed from several columns and not their own slots
    int col[MAX_ARITY] = {0}, shift[MAX_ARITY] = {0};
    uint32_t mask[MAX_ARITY] = {0};
};
constexpr uint64_t NO_KEY = ~0ull;  // a probe row without a match (keys packed from several columns are below 2^31)
namespace {
// A bijection of the 31-bit keys: two rounds of multiplicative hashing (Knuth,
// The Art of Computer Programming, vol. 3, 6.4) with the upper half of the bits
// folded into the lower after each; the odd multipliers are 2^31 times the
// fractions of the golden ratio and of the square root of two.  Keys packed side
// by side repeat the columns' patterns, which the table's own multiplicative
// hash keeps: their runs then crowd in the table (2^20 keys of 21 + 6 bits:
// insert 0.11 ms, count 0.12; mixed 0.06 and 0.10).
__device__ __forceinline__ uint32_t mix_key(uint32_t x) {
    constexpr uint32_t M = 0x7FFFFFFFu;
    x = (x * 0x4F1BBCDDu) & M;
    x ^= x >> 16;
    x = (x * 0x3504F335u) & M;
    return x ^ (x >> 16);
}
// (packed key << 32) | row
__global__ void k_pack_rows(RelView in, KeyPack kp, uint64_t n, uint64_t *__restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        uint32_t key = 0, extra = 0;
        for (int t = 0; t < kp.n; ++t) {
            const uint32_t v = col_value(in, kp.col[t], i);
            extra |= v & ~kp.mask[t];
            key |= (v & kp.mask[t]) << kp.shift[t];
        }
        if (kp.mix) key = mix_key(key);
        out[i] = extra ? NO_KEY : ((uint64_t)key << 32) | (uint32_t)i;
    }
}
// the payloads of sorted (key << 32) | row words: column c of the row, or the
// row itself when c is negative (rows clamped: a bucket sort that did not fit
// leaves words that are no rows)
__global__ void k_row_payload(RelView in, int c, const uint64_t *__restrict__ sorted, uint64_t n,
                              uint32_t *__restrict__ payload) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        uint64_t r = (uint32_t)sorted[i];
        r = r < n ? r : n - 1;
        payload[i] = c < 0 ? (uint32_t)r : col_value(in, c, r);
    }
}
}  // namespace
// false: the build side's key columns use too many bits together
static bool key_pack(Ctx *ctx, const xlog_hip_rel *r, const std::vector<int> &rk, KeyPack &kp) {
    kp.n = (int)rk.size();
    for (int t = 0; t < kp.n; ++t) kp.col[t] = rk[t];
    if (kp.n == 1) {
        kp.mask[0] = 0xFFFFFFFFu;
        return true;
    }
    Buf<unsigned long long> used(ctx, MAX_WORDS);
    fill_u64(ctx, reinterpret_cast<uint64_t *>(used.p), 0ull, MAX_WORDS);
    hipLaunchKernelGGL(k_key_bits, dim3(grid_for(r->rows, 256 * 8, 256), r->nwords()), dim3(256), 0, ctx->stream,
                       view_of(r), r->rows, used.p);
    XH_CHECK_HIP(hipGetLastError());
    ctx->read_scalars(used.p, MAX_WORDS);
    kp.bits = 0;
    for (int t = kp.n - 1; t >= 0; --t) {
        const uint64_t w = ctx->host_scalars[rk[t] >> 1];
        const uint32_t u = r->arity == 1 || (rk[t] & 1) ? (uint32_t)w : (uint32_t)(w >> 32);
        const int len = u ? 32 - __builtin_clz(u) : 0;
        kp.mask[t] = len ? 0xFFFFFFFFu >> (32 - len) : 0u;
        kp.shift[t] = len ? kp.bits : 0;
        kp.bits += len;
        if (kp.bits > 31) return false;
    }
    // Keys of few bits are their own slots of 16 bytes (2^20 rows on 20 bits 0.22 ms, mixed 0.27; 2^24 rows on 27 bits
    // 2.69 / 3.24): at most 8 slots a row, as an index of that many runs may take 4, and neither more than a 64th of
    // the device's memory nor a quarter of what a budget leaves.
    kp.mix = (1ull << kp.bits) > std::min<uint64_t>({8 * r->rows, 1ull << 28, ctx->pool->headroom() / 64});
    return true;
}
static KeyPack on_columns(const KeyPack &kp, const std::vector<int> &cols) {
    KeyPack q = kp;
    for (int t = 0; t < q.n; ++t) q.col[t] = cols[t];
    return q;
}

// Run index over packed keys, each run's rows in input order, with payloads as
// k_row_payload.  Small build sides are sorted by buckets, as whole words (they
// are all different, so that gives that order), and indexed with nothing read
// back (the table is sized for as many runs as rows): *over then points at a
// device word to be read with the probe's total.  Its low half is not zero when
// the sort did not fit (a sample far off: keys with many rows do fit); then the
// index holds nothing and is to be built again without `small`.
static void build_row_index(Ctx *ctx, const xlog_hip_rel *r, const KeyPack &kp, int payload_col, bool small,
                            JoinIndex &J, Buf<uint64_t> &state, const uint64_t **over) {
    const uint64_t n = r->rows;
    *over = nullptr;
    J.n = n;
    Owned rows(ctx, alloc_keys(ctx, n));
    LAUNCH_1D(k_pack_rows, n, view_of(r), kp, n, rows.p);
    J.payload = Buf<uint32_t>(ctx, n);
    Owned sorted(ctx);
    if (small && bucket_sort_takes(n) && fits_memory([&] { sorted.reset(alloc_keys(ctx, n)); }) &&
        bucket_sort(ctx, rows.p, n, sorted.p, nullptr, state)) {
        rows.reset(sorted.release());
        *over = state.p;
    } else if (sorted.reset(); n <= BLOCK_SORT_KEYS) {
        rows.reset(sort_keys(ctx, rows.release(), n, true, 0, 8));
    } else {
        rows.reset(sort_keys(ctx, rows.release(), n, true, 4, 8));  // stable; digit passes
    }
    LAUNCH_1D(k_row_payload, n, view_of(r), payload_col, rows.p, n, J.payload.p);
    J.ix.direct = kp.bits < 32 && !kp.mix;
    if (!small && !J.ix.direct) {
        build_run_index(ctx, rows.p, n, J.ix);
        return;
    }
    Buf<uint32_t> run_key(ctx, n);
    Buf<uint64_t> run_start(ctx, n + 1), cnt(ctx, 2);
    fill_u64(ctx, cnt.p, n, 2);
    select_runs(ctx, rows.p, n, run_key.p, run_start.p, cnt.p);
    uint64_t slots = 1024;
    while (J.ix.direct ? slots < (1ull << kp.bits) : slots < 2 * n) slots <<= 1;
    J.ix.table = Buf<unsigned long long>(ctx, 2 * slots);
    J.ix.table_mask = slots - 1;
    J.ix.nruns = n;  // (a bound)
    // (after a sort that did not fit, the runs are of words that repeat anyhow, and inserting those would probe on and
    // on)
    run_index_insert_dev(ctx, run_key.p, run_start.p, cnt.p, n, cnt.p + 1, J.ix,
                         *over ? reinterpret_cast<const uint32_t *>(*over) : nullptr);
}
// One key column: up to 3 * 2^17 rows.  Beyond, the digit passes, few when the keys have few bits, and a table sized by
// the runs found take less (10^6 rows a side, by buckets and by digit passes: Zipf keys 213 / 157 us, 1,000 keys 162 /
// 117, ids 208 / 196, hashed 272 / 275; 4 * 10^5 rows: 153 / 138, 108 / 106, 131 / 143, 158 / 187).  Keys packed from
// several columns have most of 31 bits: buckets as far as they go (10^6 rows on ids and a column of 64 values 294 /
// 327).
static bool small_build(uint64_t n, int key_cols) {
    return n <= BLOCK_SORT_KEYS || ((key_cols > 1 || n <= (3ull << 17)) && bucket_sort_takes(n));
}

// INNER join of non-empty inputs: probe words of the left side (l's own rows
// with their key in word pcol, or packed ones) against the row index of r, the
// output values oc as in OutSpec.  Returns the output's row count.
static uint64_t row_index_join(Ctx *ctx, const uint64_t *probe, uint64_t nl, int pcol, const xlog_hip_rel *r,
                               const KeyPack &kp, int payload_col, int out_arity, const int oc[4], Buf<uint64_t> &o0,
                               Buf<uint64_t> &o1) {
    bool small = small_build(r->rows, kp.n);
    for (;;) {
        JoinIndex J;
        Buf<uint64_t> state;
        ProbeJob job;
        build_row_index(ctx, r, kp, payload_col, small, J, state, &job.also);
        job.probe = probe;
        job.n = nl;
        job.pcol = pcol;
        job.ix = &J.ix;
        job.payload = J.payload.p;
        const uint64_t total = probe_prepare(ctx, job);
        if (job.also && (uint32_t)job.also_value) {  // a bucket outgrew its region
            small = false;
            continue;
        }
        if (total == 0) return 0;
        o0 = Buf<uint64_t>(ctx, total);
        o1 = Buf<uint64_t>(ctx, out_arity > 2 ? total : 0);
        probe_emit_range(ctx, job, 0, job.tiles, total, out_arity, oc, o0.p, o1.p);
        return total;
    }
}

static void check_key_lists(const xlog_hip_rel *l, const xlog_hip_rel *r, const std::vector<int> &lk,
                            const std::vector<int> &rk, int type) {
    XH_REQUIRE(l && r, XLOG_HIP_INVALID_ARG, "join input is NULL");
    XH_REQUIRE(!lk.empty() && lk.size() == rk.size(), XLOG_HIP_INVALID_ARG,
               "join: key column lists must be non-empty and of equal length");
    for (size_t t = 0; t < lk.size(); ++t)
        XH_REQUIRE(lk[t] >= 0 && lk[t] < (int)l->arity && rk[t] >= 0 && rk[t] < (int)r->arity, XLOG_HIP_INVALID_ARG,
                   "join key column out of range");
    XH_REQUIRE(type == XLOG_HIP_JOIN_INNER || type == XLOG_HIP_JOIN_SEMI || type == XLOG_HIP_JOIN_ANTI,
               XLOG_HIP_INVALID_ARG, "unknown join type");
    XH_REQUIRE(type != XLOG_HIP_JOIN_INNER || l->arity + r->arity <= MAX_ARITY, XLOG_HIP_UNSUPPORTED,
               "join: output arity (left ++ right) above 8");
    XH_REQUIRE(l->rows < KEY_NONE && r->rows < KEY_NONE, XLOG_HIP_CAPACITY_OVERFLOW,
               "join: more than 2^32 - 2 rows on one side");
}
// The result of a join with an empty side (reference relational.rs:3920-3940).
static xlog_hip_rel *empty_side_join(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, int type) {
    if (type == XLOG_HIP_JOIN_ANTI) return rel_clone(ctx, l);
    return rel_new(ctx, type == XLOG_HIP_JOIN_INNER ? l->arity + r->arity : l->arity, 0);
}

// The join of non-empty inputs with packed keys.
static xlog_hip_rel *packed_join(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, const std::vector<int> &lk,
                                 const std::vector<int> &rk, const KeyPack &kp, int type) {
    const uint64_t nl = l->rows, nr = r->rows;
    Buf<uint64_t> probe(ctx, nl);
    LAUNCH_1D(k_pack_rows, nl, view_of(l), on_columns(kp, lk), nl, probe.p);
    if (type != XLOG_HIP_JOIN_INNER) {
        Buf<uint64_t> rows(ctx, nr);
        LAUNCH_1D(k_pack_rows, nr, view_of(r), kp, nr, rows.p);
        return key_set_join(ctx, l, probe.p, 0, rows.p, nr, 0, type, (l->flags & REL_CANONICAL) != 0);
    }
    // the payload is the one column of r that is no key, or the row's number
    int payload_col = -1, others = 0;
    for (int c = 0; c < (int)r->arity; ++c)
        if (std::find(rk.begin(), rk.end(), c) == rk.end()) {
            payload_col = c;
            ++others;
        }
    if (others > 1) payload_col = -1;
    const int oc[4] = {1, 3, 0, 0};  // (left row << 32) | payload
    Buf<uint64_t> pairs, none;
    const uint64_t n = row_index_join(ctx, probe.p, nl, 0, r, kp, payload_col, 2, oc, pairs, none);
    const uint32_t arity = l->arity + r->arity;
    if (n == 0) return rel_new(ctx, arity, 0);
    RelOwner o(rel_new(ctx, arity, n), rel_free);
    o->rows = n;
    LAUNCH_1D(k_join_rows, n, view_of(l), view_of(r), join_map(l, r->arity, lk, rk, payload_col), pairs.p, n,
              out_of(o.get()));
    return o.release();
}
// Keys that do not pack, and joins whose packed keys, set or table do not fit
// the device (its budget), go through the dictionaries.
static xlog_hip_rel *op_join_keys(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, const std::vector<int> &lk,
                                  const std::vector<int> &rk, int type) {
    check_key_lists(l, r, lk, rk, type);
    if (l->rows == 0 || r->rows == 0) return empty_side_join(ctx, l, r, type);
    KeyPack kp;
    xlog_hip_rel *o = nullptr;
    if (key_pack(ctx, r, rk, kp) && fits_memory([&] { o = packed_join(ctx, l, r, lk, rk, kp, type); })) return o;
    KeyFold F;
    fold_build(ctx, r, rk, F, type == XLOG_HIP_JOIN_INNER);
    return keyed_join_probe(ctx, l, r, lk, F, type, 0);
}

static xlog_hip_rel *op_join(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, uint32_t lk, uint32_t rk,
                             int type, const std::vector<int> *out_cols) {
    XH_REQUIRE(l && r, XLOG_HIP_INVALID_ARG, "join input is NULL");
    XH_REQUIRE(lk < l->arity && rk < r->arity, XLOG_HIP_INVALID_ARG, "join key column out of range");
    if (l->arity > 2 || r->arity > 2) {
        // wider rows: the keyed join with one key column, then the projection
        xlog_hip_rel *j = op_join_keys(ctx, l, r, {(int)lk}, {(int)rk}, type);
        if (!out_cols || type != XLOG_HIP_JOIN_INNER) return j;
        std::unique_ptr<xlog_hip_rel, void (*)(xlog_hip_rel *)> jg(j, rel_free);
        return op_project(ctx, j, *out_cols);
    }
    const int pcol = probe_vidx(l->arity, lk);
    xlog_hip_rel *o = nullptr;  // (a set of keys is sized by the rows, the index below by the distinct keys)
    if ((type == XLOG_HIP_JOIN_SEMI || type == XLOG_HIP_JOIN_ANTI) && l->rows && r->rows && fits_memory([&] {
            o = key_set_join(ctx, l, l->w[0], pcol, r->w[0], r->rows, probe_vidx(r->arity, rk), type, false);
        }))
        return o;
    if (type == XLOG_HIP_JOIN_INNER && l->rows && small_build(r->rows, 1) &&
        !((r->flags & REL_CANONICAL) && r->arity == 2 && rk == 0)) {  // (those are in key order already)
        int oc[4] = {0, 0, 0, 0};
        const int out_arity = join_values(l, r->arity, rk, out_cols, oc);
        KeyPack kp;
        key_pack(ctx, r, {(int)rk}, kp);
        Buf<uint64_t> o0, o1;
        uint64_t n = 0;
        // (its table is sized for as many runs as rows: without room for that, the index below)
        if (fits_memory([&] {
                n = row_index_join(ctx, l->w[0], l->rows, pcol, r, kp, r->arity == 2 ? 1 - (int)rk : -1, out_arity, oc,
                                   o0, o1);
            })) {
            if (n == 0) return rel_new(ctx, (uint32_t)out_arity, 0);
            return rel_adopt(ctx, (uint32_t)out_arity, n, o0.release(), o1.release(), 0);
        }
        o0 = Buf<uint64_t>();
        o1 = Buf<uint64_t>();
    }
    JoinIndex J;
    build_join_index(ctx, r->w[0], r->rows, r->arity, (int)rk, (r->flags & REL_CANONICAL) != 0, J);
    return op_join_indexed(ctx, l, lk, J, r->arity, rk, type, out_cols);
}

static bool column_sorted(Ctx *ctx, const xlog_hip_rel *rel, uint32_t col) {
    if (rel->rows < 2) return true;
    Buf<uint32_t> flag(ctx, 2);
    fill_u32(ctx, flag.p, 0u, 2);
    LAUNCH_1D(k_col_unsorted, rel->rows, view_of(rel), (int)col, rel->rows, flag.p);
    ctx->read_scalars(flag.p, 1);
    return ctx->host_scalars[0] == 0;
}

// Sort-merge inner join (reference sort_merge_join_v2_inner_u32_1key,
// relational.rs:3401-3571): output columns left ++ right like the hash join.
// The reference requires both sides sorted ascending on their key and at
// most 4,000,000 row pairs; here a side whose key column is not sorted is
// sorted (stably, key word only) and there is no pair cap.  The right side's
// runs of equal keys are matched to the left rows along the merge path
// (smj_lookup); the matches are expanded by the probe's count / emit.  Rows
// come out left-row-major (in key order), right rows of a run in input order.
static xlog_hip_rel *op_sort_merge_join(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, uint32_t lk,
                                        uint32_t rk) {
    XH_REQUIRE(l && r, XLOG_HIP_INVALID_ARG, "join input is NULL");
    XH_REQUIRE(lk < l->arity && rk < r->arity, XLOG_HIP_INVALID_ARG, "join key column out of range");
    XH_REQUIRE(l->arity <= 2 && r->arity <= 2, XLOG_HIP_UNSUPPORTED, "join: input arity above 2 is not supported");
    const uint32_t arity = l->arity + r->arity;
    if (l->rows == 0 || r->rows == 0) return rel_new(ctx, arity, 0);
    // right side as (key << 32) | other column, ordered by key
    const uint64_t nr = r->rows;
    // every buffer of this operator is owned by a Buf, so an error on the way frees them
    auto adopt = [&](uint64_t *q, uint64_t count) {
        Buf<uint64_t> b;
        b.ctx = ctx;
        b.p = q;
        b.n = count;
        return b;
    };
    Buf<uint64_t> rs(ctx, nr);
    if (r->arity == 2 && rk == 0) copy_d2d(ctx, rs.p, r->w[0], nr);
    else swap_words(ctx, r->w[0], nr, rs.p);  // arity 1 keeps c0 in the low word
    if (!column_sorted(ctx, r, rk)) rs = adopt(sort_keys(ctx, rs.p, nr, false, 4, 8), nr);
    JoinIndex J;  // runs and payload only; the sort-merge lookup needs no hash table
    J.n = nr;
    Buf<uint32_t> run_key(ctx, nr);
    Buf<uint64_t> run_start(ctx, nr + 1);
    {
        Buf<uint64_t> cnt(ctx, 1);
        select_runs(ctx, rs.p, nr, run_key.p, run_start.p, cnt.p);
        J.ix.nruns = read_count(ctx, cnt.p);
    }
    fill_u64(ctx, run_start.p + J.ix.nruns, nr, 1);  // run_start[nruns] = end
    J.payload = Buf<uint32_t>(ctx, nr);
    low_words(ctx, rs.p, nr, J.payload.p);
    rs = Buf<uint64_t>();
    // left side ordered by its key column (stable: key digits only)
    const int pcol = probe_vidx(l->arity, lk);
    Buf<uint64_t> ls;
    const uint64_t *probe = l->w[0];
    if (!column_sorted(ctx, l, lk)) {
        ls = adopt(sort_keys(ctx, const_cast<uint64_t *>(l->w[0]), l->rows, false, pcol ? 0 : 4, pcol ? 4 : 8),
                   l->rows);
        probe = ls.p;
    }
    Buf<uint64_t> pre_start(ctx, l->rows);
    Buf<uint32_t> pre_cnt(ctx, l->rows);
    {
        Prof prof(ctx, XLOG_HIP_KERNEL_MERGE, 8.0 * (double)l->rows + 4.0 * (double)J.ix.nruns);
        smj_lookup(ctx, probe, l->rows, pcol, run_key.p, run_start.p, J.ix.nruns, pre_start.p, pre_cnt.p);
    }
    std::vector<int> vmap;  // value index of every output column (left ++ right)
    for (uint32_t c = 0; c < l->arity; ++c) vmap.push_back(probe_vidx(l->arity, c));
    for (uint32_t c = 0; c < r->arity; ++c) vmap.push_back(c == rk ? 2 : 3);
    int oc[4] = {0, 0, 0, 0};
    for (size_t i = 0; i < vmap.size(); ++i) oc[i] = vmap[i];
    ProbeJob job;
    job.probe = probe;
    job.n = l->rows;
    job.pcol = pcol;
    job.ix = &J.ix;
    job.payload = J.payload.p;
    job.pre_start = pre_start.p;
    job.pre_cnt = pre_cnt.p;
    const uint64_t total = probe_prepare(ctx, job);
    if (total == 0) return rel_new(ctx, arity, 0);
    Buf<uint64_t> o0(ctx, total), o1(ctx, arity > 2 ? total : 0);
    probe_emit_range(ctx, job, 0, job.tiles, total, (int)arity, oc, o0.p, o1.p);
    return rel_adopt(ctx, arity, total, o0.release(), o1.release(), 0);
}

// Nested-loop inner join (reference nested_loop_join_v2_inner_u32_1key,
// relational.rs:3041-3255): same output columns as the inner hash join, rows
// in left-row-major, right-row order; refused above rows_l * rows_r =
// 4,000,000 like the reference (NESTED_LOOP_TOTAL_THRESHOLD, provider/mod.rs:1030).
static xlog_hip_rel *op_nested_loop_join(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, uint32_t lk,
                                         uint32_t rk) {
    XH_REQUIRE(l && r, XLOG_HIP_INVALID_ARG, "join input is NULL");
    XH_REQUIRE(lk < l->arity && rk < r->arity, XLOG_HIP_INVALID_ARG, "join key column out of range");
    XH_REQUIRE(l->arity <= 2 && r->arity <= 2, XLOG_HIP_UNSUPPORTED, "join: input arity above 2 is not supported");
    const uint32_t arity = l->arity + r->arity;
    if (l->rows == 0 || r->rows == 0) return rel_new(ctx, arity, 0);
    XH_REQUIRE(l->rows <= 4000000ull / r->rows, XLOG_HIP_CAPACITY_OVERFLOW,
               "nested loop join: rows_l * rows_r exceeds 4000000");
    uint64_t *o0, *o1;
    const uint64_t n = nested_loop_join(ctx, l->w[0], l->rows, (int)l->arity, (int)lk, r->w[0], r->rows,
                                        (int)r->arity, (int)rk, &o0, &o1);
    if (n == 0) return rel_new(ctx, arity, 0);
    return rel_adopt(ctx, arity, n, o0, o1, 0);
}

// Dedup of input ordered on the key columns (reference dedup_sorted,
// relational.rs:288-420): full-row keys of arity > 1 take the full-row dedup;
// otherwise the first row of every run of adjacent rows equal on the key
// columns is kept, in input order, without sorting.
static xlog_hip_rel *op_dedup_sorted(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols) {
    XH_REQUIRE(!cols.empty(), XLOG_HIP_INVALID_ARG, "dedup needs at least one key column");
    if (in->arity > 1 && is_full_key(in, cols)) return op_dedup_full(ctx, in);
    if (in->rows <= 1) return rel_clone(ctx, in);
    std::vector<int> keys;  // distinct key columns (at most the arity, <= 4)
    for (int c : cols)
        if (std::find(keys.begin(), keys.end(), c) == keys.end()) keys.push_back(c);
    Buf<uint8_t> flags(ctx, in->rows);
    ProjSpec ks{(int)in->arity, (int)keys.size(), {0, 0, 0, 0, 0, 0, 0, 0}};
    for (int j = 0; j < ks.out_arity; ++j) ks.cols[j] = keys[j];
    LAUNCH_1D(k_group_flags, in->rows, view_of(in), ks, in->rows, flags.p);
    xlog_hip_rel *r = compact_rel(ctx, in, flags.p);
    if (in->flags & REL_CANONICAL) r->flags = REL_CANONICAL;  // a subset of a sorted set is one
    return r;
}

// One factorized TC delta step (reference fj_delta_novel_u32_recorded,
// crates/xlog-cuda/src/provider/fj_delta.rs:117-490): the set
//   { head(carry, value) : delta(carry, key), edge(key, value), head not in full }
// with the column roles of `cols`, output in full's column order (r_carry,
// r_value), canonical.  Every id must be below `domain` <= 2^16.
static xlog_hip_rel *op_fj_delta(Ctx *ctx, const xlog_hip_rel *delta, const xlog_hip_rel *edge,
                                 const xlog_hip_rel *full, const xlog_hip_fj_delta_cols &c, uint32_t domain) {
    XH_REQUIRE(delta && edge && full, XLOG_HIP_INVALID_ARG, "fj delta: input is NULL");
    XH_REQUIRE(delta->arity == 2 && edge->arity == 2 && full->arity == 2, XLOG_HIP_INVALID_ARG,
               "fj delta: delta, edge and full must be arity-2");
    auto roles_ok = [](uint32_t a, uint32_t b) { return a < 2 && b < 2 && a != b; };
    XH_REQUIRE(roles_ok(c.delta_carry, c.delta_key) && roles_ok(c.r_carry, c.r_value), XLOG_HIP_INVALID_ARG,
               "fj delta: invalid column roles (arity-2 indices, pairwise distinct)");
    XH_REQUIRE(domain > 0 && domain <= (1u << 16), XLOG_HIP_INVALID_ARG, "fj delta: domain outside (0, 2^16]");
    if (delta->rows == 0 || edge->rows == 0) {
        xlog_hip_rel *e = rel_new(ctx, 2, 0);
        e->flags = REL_CANONICAL;
        return e;
    }
    {  // every id below the domain (checked before any bitmap is touched)
        Buf<unsigned int> mx(ctx, 1);
        fill_u32(ctx, mx.p, 0u, 1);
        const xlog_hip_rel *rs[3] = {delta, edge, full};
        for (const xlog_hip_rel *r : rs)
            if (r->rows) MAX_LAUNCH_1D(k_max_u32_of_packed, r->rows, r->w[0], r->rows, mx.p);
        uint32_t h = 0;
        XH_CHECK_HIP(hipMemcpyAsync(&h, mx.p, 4, hipMemcpyDeviceToHost, ctx->stream));
        ctx->sync();
        XH_REQUIRE(h < domain, XLOG_HIP_INVALID_ARG,
                   "fj delta: id " + std::to_string(h) + " outside the domain " + std::to_string(domain));
    }
    Canon ce;  // edge as sorted unique (key << 32) | value
    canonical_keys(ctx, edge, ce);
    uint64_t *o = nullptr;
    const uint64_t n = fj_delta_step(ctx, delta->w[0], delta->rows, c.delta_carry == 0 ? 1 : 0, ce.k, ce.n,
                                     full->w[0], full->rows, c.r_carry == 0 ? 1 : 0, domain, &o);
    if (n == 0) {
        xlog_hip_rel *e = rel_new(ctx, 2, 0);
        e->flags = REL_CANONICAL;
        return e;
    }
    if (c.r_carry == 1) {  // head column order (value, carry): swap and re-sort
        uint64_t *sw = static_cast<uint64_t *>(ctx->alloc(n * sizeof(uint64_t)));
        swap_words(ctx, o, n, sw);
        ctx->free(o);
        o = sort_keys(ctx, sw, n, true);  // consumes sw
    }
    return rel_adopt(ctx, 2, n, o, nullptr, REL_CANONICAL);
}

// One sparse factorized delta step (reference fj_delta_sparse_novel_u32_recorded,
// crates/xlog-cuda/src/provider/fj_delta_sparse.rs:66-490): the set
//   { head(carry, value) : delta(carry, key), edge(key, value), head not in full }
// with no domain bound, over a device hash set filled with `full`.  The
// table is sized 2 x (|full| + candidates), the candidate count coming from
// the probe's count pass (an upper bound of the distinct candidates, which the
// reference estimates with a bitmap).  A table above max_table_bytes (when
// non-zero) declines, like the reference's Ok(None): *declined is set and no
// relation is returned.  The output is canonical in full's column order.
static xlog_hip_rel *op_fj_delta_sparse(Ctx *ctx, const xlog_hip_rel *delta, const xlog_hip_rel *edge,
                                        const xlog_hip_rel *full, const xlog_hip_fj_delta_cols &c,
                                        uint64_t max_table_bytes, bool *declined) {
    *declined = false;
    XH_REQUIRE(delta && edge && full, XLOG_HIP_INVALID_ARG, "fj delta sparse: input is NULL");
    XH_REQUIRE(delta->arity == 2 && edge->arity == 2 && full->arity == 2, XLOG_HIP_INVALID_ARG,
               "fj delta sparse: delta, edge and full must be arity-2");
    auto roles_ok = [](uint32_t a, uint32_t b) { return a < 2 && b < 2 && a != b; };
    XH_REQUIRE(roles_ok(c.delta_carry, c.delta_key) && roles_ok(c.r_carry, c.r_value), XLOG_HIP_INVALID_ARG,
               "fj delta sparse: invalid column roles (arity-2 indices, pairwise distinct)");
    auto empty = [&]() {
        xlog_hip_rel *e = rel_new(ctx, 2, 0);
        e->flags = REL_CANONICAL;
        return e;
    };
    if (delta->rows == 0 || edge->rows == 0) return empty();
    Canon ce;  // edge as sorted unique (key << 32) | value: runs of values per key
    canonical_keys(ctx, edge, ce);
    JoinIndex J;
    build_join_index(ctx, ce.k, ce.n, 2, 0, true, J);
    ProbeJob job;  // count pass only: the number of candidate tuples
    job.probe = delta->w[0];
    job.n = delta->rows;
    job.pcol = c.delta_key == 0 ? 0 : 1;
    job.ix = &J.ix;
    job.payload = J.payload.p;
    job.record_lookups = false;
    const uint64_t cand = probe_prepare(ctx, job);
    if (cand == 0) return empty();
    uint64_t slots = 1ull << 16;
    while (slots < 2 * (full->rows + cand)) slots <<= 1;
    if (max_table_bytes && slots * sizeof(uint64_t) > max_table_bytes) {
        *declined = true;
        return nullptr;
    }
    HashSet h;
    hs_init(ctx, h, slots);
    hs_insert_all(ctx, h, full->w[0], full->rows);
    h.size = full->rows;
    // the novel tuples number at most `cand`, so a limit of cand + 1 is never reached
    Buf<uint64_t> novel(ctx, cand + 1 + HS_APPEND_SLACK);
    hs_join_insert(ctx, h, delta->w[0], delta->rows, c.delta_key == 0 ? 1 : 0, c.r_carry == 0 ? 1 : 0, J.ix,
                   J.payload.p, novel.p, cand + 1);
    ctx->read_scalars(h.flags.p + 1, 2);
    XH_REQUIRE(ctx->host_scalars[0] == 0, XLOG_HIP_DEVICE_ERROR, "fj delta sparse: table overflow");
    const uint64_t n = ctx->host_scalars[1];
    if (n == 0) return empty();
    h = HashSet();
    uint64_t *s = sort_keys(ctx, novel.p, n, false);
    return rel_adopt(ctx, 2, n, s, nullptr, REL_CANONICAL);
}

// Set of the projected join, canonical: dedup_full_row(project(join(l, r))).
// When the output is (left column, right non-key column) the join is emitted
// already ordered: the probe side is first sorted by its output column (key
// word only) and the build runs are kept sorted by their payload, so each probe
// row's outputs are ascending and rows come in output-column order.  Only
// groups of probe rows that share the output column interleave; those runs
// are sorted in place (LDS bitonic sort per run), then one unique pass.  This
// replaces the radix sort of the whole join output.  Other shapes take the
// join -> sort -> unique path.
void left_keys(Ctx *ctx, const uint64_t *l, uint64_t n, int arity, int oc0, int jk, uint64_t *out);
void group_rows_async(Ctx *ctx, const uint64_t *k, uint64_t n, int32_t *gsel, uint64_t *mkeys, uint64_t *mpos,
                      uint64_t *hkeys, uint64_t *hpos, uint64_t *d_nm, uint64_t *d_nh);
void group_segments(Ctx *ctx, const uint64_t *sorted, uint64_t n, const uint64_t *head_keys, uint64_t nh,
                    uint64_t *seg, const uint64_t *d_n);
void sort_segments_async(Ctx *ctx, uint64_t *data, uint64_t n, const uint64_t *heads, uint64_t nh, uint64_t *seg,
                         unsigned long long *d_max);
void sort_segments_long(Ctx *ctx, uint64_t *data, const uint64_t *seg, uint64_t nh, uint64_t max_len);

namespace {
__global__ void k_gather_u64(const uint64_t *a, const uint64_t *b, uint64_t *out) {
    out[0] = *a;
    out[1] = *b;
}
}  // namespace

static xlog_hip_rel *op_join_project_dedup(Ctx *ctx, const xlog_hip_rel *l, const xlog_hip_rel *r, uint32_t lk,
                                           uint32_t rk, const std::vector<int> &out_cols) {
    XH_REQUIRE(l && r, XLOG_HIP_INVALID_ARG, "join input is NULL");
    XH_REQUIRE(lk < l->arity && rk < r->arity, XLOG_HIP_INVALID_ARG, "join key column out of range");
    const bool ordered = l->arity <= 2 && r->arity == 2 && out_cols.size() == 2 && out_cols[0] >= 0 &&
                         out_cols[0] < (int)l->arity && out_cols[1] == (int)l->arity + (1 - (int)rk);
    if (!ordered) {
        xlog_hip_rel *j = op_join(ctx, l, r, lk, rk, XLOG_HIP_JOIN_INNER, &out_cols);
        xlog_hip_rel *d = nullptr;
        try {
            d = op_dedup_full(ctx, j);
        } catch (...) {
            rel_free(j);
            throw;
        }
        rel_free(j);
        return d;
    }
    const uint64_t n = l->rows, nr = r->rows;
    auto empty = [&]() {
        xlog_hip_rel *e = rel_new(ctx, 2, 0);
        e->flags = REL_CANONICAL;
        return e;
    };
    if (n == 0 || nr == 0) return empty();
    // The host waits three times: for the build side's and the groups' sizes,
    // for the side probe's size (while the device runs the main count pass),
    // and for the output size (plus the sorts' histogram read-backs, which
    // their first digit pass overlaps).
    // 1. probe keys (out column << 32 | join key), ordered by the out column
    Buf<uint64_t> lk_buf;  // owns the sorted probe keys
    lk_buf.ctx = ctx;
    //    (or by the whole key, when the segment route of many keys does that in fewer passes)
    bool whole = false;
    if (l->arity == 2 && out_cols[0] == 0 && lk == 1) {
        // the rows are already (out column << 32 | join key): the sort reads them directly
        lk_buf.p = sort_keys(ctx, l->w[0], n, false, 4, 8, 0, &whole);
    } else {
        lk_buf.p = static_cast<uint64_t *>(ctx->alloc(n * sizeof(uint64_t)));
        left_keys(ctx, l->w[0], n, (int)l->arity, out_cols[0], (int)lk, lk_buf.p);
        lk_buf.p = sort_keys(ctx, lk_buf.p, n, true, 4, 8, 0, &whole);
    }
    const uint64_t *lkeys = lk_buf.p;
    // 2. build rows as (key << 32 | payload), sorted and unique, so that a probe
    //    row alone with its out column emits sorted, unique outputs
    //    (the key word's radix passes, then each run of equal keys sorted by
    //    payload in one pass; a run of more than 256 rows makes the build
    //    rows take the payload's radix passes too, after the first read-back)
    Buf<uint64_t> cnt(ctx, 5);  // unique build rows, runs, group members, groups, long run
    Buf<uint64_t> kw_buf, sk_buf;
    kw_buf.ctx = sk_buf.ctx = ctx;
    const uint64_t *sk;
    const bool canon = rk == 0 && (r->flags & REL_CANONICAL) != 0;
    if (canon) {
        sk = r->w[0];
        fill_u64(ctx, cnt.p + 4, 0ull, 1);
    } else {
        if (rk == 0) {
            kw_buf.p = sort_keys(ctx, r->w[0], nr, false, 4, 8, 0, &whole);
        } else {
            kw_buf.p = static_cast<uint64_t *>(ctx->alloc(nr * sizeof(uint64_t)));
            swap_words(ctx, r->w[0], nr, kw_buf.p);
            kw_buf.p = sort_keys(ctx, kw_buf.p, nr, true, 4, 8, 0, &whole);
        }
        if (whole) {  // the segment route ordered the build rows by the whole key
            fill_u64(ctx, cnt.p + 4, 0ull, 1);
            sk = kw_buf.p;
        } else {
            sk_buf = Buf<uint64_t>(ctx, nr);
            sort_short_runs(ctx, kw_buf.p, nr, sk_buf.p, cnt.p + 4);
            sk = sk_buf.p;
        }
    }
    Buf<uint64_t> ub;
    JoinIndex J;
    J.payload = Buf<uint32_t>(ctx, nr);
    const uint64_t *bk = sk, *d_un = nullptr;
    if (!canon && nr > 1) {
        ub = Buf<uint64_t>(ctx, nr);
        select_unique_low(ctx, sk, nr, ub.p, J.payload.p, cnt.p);  // the payloads come with the unique rows
        bk = ub.p;
        d_un = cnt.p;
    } else {
        low_words(ctx, bk, nr, J.payload.p);
    }
    RunScratch rs;
    build_run_index_async(ctx, bk, nr, d_un, rs, cnt.p + 1);
    // 3. probe rows sharing their out column (groups) can emit the same
    //    output twice and interleave: their outputs are produced on the side
    //    (probe, sort inside each group, unique) and copied into place by the
    //    main emit through the group selector
    Buf<int32_t> gsel(ctx, n);
    Buf<uint64_t> mkeys(ctx, n), mpos(ctx, n), hkeys(ctx, n), hpos(ctx, n);
    group_rows_async(ctx, lkeys, n, gsel.p, mkeys.p, mpos.p, hkeys.p, hpos.p, cnt.p + 2, cnt.p + 3);
    ctx->read_scalars(cnt.p, 5);
    uint64_t un = d_un ? ctx->host_scalars[0] : nr, nruns = ctx->host_scalars[1];
    const uint64_t nm = ctx->host_scalars[2], nh = ctx->host_scalars[3];
    if (ctx->host_scalars[4]) {  // a long run: the full sort of the build rows
        sk_buf = Buf<uint64_t>();
        sk_buf.ctx = ctx;
        sk_buf.p = sort_keys(ctx, kw_buf.p, nr, false, 0, 8);
        select_unique_low(ctx, sk_buf.p, nr, ub.p, J.payload.p, cnt.p);
        build_run_index_async(ctx, ub.p, nr, cnt.p, rs, cnt.p + 1);
        ctx->read_scalars(cnt.p, 2);
        un = ctx->host_scalars[0];
        nruns = ctx->host_scalars[1];
    }
    kw_buf = Buf<uint64_t>();
    J.n = un;
    build_run_index_finish(ctx, rs, nruns, un, J.ix);
    sk_buf = Buf<uint64_t>();
    ub = Buf<uint64_t>();
    mpos = Buf<uint64_t>();
    // 4. the side probe's count, then the main count pass (group heads count
    //    zero until their groups are known); the side total comes back while
    //    the main count runs
    const int oc[4] = {0, 3, 0, 0};  // v0 = out column (probe high word), v3 = payload
    ProbeJob side;
    if (nm) {
        side.probe = mkeys.p;
        side.n = nm;
        side.pcol = 1;
        side.ix = &J.ix;
        side.payload = J.payload.p;
        probe_count_only(ctx, side);
        probe_scan_async(ctx, side);
        ctx->post_read(side.toff.p + side.tiles, 1);
    }
    ProbeJob job;
    job.probe = lkeys;
    job.n = n;
    job.pcol = 1;
    job.ix = &J.ix;
    job.payload = J.payload.p;
    if (nm) job.gsel = gsel.p;  // gseg unset: heads deferred
    probe_count_only(ctx, job);
    // 5. group outputs: emit, sort inside each group, unique; each head then
    //    gets its group's unique words and count
    Buf<uint64_t> gseg, bag, seg, u2, nu2(ctx, 1);
    Buf<unsigned long long> mx(ctx, 1);
    uint64_t m2 = 0;
    if (nm) {
        ctx->wait_read();
        m2 = ctx->host_scalars[0];
        probe_finish(side, nm, m2);
        gseg = Buf<uint64_t>(ctx, 2 * nh);
        if (m2) {
            bag = Buf<uint64_t>(ctx, m2);
            probe_emit_range(ctx, side, 0, side.tiles, m2, 2, oc, bag.p, nullptr);
            seg = Buf<uint64_t>(ctx, 2 * nh);
            sort_segments_async(ctx, bag.p, m2, hkeys.p, nh, seg.p, mx.p);
            u2 = Buf<uint64_t>(ctx, m2);
            select_unique(ctx, bag.p, m2, u2.p, nu2.p);
            group_segments(ctx, u2.p, m2, hkeys.p, nh, gseg.p, nu2.p);
        } else {
            fill_u64(ctx, gseg.p, 0ull, 2 * nh);
        }
        probe_group_fixup(ctx, job, hpos.p, gseg.p, nh);
    }
    if (!nm || !m2) fill_u64(ctx, reinterpret_cast<uint64_t *>(mx.p), 0ull, 1);
    probe_scan_async(ctx, job);
    Buf<uint64_t> g2(ctx, 2);
    hipLaunchKernelGGL(k_gather_u64, dim3(1), dim3(1), 0, ctx->stream, job.toff.p + job.tiles,
                       reinterpret_cast<const uint64_t *>(mx.p), g2.p);
    XH_CHECK_HIP(hipGetLastError());
    ctx->read_scalars(g2.p, 2);
    uint64_t total = ctx->host_scalars[0];
    const uint64_t max_len = ctx->host_scalars[1];
    if (max_len > (uint64_t)WAVE) {
        // rare: a group with more than 64 outputs needs the block / radix
        // segment sorts; its unique words and the counts are then redone
        sort_segments_long(ctx, bag.p, seg.p, nh, max_len);
        select_unique(ctx, bag.p, m2, u2.p, nu2.p);
        group_segments(ctx, u2.p, m2, hkeys.p, nh, gseg.p, nu2.p);
        probe_count_only(ctx, job);
        probe_group_fixup(ctx, job, hpos.p, gseg.p, nh);
        probe_scan_async(ctx, job);
        ctx->read_scalars(job.toff.p + job.tiles, 1);
        total = ctx->host_scalars[0];
    }
    probe_finish(job, n, total);
    if (nm) {
        job.gseg = gseg.p;
        job.gsrc = u2.p;
    }
    if (!total) return empty();
    uint64_t *o = static_cast<uint64_t *>(ctx->alloc(total * sizeof(uint64_t)));
    try {
        probe_emit_range(ctx, job, 0, job.tiles, total, 2, oc, o, nullptr);
    } catch (...) {
        ctx->free(o);
        throw;
    }
    return rel_adopt(ctx, 2, total, o, nullptr, REL_CANONICAL);
}

static xlog_hip_rel *op_project(Ctx *ctx, const xlog_hip_rel *in, const std::vector<int> &cols) {
    XH_REQUIRE(!cols.empty() && cols.size() <= MAX_ARITY, XLOG_HIP_INVALID_ARG, "projection needs 1..8 columns");
    xlog_hip_rel *r = rel_new(ctx, (uint32_t)cols.size(), in->rows);
    r->rows = in->rows;
    ProjSpec s{(int)in->arity, (int)cols.size(), {0, 0, 0, 0, 0, 0, 0, 0}};
    for (size_t i = 0; i < cols.size(); ++i) s.cols[i] = cols[i];
    LAUNCH_1D(k_project, in->rows, view_of(in), in->rows, s, out_of(r));
    return r;
}

// a positive integer from the environment, or dflt
uint64_t env_u64(const char *name, uint64_t dflt) {
    const char *e = getenv(name);
    if (e && *e) {
        const unsigned long long v = strtoull(e, nullptr, 10);
        if (v > 0) return v;
    }
    return dflt;
}

}  // namespace xh

// ===========================================================================
// C ABI
// ===========================================================================
using namespace xh;

struct xlog_hip_ctx {
    Ctx c;
};

static Ctx *C(xlog_hip_ctx *ctx) {
    XH_REQUIRE(ctx, XLOG_HIP_INVALID_ARG, "context is NULL");
    XH_CHECK_HIP(hipSetDevice(ctx->c.device));
    return &ctx->c;
}
static void need_rel(const xlog_hip_rel *r, const char *what) {
    XH_REQUIRE(r, XLOG_HIP_INVALID_ARG, std::string(what) + " is NULL");
}

namespace xh {
// Arrow IPC stream I/O helpers (provider/io.rs:697-773)
namespace {
// Device relation from UInt32 column buffers in host memory: each column is
// copied once to a device staging buffer and packed there.
xlog_hip_rel *rel_from_ipc(Ctx *ctx, const IpcColumns &ic) {
    xlog_hip_rel *r = rel_new(ctx, ic.arity, ic.rows);
    r->rows = ic.rows;
    if (!ic.rows) return r;
    try {
        Buf<uint32_t> stage(ctx, (uint64_t)ic.arity * ic.rows);
        const uint32_t *dc[MAX_ARITY] = {nullptr};
        for (uint32_t c = 0; c < ic.arity; ++c) {
            uint32_t *d = stage.p + (uint64_t)c * ic.rows;
            XH_CHECK_HIP(hipMemcpyAsync(d, ic.cols[c], ic.rows * 4, hipMemcpyHostToDevice, ctx->stream));
            dc[c] = d;
        }
        pack_device_columns(ctx, dc, ic.arity, ic.rows, r);
        ctx->sync();  // the host bytes may go away after the call
    } catch (...) {
        rel_free(r);
        throw;
    }
    return r;
}

// All columns of a relation, column-major in host memory
std::vector<uint32_t> columns_to_host(Ctx *ctx, const xlog_hip_rel *rel) {
    std::vector<uint32_t> h((uint64_t)rel->arity * rel->rows);
    if (!rel->rows) return h;
    Buf<uint32_t> tmp(ctx, (uint64_t)rel->arity * rel->rows);
    for (uint32_t c = 0; c < rel->arity; ++c) {
        uint32_t *d = tmp.p + (uint64_t)c * rel->rows;
        if (rel->arity == 1) LAUNCH_1D(k_u64_to_u32, rel->rows, rel->w[0], rel->rows, d);
        else unpack_column(ctx, rel->w[c / 2], (c % 2) == 0, rel->rows, d);
    }
    XH_CHECK_HIP(hipMemcpyAsync(h.data(), tmp.p, h.size() * 4, hipMemcpyDeviceToHost, ctx->stream));
    ctx->sync();
    return h;
}

std::vector<uint8_t> rel_to_ipc(Ctx *ctx, const xlog_hip_rel *rel, const char *const *names) {
    const std::vector<uint32_t> h = columns_to_host(ctx, rel);
    const uint32_t *cols[4] = {nullptr, nullptr, nullptr, nullptr};
    for (uint32_t c = 0; c < rel->arity; ++c) cols[c] = h.data() + (uint64_t)c * rel->rows;
    return ipc_encode_u32(cols, rel->arity, rel->rows, names);
}

uint8_t *to_malloc(const std::vector<uint8_t> &v) {
    uint8_t *p = static_cast<uint8_t *>(malloc(v.size() ? v.size() : 1));
    XH_REQUIRE(p, XLOG_HIP_OOM, "host allocation failed");
    if (!v.empty()) memcpy(p, v.data(), v.size());
    return p;
}
}  // namespace
}  // namespace xh

extern "C" {

const char *xlog_hip_last_error(void) { return g_last_error.c_str(); }
const char *xlog_hip_version(void) { return "xlog_hip 0.1.0 (gfx950)"; }

xlog_hip_status xlog_hip_ctx_create(int device, xlog_hip_ctx **out) {
    return guarded([&] {
        XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL");
        *out = nullptr;
        int count = 0;
        XH_CHECK_HIP(hipGetDeviceCount(&count));
        XH_REQUIRE(device >= 0 && device < count, XLOG_HIP_INVALID_ARG, "device index out of range");
        XH_CHECK_HIP(hipSetDevice(device));
        std::unique_ptr<xlog_hip_ctx> h(new xlog_hip_ctx());
        Ctx &c = h->c;
        c.device = device;
        hipDeviceProp_t prop;
        XH_CHECK_HIP(hipGetDeviceProperties(&prop, device));
        c.num_cus = prop.multiProcessorCount;
        XH_CHECK_HIP(hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking));
        c.pool = new Pool(device);
        // (coherent: a kernel's stores are seen by the host while it waits; the word after the staging is host_seq)
        XH_CHECK_HIP(hipHostMalloc((void **)&c.host_scalars, (Ctx::HOST_STAGE_U64 + 8) * sizeof(uint64_t),
                                   hipHostMallocCoherent));
        c.host_seq = c.host_scalars + Ctx::HOST_STAGE_U64;
        *c.host_seq = 0;
        scan_noalloc_init(device);  // the allocation-free scan's scratch on this device
        c.tickets = static_cast<unsigned long long *>(c.alloc(16 * sizeof(unsigned long long)));
        fill_u64(&c, reinterpret_cast<uint64_t *>(c.tickets), 0ull, 16);
        XH_CHECK_HIP(hipEventCreate(&c.ev_a));
        XH_CHECK_HIP(hipEventCreate(&c.ev_b));
        XH_CHECK_HIP(hipEventCreateWithFlags(&c.ev_sync, hipEventDisableTiming));
        c.sync();
        *out = h.release();
    });
}

void xlog_hip_ctx_destroy(xlog_hip_ctx *ctx) {
    if (!ctx) return;
    Ctx &c = ctx->c;
    (void)hipSetDevice(c.device);
    (void)hipStreamSynchronize(c.stream);
    sort_state_release(&c);
    select_state_release(&c);
    if (c.tickets) c.free(c.tickets);
    if (c.prof_work) c.free(c.prof_work);
    delete c.pool;
    if (c.host_scalars) (void)hipHostFree(c.host_scalars);
    if (c.ev_a) (void)hipEventDestroy(c.ev_a);
    if (c.ev_b) (void)hipEventDestroy(c.ev_b);
    if (c.ev_sync) (void)hipEventDestroy(c.ev_sync);
    for (auto &r : c.prof_pending) {
        (void)hipEventDestroy(r.a);
        (void)hipEventDestroy(r.b);
    }
    for (hipEvent_t e : c.prof_events) (void)hipEventDestroy(e);
    (void)hipStreamDestroy(c.stream);
    delete ctx;
}

xlog_hip_status xlog_hip_synchronize(xlog_hip_ctx *ctx) { return guarded([&] { C(ctx)->sync(); }); }
void *xlog_hip_stream(xlog_hip_ctx *ctx) { return ctx ? (void *)ctx->c.stream : nullptr; }

xlog_hip_status xlog_hip_memory_stats(xlog_hip_ctx *ctx, uint64_t *in_use, uint64_t *peak, uint64_t *cached) {
    return guarded([&] {
        Ctx *c = C(ctx);
        if (in_use) *in_use = c->pool->bytes_in_use();
        if (peak) *peak = c->pool->peak_in_use();
        if (cached) *cached = c->pool->bytes_cached();
    });
}
xlog_hip_status xlog_hip_trim(xlog_hip_ctx *ctx) { return guarded([&] { C(ctx)->pool->trim(); }); }
xlog_hip_status xlog_hip_set_memory_budget(xlog_hip_ctx *ctx, uint64_t device_bytes) {
    return guarded([&] {
        Ctx *c = C(ctx);
        c->pool->set_budget((size_t)device_bytes);
        if (device_bytes && c->pool->bytes_in_use() + c->pool->bytes_cached() > device_bytes) c->pool->trim();
    });
}

xlog_hip_status xlog_hip_rel_create_empty(xlog_hip_ctx *ctx, uint32_t arity, xlog_hip_rel **out) {
    return guarded([&] {
        XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL");
        *out = rel_new(C(ctx), arity, 0);
        (*out)->flags = REL_CANONICAL;
    });
}

xlog_hip_status xlog_hip_rel_from_host_columns(xlog_hip_ctx *ctx, const uint32_t *const *cols, uint32_t arity,
                                               uint64_t rows, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL");
        XH_REQUIRE(arity >= 1 && arity <= MAX_ARITY, XLOG_HIP_INVALID_ARG, "relation arity must be 1..8");
        XH_REQUIRE(rows == 0 || cols, XLOG_HIP_INVALID_ARG, "columns are NULL");
        for (uint32_t i = 0; i < arity && rows; ++i) XH_REQUIRE(cols[i], XLOG_HIP_INVALID_ARG, "column pointer is NULL");
        const int nw = words_for(arity);
        std::vector<std::vector<uint64_t>> h(nw, std::vector<uint64_t>(rows));
        for (uint64_t i = 0; i < rows; ++i) {
            if (arity == 1) {
                h[0][i] = cols[0][i];
                continue;
            }
            for (int k = 0; k < nw; ++k)
                h[k][i] = ((uint64_t)cols[2 * k][i] << 32) | (2u * k + 1 < arity ? cols[2 * k + 1][i] : 0u);
        }
        std::unique_ptr<xlog_hip_rel, void (*)(xlog_hip_rel *)> r(rel_new(c, arity, rows), rel_free);
        r->rows = rows;
        if (rows)
            for (int k = 0; k < nw; ++k)
                XH_CHECK_HIP(hipMemcpyAsync(r->w[k], h[k].data(), rows * 8, hipMemcpyHostToDevice, c->stream));
        c->sync();
        *out = r.release();
    });
}

xlog_hip_status xlog_hip_rel_from_device_columns(xlog_hip_ctx *ctx, const uint32_t *const *dev_cols, uint32_t arity,
                                                 uint64_t rows, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *ctxp = C(ctx);
        Ctx *ctx = ctxp;
        XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL");
        XH_REQUIRE(arity >= 1 && arity <= MAX_ARITY, XLOG_HIP_INVALID_ARG, "relation arity must be 1..8");
        XH_REQUIRE(rows == 0 || dev_cols, XLOG_HIP_INVALID_ARG, "columns are NULL");
        xlog_hip_rel *r = rel_new(ctx, arity, rows);
        r->rows = rows;
        if (rows) pack_device_columns(ctx, dev_cols, arity, rows, r);
        *out = r;
    });
}

xlog_hip_status xlog_hip_rel_from_host_packed(xlog_hip_ctx *ctx, const uint64_t *keys, uint32_t arity, uint64_t rows,
                                              xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL");
        XH_REQUIRE(arity == 1 || arity == 2, XLOG_HIP_INVALID_ARG, "packed upload supports arity 1 or 2");
        XH_REQUIRE(rows == 0 || keys, XLOG_HIP_INVALID_ARG, "keys are NULL");
        xlog_hip_rel *r = rel_new(c, arity, rows);
        r->rows = rows;
        if (rows) XH_CHECK_HIP(hipMemcpyAsync(r->w[0], keys, rows * 8, hipMemcpyHostToDevice, c->stream));
        c->sync();
        *out = r;
    });
}

xlog_hip_status xlog_hip_rel_download_column(xlog_hip_ctx *ctx, const xlog_hip_rel *rel, uint32_t col, uint32_t *host,
                                             uint64_t host_cap) {
    return guarded([&] {
        Ctx *ctxp = C(ctx);
        Ctx *ctx = ctxp;
        need_rel(rel, "relation");
        XH_REQUIRE(col < rel->arity, XLOG_HIP_INVALID_ARG, "column out of range");
        XH_REQUIRE(host_cap >= rel->rows, XLOG_HIP_CAPACITY_OVERFLOW, "host buffer too small");
        if (!rel->rows) return;
        XH_REQUIRE(host, XLOG_HIP_INVALID_ARG, "host buffer is NULL");
        Buf<uint32_t> tmp(ctx, rel->rows);
        if (rel->arity == 1) LAUNCH_1D(k_u64_to_u32, rel->rows, rel->w[0], rel->rows, tmp.p);
        else {
            unpack_column(ctx, rel->w[col / 2], (col % 2) == 0, rel->rows, tmp.p);
        }
        XH_CHECK_HIP(hipMemcpyAsync(host, tmp.p, rel->rows * 4, hipMemcpyDeviceToHost, ctx->stream));
        ctx->sync();
    });
}


// ---- Arrow IPC stream I/O (provider/io.rs:697-773) ----------------------------
xlog_hip_status xlog_hip_arrow_ipc_decode_u32(const uint8_t *ipc, uint64_t len, uint32_t *arity, uint64_t *rows,
                                              uint32_t *cols, uint64_t cols_cap) {
    return guarded([&] {
        XH_REQUIRE(arity && rows, XLOG_HIP_INVALID_ARG, "arity / rows is NULL");
        IpcColumns ic;
        ipc_decode_u32(ipc, len, ic);
        *arity = ic.arity;
        *rows = ic.rows;
        if (!cols) return;
        XH_REQUIRE(cols_cap >= (uint64_t)ic.arity * ic.rows, XLOG_HIP_CAPACITY_OVERFLOW, "column buffer too small");
        for (uint32_t c = 0; c < ic.arity; ++c) memcpy(cols + (uint64_t)c * ic.rows, ic.cols[c], ic.rows * 4);
    });
}

xlog_hip_status xlog_hip_arrow_ipc_encode_u32(const uint32_t *const *cols, uint32_t arity, uint64_t rows,
                                              const char *const *names, uint8_t **ipc, uint64_t *len) {
    return guarded([&] {
        XH_REQUIRE(ipc && len, XLOG_HIP_INVALID_ARG, "ipc / len is NULL");
        const std::vector<uint8_t> v = ipc_encode_u32(cols, arity, rows, names);
        *ipc = to_malloc(v);
        *len = v.size();
    });
}

void xlog_hip_bytes_free(uint8_t *p) { free(p); }

xlog_hip_status xlog_hip_rel_from_arrow_ipc(xlog_hip_ctx *ctx, const uint8_t *ipc, uint64_t len, xlog_hip_rel **out) {
    return guarded([&] {
        XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL");
        IpcColumns ic;
        ipc_decode_u32(ipc, len, ic);
        *out = rel_from_ipc(C(ctx), ic);
    });
}

xlog_hip_status xlog_hip_rel_to_arrow_ipc(xlog_hip_ctx *ctx, const xlog_hip_rel *rel, const char *const *names,
                                          uint8_t **ipc, uint64_t *len) {
    return guarded([&] {
        need_rel(rel, "relation");
        XH_REQUIRE(ipc && len, XLOG_HIP_INVALID_ARG, "ipc / len is NULL");
        const std::vector<uint8_t> v = rel_to_ipc(C(ctx), rel, names);
        *ipc = to_malloc(v);
        *len = v.size();
    });
}

xlog_hip_status xlog_hip_read_arrow_ipc_stream_file(xlog_hip_ctx *ctx, const char *path, xlog_hip_rel **out) {
    return guarded([&] {
        XH_REQUIRE(path && out, XLOG_HIP_INVALID_ARG, "path / out is NULL");
        const std::string where = std::string("Failed to read Arrow IPC stream from ") + path + ": ";
        const int fd = open(path, O_RDONLY);
        XH_REQUIRE(fd >= 0, XLOG_HIP_INVALID_ARG, where + strerror(errno));
        struct stat st;
        if (fstat(fd, &st) != 0) {
            const int e = errno;
            close(fd);
            throw Error{XLOG_HIP_INVALID_ARG, where + strerror(e)};
        }
        const uint64_t n = (uint64_t)st.st_size;
        void *m = n ? mmap(nullptr, n, PROT_READ, MAP_PRIVATE, fd, 0) : nullptr;
        close(fd);
        XH_REQUIRE(n == 0 || m != MAP_FAILED, XLOG_HIP_INVALID_ARG, where + strerror(errno));
        // the column buffers are uploaded straight from the mapping
        try {
            IpcColumns ic;
            ipc_decode_u32(static_cast<const uint8_t *>(m), n, ic);
            *out = rel_from_ipc(C(ctx), ic);
        } catch (...) {
            if (m) munmap(m, n);
            throw;
        }
        if (m) munmap(m, n);
    });
}

xlog_hip_status xlog_hip_write_arrow_ipc_stream_file(xlog_hip_ctx *ctx, const xlog_hip_rel *rel,
                                                     const char *const *names, const char *path) {
    return guarded([&] {
        need_rel(rel, "relation");
        XH_REQUIRE(path, XLOG_HIP_INVALID_ARG, "path is NULL");
        const std::vector<uint8_t> v = rel_to_ipc(C(ctx), rel, names);
        const std::string where = std::string("Failed to write Arrow IPC stream to ") + path + ": ";
        FILE *f = fopen(path, "wb");
        XH_REQUIRE(f, XLOG_HIP_INVALID_ARG, where + strerror(errno));
        const bool wrote = v.empty() || fwrite(v.data(), 1, v.size(), f) == v.size();
        const int e = errno;
        const bool closed = fclose(f) == 0;
        XH_REQUIRE(wrote && closed, XLOG_HIP_INVALID_ARG, where + strerror(wrote ? errno : e));
    });
}

xlog_hip_status xlog_hip_rel_download_packed(xlog_hip_ctx *ctx, const xlog_hip_rel *rel, uint64_t *host,
                                             uint64_t host_cap) {
    return guarded([&] {
        Ctx *c = C(ctx);
        need_rel(rel, "relation");
        XH_REQUIRE(rel->arity <= 2, XLOG_HIP_INVALID_ARG, "packed download supports arity 1 or 2");
        XH_REQUIRE(host_cap >= rel->rows, XLOG_HIP_CAPACITY_OVERFLOW, "host buffer too small");
        if (!rel->rows) return;
        XH_REQUIRE(host, XLOG_HIP_INVALID_ARG, "host buffer is NULL");
        XH_CHECK_HIP(hipMemcpyAsync(host, rel->w[0], rel->rows * 8, hipMemcpyDeviceToHost, c->stream));
        c->sync();
    });
}

xlog_hip_status xlog_hip_rel_num_rows(const xlog_hip_rel *rel, uint64_t *rows) {
    return guarded([&] {
        need_rel(rel, "relation");
        XH_REQUIRE(rows, XLOG_HIP_INVALID_ARG, "rows is NULL");
        *rows = rel->rows;
    });
}
xlog_hip_status xlog_hip_rel_arity(const xlog_hip_rel *rel, uint32_t *arity) {
    return guarded([&] {
        need_rel(rel, "relation");
        XH_REQUIRE(arity, XLOG_HIP_INVALID_ARG, "arity is NULL");
        *arity = rel->arity;
    });
}
xlog_hip_status xlog_hip_rel_is_canonical(const xlog_hip_rel *rel, int *canonical) {
    return guarded([&] {
        need_rel(rel, "relation");
        XH_REQUIRE(canonical, XLOG_HIP_INVALID_ARG, "canonical is NULL");
        *canonical = (rel->flags & REL_CANONICAL) ? 1 : 0;
    });
}
xlog_hip_status xlog_hip_rel_device_words(const xlog_hip_rel *rel, uint32_t word, const uint64_t **dev) {
    return guarded([&] {
        need_rel(rel, "relation");
        XH_REQUIRE(dev, XLOG_HIP_INVALID_ARG, "dev is NULL");
        XH_REQUIRE(word < (uint32_t)rel->nwords(), XLOG_HIP_INVALID_ARG, "word index out of range");
        *dev = rel->w[word];
    });
}
xlog_hip_status xlog_hip_rel_clone(xlog_hip_ctx *ctx, const xlog_hip_rel *in, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        need_rel(in, "input");
        XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL");
        *out = rel_clone(c, in);
    });
}
void xlog_hip_rel_free(xlog_hip_rel *rel) {
    if (rel && rel->ctx) (void)hipSetDevice(rel->ctx->device);
    rel_free(rel);
}

#define OUT_GUARD XH_REQUIRE(out, XLOG_HIP_INVALID_ARG, "out is NULL"); *out = nullptr

xlog_hip_status xlog_hip_sort(xlog_hip_ctx *ctx, const xlog_hip_rel *in, const uint32_t *key_cols, uint32_t n_keys,
                              xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(in, "input");
        *out = op_sort(c, in, check_cols(in, key_cols, n_keys));
    });
}
xlog_hip_status xlog_hip_dedup(xlog_hip_ctx *ctx, const xlog_hip_rel *in, const uint32_t *key_cols, uint32_t n_keys,
                               xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(in, "input");
        *out = op_dedup(c, in, check_cols(in, key_cols, n_keys));
    });
}
xlog_hip_status xlog_hip_dedup_full_row(xlog_hip_ctx *ctx, const xlog_hip_rel *in, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(in, "input");
        *out = op_dedup_full(c, in);
    });
}
xlog_hip_status xlog_hip_union(xlog_hip_ctx *ctx, const xlog_hip_rel *a, const xlog_hip_rel *b, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(a, "a");
        need_rel(b, "b");
        const xlog_hip_rel *ins[2] = {a, b};
        *out = op_union_many(c, ins, 2);
    });
}
xlog_hip_status xlog_hip_union_many(xlog_hip_ctx *ctx, const xlog_hip_rel *const *ins, uint32_t n_ins,
                                    xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        *out = op_union_many(c, ins, n_ins);
    });
}
xlog_hip_status xlog_hip_diff(xlog_hip_ctx *ctx, const xlog_hip_rel *a, const xlog_hip_rel *b, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(a, "a");
        need_rel(b, "b");
        *out = op_diff(c, a, b);
    });
}
xlog_hip_status xlog_hip_hash_join(xlog_hip_ctx *ctx, const xlog_hip_rel *left, const xlog_hip_rel *right,
                                   uint32_t left_key, uint32_t right_key, int join_type, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        *out = op_join(c, left, right, left_key, right_key, join_type, nullptr);
    });
}
xlog_hip_status xlog_hip_hash_join_keys(xlog_hip_ctx *ctx, const xlog_hip_rel *left, const xlog_hip_rel *right,
                                        const uint32_t *left_keys, const uint32_t *right_keys, uint32_t n_keys,
                                        int join_type, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(left, "left");
        need_rel(right, "right");
        XH_REQUIRE(n_keys >= 1 && left_keys && right_keys, XLOG_HIP_INVALID_ARG, "key column lists are empty or NULL");
        XH_REQUIRE(n_keys <= MAX_ARITY, XLOG_HIP_INVALID_ARG, "more key columns than columns");
        std::vector<int> lk(left_keys, left_keys + n_keys), rk(right_keys, right_keys + n_keys);
        for (uint32_t t = 0; t < n_keys; ++t)
            XH_REQUIRE(left_keys[t] < left->arity && right_keys[t] < right->arity, XLOG_HIP_INVALID_ARG,
                       "join key column out of range");
        if (n_keys == 1 && left->arity <= 2 && right->arity <= 2)
            *out = op_join(c, left, right, left_keys[0], right_keys[0], join_type, nullptr);
        else
            *out = op_join_keys(c, left, right, lk, rk, join_type);
    });
}
xlog_hip_status xlog_hip_join_index_build(xlog_hip_ctx *ctx, const xlog_hip_rel *right, const uint32_t *right_keys,
                                          uint32_t n_keys, xlog_hip_join_index **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(right, "right");
        XH_REQUIRE(n_keys >= 1 && right_keys, XLOG_HIP_INVALID_ARG, "Join requires at least one key column");
        XH_REQUIRE(n_keys <= MAX_ARITY, XLOG_HIP_INVALID_ARG, "more key columns than columns");
        for (uint32_t t = 0; t < n_keys; ++t)
            XH_REQUIRE(right_keys[t] < right->arity, XLOG_HIP_INVALID_ARG, "right key column out of range");
        XH_REQUIRE(right->rows > 0, XLOG_HIP_INVALID_ARG, "cannot build a join index for an empty relation");
        XH_REQUIRE(right->rows < KEY_NONE, XLOG_HIP_CAPACITY_OVERFLOW, "join: more than 2^32 - 2 rows on one side");
        std::unique_ptr<xlog_hip_join_index> ix(new xlog_hip_join_index);
        ix->ctx = c;
        ix->arity = right->arity;
        ix->keys.assign(right_keys, right_keys + n_keys);
        ix->rows = right->rows;
        if (n_keys == 1 && right->arity <= 2) {
            build_join_index(c, right->w[0], right->rows, right->arity, (int)right_keys[0],
                             (right->flags & REL_CANONICAL) != 0, ix->J);
        } else {
            ix->F.reset(new KeyFold());
            fold_build(c, right, std::vector<int>(right_keys, right_keys + n_keys), *ix->F, true);
        }
        *out = ix.release();
    });
}
xlog_hip_status xlog_hip_hash_join_with_index(xlog_hip_ctx *ctx, const xlog_hip_rel *left, const xlog_hip_rel *right,
                                              const uint32_t *left_keys, const uint32_t *right_keys, uint32_t n_keys,
                                              int join_type, const xlog_hip_join_index *index, uint64_t max_output,
                                              xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(left, "left");
        need_rel(right, "right");
        XH_REQUIRE(index, XLOG_HIP_INVALID_ARG, "join index is NULL");
        XH_REQUIRE(index->ctx == c, XLOG_HIP_INVALID_ARG, "join index belongs to another context");
        XH_REQUIRE(n_keys >= 1 && left_keys && right_keys, XLOG_HIP_INVALID_ARG,
                   "Join requires at least one key column");
        XH_REQUIRE(n_keys <= MAX_ARITY, XLOG_HIP_INVALID_ARG, "more key columns than columns");
        std::vector<int> lk(left_keys, left_keys + n_keys), rk(right_keys, right_keys + n_keys);
        check_key_lists(left, right, lk, rk, join_type);
        // the index must have been built over this right relation and these key columns (relational.rs:3975-3985)
        XH_REQUIRE(index->rows == right->rows, XLOG_HIP_INVALID_ARG,
                   "Join index row count does not match right relation");
        XH_REQUIRE(index->arity == right->arity &&
                       std::vector<uint32_t>(right_keys, right_keys + n_keys) == index->keys,
                   XLOG_HIP_INVALID_ARG, "Join index key columns do not match requested right_keys");
        if (left->rows == 0) {
            *out = empty_side_join(c, left, right, join_type);
            return;
        }
        if (index->F) {
            *out = keyed_join_probe(c, left, right, lk, *index->F, join_type, max_output);
        } else if (left->arity <= 2) {
            *out = op_join_indexed(c, left, left_keys[0], index->J, right->arity, right_keys[0], join_type, nullptr,
                                   max_output);
        } else {
            *out = direct_join_wide_left(c, left, left_keys[0], index->J, right->arity, right_keys[0], join_type,
                                         max_output);
        }
    });
}
void xlog_hip_join_index_free(xlog_hip_join_index *index) { delete index; }
xlog_hip_status xlog_hip_nested_loop_join(xlog_hip_ctx *ctx, const xlog_hip_rel *left, const xlog_hip_rel *right,
                                          uint32_t left_key, uint32_t right_key, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        *out = op_nested_loop_join(c, left, right, left_key, right_key);
    });
}
xlog_hip_status xlog_hip_dedup_sorted(xlog_hip_ctx *ctx, const xlog_hip_rel *in, const uint32_t *key_cols,
                                      uint32_t n_keys, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(in, "input");
        *out = op_dedup_sorted(c, in, check_cols(in, key_cols, n_keys));
    });
}
xlog_hip_status xlog_hip_fj_delta_novel(xlog_hip_ctx *ctx, const xlog_hip_rel *delta, const xlog_hip_rel *edge,
                                        const xlog_hip_rel *full, const xlog_hip_fj_delta_cols *cols, uint32_t domain,
                                        xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        XH_REQUIRE(cols, XLOG_HIP_INVALID_ARG, "column roles are NULL");
        *out = op_fj_delta(c, delta, edge, full, *cols, domain);
    });
}
xlog_hip_status xlog_hip_fj_delta_sparse_novel(xlog_hip_ctx *ctx, const xlog_hip_rel *delta, const xlog_hip_rel *edge,
                                               const xlog_hip_rel *full, const xlog_hip_fj_delta_cols *cols,
                                               uint64_t max_table_bytes, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        XH_REQUIRE(cols, XLOG_HIP_INVALID_ARG, "cols is NULL");
        need_rel(delta, "delta");
        need_rel(edge, "edge");
        need_rel(full, "full");
        bool declined = false;
        xlog_hip_rel *r = op_fj_delta_sparse(c, delta, edge, full, *cols, max_table_bytes, &declined);
        *out = declined ? nullptr : r;
    });
}
xlog_hip_status xlog_hip_sort_merge_join(xlog_hip_ctx *ctx, const xlog_hip_rel *left, const xlog_hip_rel *right,
                                         uint32_t left_key, uint32_t right_key, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        *out = op_sort_merge_join(c, left, right, left_key, right_key);
    });
}
xlog_hip_status xlog_hip_join_project(xlog_hip_ctx *ctx, const xlog_hip_rel *left, const xlog_hip_rel *right,
                                      uint32_t left_key, uint32_t right_key, const uint32_t *out_cols, uint32_t n_out,
                                      xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        XH_REQUIRE(out_cols && n_out >= 1 && n_out <= 4, XLOG_HIP_INVALID_ARG, "out_cols must list 1..4 columns");
        std::vector<int> oc(out_cols, out_cols + n_out);
        *out = op_join(c, left, right, left_key, right_key, XLOG_HIP_JOIN_INNER, &oc);
    });
}
xlog_hip_status xlog_hip_join_project_dedup(xlog_hip_ctx *ctx, const xlog_hip_rel *left, const xlog_hip_rel *right,
                                            uint32_t left_key, uint32_t right_key, const uint32_t *out_cols,
                                            uint32_t n_out, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        XH_REQUIRE(out_cols && n_out >= 1 && n_out <= 4, XLOG_HIP_INVALID_ARG, "out_cols must list 1..4 columns");
        std::vector<int> oc(out_cols, out_cols + n_out);
        *out = op_join_project_dedup(c, left, right, left_key, right_key, oc);
    });
}
xlog_hip_status xlog_hip_project(xlog_hip_ctx *ctx, const xlog_hip_rel *in, const uint32_t *cols, uint32_t n_cols,
                                 xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(in, "input");
        *out = op_project(c, in, check_cols(in, cols, n_cols));
    });
}
xlog_hip_status xlog_hip_is_sorted(xlog_hip_ctx *ctx, const xlog_hip_rel *rel, uint32_t col, int *sorted) {
    return guarded([&] {
        Ctx *c = C(ctx);
        need_rel(rel, "relation");
        XH_REQUIRE(sorted, XLOG_HIP_INVALID_ARG, "sorted is NULL");
        XH_REQUIRE(col < rel->arity, XLOG_HIP_INVALID_ARG, "column out of range");
        *sorted = column_sorted(c, rel, col) ? 1 : 0;
    });
}
xlog_hip_status xlog_hip_exclusive_scan_u32(xlog_hip_ctx *ctx, uint32_t *dev, uint64_t n, uint64_t *total) {
    return guarded([&] {
        Ctx *ctxp = C(ctx);
        Ctx *ctx = ctxp;
        XH_REQUIRE(n == 0 || dev, XLOG_HIP_INVALID_ARG, "array is NULL");
        if (n == 0) { if (total) *total = 0; return; }
        Buf<unsigned long long> tot(ctx, 1);
        scan_u32_inplace(ctx, dev, n, tot.p);
        ctx->read_scalars(tot.p, 1);
        if (total) *total = ctx->host_scalars[0];
    });
}
xlog_hip_status xlog_hip_exclusive_scan_u32_noalloc(xlog_hip_ctx *ctx, uint32_t *dev, uint64_t n, uint64_t *total) {
    return guarded([&] {
        Ctx *c = C(ctx);
        XH_REQUIRE(n == 0 || dev, XLOG_HIP_INVALID_ARG, "array is NULL");
        scan_u32_inplace_noalloc(c, dev, n, total);
    });
}
xlog_hip_status xlog_hip_compact(xlog_hip_ctx *ctx, const xlog_hip_rel *in, const uint8_t *dev_mask, xlog_hip_rel **out) {
    return guarded([&] {
        Ctx *c = C(ctx);
        OUT_GUARD;
        need_rel(in, "input");
        XH_REQUIRE(in->rows == 0 || dev_mask, XLOG_HIP_INVALID_ARG, "mask is NULL");
        *out = compact_rel(c, in, dev_mask);
        if (in->flags & REL_CANONICAL) (*out)->flags = REL_CANONICAL;
    });
}

xlog_hip_status xlog_hip_fixpoint(xlog_hip_ctx *ctx, const int32_t *plan, uint32_t n_preds,
                                  const xlog_hip_rel *const *rels, xlog_hip_rel **out, xlog_hip_fixpoint_stats *stats) {
    return guarded([&] { run_fixpoint(C(ctx), plan, n_preds, rels, out, stats); });
}

xlog_hip_status xlog_hip_fixpoint_tc(xlog_hip_ctx *ctx, const xlog_hip_rel *edge, xlog_hip_rel **reach,
                                     xlog_hip_fixpoint_stats *stats) {
    return guarded([&] {
        Ctx *c = C(ctx);
        need_rel(edge, "edge");
        XH_REQUIRE(reach, XLOG_HIP_INVALID_ARG, "reach is NULL");
        // preds: 0 = edge, 1 = reach ; vars X=0 Y=1 Z=2
        static const int32_t plan[] = {2, 1, 0, 1, 1, 0, 0, 1, 1, 0, 2, 2, 1, 0, 1, 0, 1, 2};
        const xlog_hip_rel *rels[2] = {edge, nullptr};
        xlog_hip_rel *outs[2] = {nullptr, nullptr};
        run_fixpoint(c, plan, 2, rels, outs, stats);
        *reach = outs[1];
    });
}

xlog_hip_status xlog_hip_rel_digest(xlog_hip_ctx *ctx, const xlog_hip_rel *rel, uint64_t *digest) {
    return guarded([&] {
        Ctx *c = C(ctx);
        need_rel(rel, "relation");
        XH_REQUIRE(digest, XLOG_HIP_INVALID_ARG, "digest is NULL");
        XH_REQUIRE(rel->arity <= 2, XLOG_HIP_UNSUPPORTED, "digest supports arity 1 or 2");
        std::vector<uint64_t> h(rel->rows);
        if (rel->rows) {
            XH_CHECK_HIP(hipMemcpyAsync(h.data(), rel->w[0], rel->rows * 8, hipMemcpyDeviceToHost, c->stream));
            c->sync();
        }
        uint64_t x = 0xcbf29ce484222325ULL;
        for (uint64_t k : h)
            for (int b = 0; b < 8; ++b) { x ^= (k >> (8 * b)) & 255; x *= 0x100000001b3ULL; }
        *digest = x;
    });
}

}  // extern "C"

// ---- kernel timing -----------------------------------------------------------
unsigned long long *xh::Prof::work(double bytes_per_unit) {
    if (!on) return nullptr;
    constexpr uint64_t total = (uint64_t)Ctx::PROF_WORK_SLOTS * Ctx::PROF_WORK_SPREAD;
    if (!ctx->prof_work) {
        ctx->prof_work = static_cast<unsigned long long *>(ctx->alloc(total * sizeof(uint64_t)));
        fill_u64(ctx, reinterpret_cast<uint64_t *>(ctx->prof_work), 0ull, total);
    }
    if (ctx->prof_work_next >= Ctx::PROF_WORK_SLOTS) return nullptr;
    rec.work_slot = ctx->prof_work_next++;
    rec.bytes_per_work = bytes_per_unit;
    return ctx->prof_work + (uint64_t)rec.work_slot * Ctx::PROF_WORK_SPREAD;
}

void xh::Ctx::prof_resolve() {
    if (prof_pending.empty()) return;
    sync();
    std::vector<uint64_t> work;
    if (prof_work_next > 0) {
        const uint64_t n = (uint64_t)prof_work_next * PROF_WORK_SPREAD;
        std::vector<uint64_t> raw(n);
        XH_CHECK_HIP(hipMemcpy(raw.data(), prof_work, n * sizeof(uint64_t), hipMemcpyDeviceToHost));
        fill_u64(this, reinterpret_cast<uint64_t *>(prof_work), 0ull, n);
        work.assign(prof_work_next, 0);
        for (uint64_t i = 0; i < n; ++i) work[i / PROF_WORK_SPREAD] += raw[i];
        prof_work_next = 0;
    }
    for (auto &r : prof_pending) {
        float ms = 0.f;
        XH_CHECK_HIP(hipEventElapsedTime(&ms, r.a, r.b));
        if (r.kind >= 0 && r.kind < XLOG_HIP_KERNEL_KINDS) {
            prof_ms[r.kind] += ms;
            prof_bytes[r.kind] += r.bytes + (r.work_slot >= 0 ? r.bytes_per_work * (double)work[r.work_slot] : 0.0);
            prof_launches[r.kind] += 1;
        }
        prof_events.push_back(r.a);
        prof_events.push_back(r.b);
    }
    prof_pending.clear();
}

extern "C" {
xlog_hip_status xlog_hip_profile_enable(xlog_hip_ctx *ctx, int on) {
    return guarded([&] {
        Ctx *c = C(ctx);
        c->prof_resolve();
        c->profiling = on != 0;
    });
}
xlog_hip_status xlog_hip_profile_reset(xlog_hip_ctx *ctx) {
    return guarded([&] {
        Ctx *c = C(ctx);
        c->prof_resolve();
        for (int k = 0; k < XLOG_HIP_KERNEL_KINDS; ++k) {
            c->prof_ms[k] = 0;
            c->prof_bytes[k] = 0;
            c->prof_launches[k] = 0;
        }
    });
}
xlog_hip_status xlog_hip_profile_read(xlog_hip_ctx *ctx, uint32_t kind, uint64_t *launches, double *total_ms,
                                      double *algo_bytes) {
    return guarded([&] {
        Ctx *c = C(ctx);
        XH_REQUIRE(kind < XLOG_HIP_KERNEL_KINDS, XLOG_HIP_INVALID_ARG, "unknown kernel kind");
        c->prof_resolve();
        if (launches) *launches = c->prof_launches[kind];
        if (total_ms) *total_ms = c->prof_ms[kind];
        if (algo_bytes) *algo_bytes = c->prof_bytes[kind];
    });
}
}  // extern "C"
