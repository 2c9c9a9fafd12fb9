// reduce.hip -- Sum / Mean / Max (stdlib/nn/nn.cleave:111-149), the exact
// u64 sum of u32 escape counts, and the exact i64 sum of i32 arrays (the
// same counts as cleave's i32 type carries them).
//
// One launch, deterministic for a given length and device: each workgroup of a
// fixed grid folds its rows of the array's 16-byte vectors in registers, the
// wave combines lanes with cross-lane shuffles, LDS carries the 4 wave results
// to one, and the workgroup that arrives last folds the workgroups' results in
// their order (last_block.hpp).  HBM-bound from a few MB; below that, latency.
// The host-returning forms have the kernel write the result into pinned host
// memory.  With a second launch for the fold and a copy of the result, a Mean of
// 10^6 f32 took 26.7 us, now 17; Mean, Max and argmax of 10^7 together 96, now 71.
// Queued sums of f32: 2^20 6.9 -> 4.9 us, 2^23 6.8 -> 6.1, 2^25 20.7 -> 20.1, 2^28 154 ->
// 151; of u32, 2^25 21.6 -> 20.2; of f64, 2^27 156 -> 152.  max and argmax of 2^23 10.5 ->
// 9.1, 2^25 24.7 -> 24.0, 2^28 163 -> 154, unaligned 330 -> 174.
//
// Max semantics: the reference folds acc = v[0]; if v[i] > acc then acc = v[i]
// (cmpf ogt, stdlib/num/num.cleave:303).  A NaN at i > 0 never wins; a NaN at
// v[0] is the answer.  With v[0] not NaN the fold returns the first index of
// the largest non-NaN value, which is associative as (value desc, index asc)
// -- that is what the tree combines (-0 and +0 compare equal, so the earlier
// one is kept, as in the fold).
#include <algorithm>
#include <cfloat>

#include "common.hpp"
#include "last_block.hpp"

namespace {

constexpr int kThreads = 256;
// Workgroups of the running reduction that have arrived, 0 between launches; the
// allocation-free Sum has its own, as it has its own workspace.
static __device__ uint32_t g_arrived[2][ch::kTreeWords];

// Native clang vectors (register-promoted; HIP's float4/uint4 structs are not
// always).  Loads are non-temporal: the data is read once.
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// The array as rows of kThreads vectors, read U rows at a time (fold_rows).
//   Sums      U = 4, up to two workgroups a CU: workgroup b takes rows [4 b, 4 b + 4),
//             then those a grid further on, so neighbours read neighbouring 16 KiB.
//             2^25 / 2^28 f32 20.2 / 151 us; U = 8 with four a CU 20.6 / 156, one 20.7 /
//             151, eight 20.7 / 153; U = 4 with four 20.5 / 154; U = 2 with four 20.0 /
//             152, slower to 2^24; a run of rows a workgroup, U = 8, four a CU 21.6 / 156.
//             Unaligned, a row of single elements: U = 8, four a CU (2^25 f32 22 us; 40 so).
//   Maximum   Grids and U alike, but workgroup b of G takes the run [R b / G, R (b + 1) / G)
//             of R rows, its elements in ascending order.  2^18 / 2^23 / 2^25 / 2^28 f32
//             6.9 / 9.1 / 24.0 / 154 us; U = 8 with four a CU 7.2 / 9.2 / 23.7 / 161, with two
//             7.3 / 8.7 / 23.3 / 157, eight 7.3 / 11.1 / 24.7 / 161; U = 4 with four 6.9 / 9.1 /
//             24.9 / 159; U = 16 with two 7.7 / 8.6 / 22.8 / 156.  Unaligned 6.9 / 10.2 / 24.8 /
//             174; U = 4 with two 6.7 / 14.7 / 43 / 304, U = 16 with four 7.2 / 10.3 / 24.8 / 171.
struct Rows {
    int64_t begin, end, step;
};
template <int U, bool RUN>
__device__ __forceinline__ Rows my_rows(int64_t nvec) {
    const int64_t rows = (nvec + kThreads - 1) / kThreads;
    if constexpr (RUN) return {rows * blockIdx.x / gridDim.x, rows * (blockIdx.x + 1) / gridDim.x, U};
    return {(int64_t)U * blockIdx.x, rows, (int64_t)U * gridDim.x};
}
constexpr int kVectorUnroll = 4, kScalarUnroll = 8;
constexpr int kMinRows = 4;                                      // a workgroup
constexpr int kVectorPerCu = 2, kScalarPerCu = 4;  // workgroups
unsigned row_blocks(int64_t nvec, int per_cu) {
    const int64_t rows = (nvec + kThreads - 1) / kThreads, want = (rows + kMinRows - 1) / kMinRows;
    const int64_t most = ch::kTreeArity * ch::kTreeGroups;  // of the arrival tree
    const int64_t cap = std::min<int64_t>(per_cu * (int64_t)ch::num_cus(), most);
    return (unsigned)(want < 1 ? 1 : want < cap ? want : cap);
}
unsigned grid_for(int64_t len, int per_vector, bool aligned) {
    return aligned ? row_blocks(len / per_vector, kVectorPerCu) : row_blocks(len, kScalarPerCu);
}

// ---- sum f32 / f64 ------------------------------------------------------------
// One 16-byte vector per load: 4 floats or 2 doubles.
template <class T>
struct Vec16 {
    static constexpr int kN = 16 / sizeof(T);
    typedef T type __attribute__((ext_vector_type(kN)));
};

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

template <class T>
__device__ T block_sum(T v) {
    __shared__ T part[kThreads / 64];
    v = wave_sum(v);
    __syncthreads();  // the last use's reads of part
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    T r = T(0);
    if (threadIdx.x == 0)
        for (int w = 0; w < kThreads / 64; ++w) r += part[w];
    return r;  // valid in thread 0
}

// Calls fold(vector, slot) for this workgroup's vectors in ascending order per
// thread, U loads (the slots) in flight.
template <class VT, int U, bool RUN, class Fold>
__device__ __forceinline__ void fold_rows(const void* x, int64_t nvec, Fold fold) {
    const VT* p = reinterpret_cast<const VT*>(x);
    const Rows r = my_rows<U, RUN>(nvec);
    VT v[U];
    int64_t row = r.begin;
    for (; row + U <= r.end && (row + U) * kThreads <= nvec; row += r.step) {
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(p + (row + u) * kThreads + threadIdx.x);
#pragma unroll
        for (int u = 0; u < U; ++u) fold(v[u], u);
    }
    if (row >= r.end) return;
    // at most U rows are left, the last of which may be short
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t i = (row + u) * kThreads + threadIdx.x;
        if (row + u < r.end && i < nvec) v[u] = __builtin_nontemporal_load(p + i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t i = (row + u) * kThreads + threadIdx.x;
        if (row + u < r.end && i < nvec) fold(v[u], u);
    }
}

// The last workgroup's partials t, t + 256, ... of thread t in that order, all
// loads of a run of kFoldLoads in flight together.
constexpr int kFoldLoads = 4;
template <class U, class Fold>
__device__ __forceinline__ void fold_partials(const U* partial, Fold fold) {
    const int n = (int)gridDim.x;
    for (int i0 = threadIdx.x; i0 < n; i0 += kThreads * kFoldLoads) {
        U v[kFoldLoads];
#pragma unroll
        for (int u = 0; u < kFoldLoads; ++u) v[u] = ch::fetch(partial + min(i0 + u * kThreads, n - 1));
#pragma unroll
        for (int u = 0; u < kFoldLoads; ++u)
            if (i0 + u * kThreads < n) fold(v[u]);
    }
}

// Each lane keeps an accumulator per slot and vector element, and folds the slots'
// into one per element, (c0 + c1) + (c2 + c3), every kChain trips, so that no chain of
// adds grows with the array; at the end (a0 + a1) + (a2 + a3) for f32, a0 + a1 for f64.
constexpr int kChain = 16;
template <class T>
__global__ __launch_bounds__(kThreads) void sum_kernel(const T* __restrict__ x, int64_t n, T* partial,
                                                       T* __restrict__ out, int aligned, int counter) {
    constexpr int V = Vec16<T>::kN;
    typedef typename Vec16<T>::type VT;
    static_assert(kVectorUnroll == 4, "the fold of the slots");
    T chain[kVectorUnroll][V], acc[V], lane;
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = chain[0][e] = chain[1][e] = chain[2][e] = chain[3][e] = T(0);
    int trips = 0;
    auto fold_slots = [&]() {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            acc[e] += (chain[0][e] + chain[1][e]) + (chain[2][e] + chain[3][e]);
            chain[0][e] = chain[1][e] = chain[2][e] = chain[3][e] = T(0);
        }
    };
    auto next_trip = [&](bool last_slot) {
        if (last_slot && ++trips % kChain == 0) fold_slots();
    };
    if (aligned) {
        fold_rows<VT, kVectorUnroll, false>(x, n / V, [&](VT v, int slot) {
#pragma unroll
            for (int e = 0; e < V; ++e) chain[slot][e] += v[e];
            next_trip(slot == kVectorUnroll - 1);
        });
        if (blockIdx.x == 0 && threadIdx.x < (n % V)) chain[0][0] += x[n / V * V + threadIdx.x];
    } else {
        fold_rows<T, kScalarUnroll, false>(x, n, [&](T v, int slot) {
            chain[slot % kVectorUnroll][0] += v;
            next_trip(slot == kScalarUnroll - 1);
        });
    }
    fold_slots();
    if constexpr (V == 4) lane = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    else lane = acc[0] + acc[1];
    T r = block_sum(lane);
    if (gridDim.x == 1) {
        if (threadIdx.x == 0) *out = r;
        return;
    }
    if (threadIdx.x == 0) ch::publish(partial + blockIdx.x, r);
    if (!ch::last_block_tree(g_arrived[counter])) return;
    T total = T(0);
    fold_partials(partial, [&](T v) { total += v; });
    r = block_sum(total);
    if (threadIdx.x == 0) *out = r;
}

// ---- max / argmax f32 / f64 -------------------------------------------------
template <class T>
struct Best {
    T v;
    int64_t i;
};
template <class T>
__device__ __forceinline__ void take_better(Best<T>& a, T v, int64_t i) {
    // Comparisons involving NaN are false, so a NaN candidate never wins.
    if (v > a.v || (v == a.v && i < a.i)) {
        a.v = v;
        a.i = i;
    }
}
template <class T>
__device__ __forceinline__ Best<T> wave_best(Best<T> b) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        T v = __shfl_xor(b.v, o);
        int64_t i = __shfl_xor(b.i, o);
        take_better(b, v, i);
    }
    return b;
}
template <class T>
__device__ Best<T> block_best(Best<T> b) {
    __shared__ T pv[kThreads / 64];
    __shared__ int64_t pi[kThreads / 64];
    b = wave_best(b);
    __syncthreads();  // the last use's reads of pv, pi
    if ((threadIdx.x & 63) == 0) {
        pv[threadIdx.x >> 6] = b.v;
        pi[threadIdx.x >> 6] = b.i;
    }
    __syncthreads();
    Best<T> r{-INFINITY, INT64_MAX};
    if (threadIdx.x == 0)
        for (int w = 0; w < kThreads / 64; ++w) take_better(r, pv[w], pi[w]);
    return r;
}

// A thread meets its vectors in ascending order, so in one of its element
// slots a later value replaces the best only if it is greater: a compare and
// two selects an element, where the full rule takes seven operations.
// -infinity never replaces the initial one; if nothing else is there the
// fold's own answer, v[0], is taken at the end.
template <class T>
__global__ __launch_bounds__(kThreads) void max_kernel(const T* __restrict__ x, int64_t n, T* pv, int64_t* pi,
                                                       T* __restrict__ out_v, int64_t* __restrict__ out_i,
                                                       int aligned) {
    constexpr int V = Vec16<T>::kN;
    typedef typename Vec16<T>::type VT;
    constexpr uint32_t kNone = 0xFFFFFFFFu;
    T bv[V];
    uint32_t bk[V];  // how many vectors the thread had met
    uint32_t met = 0;
#pragma unroll
    for (int e = 0; e < V; ++e) bv[e] = T(-INFINITY), bk[e] = kNone;
    Best<T> b{-INFINITY, INT64_MAX};
    const int64_t first = my_rows<kVectorUnroll, true>(aligned ? n / V : n).begin * kThreads + threadIdx.x;
    auto index = [&](uint32_t k) { return first + (int64_t)k * kThreads; };  // of the vector
    if (aligned) {
        fold_rows<VT, kVectorUnroll, true>(x, n / V, [&](VT v, int) {
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (v[e] > bv[e]) bv[e] = v[e], bk[e] = met;
            ++met;
        });
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (bk[e] != kNone) take_better(b, bv[e], V * index(bk[e]) + e);
        if (blockIdx.x == 0 && threadIdx.x < (n % V)) take_better(b, x[n / V * V + threadIdx.x], n / V * V + threadIdx.x);
    } else {
        fold_rows<T, kScalarUnroll, true>(x, n, [&](T v, int) {
            if (v > bv[0]) bv[0] = v, bk[0] = met;
            ++met;
        });
        if (bk[0] != kNone) take_better(b, bv[0], index(bk[0]));
    }
    Best<T> r = block_best(b);
    if (gridDim.x > 1) {
        if (threadIdx.x == 0) {
            ch::publish(pv + blockIdx.x, r.v);
            ch::publish(pi + blockIdx.x, r.i);
        }
        if (!ch::last_block_tree(g_arrived[0])) return;
        b = Best<T>{-INFINITY, INT64_MAX};
        const int parts = (int)gridDim.x;
        for (int i0 = threadIdx.x; i0 < parts; i0 += kThreads * kFoldLoads) {
            T v[kFoldLoads];
            int64_t ix[kFoldLoads];
#pragma unroll
            for (int u = 0; u < kFoldLoads; ++u) {
                const int i = min(i0 + u * kThreads, parts - 1);
                v[u] = ch::fetch(pv + i);
                ix[u] = ch::fetch(pi + i);
            }
#pragma unroll
            for (int u = 0; u < kFoldLoads; ++u) take_better(b, v[u], ix[u]);  // the last one again changes nothing
        }
        r = block_best(b);
    }
    if (threadIdx.x == 0) {
        T x0 = x[0];
        // nothing compares > NaN, so the fold keeps a NaN v[0]; and a best of
        // -infinity means that every other element is NaN or -infinity too
        if (x0 != x0 || !(r.v > T(-INFINITY))) {
            r.v = x0;
            r.i = 0;
        }
        if (out_v) *out_v = r.v;
        if (out_i) *out_i = r.i;
    }
}

// ---- u64 sum of u32 -----------------------------------------------------------
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ uint64_t block_sum_u64(uint64_t v) {
    __shared__ uint64_t part[kThreads / 64];
    v = wave_sum_u64(v);
    __syncthreads();  // the last use's reads of part
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    uint64_t r = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kThreads / 64; ++w) r += part[w];
    return r;
}

// Signed: each element is sign-extended to 64 bits, so the u64 total is the
// two's-complement bits of the exact i64 sum.
template <bool Signed>
__device__ __forceinline__ uint64_t widen(uint32_t v) {
    return Signed ? (uint64_t)(int64_t)(int32_t)v : (uint64_t)v;
}

template <bool Signed>
__global__ __launch_bounds__(kThreads) void sum_u32_kernel(const uint32_t* __restrict__ x, int64_t n,
                                                           uint64_t* partial, uint64_t* __restrict__ out,
                                                           int aligned) {
    uint64_t acc = 0;
    if (aligned) {
        // Add in 64 bits (mod 2^64, exact for both forms).
        fold_rows<u4, kVectorUnroll, false>(x, n / 4, [&](u4 v, int) {
            acc += (widen<Signed>(v[0]) + widen<Signed>(v[1])) + (widen<Signed>(v[2]) + widen<Signed>(v[3]));
        });
        if (blockIdx.x == 0 && threadIdx.x < (n & 3)) acc += widen<Signed>(x[n / 4 * 4 + threadIdx.x]);
    } else {
        fold_rows<uint32_t, kScalarUnroll, false>(x, n, [&](uint32_t v, int) { acc += widen<Signed>(v); });
    }
    uint64_t r = block_sum_u64(acc);
    if (gridDim.x > 1) {
        if (threadIdx.x == 0) ch::publish(partial + blockIdx.x, r);
        if (!ch::last_block_tree(g_arrived[0])) return;
        uint64_t total = 0;
        fold_partials(partial, [&](uint64_t v) { total += v; });
        r = block_sum_u64(total);
    }
    if (threadIdx.x == 0) *out = r;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Queues the sum of x into *out, a word that the device can write; the
// partials (one of T a workgroup, never more than ch::kNoAllocFloats) in part.
template <class T>
int32_t queue_sum(const T* x, int64_t len, T* part, T* out, int counter) {
    constexpr int V = Vec16<T>::kN;
    const int aligned = aligned16(x);
    const unsigned blocks = grid_for(len, V, aligned);
    sum_kernel<T><<<blocks, kThreads, 0, ch::stream()>>>(x, len, part, out, aligned, counter);
    CH_LAUNCHED("sum_kernel");
    return CLEAVE_HIP_OK;
}

// Workspace of the partials of any reduction here: 16 bytes a workgroup.
char* partials() { return (char*)ch::scratch(0, 16 * 4 * (size_t)ch::num_cus()); }

template <class T>
int32_t check_sum(const char* fn, const T* x, int64_t len, const void* out) {
    CH_REQUIRE(len >= 1, "%s: length must be >= 1 (sum reads v[0])", fn);
    CH_REQUIRE(x && out, "%s: null buffer", fn);
    CH_INIT_OR_RETURN();
    CH_DEVICE(fn, x, len * sizeof(T));
    return CLEAVE_HIP_OK;
}

// Sum into a device scalar (out_dev), or into the library's host word.
template <class T>
int32_t run_sum(const char* fn, const T* x, int64_t len, T* out, bool host) {
    int32_t st = check_sum(fn, x, len, out);
    if (st != CLEAVE_HIP_OK) return st;
    if (!host) CH_DEVICE(fn, out, sizeof(T));
    char* part = partials();
    if (!part) return CLEAVE_HIP_ERR_OOM;
    return queue_sum<T>(x, len, (T*)part, out, 0);
}

// max_of / argmax likewise: partial indices, then values.
template <class T>
int32_t run_max(const char* fn, const T* x, int64_t len, T* out_max, int64_t* out_argmax, bool host) {
    constexpr int V = Vec16<T>::kN;
    CH_REQUIRE(len >= 1, "%s: length must be >= 1 (max_of reads v[0])", fn);
    CH_REQUIRE(x && (out_max || out_argmax), "%s: null buffer", fn);
    CH_INIT_OR_RETURN();
    CH_DEVICE(fn, x, len * sizeof(T));
    if (!host && out_max) CH_DEVICE(fn, out_max, sizeof(T));
    if (!host && out_argmax) CH_DEVICE(fn, out_argmax, 8);
    const int aligned = aligned16(x);
    const unsigned blocks = grid_for(len, V, aligned);
    char* base = partials();
    if (!base) return CLEAVE_HIP_ERR_OOM;
    int64_t* pi = (int64_t*)base;
    T* pv = (T*)(base + sizeof(int64_t) * blocks);
    max_kernel<T><<<blocks, kThreads, 0, ch::stream()>>>(x, len, pv, pi, out_max, out_argmax, aligned);
    CH_LAUNCHED("max_kernel");
    return CLEAVE_HIP_OK;
}

template <bool Signed>
int32_t run_sum_u32(const char* fn, const uint32_t* x, int64_t len, uint64_t* out, bool host) {
    CH_REQUIRE(len >= 0, "%s: negative length", fn);
    CH_REQUIRE(x && out, "%s: null buffer", fn);
    CH_INIT_OR_RETURN();
    CH_DEVICE(fn, x, len * 4);
    if (!host) CH_DEVICE(fn, out, 8);
    const int aligned = aligned16(x);
    const unsigned blocks = grid_for(len, 4, aligned);
    uint64_t* part = (uint64_t*)partials();
    if (!part) return CLEAVE_HIP_ERR_OOM;
    sum_u32_kernel<Signed><<<blocks, kThreads, 0, ch::stream()>>>(x, len, part, out, aligned);
    CH_LAUNCHED("sum_u32_kernel");
    return CLEAVE_HIP_OK;
}

// Host-returning forms: queue the reduction into a pinned host word of the
// library, wait for the stream and read it, without a copy of its own.  `bad`
// comes back after an error (NaN, or -1 for an index).
template <class R, class Queue>
R reduce_to_host(Queue queue, R bad) {
    ch::clear_error();
    if (ch::ensure_init() != CLEAVE_HIP_OK) return bad;
    R* h = (R*)ch::host_word();
    if (!h) return bad;
    if (queue(h) != CLEAVE_HIP_OK) return bad;
    if (ch::check_hip(hipStreamSynchronize(ch::stream()), "hipStreamSynchronize") != CLEAVE_HIP_OK) return bad;
    return *(volatile R*)h;
}

}  // namespace

extern "C" {

int32_t cleave_hip_reduce_sum_f32(const float* x, int64_t len, float* out_dev) {
    return run_sum<float>("cleave_hip_reduce_sum_f32", x, len, out_dev, false);
}

int32_t cleave_hip_reduce_sum_f64(const double* x, int64_t len, double* out_dev) {
    return run_sum<double>("cleave_hip_reduce_sum_f64", x, len, out_dev, false);
}

// cleave_hip_reduce_sum_f32 with its partials in the library's static
// workspace instead of allocated scratch: the same kernel, grid and result,
// and no hipMalloc/hipFree on any call.  The partials are all written before
// the last workgroup reads them, so nothing needs clearing between calls.
int32_t cleave_hip_reduce_sum_f32_noalloc(const float* x, int64_t len, float* out_dev) {
    const char* fn = "cleave_hip_reduce_sum_f32_noalloc";
    const int32_t st = check_sum(fn, x, len, out_dev);
    if (st != CLEAVE_HIP_OK) return st;
    CH_DEVICE(fn, out_dev, 4);
    float* part = ch::noalloc_workspace();
    if (!part) return ch::fail(CLEAVE_HIP_ERR_RUNTIME, "%s: the static workspace has no device address", fn);
    CH_REQUIRE(4 * ch::num_cus() <= ch::kNoAllocFloats, "%s: %d partial sums exceed the static workspace of %d floats",
               fn, 4 * ch::num_cus(), ch::kNoAllocFloats);
    return queue_sum<float>(x, len, part, out_dev, 1);
}

int32_t cleave_hip_reduce_max_f32(const float* x, int64_t len, float* max_dev, int64_t* argmax_dev) {
    return run_max<float>("cleave_hip_reduce_max_f32", x, len, max_dev, argmax_dev, false);
}

int32_t cleave_hip_reduce_max_f64(const double* x, int64_t len, double* max_dev, int64_t* argmax_dev) {
    return run_max<double>("cleave_hip_reduce_max_f64", x, len, max_dev, argmax_dev, false);
}

int32_t cleave_hip_reduce_sum_u32_u64(const uint32_t* x, int64_t len, uint64_t* out_dev) {
    return run_sum_u32<false>("cleave_hip_reduce_sum_u32_u64", x, len, out_dev, false);
}

int32_t cleave_hip_reduce_sum_i32_i64(const int32_t* x, int64_t len, int64_t* out_dev) {
    return run_sum_u32<true>("cleave_hip_reduce_sum_i32_i64", reinterpret_cast<const uint32_t*>(x), len,
                             reinterpret_cast<uint64_t*>(out_dev), false);
}

// Host-returning forms (synchronise).
float cleave_hip_sum_f32(const float* x, int64_t len) {
    return reduce_to_host<float>([&](float* h) { return run_sum<float>("cleave_hip_sum_f32", x, len, h, true); }, NAN);
}

float cleave_hip_mean_f32(const float* x, int64_t len) {
    float s = cleave_hip_sum_f32(x, len);
    return s / (float)len;  // sum(v) / sitofp(N), stdlib/nn/nn.cleave:135-138
}

float cleave_hip_max_of_f32(const float* x, int64_t len) {
    return reduce_to_host<float>(
        [&](float* h) { return run_max<float>("cleave_hip_max_of_f32", x, len, h, nullptr, true); }, NAN);
}

int64_t cleave_hip_argmax_f32(const float* x, int64_t len) {
    return reduce_to_host<int64_t>(
        [&](int64_t* h) { return run_max<float>("cleave_hip_argmax_f32", x, len, nullptr, h, true); }, -1);
}

double cleave_hip_sum_f64(const double* x, int64_t len) {
    return reduce_to_host<double>([&](double* h) { return run_sum<double>("cleave_hip_sum_f64", x, len, h, true); },
                                  NAN);
}

double cleave_hip_mean_f64(const double* x, int64_t len) {
    double s = cleave_hip_sum_f64(x, len);
    return s / (double)len;  // sum(v) / N.to() on f64, stdlib/nn/nn.cleave:135-138
}

double cleave_hip_max_of_f64(const double* x, int64_t len) {
    return reduce_to_host<double>(
        [&](double* h) { return run_max<double>("cleave_hip_max_of_f64", x, len, h, nullptr, true); }, NAN);
}

int64_t cleave_hip_argmax_f64(const double* x, int64_t len) {
    return reduce_to_host<int64_t>(
        [&](int64_t* h) { return run_max<double>("cleave_hip_argmax_f64", x, len, nullptr, h, true); }, -1);
}

int64_t cleave_hip_sum_i32_i64(const int32_t* x, int64_t len) {
    return reduce_to_host<int64_t>(
        [&](int64_t* h) {
            return run_sum_u32<true>("cleave_hip_sum_i32_i64", reinterpret_cast<const uint32_t*>(x), len,
                                     reinterpret_cast<uint64_t*>(h), true);
        },
        0);
}

uint64_t cleave_hip_sum_u32_u64(const uint32_t* x, int64_t len) {
    return reduce_to_host<uint64_t>(
        [&](uint64_t* h) { return run_sum_u32<false>("cleave_hip_sum_u32_u64", x, len, h, true); }, 0);
}

}  // extern "C"
