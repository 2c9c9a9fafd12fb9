// last_block.hpp -- one launch for a reduction over workgroups: every
// workgroup publishes its partial result, and the one that arrives last folds
// them all.
//
// A second launch for the fold costs 3-5 us on MI355X however little it reads.
// Which workgroup is last changes from call to call, the order in which it
// adds does not, so results stay deterministic.
//
// Partials cross workgroups on different XCDs, whose L2s do not see each
// other's lines.  They go through agent-scope atomic stores and loads, which
// write and read past the L2, and not through a device fence: __threadfence()
// writes the whole L2 back, and with one in each wave the column sums of
// 20000 x 1000 took 67 us instead of 21.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

namespace ch {

// *p = v, for fetch() in any workgroup once last_block() has told it to.  U is
// a whole number of 32-bit words; 16-byte vectors go as two 64-bit ones.
template <class U>
__device__ __forceinline__ void publish(U* p, U v) {
    static_assert(sizeof(U) % 4 == 0, "whole words");
    if constexpr (sizeof(U) % 8 == 0) {
        uint64_t w[sizeof(U) / 8];
        __builtin_memcpy(w, &v, sizeof(U));
#pragma unroll
        for (unsigned i = 0; i < sizeof(U) / 8; ++i)
            __hip_atomic_store(reinterpret_cast<uint64_t*>(p) + i, w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        uint32_t w;
        static_assert(sizeof(U) == 4, "one word");
        __builtin_memcpy(&w, &v, 4);
        __hip_atomic_store(reinterpret_cast<uint32_t*>(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
template <class U>
__device__ __forceinline__ U fetch(const U* p) {
    U v;
    if constexpr (sizeof(U) % 8 == 0) {
        uint64_t w[sizeof(U) / 8];
#pragma unroll
        for (unsigned i = 0; i < sizeof(U) / 8; ++i)
            w[i] = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p) + i, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
        __builtin_memcpy(&v, w, sizeof(U));
    } else {
        static_assert(sizeof(U) == 4, "one word");
        const uint32_t w =
            __hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_memcpy(&v, &w, 4);
    }
    return v;
}

// True in every thread of the workgroup that is the last of `total` to call
// this with `counter` (0 before the launch, 0 again after it); fetch() then
// returns what any of them published before its call.  Each wave waits for its
// own stores to complete (vmcnt counts them; they complete past the L2), the
// barrier gathers the waves, and only then does the workgroup arrive.  The
// counters are the library's, one per concurrent fold of a launch, and
// launches follow each other on the library's one stream.
__device__ __forceinline__ bool last_block(uint32_t* counter, uint32_t total) {
    __shared__ uint32_t arrived;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        arrived = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != total - 1) return false;
    if (threadIdx.x == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// The same for up to kTreeGroups * kTreeArity workgroups of a 1-D grid (all of
// it): arrivals at one address are served one after the other, about 10 ns
// each (a thousand took 10 us), so workgroups arrive in groups of kTreeArity
// at counters a cache line apart, and the groups' last ones at the root.
// `counters`: kTreeWords words.
constexpr unsigned kTreeArity = 32, kTreeGroups = 64, kTreeWords = 32 * (kTreeGroups + 1);
__device__ __forceinline__ bool last_block_tree(uint32_t* counters) {
    const unsigned group = blockIdx.x / kTreeArity, groups = (gridDim.x + kTreeArity - 1) / kTreeArity;
    const unsigned left = gridDim.x - group * kTreeArity;
    if (!last_block(counters + 32 * (group + 1), left < kTreeArity ? left : kTreeArity)) return false;
    __syncthreads();  // the first arrival's word in LDS is read by all before the next
    return last_block(counters, groups);
}

}  // namespace ch
