// Results that all workgroups of a launch contribute to, finished by the one that ends last
// (kernels_tau.hip, kernels_tools.hip).
#pragma once
#include "spamm_internal.h"

namespace spamm {

template <typename T>
__device__ __forceinline__ T agent_load(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void agent_store(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// True in every thread of the workgroup that finishes last.  What workgroups hand to it goes through
// agent-scope atomics only, which are performed where all XCDs see them: once a wave's have returned
// (the wait on the counter) and the workgroup has met, one relaxed add on the ticket says so.  (A
// release fence writes the XCD's whole L2 back: in every wave it took 25 us of a pass of 1100 waves,
// in one thread per workgroup still 2.)  The tickets are put back for the next launch.
//
// Adds to one address are performed one after the other, some 9 ns each, and workgroups of one size end together: so
// beyond TICKET_DIRECT of them a workgroup adds to the ticket of its group, and the last of a group to the common one
// (whole calls: 206 workgroups, selection of three passes 41.0 -> 38.5 us, count 20.6 -> 19.1; 1024, dropped bound 28.8 -> 19.3).
constexpr unsigned int TICKET_GROUPS = 16, TICKET_DIRECT = 48;
struct alignas(128) Ticket {
    unsigned int n;
};
struct Tickets {
    Ticket t[1 + TICKET_GROUPS];            // the common one, the groups'; zero between launches
};

__device__ __forceinline__ bool last_workgroup(Tickets *tickets) {
    __shared__ unsigned int s_last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned int g = blockIdx.x % TICKET_GROUPS, all = gridDim.x;
        const bool grouped = all > TICKET_DIRECT;
        bool last = true;
        if (grouped)
            last = __hip_atomic_fetch_add(&tickets->t[1 + g].n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (all - g + TICKET_GROUPS - 1) / TICKET_GROUPS - 1;
        if (last)
            last = __hip_atomic_fetch_add(&tickets->t[0].n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (grouped ? TICKET_GROUPS : all) - 1;
        s_last = last;
    }
    __syncthreads();
    if (s_last && threadIdx.x <= TICKET_GROUPS) agent_store(&tickets->t[threadIdx.x].n, 0u);
    return s_last != 0;
}

// A result for the host, which waits for `seq` to appear (pinned, coherent memory): by one thread, the
// result's words first.
template <typename T>
__device__ __forceinline__ void publish_result(T *host_out, const T &v, unsigned long long *host_seq, unsigned long long seq) {
    static_assert(sizeof(T) % 8 == 0, "results are whole 64-bit words");
    struct Words {
        unsigned long long w[sizeof(T) / 8];
    };
    const Words words = __builtin_bit_cast(Words, v);
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 8; i++)
        __hip_atomic_store(reinterpret_cast<unsigned long long *>(host_out) + i, words.w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(host_seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace spamm
