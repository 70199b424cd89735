// The end of a synchronous operation by the workgroup of its last launch that finishes last, instead of a launch behind it
// (publish_kernel in runtime.hip), which costs 2.6 to 3 us where a whole operation takes 8 to 15: a call of 4096 x 4096 Q8_0 by
// one row 15.4 -> 13.6 us, 2048 x 7168 Q4_K by 19 20.0 -> 18.7, an output head and its greedy selection 219 -> 216.
//
// A device-wide release fence in every workgroup, which writes back a whole L2, would cost more than the launch (256
// workgroups of a launch of a few microseconds: 25 us against 10). It is not needed where every store of the launch that
// somebody else may read goes through the L2s to memory by itself (agent scope): when a wave's stores have been
// acknowledged they are where every compute unit and every other launch finds them. Then the workgroup counts itself:
// sixteen counters on lines of their own and one for the counters, since additions to one address take 11 ns each (256
// workgroups: 10.5 us with one counter, 9.0 so, 10.9 with the launch; 1024: 19.4, 9.4 and 11.0). The counters' counter is the
// word behind the status word, and both are one atomic of eight bytes, so that the last workgroup has the status with its
// count and not by a load behind it: a call of 4096 x 4096 Q8_0 by one row 13.80 -> 13.62 us, by eight 18.5 -> 18.1. It resets what it
// counted with and publishes what publish_kernel does. Nobody waits for anybody.
#pragma once
#include "common.hpp"
#include "launch.hpp"
#include "../host/publication.h"

namespace yvex {

constexpr unsigned kArrivalLeaves = 16u, kArrivalPitch = 32u;        // counters and the words between them
static_assert(kArrivalLeaves * kArrivalPitch * 4u == YVEX_HIP_ARRIVAL_BYTES, "a line a counter");

// What a launch publishes with; without `host` somebody else does.
struct Publication {
    unsigned *arrivals, *host;
    unsigned sequence;
    int clear;
};

// A launch wrapper's offer to end the operation. A launch of many more workgroups takes so long, and stores so much, that the
// two microseconds do not show; some kernels draw the line sooner, where they are launched.
struct Publisher {
    Publication terms;
    bool taken;
};
constexpr uint64_t kPublishingGroups = 2048u;

inline Publication take_publication(Publisher *publisher, uint64_t groups, uint64_t most = kPublishingGroups)
{
    if (!publisher || groups > most) return Publication{nullptr, nullptr, 0u, 0};
    publisher->taken = true;
    return publisher->terms;
}

inline Publisher publisher_of(const yvex_hip_publication &p)
{
    return Publisher{Publication{p.arrivals, p.host, p.sequence, p.clear}, false};
}

// An output of a launch that may publish.
template <typename T>
__device__ __forceinline__ void store_published(const Publication &p, T *at, T value)
{
    if (p.host) __hip_atomic_store(at, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *at = value;
}

// The sequence number and the status word as one store of eight bytes: whoever sees the one sees the other.
__device__ __forceinline__ void publish_status(unsigned *host, unsigned sequence, int raised)
{
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(host),
                       (unsigned long long)(unsigned)raised << 32 | sequence, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Behind the last store of workgroup `group` of `groups`, by all of its threads.
__device__ __forceinline__ void publish_when_last(const Publication &p, int *status, unsigned group, unsigned groups)
{
    if (!p.host) return;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wave's stores, and what it raised, are in memory
#endif
    __syncthreads();
    if (threadIdx.x != 0u) return;
    const unsigned leaf = group % kArrivalLeaves, leaves = groups < kArrivalLeaves ? groups : kArrivalLeaves;
    const unsigned members = (groups - leaf + kArrivalLeaves - 1u) / kArrivalLeaves;
    unsigned *const counter = p.arrivals + leaf * kArrivalPitch;
    if (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != members) return;
    __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the status word below, the counters that are complete above
    const unsigned long long word = __hip_atomic_fetch_add(reinterpret_cast<unsigned long long *>(status), 1ull << 32,
                                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((unsigned)(word >> 32) + 1u != leaves) return;
    const int raised = (int)(unsigned)word;
    __hip_atomic_store(status + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (p.clear && raised) __hip_atomic_store(status, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    publish_status(p.host, p.sequence, raised);
}

}  // namespace yvex
