// grid_sync.hpp -- workgroups of one launch that need each other's results.
//
//   last_workgroup   the ticket by which the last workgroup of a launch knows
//                    that all others have stored theirs, and then folds their
//                    partials (st_part, ld_part, part_sum) or scans their
//                    counts (part_excl_scan): in reductions, frontier scans
//                    and conversions, PageRank and delta PageRank tails;
//   grid_barrier     the grid-wide barrier of the persistent cooperative
//                    launches (the fused push, the k-core peeling), and
//                    block_read, by which a block reads after it what all of
//                    its waves need.
//
// Every word one block writes and another reads inside such a launch is
// accessed with agent-scope atomics or coherent loads and stores; before
// counting itself or arriving at the barrier each wave (for the ticket thread
// 0, which stores the workgroup's results) waits until its memory operations
// are acknowledged, so after it every block sees them.  No acquire/release
// fence is used: on this part each would write back or invalidate an XCD's L2.
#pragma once
#include "device.hpp"

namespace gpr {

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima): waits until
// this wave's earlier memory operations, stores and atomics included, are
// acknowledged
constexpr int WAIT_VM0 = 0x0f70;

constexpr int GS_GROUP = 16;            // blocks per first-level barrier counter
constexpr int GS_MAX_GROUPS = 64;
constexpr int GS_LINE = 16;             // u64 per 128-byte line: one counter per line

__device__ __forceinline__ unsigned long long ld_agent(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ unsigned long long bcast64(unsigned long long v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// Whether this workgroup is the last of its launch to get here, in every
// thread (all call it).  Thread 0's earlier stores are acknowledged before
// it counts itself, so what every workgroup's thread 0 stored with
// agent-scope stores can be read by the last one with agent-scope loads: a
// reduction of per-workgroup partials then needs no launch of its own (a
// launch in a stream costs about 6 us, most of a small graph's iteration).
// Atomics on one address go one after another, about 12 ns each (50 us for
// 4096 workgroups of a kernel that takes 10), so above LW_GROUPS workgroups
// each counts on one of LW_GROUPS lines and the last of a line on the top
// one.  All counters are zero again when the launch ends.
constexpr unsigned LW_GROUPS = 64;
constexpr unsigned LW_LINE = 32;                                   // u32 per 128-byte line
constexpr size_t LW_WORDS = (LW_GROUPS + 1) * (size_t)LW_LINE;     // top, then the groups
__device__ __forceinline__ bool count_zeroed(unsigned int *c, unsigned int all) {
    if (__hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != all - 1) return false;
    __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}
__device__ __forceinline__ bool last_workgroup(unsigned int *ticket, int *s_last) {
    if (threadIdx.x == 0) {
        __builtin_amdgcn_s_waitcnt(WAIT_VM0);
        bool l = true;
        unsigned int tops = gridDim.x;
        if (gridDim.x > LW_GROUPS) {
            const unsigned grp = blockIdx.x % LW_GROUPS;
            tops = LW_GROUPS;
            l = count_zeroed(ticket + (1 + grp) * LW_LINE,
                             gridDim.x / LW_GROUPS + (grp < gridDim.x % LW_GROUPS ? 1u : 0u));
        }
        *s_last = l && count_zeroed(ticket, tops);
    }
    __syncthreads();
    return *s_last != 0;
}
template <class T> __device__ __forceinline__ void st_part(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ T ld_part(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread t's share of a sum of partials, p[S*i] for i = t, t + NT, ... below
// count, in that order, PART_U loads in flight (each takes about 0.7 us;
// with them and half the workgroups, k_pr_update takes 13.5 us at 1.5M
// vertices instead of 16.3).
constexpr int PART_U = 8;
template <int NT, int S, class T> __device__ __forceinline__ T part_sum(const T *p, uint32_t count) {
    T s = T(0);
    for (uint32_t i = threadIdx.x; i < count; i += NT * PART_U) {
        T v[PART_U];
#pragma unroll
        for (int u = 0; u < PART_U; ++u) v[u] = ld_part(&p[(size_t)S * (i + u * NT < count ? i + u * NT : i)]);
#pragma unroll
        for (int u = 0; u < PART_U; ++u)
            if (i + u * NT < count) s += v[u];
    }
    return s;
}

// Exclusive prefix sum in place of count per-workgroup counts (st_part), by
// the last workgroup; returns the total.  A scan in a launch of its own costs
// 2 us and a gap of 4 - 8 in a traversal step.
template <int NT>
__device__ __forceinline__ unsigned long long part_excl_scan(unsigned long long *a, uint32_t count) {
    __shared__ unsigned long long wsum[NT / 64];
    const unsigned w = threadIdx.x / 64;
    unsigned long long carry = 0;
    for (uint64_t b = 0; b < count; b += NT * PART_U) {
        const uint64_t i0 = b + threadIdx.x * PART_U;
        unsigned long long v[PART_U], s = 0;
#pragma unroll
        for (int u = 0; u < PART_U; ++u) v[u] = ld_part(&a[i0 + u < count ? i0 + u : 0]);
#pragma unroll
        for (int u = 0; u < PART_U; ++u) {
            if (i0 + u >= count) v[u] = 0;
            s += v[u];
        }
        const unsigned long long inc = wave_incl_scan(s);
        if (lane() == 63) wsum[w] = inc;
        __syncthreads();      // every read of this step precedes its writes
        unsigned long long off = carry, tot = 0;
        for (unsigned j = 0; j < NT / 64; ++j) {
            if (j < w) off += wsum[j];
            tot += wsum[j];
        }
        unsigned long long run = off + inc - s;
#pragma unroll
        for (int u = 0; u < PART_U; ++u) {
            if (i0 + u < count) a[i0 + u] = run;
            run += v[u];
        }
        carry += tot;
        __syncthreads();
    }
    return carry;
}

// Grid barrier in two levels.  Block b arrives on the counter of group
// b % ngroups (at most GS_GROUP blocks each); the last block of a group to
// arrive at level `lvl` counts the group on `arrive`, and level `lvl` ends
// when (lvl+1)*ngroups groups are counted.  All counters are monotonic.
// Returns false (in every thread) when the error flag is set or the wait saw
// no new arrival for `spin_limit` polls in a row.
__device__ __forceinline__ bool grid_barrier(unsigned long long *arrive, unsigned int *error, unsigned long long *group,
                                             unsigned lvl, unsigned spin_limit, int *s_ok) {
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned ngroups = (gridDim.x + GS_GROUP - 1) / GS_GROUP;
        const unsigned grp = blockIdx.x % ngroups;
        const unsigned gsize = gridDim.x / ngroups + (grp < gridDim.x % ngroups ? 1u : 0u);
        const unsigned long long got = __hip_atomic_fetch_add(&group[grp * GS_LINE], 1ull, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_AGENT);
        if (got + 1 == (unsigned long long)(lvl + 1) * gsize)
            __hip_atomic_fetch_add(arrive, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long target = (unsigned long long)(lvl + 1) * ngroups;
        unsigned long long seen = ~0ull;
        unsigned spin = 0;
        int ok = 1;
        for (;;) {
            const unsigned long long a = ld_agent(arrive);
            if (a >= target) break;
            if (__hip_atomic_load(error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                ok = 0;
                break;
            }
            if (a != seen) {
                seen = a;
                spin = 0;
            } else if (++spin > spin_limit) {
                __hip_atomic_fetch_or(error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ok = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        *s_ok = ok;
    }
    __syncthreads();
    return *s_ok != 0;
}

// K words that every block reads after a barrier, by one lane of the block
// each and handed on through LDS (s: K words): a read by every wave of a
// 256-block grid of 1024 threads is 4096 requests for one line, about 10 us.
// All threads call it.
template <int K>
__device__ __forceinline__ void block_read(const unsigned long long *const (&p)[K], unsigned long long *s,
                                           unsigned long long (&v)[K]) {
    __syncthreads();   // the last values are read
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] = ld_agent(p[k]);
#pragma unroll
        for (int k = 0; k < K; ++k) s[k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = s[k];
}

} // namespace gpr
