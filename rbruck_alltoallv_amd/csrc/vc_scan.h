// vc_scan.h — wavefront-level prefix sums (64 lanes) and their workgroup composition.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vc_common.h"

#define VC_WAVE 64
#define VC_WAVES_PER_BLOCK (VC_THREADS / VC_WAVE)

// One step of a sum over lanes by data-parallel primitives: v plus the value CTRL fetches from another lane (0 for lanes it
// gives none, and in the rows of 16 lanes ROWS leaves out).  A few cycles; a lane exchange through LDS is about a hundred.
template <int CTRL, int ROWS>
__device__ __forceinline__ int64_t vc_dpp_add(int64_t v) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, false);
    return v + (((int64_t)hi << 32) | (unsigned)lo);
}

template <int CTRL, int ROWS>
__device__ __forceinline__ int64_t vc_dpp_max(int64_t v) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, false);
    const int64_t u = ((int64_t)hi << 32) | (unsigned)lo;
    return u > v ? u : v;
}

#define VC_DPP_SHR(n) (0x110 | (n))           // from n lanes below, inside a row of 16
#define VC_DPP_BCAST15 0x142                  // last lane of a row to the next row
#define VC_DPP_BCAST31 0x143                  // lane 31 to the upper half

// Inclusive prefix sum across each half (32 lanes) of a wavefront.
__device__ __forceinline__ int64_t vc_half_inclusive_scan(int64_t v) {
    v = vc_dpp_add<VC_DPP_SHR(1), 0xf>(v);
    v = vc_dpp_add<VC_DPP_SHR(2), 0xf>(v);
    v = vc_dpp_add<VC_DPP_SHR(4), 0xf>(v);
    v = vc_dpp_add<VC_DPP_SHR(8), 0xf>(v);
    return vc_dpp_add<VC_DPP_BCAST15, 0xa>(v);
}

// Inclusive prefix sum across the 64 lanes of a wavefront (lane 63: the sum of all).
__device__ __forceinline__ int64_t vc_wave_inclusive_scan(int64_t v) { return vc_dpp_add<VC_DPP_BCAST31, 0xc>(vc_half_inclusive_scan(v)); }

// Lane 63 receives the maximum of the wavefront's values, none of them negative.
__device__ __forceinline__ int64_t vc_wave_max_last(int64_t v) {
    v = vc_dpp_max<VC_DPP_SHR(1), 0xf>(v);
    v = vc_dpp_max<VC_DPP_SHR(2), 0xf>(v);
    v = vc_dpp_max<VC_DPP_SHR(4), 0xf>(v);
    v = vc_dpp_max<VC_DPP_SHR(8), 0xf>(v);
    v = vc_dpp_max<VC_DPP_BCAST15, 0xa>(v);
    return vc_dpp_max<VC_DPP_BCAST31, 0xc>(v);
}

// Lane 63 receives the sum, or the maximum, of the wavefront's values: 32 bits, an instruction a step.
template <int CTRL, int ROWS, bool MAX> __device__ __forceinline__ unsigned vc_dpp_join(unsigned v) {
    const unsigned u = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
    return MAX ? (u > v ? u : v) : v + u;
}

template <bool MAX> __device__ __forceinline__ unsigned vc_wave_join_last(unsigned v) {
    v = vc_dpp_join<VC_DPP_SHR(1), 0xf, MAX>(v);
    v = vc_dpp_join<VC_DPP_SHR(2), 0xf, MAX>(v);
    v = vc_dpp_join<VC_DPP_SHR(4), 0xf, MAX>(v);
    v = vc_dpp_join<VC_DPP_SHR(8), 0xf, MAX>(v);
    v = vc_dpp_join<VC_DPP_BCAST15, 0xa, MAX>(v);
    return vc_dpp_join<VC_DPP_BCAST31, 0xc, MAX>(v);
}

// Lane 63's value, in every lane.
__device__ __forceinline__ int64_t vc_last_lane(int64_t v) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)v, VC_WAVE - 1), hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), VC_WAVE - 1);
    return (int64_t)((unsigned long long)hi << 32 | lo);
}

// Exclusive prefix sum across a 256-thread workgroup; `total` receives the sum of all
// lanes.  `lds` must hold VC_WAVES_PER_BLOCK int64 and is safe to reuse after return.
__device__ __forceinline__ int64_t vc_block_exclusive_scan(int64_t v, int64_t *lds, int64_t &total) {
    const int lane = threadIdx.x & (VC_WAVE - 1);
    const int wave = threadIdx.x / VC_WAVE;
    int64_t incl = vc_wave_inclusive_scan(v);
    __syncthreads();                       // protects lds from the previous use
    if (lane == VC_WAVE - 1) lds[wave] = incl;
    __syncthreads();
    int64_t before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < VC_WAVES_PER_BLOCK; k++) {
        int64_t t = lds[k];
        if (k < wave) before += t;
        all += t;
    }
    total = all;
    return before + incl - v;
}

// Sum across a 256-thread workgroup (every thread gets the result).
__device__ __forceinline__ int64_t vc_block_sum(int64_t v, int64_t *lds) {
    int64_t total;
    (void)vc_block_exclusive_scan(v, lds, total);
    return total;
}

// Five totals of a 256-thread workgroup at once (one barrier): sums of v[0], v[1], v[2], maxima of v[3], v[4] (not negative).
// Thread 0 receives them; lds holds 5 * VC_WAVES_PER_BLOCK int64.
__device__ __forceinline__ void vc_block_totals(int64_t v[5], int64_t *lds) {
    const int wave = threadIdx.x / VC_WAVE;
#pragma unroll
    for (int k = 0; k < 5; k++) v[k] = k < 3 ? vc_wave_inclusive_scan(v[k]) : vc_wave_max_last(v[k]);
    if ((threadIdx.x & (VC_WAVE - 1)) == VC_WAVE - 1)
#pragma unroll
        for (int k = 0; k < 5; k++) lds[k * VC_WAVES_PER_BLOCK + wave] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < 5; k++) {
            v[k] = lds[k * VC_WAVES_PER_BLOCK];
#pragma unroll
            for (int q = 1; q < VC_WAVES_PER_BLOCK; q++) {
                const int64_t u = lds[k * VC_WAVES_PER_BLOCK + q];
                v[k] = k < 3 ? v[k] + u : (u > v[k] ? u : v[k]);
            }
        }
}

// Workgroups count themselves on one of VC_TICKETS words, each in a cache line of its own, and the last of a word on the word
// behind them: atomics on one word go one after the other, about 10 ns each (2048 workgroups on one word: +20 us).  A grid of no more
// than VC_TICKETS workgroups uses that word alone.
#define VC_TICKETS 64
#define VC_TICKET_STRIDE 32
static_assert((VC_TICKETS + 1) * VC_TICKET_STRIDE * sizeof(unsigned) <= VC_TICKET_BYTES, "room for the counts");

// Called by one thread of every workgroup of a one-dimensional grid: true for the last one.  The words are zero before and after.
__device__ __forceinline__ bool vc_last_workgroup(unsigned *ticket) {
    unsigned *const top = ticket + VC_TICKETS * VC_TICKET_STRIDE;
    unsigned of_top = gridDim.x;
    if (gridDim.x > VC_TICKETS) {
        const unsigned mine = blockIdx.x % VC_TICKETS;
        unsigned *const word = ticket + mine * VC_TICKET_STRIDE;
        if (__hip_atomic_fetch_add(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != (gridDim.x - mine + VC_TICKETS - 1) / VC_TICKETS - 1) return false;
        __hip_atomic_store(word, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        of_top = VC_TICKETS;
    }
    if (__hip_atomic_fetch_add(top, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != of_top - 1) return false;
    __hip_atomic_store(top, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// ---- a kernel that tells the host itself that it is done (VcSignal) ----
// Everything it writes is stored with vc_store_through, past the caches.
template <class V> __device__ __forceinline__ void vc_store_through(V *p, V v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }

// Called by all threads of every workgroup after their last store.
__device__ __forceinline__ void vc_signal(const VcSignal &sig) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wavefront's stores have been performed
    __syncthreads();
    if (threadIdx.x == 0 && (gridDim.x == 1 || vc_last_workgroup(sig.ticket))) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the counts are zero again when the host goes on
        vc_store_through(sig.word, sig.value);
    }
}
