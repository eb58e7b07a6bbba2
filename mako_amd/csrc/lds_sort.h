// Weights sorted by one workgroup in LDS.
#pragma once

#include "workgroup_state.h"

namespace mako {

// The sort of a worker's share, and of what a wide top-k keeps, in LDS: up to kSegCap entries (bits(q), idx), entry t * kThreads + tid in this thread's k[t] / id[t], all with
// key_lo <= bits(q) < key_hi, are dropped into kFine value buckets (descending), and every entry finds its place by counting
// the entries of its own bucket that precede it under (q desc, idx asc); they go to kout / iout as ~bits(q) and token id.
// Returns false when a bucket is too crowded to be ranked by counting.  hist must be zero and sm.flag 0 on entry, behind a
// barrier.
// sorted_lds (optional, n words of LDS: outside the sort's own, or, of more than kSortedRoom entries, over A): receives the
// sorted ~bits(q) as well, and the function then returns behind a barrier that orders LDS only: the caller goes on from the copy instead of waiting
// for the stores to kout and reading them back.
// (An entry moves as one 64-bit value, the weight above the complement of its token id, so that one comparison orders two of
// them; and whoever counts may read past the bucket's end, where all there is is smaller.  With the two halves compared and the
// reads held inside the bucket the counting took 4.3 of a worker's 11.7 us for 4 400 entries; 2.2 of 9.7 so.)
constexpr uint32_t kSortPer = kSegCap / (uint32_t)kThreads;
constexpr uint32_t kFinePer = kFine / (uint32_t)kThreads; // buckets a thread
static_assert(kSegCap % (uint32_t)kThreads == 0 && kFine % (uint32_t)kThreads == 0, "whole rounds of the workgroup");
__device__ bool lds_bucket_sort(const uint32_t (&k)[kSortPer], const uint32_t (&id)[kSortPer], uint32_t n, uint32_t key_lo, uint32_t key_hi,
                                uint32_t* kout, uint32_t* iout, unsigned long long* dyn, FinishShared& sm, uint32_t* sorted_lds = nullptr)
{
    typedef unsigned long long u64;
    constexpr uint32_t kTrip = 4;
    const lds_ptr<u64> A = as_lds(dyn); // [kSegCap + kTrip] bucket after bucket (any order inside a bucket)
    const lds_ptr<uint32_t> hist = (lds_ptr<uint32_t>)(A + kSegCap + kTrip);
    const uint32_t tid = threadIdx.x;
    // 1. buckets by value, heaviest first
    const uint32_t range = key_hi - key_lo; // > 0
    const uint32_t shift = range > kFine ? 32u - (uint32_t)__clz((range - 1u) >> 11) : 0u; // (range - 1) >> shift < kFine
    uint32_t pib[kSortPer];
#pragma unroll
    for (uint32_t t = 0; t < kSortPer; ++t) {
        pib[t] = 0;
        if (t * kThreads + tid < n)
            pib[t] = __hip_atomic_fetch_add(&hist[(key_hi - 1u - k[t]) >> shift], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    lds_barrier();
    {
        uint32_t c[kFinePer], mine = 0, most = 0;
#pragma unroll
        for (uint32_t j = 0; j < kFinePer; ++j) {
            c[j] = hist[kFinePer * tid + j];
            mine += c[j];
            most = max(most, c[j]);
        }
        if (most > 64u)
            sm.flag = 1;
        uint32_t total;
        uint32_t ex = block_excl_scan_u32(mine, total, sm.bs); // (barriers: all counts are read before)
#pragma unroll
        for (uint32_t j = 0; j < kFinePer; ++j) {
            hist[kFinePer * tid + j] = ex;
            ex += c[j];
        }
        if (tid == 0)
            hist[kFine] = total;
    }
    lds_barrier();
    MAKO_STAMP(14);
    if (sm.flag)
        return false;
#pragma unroll
    for (uint32_t t = 0; t < kSortPer; ++t)
        if (t * kThreads + tid < n)
            A[hist[(key_hi - 1u - k[t]) >> shift] + pib[t]] = ((u64)k[t] << 32) | (u64)~id[t];
    if (tid < kTrip)
        A[n + tid] = 0ull;
    lds_barrier();
    MAKO_STAMP(15);
    // 2. rank inside the bucket, and out
    const bool over = kSortedRoom < kSegCap && n > kSortedRoom; // uniform
    uint32_t place[(kSortPer + 1u) / 2u]; // (two to a word)
#pragma unroll
    for (uint32_t t = 0; t < kSortPer; ++t) {
        const uint32_t s = t * kThreads + tid;
        if (s < n) {
            const u64 me = A[s];
            const uint32_t b = (key_hi - 1u - (uint32_t)(me >> 32)) >> shift;
            const uint32_t lo = hist[b], hi = hist[b + 1u];
            // (four entries per trip: a bucket rarely holds more)
            uint32_t at = lo;
            for (uint32_t x = lo; x < hi; x += kTrip) {
                u64 o[kTrip];
#pragma unroll
                for (uint32_t u = 0; u < kTrip; ++u)
                    o[u] = A[x + u]; // (x + u < n + kTrip)
#pragma unroll
                for (uint32_t u = 0; u < kTrip; ++u)
                    at += o[u] > me ? 1u : 0u;
            }
            kout[at] = ~(uint32_t)(me >> 32);
            iout[at] = ~(uint32_t)me;
            if (sorted_lds && !over)
                sorted_lds[at] = ~(uint32_t)(me >> 32);
            place[t / 2u] = t % 2u ? place[t / 2u] | (at << 16) : at;
        }
    }
    if (sorted_lds && over) { // (every entry has its place: the copy may go over them, once all weights are in registers)
        uint32_t w[kSortPer];
#pragma unroll
        for (uint32_t t = 0; t < kSortPer; ++t)
            w[t] = (uint32_t)(A[min(t * kThreads + tid, n - 1u)] >> 32);
        lds_barrier();
#pragma unroll
        for (uint32_t t = 0; t < kSortPer; ++t)
            if (t * kThreads + tid < n)
                sorted_lds[t % 2u ? place[t / 2u] >> 16 : place[t / 2u] & 0xffffu] = ~w[t];
    }
    if (sorted_lds) // uniform
        lds_barrier();
    else
        __syncthreads();
    return true;
}

} // namespace mako
