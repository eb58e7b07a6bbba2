// The candidate lists scan_kernel left of a row: their weights, and the heaviest of them in order.
#pragma once

#include "row_records.h"

namespace mako {

// (MAKO_TOPK_PART: __attribute__((noinline)) for a translation unit whose top-k code sits inside an out-of-line
// function: each part then has the register file to itself instead of spilling inside its loops.  No source sets it
// today: every kernel has its top-k rows in line.)
#ifndef MAKO_TOPK_PART
#define MAKO_TOPK_PART
#endif
// Keys (bits(q) << 32 | ~token id, 0 = not a candidate) of candidates t * kThreads + tid of the row's flattened
// candidate list (all slices; sm.soff holds the slices' offsets), t < ITEMS.  Positions first, then every load
// from a clamped position with no branch in between (a branch around each load would make it wait for the one
// before), then the weights of the candidates that exist.
template <int ITEMS>
__device__ __forceinline__ void candidate_keys(const Scratch& sc, uint32_t row, uint32_t slices, uint32_t n_cands, float m,
                                               float inv_t, float floor_q, const FinishShared& sm,
                                               unsigned long long (&key)[ITEMS])
{
    const uint32_t tid = threadIdx.x;
    size_t at[ITEMS];
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t) {
        const uint32_t e = t * (uint32_t)kThreads + tid, c = e < n_cands ? e : 0u; // (past the end: candidate 0, a short search)
        uint32_t s = 0;
        while (s + 1 < slices && c >= sm.soff[s + 1]) // slice holding candidate c
            ++s;
        at[t] = ((size_t)row * sc.slices_cap + s) * kCap + (c - sm.soff[s]);
    }
    float w[ITEMS];
    uint32_t id[ITEMS];
    const global_ptr<const float> cand_w = as_global(sc.cand_w);
    const global_ptr<const uint32_t> cand_i = as_global(sc.cand_i);
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t)
        w[t] = cand_w[at[t]];
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t)
        id[t] = cand_i[at[t]];
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t) {
        key[t] = 0;
        if (t * (uint32_t)kThreads < n_cands) { // uniform: whole trips past the end of the list are skipped
            const float q = weight_of(w[t], m, inv_t, sm.tab);
            if (t * (uint32_t)kThreads + tid < n_cands && q >= floor_q && q > 0.0f)
                key[t] = ((unsigned long long)__float_as_uint(q) << 32) | (unsigned long long)(kNone - id[t]);
        }
    }
}

// The same keys from the candidate lists read as SLOTS: thread tid takes entries (tid % 128) + 128 t, t < 4, of slice
// tid / 128 (in a workgroup of 1024; an eighth of the threads to a slice in any), whether or not the slice emitted that many.  Where the lists end is not needed to ask for them, so the
// loads go out together with the loads of the slices' records instead of one trip to memory behind them; and
// since every slice's list starts at t = 0, the trips past the longest list are skipped by whole waves.
// For rows of at most eight slices.
constexpr uint32_t kSlotThreads = (uint32_t)kThreads / 8u;
constexpr int kPrefetchItems = (int)(kCap / kSlotThreads);
struct CandSlots {
    float w[kPrefetchItems];
    uint32_t id[kPrefetchItems];
};
__device__ __forceinline__ bool slots_cover(uint32_t slices) { return slices <= 8u; }
__device__ __forceinline__ void fetch_candidate_slots(const Scratch& sc, uint32_t row, uint32_t slices, CandSlots& c)
{
    static_assert(kCap == (uint32_t)kPrefetchItems * kSlotThreads && kSortMax == (uint32_t)(kPrefetchItems * kThreads), "eight slices' lists, one entry after the other");
    const uint32_t sl = min(threadIdx.x / kSlotThreads, slices - 1u), i0 = threadIdx.x % kSlotThreads;
    const size_t base = ((size_t)row * sc.slices_cap + sl) * kCap + i0;
    const global_ptr<const float> cand_w = as_global(sc.cand_w);
    const global_ptr<const uint32_t> cand_i = as_global(sc.cand_i);
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)kPrefetchItems; ++t) {
        c.w[t] = cand_w[base + kSlotThreads * t];
        c.id[t] = cand_i[base + kSlotThreads * t];
    }
}
// (sm.soff as candidate_bound() leaves it)
__device__ __forceinline__ void keys_from_slots(const CandSlots& c, uint32_t slices, float m, float inv_t, float floor_q,
                                                const FinishShared& sm, unsigned long long (&key)[kPrefetchItems])
{
    const uint32_t sl = min(threadIdx.x / kSlotThreads, slices - 1u), i0 = threadIdx.x % kSlotThreads;
    const uint32_t emitted = threadIdx.x / kSlotThreads < slices ? sm.soff[sl + 1] - sm.soff[sl] : 0u;
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)kPrefetchItems; ++t) {
        key[t] = 0;
        if (i0 + kSlotThreads * t < emitted) {
            const float q = weight_of(c.w[t], m, inv_t, sm.tab);
            if (q >= floor_q && q > 0.0f)
                key[t] = ((unsigned long long)__float_as_uint(q) << 32) | (unsigned long long)(kNone - c.id[t]);
        }
    }
}

// Fast route for rows that need only a few of their candidates.  Every thread weights up to kPrefetchItems candidates;
// those at or above a weight threshold (at most kSmall of them) are ordered by (q desc, idx asc) by counting, for
// each, the entries that precede it, and left in LDS as kf[i] = ~bits(q_i), jf[i] = token id.
//   top_k > 0:  the threshold is the lower edge of the quarter-binade bin that holds the top_k-th largest weight
//               (one histogram over bits(q) >> 21), so the list is a superset of the row's top_k candidates.
//   top_k == 0: the threshold is thr_bits, below which the nucleus cannot reach (from the row's histogram).
// Returns the number of entries in the list, or kNone when they exceed kSmall (nothing is written then);
// n_valid receives the number of candidates that have a weight at all.
// `pre` (when have_pre): the row's candidate slots as fetch_candidate_slots() loaded them.
__device__ MAKO_TOPK_PART uint32_t small_candidates(const Scratch& sc, uint32_t row, uint32_t slices, uint32_t n_cands, float m, float inv_t,
                                     float floor_q, uint32_t top_k, uint32_t thr_bits, uint32_t* kf, uint32_t* jf,
                                     uint32_t& n_valid, const FinishLds& L, bool have_pre = false,
                                     const CandSlots& pre = CandSlots{})
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    uint32_t* hist = reinterpret_cast<uint32_t*>(L.sortk);             // [512]
    unsigned long long* sel = L.sortk + 256;                           // [kSmall]
    uint32_t* rank = reinterpret_cast<uint32_t*>(L.sortk + 256 + kSmall); // [kSmall]
    uint32_t* counter = rank + kSmall;
    // (cleared before the candidates are fetched: the barrier behind their weights then covers this too)
    if (tid < 512)
        hist[tid] = 0;
    if (tid < kSmall)
        rank[tid] = 0;
    if (tid == 0)
        *counter = 0;
    constexpr uint32_t kItems = (uint32_t)kPrefetchItems;
    unsigned long long key[kItems];
    if (have_pre) // uniform
        keys_from_slots(pre, slices, m, inv_t, floor_q, sm, key);
    else
        candidate_keys<kPrefetchItems>(sc, row, slices, n_cands, m, inv_t, floor_q, sm, key);
    MAKO_STAMP(17);
    lds_barrier();
    uint32_t n_list;
    if (top_k > 0) {
#pragma unroll
        for (uint32_t t = 0; t < kItems; ++t)
            if (key[t])
                atomicAdd(&hist[min((uint32_t)(key[t] >> 53), 511u)], 1u);
        lds_barrier();
        if (wave_id() == 0) {
            // one wave finds the bin of the top_k-th weight: eight bins per lane from the top down, a scan over the
            // lanes' counts, then the lane that holds the bin goes through its eight
            uint32_t c[8], mine = 0;
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                c[j] = hist[511u - (lane_id() * 8u + j)];
                mine += c[j];
            }
            const uint32_t upto = __ockl_wfscan_add_u32(mine, true);
            const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)upto, kWave - 1);
            uint32_t above = upto - mine, bits = 0, taken = 0;
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                if (above < top_k && top_k <= above + c[j]) {
                    bits = (511u - (lane_id() * 8u + j)) << 21;
                    taken = above + c[j];
                }
                above += c[j];
            }
            const unsigned long long hit = __ballot(taken != 0);
            const int owner = hit ? __ffsll((long long)hit) - 1 : 0;
            if (lane_id() == owner) {
                sm.flag = hit ? bits : 0u; // 0 when the row has fewer than top_k candidates
                sm.ticket = hit ? taken : 0u;
                sm.aux = total;
            }
        }
        lds_barrier();
        n_valid = sm.aux;
        thr_bits = sm.flag;
        n_list = n_valid < top_k ? n_valid : sm.ticket;
    } else {
        uint32_t mine = 0, ge = 0;
#pragma unroll
        for (uint32_t t = 0; t < kItems; ++t) {
            mine += key[t] != 0;
            ge += key[t] != 0 && (uint32_t)(key[t] >> 32) >= thr_bits;
        }
        const uint32_t both = block_sum_u32((mine << 16) | ge, sm.bs); // each below 65536
        n_valid = both >> 16;
        n_list = both & 0xffffu;
    }
    MAKO_STAMP(18);
    if (n_list > kSmall)
        return kNone;
    // compaction in any order: the keys are distinct, the ranks below put them in place
    const unsigned long long lower = (1ull << lane_id()) - 1ull;
#pragma unroll
    for (uint32_t t = 0; t < kItems; ++t) {
        const bool keep = key[t] != 0 && (uint32_t)(key[t] >> 32) >= thr_bits;
        const unsigned long long bal = __ballot(keep);
        if (bal) {
            uint32_t base = 0;
            if (lane_id() == (uint32_t)__ffsll((long long)bal) - 1u)
                base = atomicAdd(counter, (uint32_t)__popcll(bal));
            base = (uint32_t)__builtin_amdgcn_readlane((int)base, __ffsll((long long)bal) - 1);
            if (keep)
                sel[base + (uint32_t)__popcll(bal & lower)] = key[t];
        }
    }
    __syncthreads();
    MAKO_STAMP(19);
    {
        const uint32_t e = tid & (kSmall - 1u), part = tid / kSmall; // kParts threads share the comparisons of an entry
        constexpr uint32_t kParts = (uint32_t)kThreads / kSmall;
        const unsigned long long my = e < n_list ? sel[e] : ~0ull;
        // each of them takes its part of the list; waves whose entries lie past its end have nothing to count
        const uint32_t chunk = (n_list + kParts - 1u) / kParts, jb = part * chunk, je = min(n_list, jb + chunk);
        uint32_t r = 0;
        if ((e & ~(kWave - 1u)) < n_list) {
#pragma unroll 4
            for (uint32_t j = jb; j < je; ++j)
                r += sel[j] > my;
        }
        if (r)
            atomicAdd(&rank[e], r);
        __syncthreads();
        if (tid < n_list) {
            const uint32_t at = rank[tid];
            kf[at] = ~(uint32_t)(my >> 32);
            jf[at] = kNone - (uint32_t)my;
        }
    }
    __syncthreads();
    return n_list;
}

} // namespace mako
