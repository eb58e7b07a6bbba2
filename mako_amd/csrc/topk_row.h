// Top-k rows resolved from the candidate lists scan_kernel left.
#pragma once

#include "topk_candidates.h"
#include "whole_row.h"

namespace mako {

static_assert(kThreads == 1024, "the lists below and the whole-row path's sort have an entry of every 1 024 for each thread");

// The row's candidates (all slices) weighted, sorted by (q desc, idx asc) and left in LDS as kf[i] = ~bits(q_i),
// jf[i] = token id, invalid ones (q not a candidate) last.  Returns the number of valid candidates.
template <int ITEMS>
__device__ MAKO_TOPK_PART uint32_t sort_candidates(const Scratch& sc, uint32_t row, uint32_t slices, uint32_t n_cands, float m, float inv_t,
                                    float floor_q, uint32_t* kf, uint32_t* jf, const FinishLds& L)
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    unsigned long long key[ITEMS];
    candidate_keys<ITEMS>(sc, row, slices, n_cands, m, inv_t, floor_q, sm, key);
    bitonic_sort_regs<ITEMS>(key, as_lds(L.sortk));
    uint32_t nv = 0;
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t) {
        kf[t * 1024u + tid] = ~(uint32_t)(key[t] >> 32);
        jf[t * 1024u + tid] = kNone - (uint32_t)key[t];
        nv += key[t] != 0;
    }
    return block_sum_u32(nv, sm.bs); // (its barriers publish kf / jf)
}

// A top-k row (top_k <= kTopKFast) from the candidates scan_kernel left: weights of the candidates, the top_k-th
// weight's neighbourhood ordered by (q desc, idx asc) in LDS, the certificate that nothing left behind in a slice can
// reach the top_k-th weight, then top-p, total and draw by one wave.  A row that cannot be certified takes the
// whole-row path: here and now (INLINE_GENERAL), or through sort_kernel's work list.
#ifndef MAKO_TOPK_GENERAL_SITE
#define MAKO_TOPK_GENERAL_SITE 1 // (the general_row instance a top-k row falls back to: 0 where one exists anyway)
#endif
__device__ __forceinline__ void topk_row(const mako_sample_desc& d, const Scratch& sc, uint32_t row, uint32_t slices,
                                         const mako_sampling_params& P, float m, uint32_t argidx, uint32_t n_cands,
                                         const SliceStat& lane_stat, const FinishLds& L, bool have_pre = false,
                                         const CandSlots& pre = CandSlots{})
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    // ---- top-k rows: weights of the row's candidates, sorted by (q desc, idx asc) in LDS ----
    const float inv_t = 1.0f / P.temperature;
    const float floor_q = (1.0f < P.min_p) ? 1.0f : P.min_p;
    const float q_bound = candidate_bound(lane_stat, slices, m, inv_t, floor_q, sm);
    MAKO_STAMP(3);
    uint32_t* kf = reinterpret_cast<uint32_t*>(L.sortk + kSortMax); // upper half of the dynamic block
    uint32_t* jf = kf + kSortMax;
    uint32_t n_valid = 0;
    // the top_k-th weight's neighbourhood only
    uint32_t n_list = small_candidates(sc, row, slices, n_cands, m, inv_t, floor_q, P.top_k, 0u, kf, jf, n_valid, L, have_pre, pre);
    if (n_list == kNone)
        n_valid = n_cands <= 1024u ? sort_candidates<1>(sc, row, slices, n_cands, m, inv_t, floor_q, kf, jf, L)
                                   : sort_candidates<4>(sc, row, slices, n_cands, m, inv_t, floor_q, kf, jf, L);
    MAKO_STAMP(4);
    // top-k of the row = top-k of the candidates, provided nothing left behind can tie with or beat the k-th
    bool ok = n_valid >= P.top_k ? q_bound < __uint_as_float(~kf[P.top_k - 1]) : q_bound == 0.0f;
    if (ok && n_valid == 0) {
        fallback_row(d, row, argidx);
        return;
    }
    // (sampler.cpp:40-43; at most top_k <= kTopKFast <= kGroup entries.  A top-p cut too close to call is left to the
    // whole-row path, which can sum in the reference's order.)
    static_assert(kTopKFast <= kGroup, "top-k rows end in sorted_tail's short-list path");
    if (ok)
        [[clang::always_inline]] ok = sorted_tail<false, true>(d, row, P, kf, jf, min(P.top_k, n_valid), false, 0.0, MAKO_PATH_TOPK, L);
    if (ok)
        return;
    __syncthreads(); // (the lists in LDS are done with)
    // (where the whole-row path is a called function the views it receives by reference live in scratch memory: a copy
    // made here, so that only the rows that come this way store one)
    const FinishLds views = L;
    general_row<MAKO_TOPK_GENERAL_SITE>(d, sc, row, P, m, argidx, views);
}

} // namespace mako
