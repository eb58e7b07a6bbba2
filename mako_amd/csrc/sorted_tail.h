// Sorted candidate lists (and lists in token order): top-p cut, exact fp32 total and walk.
#pragma once

#include "generic_replay.h"
#include "group_chain.h"

namespace mako {

constexpr uint32_t kSeqMax = 1024; // lists up to this long get their total and walk entry by entry

// The band for a top-p cut in a sorted list of n weights q_at(0 .. n).  When total64 is the sum of
// exactly these weights and the lightest one's last bit still lies within 53 bits of the total's first, no fp64
// addition of any of these sums can round, whatever the order: all of them are exact, the reference's too, and the
// comparison with `want` is the reference's (band 0).
template <typename Get>
__device__ __forceinline__ double cut_band(bool have_total, uint32_t n_vocab, uint32_t n, Get q_at, double total64)
{
    if (have_total)
        return order_band(n_vocab, total64);
    return total64 <= (double)q_at(n - 1u) * 0x1p29 ? 0.0 : order_band(n, total64);
}

// q_at(0) + q_at(1) + ... as the reference's loop adds them: one wave, one fp64 addition after the other, 256
// entries per round (lane l brings entries 4l .. 4l+3, handed round lane by lane).  Stops after the round in which
// the sum reaches `want` and returns in n_added how many entries the reference's `while (n < k && sum < want)` adds
// (n, if the sum stays below `want`; pass +inf for a plain total).  Every lane returns the sum.  One wave calls it.
template <typename Get>
__device__ MAKO_RARE_CALL double wave_sequential_sum(Get q_at, uint32_t n, double want, uint32_t& n_added)
{
    double cum = 0.0;
    n_added = n;
    for (uint32_t base = 0; base < n; base += 4u * kWave) {
        float q[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t i = base + lane_id() * 4u + j;
            q[j] = i < n ? q_at(i) : 0.0f;
        }
        const double before = cum;
        for (uint32_t l = 0; l < kWave; ++l) {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                cum += (double)__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(q[j]), l));
        }
        if (cum >= want) { // (uniform) the reference stopped inside this round: again, entry by entry
            cum = before;
            uint32_t k = 0;
            for (; k < 4u * kWave && base + k < n && cum < want; ++k)
                cum += (double)__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(q[k & 3u]), k >> 2));
            n_added = base + k;
            break;
        }
    }
    return cum;
}

// The reference's `total` (src/gen/sampler.cpp:46-48) over n weights in the order q_at gives them.  All threads call,
// all get it.
template <typename Get>
__device__ MAKO_RARE_CALL double reference_total(Get q_at, uint32_t n, FinishShared& sm)
{
    __syncthreads();
    if (wave_id() == 0) {
        uint32_t added;
        const double t = wave_sequential_sum(q_at, n, (double)INFINITY, added);
        if (lane_id() == 0)
            sm.bs.f64[0] = t;
    }
    __syncthreads();
    const double t = sm.bs.f64[0];
    __syncthreads();
    return t;
}

// Tail of every path that ends with a list sorted by (q desc, idx asc): kf[i] = ~bits(q_i), jf[i] = token id,
// n1 entries (already cut to top_k).  Applies top-p (src/gen/sampler.cpp:44-61) against total64 (the fp64 sum over
// the row's candidates; summed from the list when !have_total), then the exact fp32 total (:80-82) and walk
// (:64-73).  All threads of the workgroup must call it.
//
// When `need_cut` the list is only the heaviest part of the row's candidates and every candidate missing from
// it weighs at most q_bound: the nucleus must then end inside the list, at an entry strictly heavier than
// q_bound.  If it does not, nothing is written and false is returned (the caller widens the list).
//
// A cut that the sums here cannot tell from its neighbour with certainty (see order_band) is not made: nothing is
// written and false is returned.  The caller then either widens (need_cut) or calls the EXACT instance with, as
// total64, the reference's own total (reference_total() over the candidates in the reference's order): the cut is
// then made by the reference's running sum, entry by entry.  EXACT on a whole list always succeeds.  (An instance of
// its own, so that the usual one carries none of its code: sorted_tail_exact().)
//
// `recs` (`t_groups` of them) describe a list whose groups were prepared by sort_kernel's workers; without them the list is
// cut into groups of kGroup here.
// SHORT_ONLY: the caller's lists never exceed kGroup entries; the code for longer ones is left out.
// UNSORTED (with PLANNED): some of the workers' shares may have been left unsorted, as one record each
// (unsorted_shares.h); a row whose records of that kind cannot all be applied is given up (false).
// UNORDERED (with PLANNED, without a top-p): the list is in token order, not sorted (a row that is neither cut to a
// top-k nor to a nucleus: src/gen/sampler.cpp:79-83 and :64-72 over the candidates as they come); nothing here needs
// the order.
template <bool PLANNED = false, bool SHORT_ONLY = false, bool EXACT = false, bool UNSORTED = false, bool UNORDERED = false>
__device__ bool sorted_tail(const mako_sample_desc& d, uint32_t row, const mako_sampling_params& P, const uint32_t* kf_ptr,
                            const uint32_t* jf, uint32_t n1_arg, bool have_total, double total64, uint32_t path,
                            const FinishLds& L, bool need_cut = false, float q_bound = 0.0f, const GroupRec* recs = nullptr,
                            uint32_t t_groups = 0)
{
    assume_lds(L);
    constexpr bool exact = EXACT;
    using namespace seqfp;
    // (a planned row's list is in device memory; the other callers may hand over a list in LDS)
    const typename std::conditional<PLANNED, GlobalKeys, AnyKeys>::type kf{kf_ptr};
    const float u_row = d.u[row]; // (asked for here, wanted much later)
    const uint32_t n1 = uniform_u32(n1_arg);
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    auto qat = [=](uint32_t i) { return __uint_as_float(~kf[i]); };
    // (UNORDERED: a list in token order, whose entry i is token i: jf is not read)
    auto idat = [=](uint32_t i) {
        if constexpr (UNORDERED)
            return i;
        else
            return jf[i];
    };
    const GroupLds G = group_lds(L);
    const bool topp_active = P.top_p < 1.0f;
    if (!PLANNED && !SHORT_ONLY && n1 > kGroup * kMaxGroups) {
        // oversized lists take the generic windowed replay
        uint32_t n = n1;
        if (topp_active) {
            if (!have_total) {
                double part = 0;
                for (uint32_t i = tid; i < n; i += kThreads)
                    part += (double)qat(i);
                total64 = block_sum_f64(part, sm.bs);
            }
            const double want = (double)P.top_p * total64;
            uint32_t keep = kNone;
            if (exact) {
                if (wave_id() == 0) {
                    uint32_t added;
                    const double cum = wave_sequential_sum(qat, n, want, added);
                    if (lane_id() == 0)
                        sm.aux = cum >= want ? added : kNone;
                }
                __syncthreads();
                keep = sm.aux;
            } else {
                const double band = cut_band(have_total, d.n_vocab, n, qat, total64);
                double carry = 0;
                if (tid == 0)
                    sm.aux = 0; // set: the cut is too close to `want` to call
                for (uint32_t base = 0; base < n; base += kThreads) {
                    const uint32_t i = base + tid;
                    const double q = i < n ? (double)qat(i) : 0.0;
                    double tile;
                    const double incl = carry + block_incl_scan_f64(q, tile, sm.bs);
                    const uint32_t hit = (i < n && incl >= want) ? i : kNone;
                    const uint32_t first = block_min_u32(hit, sm.bs);
                    if (first != kNone) {
                        keep = first + 1;
                        if (i == first && P.top_p > 0.0f && band != 0.0 && !(incl - want > band && want - (incl - q) > band))
                            sm.aux = 1;
                        break;
                    }
                    carry += tile;
                }
                __syncthreads();
                if (sm.aux || keep == kNone) // (a list that never reaches `want`: the reference's sum might)
                    return false;
            }
            if (need_cut && keep == kNone)
                return false;
            n = keep == kNone ? n : keep;
        }
        if (need_cut && !(q_bound < qat(n - 1)))
            return false;
        // (a call: so long a list is rare, and the code for it, in line, costs every other list registers)
        MAKO_CALL draw_from_list(d, row, qat, idat, n, path, sm);
        return true;
    }

    if (!PLANNED && n1 <= kGroup) {
        // short list: one wave does everything, the chain of fp32 roundings replayed with real additions.
        // (Verification too: 256 rows cut to 40 candidates under masks, each with a draft, take plan_kernel 10 us; sorting
        // all of a row's candidates and replaying the sum in windows of the whole workgroup took it 80.)
        MAKO_STAMP(5);
        __syncthreads(); // the list is published; sm.flag is free
        if (wave_id() == 0) {
            float q[4];
            load_span(kf, 0, n1, q);
            double p[4];
            p[0] = (double)q[0];
            p[1] = p[0] + (double)q[1];
            p[2] = p[1] + (double)q[2];
            p[3] = p[2] + (double)q[3];
            const double incl = __ockl_wfscan_add_f64(p[3], true);
            if (!have_total)
                total64 = readlane_f64(incl, kWave - 1);
            uint32_t n = n1;
            bool ok = true;
            if (topp_active && exact) {
                const double want = (double)P.top_p * total64;
                uint32_t added;
                const double cum = wave_sequential_sum(qat, n1, want, added);
                if (cum >= want)
                    n = max(added, 1u); // (sampler.cpp:58: never fewer than one)
                else
                    ok = !need_cut;
            } else if (topp_active) {
                const double want = (double)P.top_p * total64;
                const double band = cut_band(have_total, d.n_vocab, n1, qat, total64);
                const double base = incl - p[3];
                uint32_t hit = kNone;
                bool clear = true; // both neighbours of the cut clear `want` by more than the band
#pragma unroll
                for (int j = 3; j >= 0; --j)
                    if (base + p[j] >= want) {
                        hit = lane_id() * 4u + (uint32_t)j;
                        clear = !(P.top_p > 0.0f) || band == 0.0 || (base + p[j] - want > band && want - (j ? base + p[j - 1] : base) > band);
                    }
                const unsigned long long bal = __ballot(hit != kNone && hit < n1);
                if (bal) {
                    const int src = __ffsll((long long)bal) - 1;
                    n = (uint32_t)__builtin_amdgcn_readlane((int)hit, src) + 1u;
                    ok = __builtin_amdgcn_readlane((int)clear, src) != 0;
                } else {
                    ok = false; // (a list that never reaches `want`: the reference's sum might)
                }
            }
            if (ok && need_cut && !(q_bound < qat(n - 1)))
                ok = false;
            if (ok) {
                float x[4]; // (entry 64 j + lane)
                load_span_lanes(kf, 0, n, x);
                const float total = lanes_sum(x, n, 0.0f);
                const float span = total - 0.0f;
                const float prod = u_row * span;
                float r = prod + 0.0f;
                uint32_t pos = n - 1, accepted = 0;
                bool walks = true, keeps_draft = false;
                float q_draft = 0.0f;
                if (d.draft) { // uniform
                    // Verification (src/gen/sampler.cpp:93-106): the draft's place in the list, one entry per lane and
                    // ballot.  A rejected draft leaves the list for the redraw: as a weight of 0.0f it neither stops the
                    // walk nor changes r; only where the list would begin or end with it is the place next to it meant.
                    const int32_t draft = d.draft[row];
                    uint32_t pd = kNone;
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t i = j * kWave + (uint32_t)lane_id();
                        const unsigned long long at = __ballot(i < n && (int32_t)idat(min(i, n - 1u)) == draft);
                        if (at)
                            pd = j * kWave + (uint32_t)__ffsll((long long)at) - 1u;
                    }
                    q_draft = pd == kNone ? 0.0f : qat(pd);
                    accepted = r < q_draft ? 1u : 0u;
                    const uint32_t others = pd == kNone ? n : n - 1u;
                    if (accepted || others == 0u) { // (the draft, also where it is the only candidate)
                        keeps_draft = true;
                        walks = false;
                    } else {
                        const float rest = total - q_draft;
                        const float span2 = rest - 0.0f;
                        const float prod2 = d.u2[row] * span2;
                        r = prod2 + 0.0f;
                        if (pos == pd)
                            pos = n - 2u;
#pragma unroll
                        for (uint32_t j = 0; j < 4; ++j)
                            x[j] = j * kWave + (uint32_t)lane_id() == pd ? 0.0f : x[j];
                        if (r < 0.0f) {
                            pos = pd == 0u ? 1u : 0u;
                            walks = false;
                        }
                    }
                } else if (r < 0.0f) {
                    pos = 0;
                    walks = false;
                }
                if (walks && r == r && r != INFINITY)
                    walk_lanes(x, n, 0u, r, pos);
                if (d.out_cand_idx && d.out_cand_q)
                    for (uint32_t j = lane_id(); j < n && j < d.cand_cap; j += kWave) {
                        d.out_cand_idx[(size_t)row * d.cand_cap + j] = (int32_t)idat(j);
                        d.out_cand_q[(size_t)row * d.cand_cap + j] = qat(j);
                    }
                if (lane_id() == 0) {
                    RowOut o;
                    o.token = keeps_draft ? d.draft[row] : (int32_t)idat(pos);
                    o.n_cand = n;
                    o.total = total;
                    o.q = keeps_draft ? q_draft : qat(pos);
                    o.path = path;
                    o.accepted = accepted;
                    write_row(d, row, o);
                }
            }
            if (lane_id() == 0)
                sm.flag = ok;
        }
        __syncthreads();
        MAKO_STAMP(9);
        return sm.flag != 0;
    }
    if constexpr (SHORT_ONLY)
        return false; // (not reached)

    // group records: fp64 sums (and, from the workers, the increments)
    MAKO_STAMP(5);
    const uint32_t groups1 = PLANNED ? t_groups : (n1 + kGroup - 1) / kGroup;
    if (tid == 0) {
        G.misc()[3] = 0; // slots in use
        G.misc()[7] = 0; // increments to be made for the running sum
        G.misc()[8] = 0; // and for the walk
        if (UNSORTED) {
            sm.ticket = 0; // set: a record of an unsorted share where the code below needs the list itself
            sm.flag = 0;   // set: the list has such records
        }
    }
    // (the list's first entries, which sum and walk go through one by one, in the same trip to memory)
    float* const head = G.head();
    static_assert(kHeadLen % (uint32_t)kThreads == 0 && kSeqMax <= kHeadLen && kHeadStaged <= kHeadGroups, "whole rounds of the workgroup");
    uint32_t head_raw[kHeadLen / kThreads];
#pragma unroll
    for (uint32_t t = 0; t < kHeadLen / kThreads; ++t)
        head_raw[t] = kf[min(t * kThreads + tid, n1 - 1u)];
    if constexpr (PLANNED) {
        const global_ptr<const u32x4> rp = (global_ptr<const u32x4>)(as_global(recs) + min(tid, groups1 ? groups1 - 1u : 0u));
        const u32x4 r0 = rp[0], r1 = rp[1];
        lds_barrier(); // (misc[3] is published; the loads stay in flight)
        if (tid < groups1) {
            G.pg()[tid + 1] = __longlong_as_double((long long)(((unsigned long long)r0.y << 32) | r0.x));
            G.inc()[tid] = make_float2(__uint_as_float(r0.z), __uint_as_float(r0.w));
            // (clamped into the list: a record is only ever read, never trusted for addressing)
            const uint32_t st = min(r1.z, n1), pk = r1.w & ((1u << kSlotShift) - 1u);
            const uint32_t len = min(pk & kLenMask, min(kGroup, n1 - st));
            G.winc()[tid] = make_float2(__uint_as_float(r1.x), __uint_as_float(r1.y));
            G.start()[tid] = st;
            G.pack()[tid] = (pk & ~kLenMask) | len;
            // (the short lists' head and the candidates written out are read entry by entry: no unsorted share may lie
            // there, wherever the plan expected it to lie)
            if (UNSORTED && (pk & kOpaque)) {
                sm.flag = 1;
                if (tid < kHeadGroups || st < kHeadGroups * kGroup || (d.out_cand_idx && d.out_cand_q && st < d.cand_cap))
                    sm.ticket = 1;
            }
        }
    } else {
        __syncthreads();
        if (tid < groups1) {
            G.start()[tid] = tid * kGroup;
            G.pack()[tid] = min(kGroup, n1 - tid * kGroup); // (no exponents: the increments are made below)
            G.inc()[tid] = G.winc()[tid] = make_float2(INFINITY, INFINITY);
        }
        for (uint32_t g0 = wave_id() * 4u; g0 < groups1; g0 += kWaves * 4u) {
            float q[4][4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t g = min(g0 + u, groups1 - 1u);
                load_span(kf, g * kGroup, min(kGroup, n1 - g * kGroup), q[u]);
            }
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const double s = __ockl_wfred_add_f64((((double)q[u][0] + (double)q[u][1]) + (double)q[u][2]) + (double)q[u][3]);
                if (lane_id() == 0 && g0 + u < groups1)
                    G.pg()[g0 + u + 1] = s;
            }
        }
    }
#pragma unroll
    for (uint32_t t = 0; t < kHeadLen / kThreads; ++t)
        head[t * kThreads + tid] = __uint_as_float(~head_raw[t] & (t * kThreads + tid < n1 ? 0xffffffffu : 0u));
    if (tid < kWave)
        head[kHeadLen + tid] = 0.0f;
    __syncthreads();
    if (UNSORTED && sm.ticket)
        return false;
    const uint32_t path_out = (UNSORTED && path == MAKO_PATH_SORTED && sm.flag) ? MAKO_PATH_SUMMED : path;
    {
        const double v = tid < groups1 ? G.pg()[tid + 1] : 0.0;
        double all;
        const double incl = block_incl_scan_f64(v, all, sm.bs);
        if (tid < groups1)
            G.pg()[tid + 1] = incl;
        if (tid == 0)
            G.pg()[0] = 0.0;
        if (!have_total)
            total64 = all;
    }
    __syncthreads();

    // top-p: first entry at which the running fp64 sum reaches top_p * total
    MAKO_STAMP(6);
    uint32_t n = n1, groups = uniform_u32(groups1);
    if (topp_active) {
        const double want = (double)P.top_p * total64;
        uint32_t hitg = (tid < groups1 && G.pg()[tid + 1] >= want) ? tid : kNone;
        if (exact) {
            // the reference's own running sum decides; the group it ends in follows from the entry
            if (wave_id() == 0) {
                uint32_t added;
                const double cum = wave_sequential_sum(qat, n1, want, added);
                if (lane_id() == 0)
                    G.misc()[0] = cum >= want ? max(added, 1u) : kNone;
            }
            __syncthreads();
            const uint32_t n_ref = G.misc()[0];
            hitg = kNone;
            if (n_ref != kNone && tid < groups1) {
                const uint32_t st = G.start()[tid], len = G.pack()[tid] & kLenMask;
                if (st < n_ref && n_ref <= st + len)
                    hitg = tid;
            }
            __syncthreads();
        }
        const uint32_t gs = block_min_u32(hitg, sm.bs);
        if (gs == kNone && (need_cut || !exact))
            return false; // (a list that never reaches `want`: a partial one is widened, a whole one decided exactly)
        if (UNSORTED && gs != kNone && (G.pack()[gs] & kOpaque))
            return false; // (the cut falls into a share that was left unsorted)
        if (gs != kNone && exact) {
            const uint32_t st = G.start()[gs], len = G.pack()[gs] & kLenMask, keep = G.misc()[0] - st;
            __syncthreads();
            if (tid == 0 && keep != len)
                G.pack()[gs] = keep; // (no exponents: both increments are made again, or the group is replayed)
            __syncthreads();
            n = uniform_u32(G.misc()[0]);
            groups = uniform_u32(gs + 1u);
        } else if (gs != kNone) {
            const double band = cut_band(have_total, d.n_vocab, n1, qat, total64);
            if (wave_id() == 0) {
                const uint32_t st = G.start()[gs], len = G.pack()[gs] & kLenMask;
                float q[4];
                load_span(kf, st, len, q);
                double p[4];
                p[0] = (double)q[0];
                p[1] = p[0] + (double)q[1];
                p[2] = p[1] + (double)q[2];
                p[3] = p[2] + (double)q[3];
                const double incl = __ockl_wfscan_add_f64(p[3], true);
                const double base = G.pg()[gs] + (incl - p[3]);
                uint32_t hit = kNone;
                bool clear = true; // both neighbours of the cut clear `want` by more than the band
#pragma unroll
                for (int j = 3; j >= 0; --j)
                    if (base + p[j] >= want) {
                        hit = lane_id() * 4u + (uint32_t)j;
                        clear = !(P.top_p > 0.0f) || band == 0.0 || (base + p[j] - want > band && want - (j ? base + p[j - 1] : base) > band);
                    }
                const unsigned long long bal = __ballot(hit != kNone && hit < len);
                uint32_t keep = len;
                bool ok = false; // (no entry of the group reaches `want` although its sum does: too close to call)
                if (bal) {
                    const int src = __ffsll((long long)bal) - 1;
                    keep = (uint32_t)__builtin_amdgcn_readlane((int)hit, src) + 1u;
                    ok = __builtin_amdgcn_readlane((int)clear, src) != 0;
                }
                // (the shortened group's increment for the running sum is made again from the entries at hand, for the
                // binade its old one was for; the walk's is not)
                const uint32_t eg_cut = (uniform_u32(G.pack()[gs]) >> kSumExpShift) & 0xffu;
                float2 cut_inc = make_float2(INFINITY, INFINITY);
                double cut_mass = 0.0;
                if (ok && keep != len) { // uniform
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)
                        q[j] = lane_id() * 4u + j < keep ? q[j] : 0.0f;
                    cut_inc = span_incs(q, (int)eg_cut);
                    cut_mass = __ockl_wfred_add_f64((((double)q[0] + (double)q[1]) + (double)q[2]) + (double)q[3]);
                }
                if (lane_id() == 0) {
                    G.misc()[0] = ok ? st + keep : kNone;
                    if (ok && keep != len) {
                        G.pack()[gs] = keep | (eg_cut << kSumExpShift);
                        G.inc()[gs] = cut_inc;
                        G.pg()[gs + 1u] = G.pg()[gs] + cut_mass; // (the guesses' sums end with the list)
                    }
                }
            }
            __syncthreads();
            if (G.misc()[0] == kNone)
                return false;
            n = uniform_u32(G.misc()[0]);
            groups = uniform_u32(gs + 1u);
        }
    }
    if (n < 1)
        n = 1;
    // (values merged over branches the compiler cannot see as uniform: back to scalar registers)
    n = uniform_u32(n);
    groups = uniform_u32(groups);
    if (need_cut && !(q_bound < qat(n - 1)))
        return false;
    __syncthreads();

    // candidates and the row's results, once total and position are known
    auto emit = [&](float total, uint32_t pos, uint32_t accepted, bool keeps_draft, float q_draft) __attribute__((always_inline)) {
        if (d.out_cand_idx && d.out_cand_q)
            for (uint32_t j = tid; j < n && j < d.cand_cap; j += kThreads) {
                d.out_cand_idx[(size_t)row * d.cand_cap + j] = (int32_t)idat(j);
                d.out_cand_q[(size_t)row * d.cand_cap + j] = qat(j);
            }
        if (tid == 0) {
            RowOut o;
            o.token = keeps_draft ? d.draft[row] : (int32_t)idat(pos);
            o.n_cand = n;
            o.total = total;
            o.q = keeps_draft ? q_draft : qat(pos);
            o.path = path_out;
            o.accepted = accepted;
            write_row(d, row, o);
        }
    };
    // Verification (src/gen/sampler.cpp:93-106): where the draft is in the list (kNone: nowhere) ...
    auto find_draft = [&]() __attribute__((always_inline)) {
        const uint32_t draft = (uint32_t)d.draft[row];
        if constexpr (UNORDERED)
            return draft < n ? draft : kNone;
        constexpr uint32_t kTrip = 8;
        uint32_t at = kNone;
        for (uint32_t base = 0; base < n; base += kTrip * kThreads) {
            uint32_t id[kTrip];
#pragma unroll
            for (uint32_t t = 0; t < kTrip; ++t)
                id[t] = idat(min(base + t * kThreads + tid, n - 1u));
#pragma unroll
            for (uint32_t t = 0; t < kTrip; ++t)
                at = id[t] == draft && base + t * kThreads + tid < n ? base + t * kThreads + tid : at;
        }
        return block_min_u32(at, sm.bs);
    };
    // ... and the end of a redraw's walk: a rejected draft leaves the list as a weight of 0.0f, which can neither stop the
    // walk nor change r; only where the walk would run off its list onto the draft, the candidate in front of it is meant
    // (the draft itself, if there is no other).
    auto redrawn_end = [&](uint32_t pos, uint32_t dp) __attribute__((always_inline)) {
        if (pos != dp) // uniform
            return pos;
        uint32_t before = 0; // (index + 1 of the last candidate in front of it)
        for (uint32_t i = tid; i < dp; i += kThreads)
            before = qat(i) > 0.0f ? i + 1u : before;
        before = kNone - block_min_u32(kNone - before, sm.bs);
        return before ? before - 1u : dp;
    };

    MAKO_STAMP(7);
    if (n <= kSeqMax) {
        // A nucleus this short is gone through entry by entry in LDS, once for the total and once for the walk (two
        // nanoseconds an entry each way): the increments of groups only pay on longer lists.
        const uint32_t dp = d.draft ? find_draft() : kNone;
        if (wave_id() == 0) {
            const float S = sum_lds(head, n, 0.0f);
            const float span = S - 0.0f;
            const float prod = u_row * span;
            float r = prod + 0.0f;
            uint32_t at = n - 1, kept = 0;
            if (d.draft) {
                const float q_draft = dp == kNone ? 0.0f : head[dp];
                if (r < q_draft) {
                    kept = 1;
                } else {
                    const float rest = S - q_draft;
                    const float span2 = rest - 0.0f;
                    const float prod2 = d.u2[row] * span2;
                    r = prod2 + 0.0f;
                    if (dp != kNone && lane_id() == 0)
                        head[dp] = 0.0f;
                }
            }
            if (!kept) {
                if (r < 0.0f)
                    at = 0;
                else if (r == r && r != INFINITY)
                    walk_lds(head, n, r, at);
            }
            if (lane_id() == 0) {
                G.misc()[1] = __float_as_uint(S);
                G.misc()[2] = at;
                G.misc()[4] = kept;
            }
        }
        __syncthreads();
        MAKO_STAMP(9);
        const float S = __uint_as_float(G.misc()[1]);
        uint32_t pos = G.misc()[2];
        const bool kept = G.misc()[4] != 0u;
        if (d.draft && !kept)
            pos = redrawn_end(pos, dp);
        emit(S, pos, kept ? 1u : 0u, kept, (kept && dp != kNone) ? qat(dp) : 0.0f);
        return true;
    }

    // The exact fp32 total, then the walk from u times it (group_chain.h).  Where the binades change, and where the walk
    // ends, is known beforehand but for what the fp64 sums leave open: those groups' entries are fetched now, by all the
    // waves, the sum's increments that are missing are made, and while one wave then chains the running sum the others see to
    // those for the walk.
    const double r0_raw = (double)u_row * G.pg()[groups], r0_guess = r0_raw == r0_raw ? r0_raw : 0.0;
    // (the sum's leading groups: up to the last of the first two in which it changes binade; the second costs half a
    // microsecond one by one, a replay nearly one)
    const uint32_t lead = min(groups, sum_changes_binade(G, min(1u, groups - 1u)) ? 2u : 1u);
    // A walk that is expected to end within the staged head goes through it one by one: a replay for every binade r falls
    // through costs a microsecond, twelve groups at two nanoseconds an entry six.
    const double head_mass = G.pg()[min(kHeadStaged, groups)];
    bool head_walk = r0_guess * 1.001 <= head_mass || groups <= kHeadStaged;
    plan_groups<UNSORTED>(G, lead, 0u, groups, true, !head_walk, r0_guess, LeftOut{});
    __syncthreads();
    MAKO_STAMP(13);
    fill_staged(kf, G);
    // (what a worker left for another binade than is expected now: none in most rows, four in some, and the trip is only taken
    // for some.  Left to the chain to replay instead, tail_kernel took 22.9 us on the 64-row decode batch, 22.4 so)
    build_incs(kf, r0_guess, G, true, !PLANNED, (uint32_t)wave_id(), (uint32_t)kWaves);
    if (!PLANNED)
        __syncthreads();
    else
        lds_barrier();
    if (wave_id() == 0) {
        float S = 0.0f;
        const bool ok = chain_sum<UNSORTED>(kf, G, groups, lead, lead == groups ? n : uniform_u32(G.start()[lead]), S);
        MAKO_STAMP(15);
        if (lane_id() == 0)
            G.misc()[1] = ok ? __float_as_uint(S) : 0xffffffffu; // (a sum of weights is never a NaN)
    } else if (PLANNED) {
        build_incs(kf, r0_guess, G, false, true, (uint32_t)wave_id() - 1u, (uint32_t)kWaves - 1u);
    }
    __syncthreads();
    MAKO_STAMP(8);
    if (UNSORTED && G.misc()[1] == 0xffffffffu)
        return false;
    const float total = __uint_as_float(G.misc()[1]);
    const float span = total - 0.0f;
    const float prod = u_row * span;
    float r = prod + 0.0f;

    // (all the waves: the increments of the groups from `from` on for a walk that is at r_here in front of that group, and
    // the entries of the groups it is expected to replay)
    LeftOut out;
    auto prepare_walk = [&](uint32_t from, double r_here) __attribute__((always_inline)) {
        __syncthreads();
        if (tid == 0)
            G.misc()[3] = G.misc()[7] = G.misc()[8] = 0;
        if (tid < groups)
            G.pack()[tid] &= (1u << kSlotShift) - 1u;
        const double r0_here = r_here + G.pg()[from];
        __syncthreads();
        plan_groups<UNSORTED>(G, 0u, from, groups, false, true, r0_here, out);
        __syncthreads();
        fill_staged(kf, G, out);
        build_incs(kf, r0_here, G, false, true, (uint32_t)wave_id(), (uint32_t)kWaves);
        __syncthreads();
    };
    uint32_t dp = kNone;
    if (d.draft) { // uniform
        dp = find_draft();
        const float q_draft = dp == kNone ? 0.0f : qat(dp);
        if (r < q_draft) {
            emit(total, dp == kNone ? 0u : dp, 1u, true, q_draft);
            return true;
        }
        const float rest = total - q_draft;
        const float span2 = rest - 0.0f;
        const float prod2 = d.u2[row] * span2;
        r = prod2 + 0.0f;
        if (q_draft > 0.0f) { // (it is a candidate: its group is gone through without it, the sums behind it lose its weight)
            const uint32_t mine = tid < groups && G.start()[tid] <= dp && dp - G.start()[tid] < (G.pack()[tid] & kLenMask) ? tid : kNone;
            out.group = uniform_u32(block_min_u32(mine, sm.bs));
            if (out.group != kNone) {
                out.entry = dp - uniform_u32(G.start()[out.group]);
                for (uint32_t g = out.group + 1u + tid; g <= groups; g += kThreads)
                    G.pg()[g] -= (double)q_draft;
                __syncthreads();
                if (tid == 0) {
                    G.winc()[out.group] = make_float2(INFINITY, INFINITY);
                    // (nor a slot: what was fetched for the sum holds the draft, and a walk that was expected to end in the head
                    // passes it at r = 0 where nothing in it weighs anything)
                    G.pack()[out.group] &= ~(0xffu << kWalkExpShift) & ((1u << kSlotShift) - 1u);
                }
            }
        }
        const double rg = r == r ? (double)r : 0.0;
        head_walk = rg * 1.001 <= G.pg()[min(kHeadStaged, groups)] || groups <= kHeadStaged;
        if (!head_walk)
            prepare_walk(0u, rg);
        else if (q_draft > 0.0f && dp < kHeadLen && tid == 0) // (read by wave 0 alone)
            head[dp] = 0.0f;
    }

    uint32_t pos = n - 1;
    if (r < 0.0f) {
        pos = 0;
    } else if (r == r && r != INFINITY) {
        MAKO_STAMP(14);
        uint32_t first = 0; // groups already walked
        for (;;) {
            if (wave_id() == 0) {
                uint32_t at = n - 1u;
                WalkEnd end = kWalkEnd;
                if (first == 0u && head_walk) {
                    first = min(kHeadStaged, groups);
                    if (walk_lds(head, first == groups ? n : uniform_u32(G.start()[first]), r, at))
                        end = kWalkStopped;
                }
                if (end != kWalkStopped)
                    end = chain_walk<UNSORTED>(kf, G, groups, first, r, at, out);
                if (lane_id() == 0) {
                    G.misc()[0] = end;
                    G.misc()[2] = end == kWalkStopped ? at : n - 1u;
                    G.misc()[5] = first;
                    G.misc()[6] = __float_as_uint(r);
                }
            }
            __syncthreads();
            const uint32_t end = uniform_u32(G.misc()[0]);
            pos = uniform_u32(G.misc()[2]);
            if (UNSORTED && end == kWalkGaveUp)
                return false;
            if (end != kWalkRebuild)
                break;
            first = uniform_u32(G.misc()[5]);
            r = uniform_f32(__uint_as_float(G.misc()[6]));
            prepare_walk(first, (double)r);
        }
    }
    if (d.draft)
        pos = redrawn_end(pos, dp);
    MAKO_STAMP(9);
    const bool only = d.draft && pos == dp; // (the draft was the only candidate: src/gen/sampler.cpp:104-105)
    emit(total, pos, 0u, only, only ? qat(dp) : 0.0f);
    return true;
}

// The EXACT instance, out of line where the source is compiled for it (see MAKO_RARE_CALL).
template <bool PLANNED = false>
__device__ MAKO_RARE_CALL void sorted_tail_exact(const mako_sample_desc& d, uint32_t row, const mako_sampling_params& P,
                                                 const uint32_t* kf, const uint32_t* jf, uint32_t n1, double total64,
                                                 uint32_t path, const FinishLds& L)
{
    assume_lds(L);
    sorted_tail<PLANNED, false, true>(d, row, P, kf, jf, n1, true, total64, path, L, false, 0.0f);
}

} // namespace mako
