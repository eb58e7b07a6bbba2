// Rows that are cut neither to a top-k nor to a nucleus (top_k == 0, top_p >= 1, temperature > 0): the reference adds
// up and walks the candidates in token order (src/gen/sampler.cpp:29-36, :79-83, :64-72), so nothing is sorted.  A batch that
// the caller's host copy of the parameters shows to have none but rows of the whole-row class gets three launches for them
// instead of one workgroup per row on the whole-row path:
//   index_weights_kernel  a workgroup per 16 384 logits: masks and penalties as everywhere, q = expf((w - m) / T), and
//                         ~bits(q) (0.0f for a logit that is no candidate) stored at the token's own position (entry i
//                         of the list is token i: no array of token ids);
//   index_groups_kernel   a workgroup per 16 384 entries: the group records of its 64 groups of 256 (fp64 sums, the
//                         increments of the running fp32 sum and of the walk in the binades guessed from the sums before them),
//                         as sort_kernel's workers leave them for a sorted list;
//   index_tail_kernel     a workgroup per row: the exact fp32 total and the walk over the group records
//                         (sorted_tail's planned instance for lists in any order).
// Where there are, or may be, rows of other kinds beside them, the same work is done in the launches of those (beside_rows.h):
// the weights with finish_kernel's, the groups with sort_kernel's, the rest with tail_kernel's.
// A logit that is no candidate stays in the list as a weight of 0.0f: adding it changes no sum, and the walk's
// `r < q` is never true for it.  The list ends behind the row's last candidate, which is where the reference's walk
// ends when it runs off its list.  Verification works on the same list: the draft's weight is entry `draft`, and a
// rejected draft is redrawn with that entry taken as 0.0f (sorted_tail's UNORDERED instance).
// A row with up to 256 candidates (a min-p on a peaked row, a grammar's mask) needs no records: each piece leaves its candidates'
// token ids in order, and few_candidates_row() finishes the row from those.
// The other rows of the whole-row class (top-k without top-p, top-k beyond the candidate lists) only get their weights
// here (into the array general_row_from_weights() starts from), the first rounds of their nth_element (nth_steps.h), and one
// workgroup each in the last launch for the rest of the whole-row path.
#pragma once

#include "sorted_tail.h"
#include "worker_sort.h"
#include "nth_steps.h"
#include "whole_row.h"

namespace mako {

constexpr uint32_t kIndexBlock = 4096;                   // entries whose fp64 sum index_weights_kernel leaves as one number
constexpr uint32_t kIndexMaxVocab = kMaxGroups * kGroup; // the group records of a row
constexpr uint32_t kIndexFewMax = kGroup;                // candidates that a row may have to be finished from a list of them
static_assert(kIndexMaxVocab / kSliceMax <= kWorkers && kIndexMaxVocab / kIndexBlock <= kMaxSlices && kIndexMaxVocab / kIndexBlock <= (uint32_t)kWave &&
                  kSliceMax == 4u * kIndexBlock && kIndexBlock == (uint32_t)kWaves * kGroup,
              "a piece's count and last candidate travel in the plan's per-worker words, the blocks' sums in the row's part_sum, a lane each");
// The pivot of the first round of nth_element on a row that is its own list (no gaps): the median of the weights of its second
// logit, its middle and its last one.  A barrier later sm.bs.u64[0] is the pivot, [1] the first entry, sm.aux where the pivot
// is.  hl: the history's length, 0 where there is nothing to penalise.  All threads call.
__device__ __forceinline__ void first_pivot(const mako_sample_desc& d, uint32_t row, const mako_sampling_params& P, uint32_t hl, float m, FinishShared& sm)
{
    typedef unsigned long long u64;
    const uint32_t places[4] = {1u, d.n_vocab / 2u, d.n_vocab - 1u, 0u}, mine = min((uint32_t)lane_id(), 3u);
    const uint32_t at = mine == 0u ? places[0] : (mine == 1u ? places[1] : (mine == 2u ? places[2] : places[3]));
    if (hl) { // uniform
        if (threadIdx.x < 4u)
            sm.run[threadIdx.x] = 0u;
        lds_barrier();
        const global_ptr<const int32_t> ht = as_global(d.hist_tokens) + (int64_t)row * d.hist_stride;
        const global_ptr<const uint32_t> hc = d.hist_counts ? as_global(d.hist_counts) + (int64_t)row * d.hist_stride : nullptr;
        for (uint32_t h = threadIdx.x; h < hl; h += kThreads) {
            const uint32_t t = (uint32_t)ht[h];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i)
                if (t == places[i])
                    atomicAdd(&sm.run[i], hc ? hc[h] : 1u);
        }
        lds_barrier();
    }
    if (wave_id() == 0) {
        float w = as_global(d.logits)[(int64_t)row * d.logits_stride + at];
        const uint32_t word = d.mask ? as_global(d.mask)[(int64_t)row * d.mask_stride + (at >> 5)] : ~0u;
        w = (word >> (at & 31u)) & 1u ? w : -INFINITY;
        const uint32_t c = hl ? sm.run[mine] : 0u;
        if (c)
            w = penalize(w, c, P.repetition_penalty, P.presence_penalty, P.frequency_penalty);
        const uint32_t key = ~__float_as_uint(weight_of(w, m, 1.0f / P.temperature, sm.tab));
        auto entry = [&](int i) { return ((u64)(uint32_t)__builtin_amdgcn_readlane((int)key, i) << 32) | (u64)places[i]; };
        u64 med;
        uint32_t from;
        median_of_three<u64>(entry(0), entry(1), entry(2), places[0], places[1], places[2], med, from);
        if (lane_id() == 0) {
            sm.bs.u64[0] = med;
            sm.bs.u64[1] = entry(3);
            sm.aux = from;
        }
    }
}

// A thread's four bits (of the entries from `base` on), whole blocks of 256 entries at a time.
__device__ __forceinline__ void store_nth_bits(global_ptr<uint32_t> words, uint32_t base, uint32_t four)
{
    const uint32_t word = eight_nibbles(four);
    if ((lane_id() & 7) == 0)
        words[base >> 5] = word;
}

// Piece `piece` of row `row`; of a row of another kind nothing.  (ALIGNED: as load_raw() has it.  STEPS: there may
// be rows for nth_steps.h, whose bits take registers that the others can do without.)
template <bool ALIGNED, int KH, bool STEPS>
__device__ __forceinline__ void index_weights_piece(const mako_sample_desc& d_arg, const Scratch& sc_val, uint32_t slices, uint32_t row, uint32_t piece,
                                                    unsigned long long* s_dyn64, FinishShared& sm, ArgsLds& s_args)
{
    const uint32_t tid = threadIdx.x;
    const mako_sampling_params P0 = d_arg.params[row];
    if (classify(P0) != kGeneral) // uniform
        return;
    // (a row that is cut to a top-k without a top-p, or to a top-k beyond the candidate lists, is still finished by one
    // workgroup on the whole-row path, in index_tail_kernel's launch; its weights, a third of that path's time, are left
    // here where general_row_from_weights() expects them)
    const bool in_order = index_order_row(P0);
    stage_args_only(d_arg, sc_val, s_args);
    stage_params(P0, s_args);
    if (tid < 32)
        sm.tab[tid] = k_exp2_tab[tid];
    __syncthreads();
    const mako_sample_desc& d = s_args.d;
    const Scratch& sc = s_args.sc;
    const mako_sampling_params& P = s_args.P;
    if (d.force_token || d.close_token) { // a forced row needs no weights: it is not claimed, and the launch that
                                          // finishes the late rows writes its token
        int32_t ftok;
        uint32_t above;
        if (row_forced(d, sc, row, slices, ftok, above) != MAKO_FORCED_NONE)
            return;
    }
    float m;
    uint32_t argidx, n_cands, any_overflow;
    row_summary(sc, row, slices, m, argidx, n_cands, any_overflow);
    const uint32_t hl = d.hist_tokens ? min(as_global(d.hist_len)[row], (uint32_t)d.hist_stride) : 0u;
    const bool pen = d.hist_tokens && !penalties_neutral(P);
    const uint32_t lo = piece * kSliceMax, hi = min(d.n_vocab, lo + kSliceMax);
    float wv[16];
    // (a row for nth_steps.h: the first round's pivot if every logit should turn out to be a candidate)
    const bool steps = STEPS && !in_order && nth_steps_for(d.n_vocab); // uniform
    load_penalised<ALIGNED, KH>(d, row, lo, hi, kSliceMax, P, pen, hl, pen, reinterpret_cast<uint32_t*>(s_dyn64), wv, [&]() {
        if (steps)
            first_pivot(d, row, P, pen ? hl : 0u, m, sm);
    });
    const float inv_t = 1.0f / P.temperature;
    // (a weight of zero is below either)
    const float floor_p = (1.0f < P.min_p) ? 1.0f : P.min_p, floor_q = floor_p < 0x1p-149f ? 0x1p-149f : floor_p;
    NthFirst first = {0u, 0u, 0u, 0u}; // (in scalar registers)
    if (steps) {
        lds_barrier();
        first = NthFirst{uniform_u32((uint32_t)(sm.bs.u64[0] >> 32)), uniform_u32((uint32_t)sm.bs.u64[0]), uniform_u32(sm.aux),
                         uniform_u32((uint32_t)(sm.bs.u64[1] >> 32))};
    }
    // (~bits(q), at the token's own position)
    // (stores known to go to device memory: one that could go to LDS as well is waited for with the table's next read)
    const global_ptr<uint32_t> key0 = as_global(sc.key[0]) + (size_t)row * sc.vpad;
    MAKO_CHECK(sc, kCheckStage, (uint64_t)hi <= sc.vpad);
    // (a wide row: its weights counted by value)
    const bool wide = STEPS && wide_row(P0) && nth_picks_for(d.n_vocab); // uniform
    uint32_t* const bins = reinterpret_cast<uint32_t*>(s_dyn64) + 1024u; // [kNthBins], behind the sums below
    if (wide) {
        lds_barrier(); // (the penalty table is done with)
        if (tid < kNthBins)
            bins[tid] = 0u;
        lds_barrier();
    }
    uint32_t is_cand = 0; // bit j: the thread's logit j is a candidate
    double bsum[4];
#pragma unroll
    for (uint32_t b = 0; b < 4; ++b) {
        bsum[b] = 0.0;
        // (the thread's logits 4b .. 4b+3 lie in the piece's b-th 4 096, four in a row)
        const uint32_t base = elem_index(lo, tid, 4u * b);
        if (lo + b * kIndexBlock < hi) { // uniform
            uint32_t k[4];
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) {
                // (what lies past the row's end is NaN, of which the weight is zero)
                const float q = weight_of(wv[4u * b + c], m, inv_t, sm.tab);
                const bool ok = q >= floor_q; // src/gen/sampler.cpp:34-35
                k[c] = ok ? __float_as_uint(q) : 0u;
                is_cand |= (ok ? 1u : 0u) << (4u * b + c);
                bsum[b] += (double)__uint_as_float(k[c]);
                if (wide && ok)
                    atomicAdd(&bins[nth_bin(k[c])], 1u);
            }
            if (base + 3u < hi) {
                *(global_ptr<u32x4>)(key0 + base) = u32x4{~k[0], ~k[1], ~k[2], ~k[3]};
            } else {
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c)
                    if (elem_index(lo, tid, 4u * b + c) < hi)
                        key0[elem_index(lo, tid, 4u * b + c)] = ~k[c];
            }
            if (steps) { // uniform
                // who is a candidate, and who belongs left of the pivot: bits for nth_steps.h's first step
                uint32_t is = 0, left = 0;
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c) {
                    const uint32_t at = elem_index(lo, tid, 4u * b + c);
                    // (where the pivot was, the first entry is now, token 0)
                    const bool moved = at == first.from;
                    const uint32_t key = moved ? first.first_key : ~k[c];
                    const bool lighter = key < first.pivot_key || (key == first.pivot_key && (moved || at < first.pivot_id));
                    is |= (k[c] ? 1u : 0u) << c;
                    left |= (at != 0u && at < hi && lighter ? 1u : 0u) << c;
                }
                store_nth_bits(as_global(nth_bits(sc, row, 2u)), base, is);
                store_nth_bits(as_global(nth_bits(sc, row, 0u)), base, left);
            } else if (!in_order) { // uniform
                // the token ids as well: with them this is the whole-row path's list of candidates when every logit turns out
                // to be one, as the pieces' counts will tell
                const global_ptr<uint32_t> li = as_global(sc.idx[0]) + (size_t)row * sc.vpad;
                if (base + 3u < hi) {
                    *(global_ptr<u32x4>)(li + base) = u32x4{base, base + 1u, base + 2u, base + 3u};
                } else {
#pragma unroll
                    for (uint32_t c = 0; c < 4; ++c)
                        if (elem_index(lo, tid, 4u * b + c) < hi)
                            li[elem_index(lo, tid, 4u * b + c)] = elem_index(lo, tid, 4u * b + c);
                }
            }
        }
        // (four weights at a time: with all sixteen in flight the kernel needs twice the registers, and two workgroups
        // no longer share a CU)
        __builtin_amdgcn_sched_barrier(0);
    }
    // the piece's fp64 sum (an estimate for the binades only: any order of addition will do), its candidates and its
    // last one
    double* wsum = reinterpret_cast<double*>(s_dyn64); // [4][kWaves] (the penalty table is done with)
    uint32_t* wcnt = reinterpret_cast<uint32_t*>(wsum + 4 * kWaves);
    __syncthreads();
#pragma unroll
    for (uint32_t b = 0; b < 4; ++b) {
        const double s = __ockl_wfred_add_f64(bsum[b]);
        if (lane_id() == 0)
            wsum[b * kWaves + wave_id()] = s;
    }
    uint32_t cnt = __ockl_wfred_add_u32((uint32_t)__popc(is_cand));
    uint32_t last = __ockl_wfred_max_u32(is_cand ? elem_index(lo, tid, 31u - (uint32_t)__clz((int)is_cand)) + 1u : 0u);
    if (lane_id() == 0) {
        wcnt[wave_id()] = cnt;
        wcnt[kWaves + wave_id()] = last;
    }
    __syncthreads();
    if (wide && tid < kNthBins)
        nth_hist(sc, row, piece)[tid] = bins[tid];
    if (in_order) { // uniform
        // few candidates: their token ids in order (in the piece's part of idx[1]; few_candidates_row())
        const uint32_t all = __ockl_wfred_add_u32((uint32_t)lane_id() < (uint32_t)kWaves ? wcnt[min((uint32_t)lane_id(), (uint32_t)kWaves - 1u)] : 0u);
        if (all <= kIndexFewMax) { // uniform
            uint32_t* const in_front = wcnt + 2 * kWaves; // [4][kWaves] of the piece's b-th 4 096, by wave
            uint32_t mine[2], upto[2]; // (two counts a word)
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                mine[h] = (uint32_t)__popc((is_cand >> (8u * h)) & 15u) | ((uint32_t)__popc((is_cand >> (8u * h + 4u)) & 15u) << 16);
                upto[h] = __ockl_wfscan_add_u32(mine[h], true);
                if (lane_id() == kWave - 1) {
                    in_front[2u * h * kWaves + wave_id()] = upto[h] & 0xffffu;
                    in_front[(2u * h + 1u) * kWaves + wave_id()] = upto[h] >> 16;
                }
            }
            lds_barrier();
            static_assert(4 * kWaves == kWave, "a count per lane");
            const uint32_t n = in_front[lane_id()], before = __ockl_wfscan_add_u32(n, true) - n;
            uint32_t* ids = sc.idx[1] + (size_t)row * sc.vpad + lo;
#pragma unroll
            for (uint32_t b = 0; b < 4; ++b) {
                uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)before, (int)uniform_u32(b * (uint32_t)kWaves + wave_id())) +
                              (((upto[b / 2u] - mine[b / 2u]) >> (16u * (b & 1u))) & 0xffffu);
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c)
                    if ((is_cand >> (4u * b + c)) & 1u) {
                        MAKO_CHECK(sc, kCheckCompact, at < all && (uint64_t)lo + at < sc.vpad);
                        ids[at++] = elem_index(lo, tid, 4u * b + c);
                    }
            }
        }
    }
    if (tid < 4u && lo + tid * kIndexBlock < hi) { // (a sum per 4 096 entries: index_groups_kernel's workgroups may be that small)
        double s = 0.0;
        for (int w = 0; w < kWaves; ++w)
            s += wsum[tid * kWaves + w];
        sc.part_sum[(size_t)row * kMaxSlices + piece * 4u + tid] = s;
    }
    if (tid == 0) {
        cnt = last = 0;
        for (int w = 0; w < kWaves; ++w) {
            cnt += wcnt[w];
            last = max(last, wcnt[kWaves + w]);
        }
    }
    if (tid == 0) {
        BigPlan* plan = sc.plan + row;
        plan->cursor[piece] = cnt; // (the pieces' counts and last candidates travel in the plan's per-worker words)
        plan->key_lo[piece] = last;
        if (piece == 0) {
            if (STEPS) {
                plan->cap[kNthCursor] = plan->cap[kNthMet] = plan->cap[kNthMade] = 0u;
                *nth_first(plan) = first;
            }
            plan->flag = kIndexClaimed;
            plan->m = m;
            plan->argidx = argidx;
            plan->n0 = 0u;
        }
    }
}

// Workgroup p of a row leaves the records of the groups of its 4096 GPW entries, or none if few_candidates_row() does without.  Wave w
// takes the groups w, w + 16, ... (GPW of them): their entries in one trip to memory, their fp64 sums to LDS, and once
// every wave has the sums before each group, the increments from the entries it still holds.  (GPW = 4 where there are rows
// enough to fill the chip, 1 on a small batch, which waits for one workgroup's chain of dependent steps.)
template <uint32_t GPW>
__device__ __forceinline__ void index_groups_block(const mako_sample_desc& d_arg, const Scratch& sc_val, uint32_t row, uint32_t p, double* s_gs)
{
    constexpr uint32_t kSpan = kIndexBlock * GPW; // entries per workgroup
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    const mako_sampling_params P0 = d_arg.params[row];
    if (!index_order_row(P0)) // uniform
        return;
    BigPlan* plan = sc_val.plan + row;
    // (zero: index_weights_kernel left the row alone, its token is forced; a workgroup that starts late may already see
    // what this kernel's first workgroup has made of the flag)
    if (plan->flag == 0u) // uniform
        return;
    const uint32_t pieces = (d_arg.n_vocab + kSliceMax - 1u) / kSliceMax, blocks = (d_arg.n_vocab + kIndexBlock - 1u) / kIndexBlock;
    const uint32_t cnt_l = lane < pieces ? plan->cursor[min(lane, kWorkers - 1u)] : 0u;
    const uint32_t last_l = lane < pieces ? plan->key_lo[min(lane, kWorkers - 1u)] : 0u;
    const double ps = lane < blocks ? sc_val.part_sum[(size_t)row * kMaxSlices + lane] : 0.0;
    const float u_row = d_arg.u[row];
    const uint32_t n_cand = __ockl_wfred_add_u32(cnt_l), n_list = __ockl_wfred_max_u32(last_l);
    const double incl = __ockl_wfscan_add_f64(ps, true);
    const double total64 = readlane_f64(incl, kWave - 1), mass = readlane_f64(incl - ps, p * GPW);
    if (p == 0 && tid == 0) {
        plan->n0 = n_list;
        plan->groups = (n_list + kGroup - 1u) / kGroup;
        plan->total64 = total64;
        plan->thr = n_cand;
        const bool gaps_matter = n_cand < n_list && d_arg.out_cand_idx && d_arg.out_cand_q && d_arg.cand_cap;
        plan->flag = n_cand == 0u ? kIndexEmpty : (gaps_matter ? kIndexWhole : (n_cand <= kIndexFewMax ? kIndexFew : kIndexReady));
    }
    if (n_cand <= kIndexFewMax || p * kSpan >= n_list) // uniform
        return;
    const uint32_t off = p * kSpan, cnt = min(kSpan, n_list - off);
    const uint32_t groups = (cnt + kGroup - 1u) / kGroup; // <= 16 GPW <= 64
    const GlobalKeys kf{sc_val.key[0] + (size_t)row * sc_val.vpad};
    GroupRec* recs = sc_val.gt + (size_t)row * sc_val.g_cap + p * (kSpan / kGroup);
    MAKO_CHECK(sc_val, kCheckGroups, p * (kSpan / kGroup) + groups <= sc_val.g_cap && (uint64_t)off + cnt <= sc_val.vpad);
    float q[GPW][4];
    uint32_t len[GPW];
#pragma unroll
    for (uint32_t k = 0; k < GPW; ++k) {
        const uint32_t g = wave + k * (uint32_t)kWaves;
        len[k] = g < groups ? min(kGroup, cnt - g * kGroup) : 0u; // uniform per wave
        load_span(kf, off + min(g, groups - 1u) * kGroup, len[k], q[k]);
    }
    if (GPW < 4u && tid < (uint32_t)kWave)
        s_gs[tid] = 0.0;
    if (GPW < 4u)
        __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < GPW; ++k) {
        const double s = __ockl_wfred_add_f64((((double)q[k][0] + (double)q[k][1]) + (double)q[k][2]) + (double)q[k][3]);
        if (lane == 0)
            s_gs[wave + k * (uint32_t)kWaves] = len[k] ? s : 0.0;
    }
    __syncthreads();
    // the sums before and behind each group: lane g holds group g's
    const double v = s_gs[lane];
    const double upto = __ockl_wfscan_add_f64(v, true);
    const double before_l = mass + (upto - v);
    const double r0_raw = (double)u_row * total64, r0 = r0_raw == r0_raw ? r0_raw : 0.0;
#pragma unroll
    for (uint32_t k = 0; k < GPW; ++k) {
        const uint32_t g = uniform_u32(wave + k * (uint32_t)kWaves);
        if (g >= groups) // uniform per wave
            break;
        const double sum = s_gs[g], before = readlane_f64(before_l, g);
        group_record(q[k], off + g * kGroup, len[k], sum, before, before + sum, r0, recs + g);
    }
}

// A row with few candidates (a min-p leaves a peaked row a few dozen): the pieces' lists one after the other are
// the row's, in token order, which one wave adds up and walks.  All threads call.
// In line in the kernel, or at most one call away, and the tail for short lists in line here: where the tail was a called function,
// and this another, sixteen waves stored and fetched their registers at each entry for what one wave does, and from 128 rows on that
// took longer than the records.  (Peaked rows with a min-p of 0.02 to 0.1, over the group records, with the calls, and so: one of
// 129 280 31.7 us, 26.2 and 22.1, 64 of them 66, 44 and 37, 512 rows of 700 40.6, 61.0 and 28.4; without the caller's copy of the
// parameters 24 rows of 151 553 71, 48 and 41, 512 of 700 119, 147 and 111.)
__device__ __forceinline__ void few_candidates_row(const mako_sample_desc& d, const Scratch& sc, uint32_t row, const mako_sampling_params& P, const FinishLds& L)
{
    assume_lds(L);
    const uint32_t tid = threadIdx.x, lane = lane_id(), pieces = (d.n_vocab + kSliceMax - 1u) / kSliceMax;
    const uint32_t upto = __ockl_wfscan_add_u32(lane < pieces ? sc.plan[row].cursor[min(lane, kWorkers - 1u)] : 0u, true);
    const uint32_t n_cand = min((uint32_t)__builtin_amdgcn_readlane((int)upto, kWave - 1), kIndexFewMax);
    uint32_t piece = 0, before = 0;
    for (uint32_t k = 0; k < pieces; ++k) { // uniform
        const uint32_t to = (uint32_t)__builtin_amdgcn_readlane((int)upto, (int)k);
        if (tid >= to) {
            piece = k + 1u;
            before = to;
        }
    }
    const size_t at = (size_t)row * sc.vpad;
    uint32_t* kf = sc.key[1] + at;
    uint32_t* jf = sc.idx[0] + at;
    if (tid < n_cand) {
        const uint32_t id = min(sc.idx[1][at + min(piece, pieces - 1u) * kSliceMax + (tid - before)], d.n_vocab - 1u);
        kf[tid] = sc.key[0][at + id];
        jf[tid] = id;
    }
    __syncthreads();
    [[clang::always_inline]] sorted_tail<false, true>(d, row, P, kf, jf, n_cand, true, sc.plan[row].total64, MAKO_PATH_INDEXED, L);
}

// What these kernels have left of a row of theirs (flag: of its plan, which is zero again behind this), by one workgroup: the
// rest of the whole-row path, or the total and the draw.  All threads call; sm.tab must hold the exp2 table.  ALL_KINDS: rows
// that are not in token order are among them.  (Without their code, and with it, as much scratch memory either way.  With a min-p: one
// row of 129 280 21.8 us and 22.2, 64 of them 37.2 and 37.6, 512 rows of 700 28.4 and 29.0; temperature only, one row 39.1 and 39.6,
// 64 76.2 and 76.5.)
// Returns whether the row is one for few_candidates_row(), which the caller calls (from here it would be deeper in the stack).
template <bool ALL_KINDS = true>
__device__ __forceinline__ bool finish_index_row_here(const mako_sample_desc& d, const Scratch& sc, const mako_sampling_params& P, uint32_t row,
                                                      const FinishLds& L)
{
    const uint32_t tid = threadIdx.x;
    BigPlan* plan = sc.plan + row;
    const uint32_t flag = plan->flag, n0 = min(plan->n0, d.n_vocab), n_cand = plan->thr;
    const uint32_t groups = min(plan->groups, min(kMaxGroups, sc.g_cap));
    const double total64 = plan->total64;
    const float m = plan->m;
    const uint32_t argidx = plan->argidx;
    // (the pieces' counts of candidates: when every logit is one, index_weights_kernel's list is the row's list)
    const uint32_t pieces = (d.n_vocab + kSliceMax - 1u) / kSliceMax;
    const uint32_t counted = __ockl_wfred_add_u32((uint32_t)lane_id() < pieces ? plan->cursor[min((uint32_t)lane_id(), kWorkers - 1u)] : 0u);
    __syncthreads(); // (the plan has been read)
    if (tid == 0)
        plan->flag = 0;
    if (!index_order_row(P)) {
        // the whole-row path from the weights index_weights_kernel left (the group records' kernel has not touched the row)
        if constexpr (ALL_KINDS)
            if (flag == kIndexClaimed && !general_row_from_weights<0>(d, sc, row, P, m, argidx, uniform_u32(counted), L)) { // uniform
                __syncthreads();
                general_row<0>(d, sc, row, P, m, argidx, L);
            }
        return false;
    }
    if (flag == kIndexEmpty) {
        fallback_row(d, row, argidx);
        return false;
    }
    if (flag == kIndexFew)
        return true;
    if (flag == kIndexReady) {
        const uint32_t* kf = sc.key[0] + (size_t)row * sc.vpad;
        // (entry i of the list is token i: no array of token ids)
        const bool done = sorted_tail<true, false, false, false, true>(d, row, P, kf, nullptr, n0, true, total64, MAKO_PATH_INDEXED, L, false, 0.0f,
                                                                       sc.gt + (size_t)row * sc.g_cap, groups);
        if (done) {
            // (the list's length counts the gaps; the candidates are what the reference counts)
            if (tid == 0 && d.out_n_cand)
                d.out_n_cand[row] = n_cand;
            return false;
        }
    }
    if (flag == kIndexReady || flag == kIndexWhole)
        general_row<0>(d, sc, row, P, m, argidx, L);
    return false;
}
// (those of few_candidates_row() apart)
__device__ MAKO_RARE_CALL void finish_index_row(const mako_sample_desc& d, const Scratch& sc, const mako_sampling_params& P, uint32_t row,
                                                const FinishLds& L)
{
    assume_lds(L);
    (void)finish_index_row_here(d, sc, P, row, L);
}

// Rows of the kind that `want` says (kGeneral, or those of them that are in token order) by their rank among them, for ranks that
// never fall: the search goes on from the 64 rows it was in.  (From the first row for every piece, a batch of 30 000 rows of
// 400 logits, half of them such rows, took 27.0 ms; 9.4 so, and 14.0 with one workgroup a row.)  The same for the whole workgroup.
struct RankedRows {
    uint32_t base = 0, before = 0; // a multiple of 64 rows, and the rows of the kind in front of it

    template <typename Want>
    __device__ __forceinline__ bool find(const mako_sample_desc& d, uint32_t rank, Want want, uint32_t& row)
    {
        for (; base < d.n_rows; base += (uint32_t)kWave) {
            const uint32_t r = base + (uint32_t)lane_id();
            const bool is = r < d.n_rows && want(d.params[min(r, d.n_rows - 1u)]);
            const unsigned long long all = __builtin_amdgcn_ballot_w64(is);
            const uint32_t n = (uint32_t)__popcll(all);
            if (rank - before < n) {
                const unsigned long long hit = __builtin_amdgcn_ballot_w64(is && mask_rank(all) == rank - before);
                row = base + (uint32_t)__ffsll((long long)hit) - 1u;
                return true;
            }
            before += n;
        }
        return false;
    }
};

#ifdef MAKO_EMIT_INDEX_KERNELS
// grid = (rows rounded up to a multiple of eight, ceil(V / 16384)): workgroups go to the eight XCDs in turn, so that all of
// these kernels work on a row on the same one.
template <bool ALIGNED, int KH, bool STEPS>
__global__ __launch_bounds__(kThreads) void index_weights_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[];
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    if (blockIdx.x < d_arg.n_rows)
        index_weights_piece<ALIGNED, KH, STEPS>(d_arg, sc_val, slices, blockIdx.x, blockIdx.y, s_dyn64, sm, s_args);
}

// grid = (rows rounded up to a multiple of eight, ceil(V / (4096 GPW))).
template <uint32_t GPW>
__global__ __launch_bounds__(kThreads) void index_groups_kernel(mako_sample_desc d_arg, Scratch sc_val)
{
    __shared__ double s_gs[kWave];
    if (blockIdx.x < d_arg.n_rows)
        index_groups_block<GPW>(d_arg, sc_val, blockIdx.x, blockIdx.y, s_gs);
}

// grid = (rows rounded up to a multiple of eight, workgroups per row): a step of nth_steps.h.
// (Two workgroups share a CU only with 80 scalar registers each, all in all: with 82 the second half of the first step's 512
// started 16 us after the first.)
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_num_sgpr(80))) void nth_step_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t step)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[];
    __shared__ BlockScratch s_bs;
    if (blockIdx.x < d_arg.n_rows) {
        const NthMadeOf made = nth_step(d_arg, sc_val, blockIdx.x, blockIdx.y, gridDim.y, step, s_dyn64, s_bs);
        if (made != kNthNone && blockIdx.y == 0u && threadIdx.x == 0u)
            sc_val.plan[blockIdx.x].cap[kNthMade] = step;
    }
}

// grid = (1, rows).
template <bool ALL_KINDS>
__global__ __launch_bounds__(kThreads) void index_tail_kernel(mako_sample_desc d_arg, Scratch sc_val)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[];
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    const uint32_t row = blockIdx.y;
    if (classify(d_arg.params[row]) != kGeneral || sc_val.plan[row].flag == 0u) // uniform (none: its token is forced)
        return;
    MAKO_ROW(row);
    if (threadIdx.x < 32)
        sm.tab[threadIdx.x] = k_exp2_tab[threadIdx.x];
    stage_args(d_arg, sc_val, row, s_args);
    const FinishLds views = finish_lds_views(sm, s_dyn64);
    if (finish_index_row_here<ALL_KINDS>(s_args.d, s_args.sc, s_args.P, row, views)) // uniform
        few_candidates_row(s_args.d, s_args.sc, row, s_args.P, views);
}
#endif // MAKO_EMIT_INDEX_KERNELS

} // namespace mako
