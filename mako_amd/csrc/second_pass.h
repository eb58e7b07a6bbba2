// finish_kernel: the second pass over the top_k == 0 rows.
#pragma once

#include "slice_load.h"
#include "work_split.h"
#include "row_records.h"
#include "coarse_plan.h"

namespace mako {

// A workgroup's share of a top_k == 0 row's pieces, one after the other.  Of each piece: the exact fp64 sum of q over
// it, and every weight the row's plan keeps handed to the share of the worker that will sort it.
// The summation order is fixed: each thread adds its logits in index order, then lanes, then waves.
// The plan (coarse_plan()) is built while the first piece's logits are on their way; every workgroup of the row
// arrives at the same one, and the one with the row's first piece stores it for the kernels that follow and enters
// the row in their lists.
// The large batches' instance, whose workgroups go through several pieces, asks for a piece's logits ahead of the hand-over of
// the piece before it (AHEAD; where their registers are to be had: not with eight history entries a thread, and not beside
// other rows).
// `loads`: the piece's own where they have been asked for ahead, then those of piece `next` (kNone: there is none).
// (PEN: the row has penalties to apply; a compile-time fact so that each case gets straight-line code of its own.)
// (`slices`: of scan_kernel, whose records give the row maximum)
// (PLANNING: the workgroup's first piece, with which the plan is built; returns false when the row leaves for the
// whole-row path and the pass has nothing more to do for it)
template <bool ALIGNED, int KH, bool PEN, bool PLANNING, bool UNSORTED, bool AHEAD, uint32_t SORT_WAVES>
__device__ bool one_piece(const mako_sample_desc& d, const Scratch& sc, uint32_t row, uint32_t slice, uint32_t slice_len,
                          const mako_sampling_params& P, uint32_t hl, uint32_t slices, const FinishLds& L, CoarsePlan& pl,
                          float& m, uint32_t& argidx, uint32_t opaque_first, SliceLoads<KH>& loads, uint32_t next)
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    constexpr bool pen = PEN;
    BigPlan* plan = sc.plan + row;
    const uint32_t lo = slice * slice_len;
    const uint32_t hi = min(d.n_vocab, lo + slice_len);
    float wv[16];
    MAKO_STAMP(28);
    if constexpr (PLANNING) {
        PlanLoads pre;
        issue_plan_loads<UNSORTED>(d, sc, row, slices, pre);
        issue_slice<ALIGNED, KH>(d, row, lo, hi, loads);
        clear_counts<KH>(d, pen, slice_len, L.cnt);
        {
            uint32_t n_cands, any_overflow;
            row_summary_of(pre.st, slices, m, argidx, n_cands, any_overflow);
            // (a short row's only list has all that is in front of what it left out: no use for it where it is shorter than the
            // nucleus.  200 rows of 3 001 logits 52 us, 87 with a second look at those; longer rows gain nothing, four of 16 000 32.6
            // us and 34.0)
            const uint32_t narrow_max = any_overflow || n_cands > kSortMax ? 0u : (short_slice(d.n_vocab) ? min(n_cands, kSmall) : kSmall);
            coarse_plan(sc, row, slices, d.n_vocab, P, m, pre, narrow_max, UNSORTED ? opaque_first : kNone, UNSORTED ? kShareLarge : kShareSmall, pl, sm.tab);
        }
    } else {
        if (!AHEAD)
            issue_slice<ALIGNED, KH>(d, row, lo, hi, loads);
        clear_counts<KH>(d, pen, slice_len, L.cnt);
    }
    finish_penalised<ALIGNED, KH>(d, row, lo, hi, slice_len, P, hl, pen, L.cnt, loads, wv);
    MAKO_STAMP(1);
    MAKO_STAMP(24);
    const uint32_t flag = pl.flag;
    if (PLANNING && slice == 0) {
        // the row's first piece stores the plan and enters the row in the lists of sort_kernel and tail_kernel
        // (stores and counters known to be in device memory: a store that could be to LDS as well is waited for with the next
        // read of LDS, and this workgroup has the most to do of the row's: one nucleus row 14.4 -> 14.0 us)
        const global_ptr<BigPlan> plan = as_global(sc.plan + row);
        const global_ptr<uint32_t> work_n = as_global(sc.work_n), work_sort = as_global(sc.work_sort);
        auto take = [](global_ptr<uint32_t> n, uint32_t by) { return __hip_atomic_fetch_add(n, by, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
        if (tid < kWorkers) {
            plan->key_lo[tid] = pl.key_lo[tid];
            plan->stage_off[tid] = pl.stage_off[tid];
            plan->cap[tid] = pl.cap[tid];
            plan->mass[tid] = pl.mass_above[tid];
        }
        if (tid == 0) {
            plan->thr = pl.thr;
            plan->argidx = argidx;
            plan->m = m;
            plan->mass_all = pl.mass_all;
            plan->flag = flag;
            const uint32_t unsorted = (UNSORTED && flag == 1) ? pl.opq_mask : 0u;
            plan->opq_mask = unsorted;
            if (flag == 1 || flag == 3) {
                // sort_kernel's work: a workgroup per worker that sorts, and collectors whose waves take the row's unsorted
                // shares, a share at a time (work items kWorkers + c)
                const uint32_t n_unsorted = (uint32_t)__popc(unsorted);
                const uint32_t each = shares_collected(SORT_WAVES, pl.nucleus_rows), collectors = (n_unsorted + each - 1u) / each;
                if constexpr (UNSORTED) {
                    // (two lists, the costly entries in front: large_batch_lists())
                    const SortLists lists = large_batch_lists(pl.nucleus_rows);
                    if (flag == 3) {
                        work_sort[lists.sorted_at + take(work_n + 0, 1u)] = row << 8;
                    } else {
                        const uint32_t in_front = min(collectors, kCollectorsInFront);
                        uint32_t at = lists.sorted_at - take(work_n + 3, in_front) - in_front;
                        for (uint32_t c = 0; c < in_front; ++c)
                            work_sort[at++] = (row << 8) | (kWorkers + c);
                        at = lists.sorted_at + take(work_n + 0, pl.workers - n_unsorted + collectors - in_front);
                        for (uint32_t c = in_front; c < collectors; ++c)
                            work_sort[at++] = (row << 8) | (kWorkers + c);
                        for (uint32_t w = 0; w < pl.workers; ++w)
                            if (!((unsorted >> w) & 1u))
                                work_sort[at++] = (row << 8) | w;
                    }
                } else {
                    const uint32_t work = flag == 1 ? pl.workers : 1u;
                    uint32_t at = take(work_n + 0, work);
                    for (uint32_t w = 0; w < work; ++w)
                        work_sort[at++] = (row << 8) | w;
                }
                if (flag == 1)
                    as_global(sc.work_tail)[take(work_n + 1, 1u)] = row;
            }
        }
    }
    if (flag == 2) // the whole-row path starts from the logits again
        return false;
    const float inv_t = 1.0f / P.temperature;
    // (a weight of zero is below either)
    const float floor_p = (1.0f < P.min_p) ? 1.0f : P.min_p, floor_q = floor_p < 0x1p-149f ? 0x1p-149f : floor_p;
    const uint32_t thr = max(pl.thr, 1u);
    const uint32_t edge7 = uniform_u32(pl.key_lo[7]), edge15 = uniform_u32(pl.key_lo[15]), edge23 = uniform_u32(pl.key_lo[23]);
    double sum = 0;
    uint32_t qb[16];   // bits(q), 0 where q is not a candidate
    uint32_t slot[16]; // kept weights: worker << 16 | position among this workgroup's entries for that worker
    // (a piece may be shorter than the sixteen logits per thread: whole blocks past its end are skipped; the test is
    // the same for every thread)
#pragma unroll
    for (uint32_t g = 0; g < 16u; g += 4u) {
#pragma unroll
        for (uint32_t j = g; j < g + 4u; ++j) {
            qb[j] = 0u;
            slot[j] = kNone;
        }
        if (lo + (g / 4u) * kBlock < hi) {
            // (the large batches' instance: a wave whose four weights a lane all underflow to zero, as those of a peaked row far
            // below its maximum do, skips the arithmetic that would tell it so; exp_moved() returns 0 below that bound)
            bool any = !UNSORTED;
            if (UNSORTED) {
                bool under = true;
#pragma unroll
                for (uint32_t j = g; j < g + 4u; ++j)
                    under = under & ((wv[j] - m) * inv_t < -0x1.9fe368p6f);
                any = __ballot(!under) != 0ull; // uniform
            }
            if (any) {
                float q[4];
                bool keeps[4];
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    q[j] = weight_of(wv[g + j], m, inv_t, sm.tab);
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    qb[g + j] = q[j] >= floor_q ? __float_as_uint(q[j]) : 0u;
                    sum += (double)__uint_as_float(qb[g + j]);
                    keeps[j] = qb[g + j] >= thr;
                }
                // the worker whose range of bits(q) holds the weight (equal weights always meet in one share): the number of
                // workers whose lower edge lies above it, by bisection over the edges (the first two steps against edges held
                // in scalar registers, the other three from LDS), and a place among the workgroup's entries for it.
                // (Four logits side by side: one after the other, each with its own branch, they wait for three reads and an
                // atomic's answer every time.  The worker's number is kept as an offset into its words in LDS.  A flat row's
                // piece of 16 384, weights and all: 7.1 -> 6.0 us.)
                if (__ballot(keeps[0] | keeps[1] | keeps[2] | keeps[3]) != 0ull) { // uniform
                    static_assert(kWorkers == 32, "five steps");
                    const lds_ptr<const char> edges = (lds_ptr<const char>)as_lds(pl.key_lo), counts = (lds_ptr<const char>)as_lds(pl.count);
                    uint32_t w[4], place[4];
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        w[j] = qb[g + j] < edge15 ? 64u : 0u;
                        w[j] |= qb[g + j] < (qb[g + j] < edge15 ? edge23 : edge7) ? 32u : 0u;
                        place[j] = 0u;
                    }
#pragma unroll
                    for (uint32_t step = 4u; step; step >>= 1)
#pragma unroll
                        for (uint32_t j = 0; j < 4; ++j)
                            w[j] += qb[g + j] < *(lds_ptr<const uint32_t>)(edges + w[j] + 4u * (step - 1u)) ? 4u * step : 0u;
                    __builtin_amdgcn_sched_barrier(0); // (the four counters are asked for one behind the other)
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)
                        if (keeps[j])
                            place[j] = __hip_atomic_fetch_add((lds_ptr<uint32_t>)(counts + w[j]), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)
                        slot[g + j] = keeps[j] ? (w[j] << 14) | place[j] : kNone;
                }
            }
        }
    }
    MAKO_STAMP(25);
    if (AHEAD)
        __builtin_amdgcn_sched_barrier(0); // (not among the weights, whose registers these take)
    if (AHEAD && next != kNone) // uniform
        issue_slice<ALIGNED, KH>(d, row, next * slice_len, min(d.n_vocab, next * slice_len + slice_len), loads);
    // the piece's sum: wave reductions, then the waves' results in order
    {
        const double sw = __ockl_wfred_add_f64(sum);
        if (lane_id() == 0)
            sm.bs.f64[wave_id()] = sw;
    }
    lds_barrier();
    MAKO_STAMP(26);
    // One run per worker in its share of the row's staging arrays, reserved with a single atomic.  The kept weights
    // are first put in LDS (the penalty table's block, free by now) in the order of their workers, each worker's from a
    // multiple of four on, so that the runs go out as contiguous stores, four entries at a time.
    // (the reservations' answers take a trip to device memory: the entries are put in LDS order under it)
    uint32_t mine = 0, lbase_mine = 0, base_mine = 0;
    if (wave_id() == 0) {
        mine = tid < kWorkers ? pl.count[tid] : 0u;
        const uint32_t padded = (mine + 3u) & ~3u, upto = __ockl_wfscan_add_u32(padded, true);
        lbase_mine = upto - padded;
        if (tid < kWorkers) {
            pl.lbase[tid] = lbase_mine;
            if (mine)
                base_mine = __hip_atomic_fetch_add(as_global(&plan->cursor[tid]), mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (tid == kWorkers - 1u)
            pl.lbase[kWorkers] = upto;
    }
    lds_barrier(); // (not one that waits for the reservations)
    MAKO_STAMP(27);
    if (tid < kWorkers)
        pl.count[tid] = 0; // (for the workgroup's next piece)
    const global_ptr<uint32_t> kstage = as_global(sc.key[1]) + (size_t)row * sc.vpad;
    const global_ptr<uint32_t> istage = as_global(sc.idx[1]) + (size_t)row * sc.vpad;
    // (room for all a piece can hold: with half as much, a flat row's pieces, which keep nearly everything, went through
    // it twice, 2 us more each; a workgroup of 1 024 has its CU to itself anyway, and two of 512 have room for all they can hold)
    uint2* buf = reinterpret_cast<uint2*>(L.cnt); // [kPieceMax + 3 kWorkers] (weight, token id)
    static_assert(kFinishLds >= (kPieceMax + 3u * kWorkers) * sizeof(uint2), "");
    const uint32_t kept = pl.lbase[kWorkers];
    // (an entry's worker travels in the upper bits of its token id)
    constexpr uint32_t kIdBits = 27;
    static_assert(kMaxSlices * kSliceMax <= 1u << kIdBits && kWorkers <= 1u << (32u - kIdBits) && kSliceMax <= 0x10000u,
                  "a token id and a worker in a word; an entry's place fits sixteen bits beside its worker");
    // (from here on: worker << 16 | the entry's place in the workgroup's order.  The runs' starts are read for all
    // sixteen at once, kept or not: behind sixteen branches each read would be a wait of its own.)
    {
        uint32_t start[16];
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j)
            start[j] = pl.lbase[(slot[j] >> 16) & (kWorkers - 1u)];
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j)
            if (slot[j] != kNone)
                slot[j] = (slot[j] & 0xffff0000u) | (start[j] + (slot[j] & 0xffffu));
    }
    bool dropped = false;
    const uint32_t unsorted_mask = UNSORTED ? uniform_u32(pl.opq_mask) : 0u;
    if (kept) { // uniform
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j)
            if (slot[j] != kNone)
                buf[slot[j] & 0xffffu] = make_uint2(qb[j], elem_index(lo, tid, j) | ((slot[j] >> 16) << kIdBits));
        if (tid < kWorkers) { // (wave 0: where each worker's run goes and where it, or its room, ends in the workgroup's order)
            const uint32_t room = pl.cap[tid], left = room > base_mine ? room - base_mine : 0u;
            pl.run[tid] = make_uint2(pl.stage_off[tid] + base_mine - lbase_mine, lbase_mine + min(mine, left));
            dropped = mine > left;
        }
        lds_barrier();
        typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(4)));
        const uint32_t id_mask = (1u << kIdBits) - 1u;
        // (a share that is only summed has no use for the token ids)
        auto wants_ids = [&](uint32_t w) { return !UNSORTED || !((unsorted_mask >> w) & 1u); };
        for (uint32_t e = 4u * tid; e < kept; e += 4u * kThreads) { // (uniform per wave but for the last trip)
            const uint4 x0 = *reinterpret_cast<const uint4*>(buf + e), x1 = *reinterpret_cast<const uint4*>(buf + e + 2u);
            const uint32_t w = x0.y >> kIdBits;
            const uint2 run = pl.run[w];
            if (e + 4u <= run.y) {
                MAKO_CHECK(sc, kCheckStage, (uint64_t)(run.x + e) + 3u < sc.vpad && run.x + e >= pl.stage_off[w] &&
                                                run.x + e + 4u <= pl.stage_off[w] + pl.cap[w]);
                *(global_ptr<u32x4_any>)(kstage + run.x + e) = u32x4_any{x0.x, x0.z, x1.x, x1.z};
                if (wants_ids(w))
                    *(global_ptr<u32x4_any>)(istage + run.x + e) = u32x4_any{x0.y & id_mask, x0.w & id_mask, x1.y & id_mask, x1.w & id_mask};
            }
        }
        if (tid < 4u * kWorkers) { // each run's last entries, fewer than four
            const uint32_t w = tid >> 2, first = pl.lbase[w];
            const uint2 run = pl.run[w];
            const uint32_t e = first + ((run.y - first) & ~3u) + (tid & 3u);
            if (e < run.y) {
                const uint2 x = buf[e];
                MAKO_CHECK(sc, kCheckStage, (uint64_t)(run.x + e) < sc.vpad && run.x + e >= pl.stage_off[w] && run.x + e < pl.stage_off[w] + pl.cap[w]);
                kstage[run.x + e] = x.x;
                if (wants_ids(w))
                    istage[run.x + e] = x.y & id_mask;
            }
        }
        lds_barrier();
    }
    MAKO_STAMP(29);
    if (dropped) // (more weights in a range than the counts promised: the row takes the whole-row path)
        plan->overflow = 1;
    if (tid == 0) {
        double total = 0;
        for (int w = 0; w < kWaves; ++w) // waves in order: the same inputs always give the same bits
            total += sm.bs.f64[w];
        as_global(sc.part_sum)[(size_t)row * kMaxSlices + slice] = total;
    }
    lds_barrier(); // (the waves' sums have been read before the next piece's replace them)
    MAKO_STAMP(30);
    return true;
}

template <bool ALIGNED, int KH, bool PEN, bool UNSORTED, bool AHEAD, uint32_t SORT_WAVES>
__device__ void row_pieces(const mako_sample_desc& d, const Scratch& sc, uint32_t row, uint32_t first, uint32_t stride,
                           uint32_t n_pieces, uint32_t slice_len, const mako_sampling_params& P, uint32_t hl, uint32_t slices,
                           const FinishLds& L, CoarsePlan& pl, uint32_t opaque_first)
{
    assume_lds(L);
    // the workgroup's pieces in turn: first, first + stride, ...
    float m = 0.0f;
    uint32_t argidx = 0;
    SliceLoads<KH> loads;
    auto behind = [&](uint32_t slice) { return slice + stride < n_pieces ? slice + stride : kNone; };
    if (first >= n_pieces || !one_piece<ALIGNED, KH, PEN, true, UNSORTED, AHEAD, SORT_WAVES>(d, sc, row, first, slice_len, P, hl, slices, L, pl, m, argidx, opaque_first, loads,
                                                                         behind(first)))
        return;
    for (uint32_t slice = first + stride; slice < n_pieces; slice += stride)
        one_piece<ALIGNED, KH, PEN, false, UNSORTED, AHEAD, SORT_WAVES>(d, sc, row, slice, slice_len, P, hl, slices, L, pl, m, argidx, kNone, loads, behind(slice));
}

// Second pass over the top_k == 0 rows.  grid = (most pieces a row can have, rows) workgroups, of which workgroup i
// serves the i-th share of a row's pieces in row order, SecondPassCut::per_row per top_k == 0 row (find_piece): the busy
// workgroups are then the first ones dispatched and land evenly on the XCDs, shader engines and CUs, whatever the
// mix of rows.
// (UNSORTED: the instance for batches of many such rows, whose plans leave shares unsorted: unsorted_shares.h)
// (n_wgs: workgroups of the launch that are finish_kernel's.  SORT_WAVES: waves of a workgroup of the sort that follows)
template <bool ALIGNED, int KH, bool UNSORTED, bool AHEAD, uint32_t SORT_WAVES>
__device__ __forceinline__ void finish_body(const mako_sample_desc& d_arg, const Scratch& sc_arg, uint32_t slices, uint32_t n_wgs,
                                            unsigned long long* s_dyn64, FinishShared& sm, ArgsLds& s_args, CoarsePlan& s_plan)
{
#ifdef MAKO_TIMING_FINISH
    MAKO_WG_TIMER;
#endif
    // What the workgroup needs before it can ask for its logits is asked for in as few trips to memory as possible
    // (each costs most of a microsecond here, and the pass starts with nothing else to do): the rows' parameters
    // for find_piece() and the arguments' copy go out together with the cut, and the row's own parameters are then
    // taken from the lane that loaded them.
    uint32_t wg = blockIdx.y;
    const uint32_t tid = threadIdx.x;
    const bool by_lane = d_arg.n_rows <= (uint32_t)kWave; // uniform
    mako_sampling_params P_lane = mako_sampling_params{};
    if (by_lane)
        P_lane = d_arg.params[min((uint32_t)lane_id(), d_arg.n_rows - 1u)];
    stage_args_only(d_arg, sc_arg, s_args);
    // (pieces per row, their length, workgroups with work: the others leave at once)
    const uint4 cut = *reinterpret_cast<const uint4*>(sc_arg.work_n + 4);
    const uint32_t nucleus_rows = UNSORTED ? sc_arg.work_n[10] : 0u;
    // Workgroups go to the eight XCDs in turn.  The shares are dealt so that an XCD's workgroups serve consecutive
    // ones: the workgroups of a row then sit on one XCD (two where a row straddles), whose L2 fetches the row's
    // coarse counts and history once for all of them.  (Only if the grid holds every workgroup the deal names.)
    if (cut.x < cut.w) {
        // More pieces than one round of workgroups, so a row's workgroups go through several pieces each and rows that
        // need little are done long before rows that need much (a near-flat row takes twice as long as a peaked one).
        // The rows go round-robin to the XCDs (an XCD's workgroups are dispatched in order onto whichever of its CUs
        // is free, but which XCD a workgroup goes to is fixed by its number), a row's workgroups to one XCD.
        const uint32_t rowrank = (wg & 7u) + 8u * ((wg >> 3) / cut.x);
        wg = rowrank * cut.x + (wg >> 3) % cut.x;
        if (rowrank * cut.x >= cut.z)
            return;
    } else {
        const uint32_t per_xcd = (cut.z + 7u) / 8u;
        if (per_xcd * 8u <= n_wgs) {
            if ((wg >> 3) >= per_xcd)
                return;
            wg = (wg & 7u) * per_xcd + (wg >> 3);
        }
    }
    if (wg >= cut.z)
        return;
    const uint32_t pieces = cut.x, piece_len = cut.y, n_pieces = cut.w; // (pieces: workgroups per row)
    uint32_t row, piece;
    if (by_lane) {
        // find_piece() over the parameters already here: one row per lane, every wave for itself
        const uint32_t mine = ((uint32_t)lane_id() < d_arg.n_rows && classify(P_lane) == kNucleus) ? pieces : 0u;
        const uint32_t upto = __ockl_wfscan_add_u32(mine, true);
        const unsigned long long bal = __ballot(wg >= upto - mine && wg < upto);
        if (bal == 0ull)
            return;
        const int owner = __ffsll((long long)bal) - 1;
        row = (uint32_t)owner;
        piece = wg - (uint32_t)__builtin_amdgcn_readlane((int)(upto - mine), owner);
        mako_sampling_params P_row;
        uint32_t* dst = reinterpret_cast<uint32_t*>(&P_row);
        const uint32_t* src = reinterpret_cast<const uint32_t*>(&P_lane);
#pragma unroll
        for (uint32_t i = 0; i < sizeof(mako_sampling_params) / 4; ++i)
            dst[i] = (uint32_t)__builtin_amdgcn_readlane((int)src[i], owner);
        stage_params(P_row, s_args);
    } else {
        if (!find_piece(d_arg, wg, pieces, 0u, row, piece, sm.bs))
            return;
        stage_params(d_arg.params[row], s_args);
    }
    MAKO_ROW(row);
    MAKO_WG_TAG((row << 8) | piece | 0x80000000u);
    if (tid < 32)
        sm.tab[tid] = k_exp2_tab[tid];
    __syncthreads(); // (publishes the arguments, the parameters and the table)
    const mako_sample_desc& d = s_args.d;
    const Scratch& sc = s_args.sc;
    FinishLds L;
    L.sm = &sm;
    L.cnt = reinterpret_cast<uint32_t*>(s_dyn64);
    L.sortk = s_dyn64;                                             // 32 KB
    L.wcount = reinterpret_cast<uint32_t*>(s_dyn64 + kSortMax);    // next 16 KB
    const mako_sampling_params& P = s_args.P;
    MAKO_STAMP(0);
    if (d.force_token || d.close_token) { // a forced row needs no weights (plan_kernel writes its token)
        int32_t ftok;
        uint32_t above;
        if (row_forced(d, sc, row, slices, ftok, above) != MAKO_FORCED_NONE)
            return;
    }
    // (the history's length and, inside slice_partial, the history, the logits and the slices' records: one trip)
    const uint32_t hl = d.hist_tokens ? min(as_global(d.hist_len)[row], (uint32_t)d.hist_stride) : 0u;
    // (a row without history entries takes the penalising variant too when it has penalties: it finds nothing to
    // penalise, and nothing here waits for the length)
    // (shares may be left unsorted from the first position that the tail neither keeps in LDS nor writes out; never on
    // verification rows, whose replay reads the list itself)
    if (UNSORTED && tid == 0)
        s_plan.nucleus_rows = nucleus_rows; // (read behind the plan's barriers)
    const uint32_t opaque_first = (UNSORTED && !d.draft) ? max(kHeadGroups * kGroup, (d.out_cand_idx && d.out_cand_q) ? d.cand_cap : 0u) : kNone;
    if (d.hist_tokens && !penalties_neutral(P))
        row_pieces<ALIGNED, KH, true, UNSORTED, AHEAD, SORT_WAVES>(d, sc, row, piece, pieces, n_pieces, piece_len, P, hl, slices, L, s_plan, opaque_first);
    else
        row_pieces<ALIGNED, KH, false, UNSORTED, AHEAD, SORT_WAVES>(d, sc, row, piece, pieces, n_pieces, piece_len, P, hl, slices, L, s_plan, opaque_first);
}

// (its arguments by value: the cut is one trip to memory away, not two)
template <bool ALIGNED, int KH, bool UNSORTED, int THREADS = kThreads>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(4))) void finish_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[]; // (128-bit LDS operations need the alignment)
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    __shared__ CoarsePlan s_plan;
    finish_body<ALIGNED, KH, UNSORTED, UNSORTED && KH <= 2, kSortWaves>(d_arg, sc_val, slices, gridDim.y, s_dyn64, sm, s_args, s_plan);
}

} // namespace mako
