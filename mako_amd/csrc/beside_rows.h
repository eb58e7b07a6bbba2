// Batches in which rows of the whole-row class are beside rows of other kinds, or may be (the caller's host copy of the
// parameters shows them, or there is none): the kernels of index_rows.h as workgroups of the others' launches, so that a
// batch has four launches whatever its rows are.  (Launches of their own would cost a batch without such rows three times
// 2 us; one workgroup for all of a row's work, as a batch without the host copy had it, took 500 to 700 us a row.)
// Workgroups behind those of the launch's own kernel take the rows' pieces in turn; scan_kernel has counted the rows, and
// without any of them they leave at once.  (Looked for in the parameters instead, 64 rows a trip to memory, their absence kept
// finish's launch of 4 000 top-k rows 50 us, 10 without these workgroups, 12 now.)
#pragma once

#include "index_rows.h"
#include "second_pass.h"
#include "sort_kernels.h"
#include "tail_kernel.h"

namespace mako {

#ifdef MAKO_EMIT_BESIDE_FINISH
// grid = (1, finish_wgs + workgroups for the weights)
template <bool ALIGNED, int KH, bool UNSORTED>
__global__ __launch_bounds__(kThreads) void finish_beside_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices, uint32_t finish_wgs)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[]; // (128-bit LDS operations need the alignment)
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    __shared__ CoarsePlan s_plan;
    if (blockIdx.y < finish_wgs) {
        finish_body<ALIGNED, KH, UNSORTED, false, kSortBesideWaves>(d_arg, sc_val, slices, finish_wgs, s_dyn64, sm, s_args, s_plan);
        return;
    }
    const uint32_t pieces = (d_arg.n_vocab + kSliceMax - 1u) / kSliceMax;
    const uint32_t all = sc_val.work_n[8] * pieces;
    RankedRows rows;
    for (uint32_t p = blockIdx.y - finish_wgs; p < all; p += gridDim.y - finish_wgs) {
        uint32_t row;
        if (!rows.find(d_arg, p / pieces, [](const mako_sampling_params& P) { return classify(P) == kGeneral; }, row))
            return;
        index_weights_piece<ALIGNED, KH, true>(d_arg, sc_val, slices, row, p % pieces, s_dyn64, sm, s_args);
        __syncthreads(); // (the next piece's table of counts and arguments)
    }
}
#endif

#ifdef MAKO_EMIT_BESIDE_SORT
// grid = (as sort_kernel's, sort_rows + rows of workgroups for the groups)
template <bool UNSORTED>
__global__ __launch_bounds__(kThreads) void sort_beside_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices, uint32_t sort_rows, uint32_t cus)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[]; // (128-bit LDS operations need the alignment)
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    // (what either way needs first in one trip, and ahead of the branch: behind it, where stores of the other way might have
    // been, the compiler takes no scalar loads, and thousands of workgroups without work wait for nothing but this trip.
    // 8 704 of them: 31 us with vector loads, a trip of their own for the arguments and, short of registers, scratch memory; 23 now, 20.6 in
    // sort_kernel)
    const uint32_t general = sc_val.work_n[8], in_order = sc_val.work_n[9];
    SortFirstTrip first;
    fetch_sort_entry<UNSORTED>(d_arg, sc_val, min(blockIdx.y, max(sort_rows, 1u) - 1u) * gridDim.x + blockIdx.x, first);
    if (blockIdx.y < sort_rows) {
        sort_body<UNSORTED>(d_arg, sc_val, slices, first, s_dyn64, sm, s_args);
        return;
    }
    const uint32_t blocks = (d_arg.n_vocab + kIndexBlock - 1u) / kIndexBlock;
    const uint32_t all = in_order * blocks;
    const uint32_t me = (blockIdx.y - sort_rows) * gridDim.x + blockIdx.x, wgs = (gridDim.y - sort_rows) * gridDim.x;
    RankedRows rows;
    for (uint32_t p = wgs - 1u - me; p < all; p += wgs) {
        uint32_t row;
        if (!rows.find(d_arg, p / blocks, [](const mako_sampling_params& P) { return index_order_row(P); }, row))
            break;
        index_groups_block<1u>(d_arg, sc_val, row, p % blocks, reinterpret_cast<double*>(s_dyn64));
        __syncthreads();
    }
    // (nth_steps.h's steps, by as many workgroups a row as there are CUs for, since they wait for each other.  Behind the groups,
    // whose workgroups are counted from the other end)
    const uint32_t nth_rows = nth_steps_for(d_arg.n_vocab) ? general - in_order : 0u;
    if (nth_rows) { // uniform
        const uint32_t per_row = min(max(min(wgs, cus) / nth_rows, 1u), (d_arg.n_vocab + kNthChunk - 1u) / kNthChunk);
        RankedRows ranked;
        for (uint32_t p = me; p < nth_rows * per_row; p += wgs) {
            uint32_t row;
            if (!ranked.find(d_arg, p / per_row, [](const mako_sampling_params& P) { return nth_row(P); }, row))
                break;
            nth_steps_at_once(d_arg, sc_val, row, p % per_row, per_row, s_dyn64, sm.bs);
            __syncthreads();
        }
    }
}
#endif

#ifdef MAKO_EMIT_BESIDE_TAIL
// grid as tail_kernel's
template <bool UNSORTED>
__global__ __launch_bounds__(kThreads) void tail_beside_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices, uint32_t tail_cap)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[]; // (128-bit LDS operations need the alignment)
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    tail_body<UNSORTED, true>(d_arg, sc_val, slices, tail_cap, s_dyn64, sm, s_args);
}
#endif

} // namespace mako
