// Batches in which rows of the whole-row class are beside rows of other kinds, or may be (the caller's host copy of the
// parameters shows them, or there is none): the kernels of index_rows.h as workgroups of the others' launches, so that a
// batch has four launches whatever its rows are.  (Launches of their own would cost a batch without such rows three times
// 2 us; one workgroup for all of a row's work, as a batch without the host copy had it, took 500 to 700 us a row.)
// Workgroups behind those of the launch's own kernel take the rows' pieces in turn; without such rows they leave after
// a look at the parameters.
#pragma once

#include "index_rows.h"
#include "second_pass.h"
#include "sort_kernels.h"
#include "tail_kernel.h"

namespace mako {

#ifdef MAKO_EMIT_BESIDE_FINISH
// grid = (1, finish_wgs + workgroups for the weights)
template <bool VEC, int KH, bool UNSORTED>
__global__ __launch_bounds__(kThreads) void finish_beside_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices, uint32_t finish_wgs)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[]; // (128-bit LDS operations need the alignment)
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    __shared__ CoarsePlan s_plan;
    if (blockIdx.y < finish_wgs) {
        finish_body<VEC, KH, UNSORTED>(d_arg, sc_val, slices, finish_wgs, s_dyn64, sm, s_args, s_plan);
        return;
    }
    const uint32_t pieces = (d_arg.n_vocab + kSliceMax - 1u) / kSliceMax;
    RankedRows rows;
    for (uint32_t p = blockIdx.y - finish_wgs;; p += gridDim.y - finish_wgs) {
        uint32_t row;
        if (!rows.find(d_arg, p / pieces, [](const mako_sampling_params& P) { return classify(P) == kGeneral; }, row))
            return;
        index_weights_piece<VEC, KH>(d_arg, sc_val, slices, row, p % pieces, s_dyn64, sm, s_args);
        __syncthreads(); // (the next piece's table of counts and arguments)
    }
}
#endif

#ifdef MAKO_EMIT_BESIDE_SORT
// grid = (as sort_kernel's, sort_rows + rows of workgroups for the groups)
template <bool UNSORTED>
__global__ __launch_bounds__(kThreads) void sort_beside_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices, uint32_t sort_rows)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[]; // (128-bit LDS operations need the alignment)
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    if (blockIdx.y < sort_rows) {
        sort_body<UNSORTED>(d_arg, sc_val, slices, s_dyn64, sm, s_args);
        return;
    }
    const uint32_t blocks = (d_arg.n_vocab + kIndexBlock - 1u) / kIndexBlock;
    RankedRows rows;
    for (uint32_t p = (blockIdx.y - sort_rows) * gridDim.x + blockIdx.x;; p += (gridDim.y - sort_rows) * gridDim.x) {
        uint32_t row;
        if (!rows.find(d_arg, p / blocks, [](const mako_sampling_params& P) { return index_order_row(P); }, row))
            return;
        index_groups_block<1u>(d_arg, sc_val, row, p % blocks, reinterpret_cast<double*>(s_dyn64));
        __syncthreads();
    }
}
#endif

#ifdef MAKO_EMIT_BESIDE_TAIL
// grid as tail_kernel's
template <bool UNSORTED>
__global__ __launch_bounds__(kThreads) void tail_beside_kernel(mako_sample_desc d_arg, Scratch sc_val, uint32_t slices, uint32_t tail_cap,
                                                               uint32_t index_path)
{
    extern __shared__ __align__(16) unsigned long long s_dyn64[]; // (128-bit LDS operations need the alignment)
    __shared__ FinishShared sm;
    __shared__ ArgsLds s_args;
    tail_body<UNSORTED, true>(d_arg, sc_val, slices, tail_cap, index_path, s_dyn64, sm, s_args);
}
#endif

} // namespace mako
