// Launchers of the sampler's kernels.  Every kernel family is compiled as a translation unit of its own (k_*.hip):
// the compiler's register allocation for a kernel otherwise depends on which other kernels share its inlined device
// functions (sort_kernel lost 2.4 us per batch to spills when plan_kernel variants with the whole-row path were
// compiled beside it).  Each init function raises the dynamic LDS limit of its family's kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mako_sampler.h"

namespace mako {
struct Scratch;

hipError_t init_scan_kernels();
hipError_t init_finish_kernels();
hipError_t init_plan_alone();
hipError_t init_sort_kernels();
hipError_t init_tail_kernels();

// scan_kernel<aligned, kh, above, short_slice(slice_len)>, grid = (slices, rows), `lds` bytes of dynamic LDS
// (`sc`: the HOST copy of the context's record; the kernels take it by value, so that their first loads need no
// trip to memory for the record itself)
void launch_scan(bool aligned, int kh, bool above, dim3 grid, size_t lds, hipStream_t st, const mako_sample_desc& d,
                 const Scratch& sc, uint32_t slice_len, uint32_t cus);
// finish_kernel<aligned, kh> on `wgs` workgroups
// (unsorted: the instances for batches of many top_k == 0 rows, whose plans leave shares unsorted; the kernels
// of one batch must agree on it)
void launch_finish(bool aligned, int kh, bool unsorted, uint32_t wgs, hipStream_t st, const mako_sample_desc& d, const Scratch& sc,
                   uint32_t slices); // (host copy, by value)
// the large batches' instance of 512 threads, two workgroups to a CU (second_pass_halves(); histories of up to 2 048 entries)
hipError_t init_finish_halves();
void launch_finish_halves(bool aligned, uint32_t wgs, hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices);
void launch_plan_alone(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices); // (host copy, by value)
// sort_kernel's workgroup i serves entry i of the work list: `grid_rows` * kWorkers workgroups must cover the
// longest list the batch can produce (kWorkers entries per top_k == 0 row); tail_kernel takes one workgroup per possible wide row.  Workgroups beyond the lists leave at once, but each
// of them still has to be dispatched.
void launch_sort(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices, uint32_t grid_rows, bool unsorted); // (host copy)
// (tail_kernel: `tail_cap` workgroups for the possible wide rows, then one per row for what is left of every row)
void launch_tail(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices, uint32_t tail_cap, bool unsorted); // (host copy, by value)
// the three kernels of a batch with none but rows of the whole-row class (index_rows.h): the weights, the group records, the
// total and the draw
hipError_t init_index_kernels();
// (steps: there are rows for nth_steps.h, its steps or its picks)
void launch_index_weights(bool aligned, int kh, bool steps, hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices);
// a step of nth_steps.h, `wgs` workgroups per row
void launch_nth_step(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t step, uint32_t wgs);
void launch_index_finish(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, bool in_order_rows, bool other_rows);
// finish, sort and tail of a batch where such rows are, or may be, beside others (beside_rows.h): the same launches with
// `more` workgroups behind their own for those rows
hipError_t init_beside_finish();
hipError_t init_beside_sort();
hipError_t init_beside_tail();
void launch_finish_beside(bool aligned, int kh, bool unsorted, uint32_t wgs, uint32_t more, hipStream_t st, const mako_sample_desc& d,
                          const Scratch& sc, uint32_t slices);
void launch_sort_beside(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices, uint32_t grid_rows, bool unsorted,
                        uint32_t more, uint32_t cus);
void launch_tail_beside(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices, uint32_t tail_cap, bool unsorted);
} // namespace mako
