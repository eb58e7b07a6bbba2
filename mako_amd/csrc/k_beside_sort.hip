// sort_beside_kernel: the wide rows' sort and the group records of the rows in token order in one launch.
#define MAKO_EMIT_BESIDE_SORT
#include "launch.h"
#include "sampler_kernels.h"

namespace mako {
void launch_sort_beside(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices, uint32_t grid_rows, bool unsorted,
                        uint32_t more, uint32_t cus)
{
    static_assert(kSortBesideWaves == (uint32_t)kWaves, "");
    const uint32_t x = unsorted ? kSortItemsPerRow : kWorkers;
    const dim3 grid(x, grid_rows + (more + x - 1u) / x);
    if (unsorted)
        hipLaunchKernelGGL(sort_beside_kernel<true>, grid, dim3(kThreads), kSortLds, st, d, sc, slices, grid_rows, cus);
    else
        hipLaunchKernelGGL(sort_beside_kernel<false>, grid, dim3(kThreads), kSortLds, st, d, sc, slices, grid_rows, cus);
}

hipError_t init_beside_sort()
{
    const hipError_t e = hipFuncSetAttribute((const void*)sort_beside_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSortLds);
    return e != hipSuccess ? e : hipFuncSetAttribute((const void*)sort_beside_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSortLds);
}
} // namespace mako
