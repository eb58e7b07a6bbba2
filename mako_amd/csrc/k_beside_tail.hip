// tail_beside_kernel: tail_kernel for batches whose rows of the whole-row class have been begun by the launches before it.
#define MAKO_EMIT_BESIDE_TAIL
#include "launch.h"
#include "sampler_kernels.h"

namespace mako {
void launch_tail_beside(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices, uint32_t tail_cap, bool unsorted)
{
    const dim3 grid(1, tail_cap + d.n_rows);
    if (unsorted)
        hipLaunchKernelGGL(tail_beside_kernel<true>, grid, dim3(kThreads), kTailLds, st, d, sc, slices, tail_cap);
    else
        hipLaunchKernelGGL(tail_beside_kernel<false>, grid, dim3(kThreads), kTailLds, st, d, sc, slices, tail_cap);
}

hipError_t init_beside_tail()
{
    const hipError_t e = hipFuncSetAttribute((const void*)tail_beside_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds);
    return e != hipSuccess ? e : hipFuncSetAttribute((const void*)tail_beside_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds);
}
} // namespace mako
