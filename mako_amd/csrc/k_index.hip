// The kernels of the rows whose candidates stay in token order (index_rows.h): a translation unit of their own.
#define MAKO_EMIT_INDEX_KERNELS
#include "launch.h"
#include "sampler_kernels.h"

namespace mako {
namespace {
template <bool ALIGNED, bool STEPS>
void launch_weights(int kh, dim3 grid, hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices)
{
    if (kh == 2)
        hipLaunchKernelGGL((index_weights_kernel<ALIGNED, 2, STEPS>), grid, dim3(kThreads), kDynLds, st, d, sc, slices);
    else if (kh == 8)
        hipLaunchKernelGGL((index_weights_kernel<ALIGNED, 8, STEPS>), grid, dim3(kThreads), kDynLds, st, d, sc, slices);
    else
        hipLaunchKernelGGL((index_weights_kernel<ALIGNED, 0, STEPS>), grid, dim3(kThreads), kDynLds, st, d, sc, slices);
}
} // namespace

void launch_index_weights(bool aligned, int kh, bool steps, hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices)
{
    const dim3 grid((d.n_rows + 7u) & ~7u, (d.n_vocab + kSliceMax - 1u) / kSliceMax);
    if (aligned && steps)
        launch_weights<true, true>(kh, grid, st, d, sc, slices);
    else if (aligned)
        launch_weights<true, false>(kh, grid, st, d, sc, slices);
    else if (steps)
        launch_weights<false, true>(kh, grid, st, d, sc, slices);
    else
        launch_weights<false, false>(kh, grid, st, d, sc, slices);
}

void launch_nth_step(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t step, uint32_t wgs)
{
    const uint32_t rounds = kNthChunk * 8u + (d.n_vocab + 63u) / 64u * 12u + 64u, picking = step == 1u ? kNthPickedMax * 8u + 64u : 0u;
    hipLaunchKernelGGL(nth_step_kernel, dim3((d.n_rows + 7u) & ~7u, wgs), dim3(kThreads), rounds > picking ? rounds : picking, st, d, sc, step);
}

void launch_index_finish(hipStream_t st, const mako_sample_desc& d, const Scratch& sc, bool in_order_rows, bool other_rows)
{
    // (the group records are for rows in token order only: a workgroup per 16 384 entries where the rows fill the chip
    // anyway, per 4 096 on a small batch)
    if (in_order_rows && (uint64_t)d.n_rows * ((d.n_vocab + kSliceMax - 1u) / kSliceMax) >= 256u)
        hipLaunchKernelGGL(index_groups_kernel<4u>, dim3((d.n_rows + 7u) & ~7u, (d.n_vocab + kSliceMax - 1u) / kSliceMax), dim3(kThreads), 0, st, d, sc);
    else if (in_order_rows)
        hipLaunchKernelGGL(index_groups_kernel<1u>, dim3((d.n_rows + 7u) & ~7u, (d.n_vocab + kIndexBlock - 1u) / kIndexBlock), dim3(kThreads), 0, st, d, sc);
    if (other_rows)
        hipLaunchKernelGGL(index_tail_kernel<true>, dim3(1, d.n_rows), dim3(kThreads), kTailLds, st, d, sc);
    else
        hipLaunchKernelGGL(index_tail_kernel<false>, dim3(1, d.n_rows), dim3(kThreads), kTailLds, st, d, sc);
}

hipError_t init_index_kernels()
{
    const void* kernels[] = {(const void*)index_weights_kernel<true, 0, false>, (const void*)index_weights_kernel<true, 0, true>,
                             (const void*)index_weights_kernel<true, 2, false>, (const void*)index_weights_kernel<true, 2, true>,
                             (const void*)index_weights_kernel<true, 8, false>, (const void*)index_weights_kernel<true, 8, true>,
                             (const void*)index_weights_kernel<false, 0, false>, (const void*)index_weights_kernel<false, 0, true>,
                             (const void*)index_weights_kernel<false, 2, false>, (const void*)index_weights_kernel<false, 2, true>,
                             (const void*)index_weights_kernel<false, 8, false>, (const void*)index_weights_kernel<false, 8, true>};
    for (const void* k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDynLds);
        if (e != hipSuccess)
            return e;
    }
    hipError_t e = hipFuncSetAttribute((const void*)nth_step_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kNthLds);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void*)index_tail_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds);
    return e != hipSuccess ? e : hipFuncSetAttribute((const void*)index_tail_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds);
}
} // namespace mako
