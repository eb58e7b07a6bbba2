// finish_kernel for batches of many top_k == 0 rows: workgroups of 512 threads, two to a CU (79 680 bytes of LDS each).  A CU's vector
// units were busy for 54 to 57 % of the kernel's time, its LDS for 16 to 37 %: what is between is barriers and trips to memory, which
// one workgroup now fills for the other.  112 to 150 rows of 129 280 logits with histories of 1 024, in a batch of 512: 73.0 us with one
// workgroup of 1 024, 66.4 so (the batch 187.2 -> 177.3); 256 rows of 151 552, half of them flat: 104.7 and 102.  With four history
// entries a thread the next piece's loads ahead of the hand-over spill, and are worth nothing with a second workgroup on the CU
// (68.3 us with them and 28 bytes of scratch memory, 66.4 without).
#define MAKO_THREADS 512
#include "launch.h"
#include "sampler_common.h"
#include "second_pass.h"

namespace mako {
namespace {
template <bool ALIGNED, int KH>
void launch_one(uint32_t wgs, hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices)
{
    hipLaunchKernelGGL((finish_kernel<ALIGNED, KH, true>), dim3(1, wgs), dim3(kThreads), kFinishLds, st, d, sc, slices);
}
} // namespace

// (histories of up to 2 or 4 entries a thread)
void launch_finish_halves(bool aligned, uint32_t wgs, hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slices)
{
    const bool two = !d.hist_tokens || d.hist_stride <= 2 * kThreads;
    if (aligned && two)
        launch_one<true, 2>(wgs, st, d, sc, slices);
    else if (aligned)
        launch_one<true, 4>(wgs, st, d, sc, slices);
    else if (two)
        launch_one<false, 2>(wgs, st, d, sc, slices);
    else
        launch_one<false, 4>(wgs, st, d, sc, slices);
}

hipError_t init_finish_halves()
{
    for (const void* k : {(const void*)finish_kernel<true, 2, true>, (const void*)finish_kernel<false, 2, true>,
                          (const void*)finish_kernel<true, 4, true>, (const void*)finish_kernel<false, 4, true>}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFinishLds);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}
} // namespace mako
