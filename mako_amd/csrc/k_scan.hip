// scan_kernel's variants: the only kernels that stream the logits.
#include "launch.h"
#include "sampler_kernels.h"

namespace mako {
namespace {
template <bool ALIGNED, int KH, bool ABOVE, bool SHORT>
void launch_one(dim3 grid, size_t lds, hipStream_t st, const mako_sample_desc& d, const Scratch& sc, uint32_t slice_len,
                uint32_t cus)
{
    hipLaunchKernelGGL((scan_kernel<ALIGNED, KH, ABOVE, SHORT>), grid, dim3(kThreads), lds, st, d, sc, slice_len, cus);
}
template <bool ALIGNED, int KH>
void launch_kh(bool above, dim3 grid, size_t lds, hipStream_t st, const mako_sample_desc& d, const Scratch& sc,
               uint32_t slice_len, uint32_t cus)
{
    if (short_slice(slice_len) && above) // (a row of one slice)
        launch_one<ALIGNED, KH, true, true>(grid, lds, st, d, sc, slice_len, cus);
    else if (short_slice(slice_len))
        launch_one<ALIGNED, KH, false, true>(grid, lds, st, d, sc, slice_len, cus);
    else if (above)
        launch_one<ALIGNED, KH, true, false>(grid, lds, st, d, sc, slice_len, cus);
    else
        launch_one<ALIGNED, KH, false, false>(grid, lds, st, d, sc, slice_len, cus);
}
template <bool ALIGNED>
void launch_aligned(int kh, bool above, dim3 grid, size_t lds, hipStream_t st, const mako_sample_desc& d, const Scratch& sc,
                uint32_t slice_len, uint32_t cus)
{
    if (kh == 2)
        launch_kh<ALIGNED, 2>(above, grid, lds, st, d, sc, slice_len, cus);
    else if (kh == 8)
        launch_kh<ALIGNED, 8>(above, grid, lds, st, d, sc, slice_len, cus);
    else
        launch_kh<ALIGNED, 0>(above, grid, lds, st, d, sc, slice_len, cus);
}
} // namespace

void launch_scan(bool aligned, int kh, bool above, dim3 grid, size_t lds, hipStream_t st, const mako_sample_desc& d,
                 const Scratch& sc, uint32_t slice_len, uint32_t cus)
{
    if (aligned)
        launch_aligned<true>(kh, above, grid, lds, st, d, sc, slice_len, cus);
    else
        launch_aligned<false>(kh, above, grid, lds, st, d, sc, slice_len, cus);
}

hipError_t init_scan_kernels()
{
    const void* kernels[] = {(const void*)scan_kernel<true, 0, false>, (const void*)scan_kernel<false, 0, false>,
                             (const void*)scan_kernel<true, 2, false>, (const void*)scan_kernel<false, 2, false>,
                             (const void*)scan_kernel<true, 8, false>, (const void*)scan_kernel<false, 8, false>,
                             (const void*)scan_kernel<true, 0, true>,  (const void*)scan_kernel<false, 0, true>,
                             (const void*)scan_kernel<true, 2, true>,  (const void*)scan_kernel<false, 2, true>,
                             (const void*)scan_kernel<true, 8, true>,  (const void*)scan_kernel<false, 8, true>,
                             (const void*)scan_kernel<true, 0, false, true>, (const void*)scan_kernel<false, 0, false, true>,
                             (const void*)scan_kernel<true, 2, false, true>, (const void*)scan_kernel<false, 2, false, true>,
                             (const void*)scan_kernel<true, 8, false, true>, (const void*)scan_kernel<false, 8, false, true>,
                             (const void*)scan_kernel<true, 0, true, true>, (const void*)scan_kernel<false, 0, true, true>,
                             (const void*)scan_kernel<true, 2, true, true>, (const void*)scan_kernel<false, 2, true, true>,
                             (const void*)scan_kernel<true, 8, true, true>, (const void*)scan_kernel<false, 8, true, true>};
    for (const void* k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDynLds);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}
} // namespace mako
