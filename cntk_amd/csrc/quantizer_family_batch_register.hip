// Kernel family of the per-column gradient quantizer (gfx950): the members of a gradient set whose columns stay in registers, quantized or
// reduced by one grid per workgroup size.
// The launchers of one family, instantiated here and nowhere else; quantizer_launch.h declares the functions and chooses
// between the families.
#include "quantizer_launch.h"

namespace cntkq {

template <int NBITS, bool ZT>
struct RegBatchLauncher
{
    static hipError_t run(hipStream_t s, LaunchEvents ev, const QuantizeBatchEntry* entries, const uint32_t* begins, uint32_t count,
                          uint32_t total_blocks, size_t lds, uint32_t threads, bool wide)
    {
        if constexpr (NBITS >= 32)
            return hipErrorInvalidValue;
        else
        {
            if (threads == 1024)
                hipExtLaunchKernelGGL((quantize_reg_batch_kernel<NBITS, ZT, 1024, false>), dim3(total_blocks), dim3(1024), lds, s, ev.start, ev.stop, 0,
                                      entries, begins, count);
            else if (wide)
                hipExtLaunchKernelGGL((quantize_reg_batch_kernel<NBITS, ZT, 256, true>), dim3(total_blocks), dim3(256), lds, s, ev.start, ev.stop, 0,
                                      entries, begins, count);
            else
                hipExtLaunchKernelGGL((quantize_reg_batch_kernel<NBITS, ZT, 256, false>), dim3(total_blocks), dim3(256), lds, s, ev.start, ev.stop, 0,
                                      entries, begins, count);
            return hipGetLastError();
        }
    }
};

template <int NBITS, bool ZT>
struct StripeRegBatchLauncher
{
    static hipError_t run(hipStream_t s, LaunchEvents ev, const StripeBatchEntry* entries, const uint32_t* begins, uint32_t count,
                          uint32_t total_blocks, size_t lds, uint32_t threads, bool wide, bool one)
    {
        if constexpr (NBITS >= 32)
            return hipErrorInvalidValue;
        else
        {
            if (one && threads == 1024)
                hipExtLaunchKernelGGL((stripe_one_reg_batch_kernel<NBITS, ZT, 1024, false>), dim3(total_blocks), dim3(1024), lds, s, ev.start, ev.stop,
                                      0, entries, begins, count);
            else if (one && wide)
                hipExtLaunchKernelGGL((stripe_one_reg_batch_kernel<NBITS, ZT, 256, true>), dim3(total_blocks), dim3(256), lds, s, ev.start, ev.stop, 0,
                                      entries, begins, count);
            else if (one)
                hipExtLaunchKernelGGL((stripe_one_reg_batch_kernel<NBITS, ZT, 256, false>), dim3(total_blocks), dim3(256), lds, s, ev.start, ev.stop, 0,
                                      entries, begins, count);
            else if (threads == 1024)
                hipExtLaunchKernelGGL((stripe_reduce_reg_batch_kernel<NBITS, ZT, 1024, false>), dim3(total_blocks), dim3(1024), lds, s, ev.start,
                                      ev.stop, 0, entries, begins, count);
            else if (wide)
                hipExtLaunchKernelGGL((stripe_reduce_reg_batch_kernel<NBITS, ZT, 256, true>), dim3(total_blocks), dim3(256), lds, s, ev.start,
                                      ev.stop, 0, entries, begins, count);
            else
                hipExtLaunchKernelGGL((stripe_reduce_reg_batch_kernel<NBITS, ZT, 256, false>), dim3(total_blocks), dim3(256), lds, s, ev.start,
                                      ev.stop, 0, entries, begins, count);
            return hipGetLastError();
        }
    }
};

hipError_t family_batch_reg_quantize(size_t nbits, bool zt, hipStream_t s, LaunchEvents ev, const QuantizeBatchEntry* entries, const uint32_t* begins, uint32_t count, uint32_t total_blocks, size_t lds, uint32_t threads, bool wide)
{
    return dispatch_nbits<RegBatchLauncher>(nbits, zt, s, ev, entries, begins, count, total_blocks, lds, threads, wide);
}

hipError_t family_batch_reg_stripe(size_t nbits, bool zt, hipStream_t s, LaunchEvents ev, const StripeBatchEntry* entries, const uint32_t* begins, uint32_t count, uint32_t total_blocks, size_t lds, uint32_t threads, bool wide, bool one)
{
    return dispatch_nbits<StripeRegBatchLauncher>(nbits, zt, s, ev, entries, begins, count, total_blocks, lds, threads, wide, one);
}

} // namespace cntkq
