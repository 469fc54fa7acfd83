// The kernels of short columns by groups of lanes: stripe reduction, float and double columns.
#include "quantizer_launch.h"

namespace cntkq {

namespace {

template <int NBITS, bool ZT, typename E, int CHAIN>
hipError_t launch_lanes_stripe(hipStream_t s, LaunchEvents ev, const StripeSources& src, E* stripe_res, char* q_out, E* agg_out, const LanesGeom& t)
{
    hipExtLaunchKernelGGL((stripe_lanes_kernel<NBITS, ZT, CHAIN, E>), dim3(lanes_blocks(t)),
                          dim3(kLanesThreads), lanes_lds_bytes<E>(t, src.workers), s, ev.start, ev.stop, 0, src, stripe_res, q_out, agg_out, t);
    return hipGetLastError();
}

template <int NBITS, bool ZT>
struct StripeLanesLauncher
{
    template <typename E>
    static hipError_t run(hipStream_t s, LaunchEvents ev, const StripeSources& src, E* stripe_res, char* q_out, E* agg_out, const LanesGeom& t)
    {
        if constexpr (NBITS >= Word<E>::kBits)
            return hipErrorInvalidValue;
        else
        {
#define CNTKQ_BODY(C) return launch_lanes_stripe<NBITS, ZT, E, C>(s, ev, src, stripe_res, q_out, agg_out, t);
            CNTKQ_LANES_CHAINS(E, CNTKQ_BODY)
            return hipErrorInvalidValue;
#undef CNTKQ_BODY
        }
    }
};

} // namespace

hipError_t family_lanes_stripe(size_t nbits, bool zt, hipStream_t s, LaunchEvents ev, const StripeSources& src, float* stripe_res, char* q_out,
                               float* agg_out, const LanesGeom& t)
{
    return dispatch_nbits<StripeLanesLauncher>(nbits, zt, s, ev, src, stripe_res, q_out, agg_out, t);
}

hipError_t family_lanes_stripe(size_t nbits, bool zt, hipStream_t s, LaunchEvents ev, const StripeSources& src, double* stripe_res, char* q_out,
                               double* agg_out, const LanesGeom& t)
{
    return dispatch_nbits<StripeLanesLauncher>(nbits, zt, s, ev, src, stripe_res, q_out, agg_out, t);
}

} // namespace cntkq
