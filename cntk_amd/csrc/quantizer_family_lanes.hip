// The kernels of short columns by groups of lanes: quantize, float and double columns.
#include "quantizer_launch.h"

namespace cntkq {

namespace {

template <int NBITS, bool ZT, typename E, int CHAIN>
hipError_t launch_lanes_quantize(hipStream_t s, LaunchEvents ev, const E* g, const E* r_in, E* r_out, char* q, const LanesGeom& t)
{
    hipExtLaunchKernelGGL((quantize_lanes_kernel<NBITS, ZT, CHAIN, E>), dim3(lanes_blocks(t)),
                          dim3(kLanesThreads), lanes_lds_bytes<E>(t, 0), s, ev.start, ev.stop, 0, g, r_in, r_out, q, t);
    return hipGetLastError();
}

template <int NBITS, bool ZT>
struct LanesLauncher
{
    template <typename E>
    static hipError_t run(hipStream_t s, LaunchEvents ev, const E* g, const E* r_in, E* r_out, char* q, const LanesGeom& t)
    {
        if constexpr (NBITS >= Word<E>::kBits)
            return hipErrorInvalidValue;
        else
        {
#define CNTKQ_BODY(C) return launch_lanes_quantize<NBITS, ZT, E, C>(s, ev, g, r_in, r_out, q, t);
            CNTKQ_LANES_CHAINS(E, CNTKQ_BODY)
            return hipErrorInvalidValue;
#undef CNTKQ_BODY
        }
    }
};

} // namespace

hipError_t family_lanes_quantize(size_t nbits, bool zt, hipStream_t s, LaunchEvents ev, const float* g, const float* r_in, float* r_out, char* q,
                                 const LanesGeom& t)
{
    return dispatch_nbits<LanesLauncher>(nbits, zt, s, ev, g, r_in, r_out, q, t);
}

hipError_t family_lanes_quantize(size_t nbits, bool zt, hipStream_t s, LaunchEvents ev, const double* g, const double* r_in, double* r_out, char* q,
                                 const LanesGeom& t)
{
    return dispatch_nbits<LanesLauncher>(nbits, zt, s, ev, g, r_in, r_out, q, t);
}

} // namespace cntkq
