// The int8 LDS-ring GEMM over a row-major [K,N] B read in place: its
// instantiations, in a source of their own so that they build beside the rest.
#include "gemm_i8_ring.hpp"

namespace nnops_amd {

void launch_ring_trb(const GemmI8Kern& k, const RingPlan& r, const RingSplit& sk, hipStream_t s)
{
    launch_ring_tiles<false, true>(k, r, sk, s);
}

}  // namespace nnops_amd
