// Ring GEMM kernels: plain, K not a multiple of 64.
#include "gemm_ring.h"

namespace moe {

template void launch_ring<false, false, true>(const GemmParams&, RingKernel, unsigned, hipStream_t);

}  // namespace moe
