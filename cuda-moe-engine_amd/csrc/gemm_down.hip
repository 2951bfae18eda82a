// Ring GEMM kernels: plain.
#include "gemm_ring.h"

namespace moe {

template void launch_ring<false, false, false>(const GemmParams&, RingKernel, unsigned, hipStream_t);

}  // namespace moe
