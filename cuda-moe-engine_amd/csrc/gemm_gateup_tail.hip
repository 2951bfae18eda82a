// Ring GEMM kernels: gate/up + SwiGLU, K not a multiple of 64.
#include "gemm_ring.h"

namespace moe {

template void launch_ring<true, false, true>(const GemmParams&, RingKernel, unsigned, hipStream_t);

}  // namespace moe
