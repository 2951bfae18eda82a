// Ring GEMM kernels: gate/up + SwiGLU, packed rows.
#include "gemm_ring.h"

namespace moe {

template void launch_ring<true, false, false>(const GemmParams&, RingKernel, unsigned, hipStream_t);

}  // namespace moe
