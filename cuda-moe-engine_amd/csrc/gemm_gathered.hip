// Ring GEMM kernels: gate/up + SwiGLU, rows gathered from x.
#include "gemm_ring.h"

namespace moe {

template void launch_ring<true, true, false>(const GemmParams&, RingKernel, unsigned, hipStream_t);

}  // namespace moe
