// Ring GEMM kernel: gate/up + SwiGLU with column pieces, K not a multiple of 64.
#include "gemm_ring.h"

namespace moe {

template void launch_pieces<false, true>(const GemmParams&, unsigned, hipStream_t);

}  // namespace moe
