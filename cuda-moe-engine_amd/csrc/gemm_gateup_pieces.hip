// Ring GEMM kernel: gate/up + SwiGLU with column pieces, packed rows.
#include "gemm_ring.h"

namespace moe {

template void launch_pieces<false, false>(const GemmParams&, unsigned, hipStream_t);

}  // namespace moe
