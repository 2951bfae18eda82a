// Ring GEMM kernel: gate/up + SwiGLU with column pieces, rows gathered from x.
#include "gemm_ring.h"

namespace moe {

template void launch_pieces<true, false>(const GemmParams&, unsigned, hipStream_t);

}  // namespace moe
