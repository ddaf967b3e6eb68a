// Prefill GEMM kernels for K = 8 bits per weight (all codebooks): the narrow core
// and the 256-row wide one.
#include "gemm_wide.hpp"

namespace stx {
STX_INSTANTIATE_GEMM_NARROW(8)
STX_INSTANTIATE_GEMM_WIDE(8)
}  // namespace stx
