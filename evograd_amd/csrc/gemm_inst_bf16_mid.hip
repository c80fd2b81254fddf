// Instantiations of the 128 x 128 product kernel (gemm_mid.hpp), bf16 operands.
#include "gemm_mid.hpp"

namespace eg {
namespace gk {
EG_MID_ALL_KERNELS(template, bf16_t)
}  // namespace gk
}  // namespace eg
