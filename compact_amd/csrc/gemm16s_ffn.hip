// Instantiations of the 128 x 128 tiles of the 16x16x32 loop
// (gemm16s_kernel.h): F1 and B1 on a bf16 cache or none.

#include "gemm16s_kernel.h"

namespace cpt {
namespace gemm {

CPT_ST16_INST_FFN(CPT_ST16_DEFINE)

}  // namespace gemm
}  // namespace cpt
