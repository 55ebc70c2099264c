// Instantiations of the 128 x 128 tiles of the 16x16x32 loop
// (gemm16s_kernel.h): F1 without codec, B1 on a bf16 cache.

#include "gemm16s_kernel.h"

namespace cpt {
namespace gemm {

CPT_ST16_INST_GLU(CPT_ST16_DEFINE, kBF16)
CPT_ST16_INST_GLU(CPT_ST16_DEFINE, kF16)
CPT_ST16_INST_DGLU(CPT_ST16_DEFINE)

}  // namespace gemm
}  // namespace cpt
