// Instantiations of the 128 x 128 tiles of the 16x16x32 loop
// (gemm16s_kernel.h): the plain store, fp16.

#include "gemm16s_kernel.h"

namespace cpt {
namespace gemm {

CPT_ST16_INST_STORE(CPT_ST16_DEFINE, kF16)

}  // namespace gemm
}  // namespace cpt
