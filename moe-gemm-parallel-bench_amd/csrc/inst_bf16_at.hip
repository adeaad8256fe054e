// Compiled bf16 kernels for transposed operands: M-contiguous A.
#include "registry.h"
namespace moegemm {
MOEGEMM_MENU_AT(MOEGEMM_INST16_TR, EBf16)
}  // namespace moegemm
