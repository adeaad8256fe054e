// Compiled f16 kernels for transposed operands: K-contiguous B.
#include "registry.h"
namespace moegemm {
MOEGEMM_MENU_BT(MOEGEMM_INST16_TR, EF16)
}  // namespace moegemm
