// Compiled f16 general kernels (operands outside the LDS-DMA layouts).
#include "registry.h"
namespace moegemm {
MOEGEMM_MENU_16BIT(MOEGEMM_INST16_GEN, EF16)
}  // namespace moegemm
