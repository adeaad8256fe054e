// Compiled bf16 kernels for operands staged element by element.
#include "registry.h"
namespace moegemm {
MOEGEMM_MENU_16BIT(MOEGEMM_INST_PLAIN, EBf16)
}  // namespace moegemm
