// Compiled f32 kernels for operands staged element by element.
#include "registry.h"
namespace moegemm {
MOEGEMM_MENU_F32(MOEGEMM_INST_PLAIN, EF32)
}  // namespace moegemm
