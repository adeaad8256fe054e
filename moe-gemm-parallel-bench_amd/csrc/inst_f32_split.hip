// Compiled f32 split-K kernels.
#include "registry.h"
namespace moegemm {
MOEGEMM_MENU_F32(MOEGEMM_INST32_SPLIT, EF32)
}  // namespace moegemm
