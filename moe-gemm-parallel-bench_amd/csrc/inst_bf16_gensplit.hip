// Compiled bf16 split-K kernels of the general tile.
#include "registry.h"
namespace moegemm {
MOEGEMM_MENU_GEN_SPLIT(MOEGEMM_INST16_GENSPLIT, EBf16)
}  // namespace moegemm
