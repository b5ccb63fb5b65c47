// complex64 register pass with 4 register bits: the lean variant.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, float, kTileBitsC64, 4, V_LEAN, false)
}  // namespace aerhip
