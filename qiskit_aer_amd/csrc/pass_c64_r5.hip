// complex64 register pass with 5 register bits: the lean variant.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, float, kTileBitsC64, 5, V_LEAN, false)
}  // namespace aerhip
