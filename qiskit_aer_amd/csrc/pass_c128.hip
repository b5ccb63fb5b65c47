// complex128 register passes with 3 register bits: the lean variants.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, double, kTileBitsC128, 3, V_LEAN, false)
AERHIP_REG_PASS(, double, kTileBitsC128, 3, V_LEAN, true)
}  // namespace aerhip
