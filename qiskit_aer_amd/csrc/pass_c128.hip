// complex128 register passes with 3 register bits: the lean variants.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, double, kTileBitsC128, 3, false, false)
AERHIP_REG_PASS(, double, kTileBitsC128, 3, false, true)
}  // namespace aerhip
