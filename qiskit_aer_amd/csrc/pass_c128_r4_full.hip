// complex128 register pass with 4 register bits: the full variant.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, double, kTileBitsC128, 4, V_FULL, false)
}  // namespace aerhip
