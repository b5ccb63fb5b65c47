// complex128 register pass with 3 register bits: the variant with 4x4 gates.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, double, kTileBitsC128, 3, V_GATES, false)
}  // namespace aerhip
