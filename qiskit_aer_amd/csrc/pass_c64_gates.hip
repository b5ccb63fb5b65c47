// complex64 register pass with 4 register bits: the variant with 4x4 gates.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, float, kTileBitsC64, 4, V_GATES, false)
}  // namespace aerhip
