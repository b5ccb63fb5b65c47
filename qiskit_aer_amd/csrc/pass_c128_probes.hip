// complex128 register pass with 3 register bits: the variant with probes.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, double, kTileBitsC128, 3, V_PROBES, false)
}  // namespace aerhip
