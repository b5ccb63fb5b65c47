// complex64 register pass with 4 register bits: the variant with probes.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_REG_PASS(, float, kTileBitsC64, 4, V_PROBES, false)
}  // namespace aerhip
