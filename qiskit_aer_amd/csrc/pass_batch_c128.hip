// complex128 batched-circuit kernel.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_BATCH(, double, kTileBitsC128, 3)
}  // namespace aerhip
