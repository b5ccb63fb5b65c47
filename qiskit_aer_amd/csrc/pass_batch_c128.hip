// complex128 batched-circuit kernel: every pass kind.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_BATCH(, double, kTileBitsC128, 3, V_FULL)
}  // namespace aerhip
