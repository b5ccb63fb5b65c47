// complex64 batched-circuit kernel: every pass kind.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_BATCH(, float, kTileBitsC64, 4, V_FULL)
}  // namespace aerhip
