// complex64 batched-circuit kernel.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_BATCH(, float, kTileBitsC64, 4)
}  // namespace aerhip
