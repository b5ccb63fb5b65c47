// complex128 batched-circuit kernel: register passes of lean ops and probes.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_BATCH(, double, kTileBitsC128, 3, V_PROBES)
}  // namespace aerhip
