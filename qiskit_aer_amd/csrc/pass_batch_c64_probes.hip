// complex64 batched-circuit kernel: register passes of lean ops and probes.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_BATCH(, float, kTileBitsC64, 4, V_PROBES)
}  // namespace aerhip
