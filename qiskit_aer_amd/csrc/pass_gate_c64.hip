// complex64 gate pass on tiles of 2^12 amplitudes.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_GATE_PASS(, float, kTileBitsC64, kGateRegBits, false)
}  // namespace aerhip
