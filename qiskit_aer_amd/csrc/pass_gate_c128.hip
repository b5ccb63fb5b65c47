// complex128 gate pass on tiles of 2^12 amplitudes.
#include "pass_kernels.hpp"

namespace aerhip {
AERHIP_GATE_PASS(, double, kGateTileC128, kGateRegBits, false)
}  // namespace aerhip
