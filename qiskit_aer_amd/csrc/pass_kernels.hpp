// The pass kernels the engine launches, declared here and compiled in
// translation units of their own (pass_*.hip), which hipcc builds in parallel.
#pragma once

#include "batch.hpp"
#include "gate_pass.hpp"
#include "reg_pass.hpp"
#include "tile_pass.hpp"

namespace aerhip {

constexpr uint32_t kTileBitsC128 = 11;  // 2^11 x 16 B = 32 KiB of LDS
constexpr uint32_t kTileBitsC64 = 12;   // 2^12 x 8 B  = 32 KiB of LDS

constexpr uint32_t kGateTileC128 = 12;  // 2^12 x 8 B = 32 KiB of LDS per component
constexpr uint32_t kGateRegBits = 4;
static_assert(kGateTileC128 == kTileBitsC64, "gate passes of both types launch workgroups of one size");
static_assert(kGateTileC128 == kTileBitsC128 + 1, "a complex128 gate tile fills two probe partials");

#define AERHIP_REG_PASS(EXT, T, B, R, V, WIDE)                                                        \
  EXT template __global__ void k_reg_pass<T, B, R, V, WIDE>(                                          \
      cx<T> *__restrict__, const PassDesc *__restrict__, const ROp<T> *__restrict__,                     \
      const TileOp *__restrict__, const cx<double> *__restrict__, double *__restrict__, uint64_t,        \
      uint32_t, uint32_t, uint32_t);
#define AERHIP_BATCH(EXT, T, B, R, V)                                                                    \
  EXT template __global__ void k_batch<T, B, R, V>(                                                      \
      cx<T> *__restrict__, const BatchCircuit *__restrict__, const BatchGroups, uint32_t,                \
      const PassDesc *__restrict__, const ROp<T> *__restrict__, const TileOp *__restrict__,              \
      const cx<double> *__restrict__, double *__restrict__);

#define AERHIP_GATE_PASS(EXT, T, B, R, PROBES)                                                           \
  EXT template __global__ void k_gate_pass<T, B, R, PROBES>(                                             \
      cx<T> *__restrict__, const PassDesc *__restrict__, const ROp<T> *__restrict__,                     \
      const cx<double> *__restrict__, double *__restrict__, uint64_t, uint32_t, uint32_t, uint32_t);

AERHIP_GATE_PASS(extern, double, kGateTileC128, kGateRegBits, false)
AERHIP_GATE_PASS(extern, double, kGateTileC128, kGateRegBits, true)
AERHIP_GATE_PASS(extern, float, kTileBitsC64, kGateRegBits, false)
AERHIP_GATE_PASS(extern, float, kTileBitsC64, kGateRegBits, true)
AERHIP_REG_PASS(extern, double, kTileBitsC128, 3, V_LEAN, false)
AERHIP_REG_PASS(extern, double, kTileBitsC128, 3, V_LEAN, true)
AERHIP_REG_PASS(extern, double, kTileBitsC128, 3, V_GATES, false)
AERHIP_REG_PASS(extern, double, kTileBitsC128, 3, V_PROBES, false)
AERHIP_REG_PASS(extern, double, kTileBitsC128, 3, V_FULL, false)
AERHIP_REG_PASS(extern, double, kTileBitsC128, 4, V_LEAN, false)
AERHIP_REG_PASS(extern, double, kTileBitsC128, 4, V_FULL, false)
AERHIP_REG_PASS(extern, float, kTileBitsC64, 4, V_LEAN, false)
AERHIP_REG_PASS(extern, float, kTileBitsC64, 4, V_GATES, false)
AERHIP_REG_PASS(extern, float, kTileBitsC64, 4, V_FULL, false)
AERHIP_REG_PASS(extern, float, kTileBitsC64, 5, V_LEAN, false)
AERHIP_REG_PASS(extern, float, kTileBitsC64, 5, V_FULL, false)
AERHIP_BATCH(extern, double, kTileBitsC128, 3, V_PROBES)
AERHIP_BATCH(extern, double, kTileBitsC128, 3, V_FULL)
AERHIP_BATCH(extern, float, kTileBitsC64, 4, V_FULL)

}  // namespace aerhip
