// Batched circuits (gfx950).
//
// Many independent statevectors of different sizes advance together: pass p of
// every circuit that has one is a single launch, with one workgroup per tile.
// The circuits are ordered by size, then by their number of passes, so that the
// circuits of one size that are still running are a range (BatchGroup) and a
// workgroup finds its circuit and tile from its index.  One workgroup per
// circuit instead leaves the device waiting for the largest ones: 512 circuits
// of 10 to 20 qubits with 64 Pauli strings each took 192 ms that way (with a
// sweep per string), 18 ms this way.
#pragma once

#include "reg_pass.hpp"

namespace aerhip {

struct BatchCircuit {
  uint64_t sv_off;      // first amplitude of the circuit's state in the batch buffer
  uint32_t num_qubits;
  uint32_t pass_begin;  // passes[pass_begin .. + pass_count)
  uint32_t pass_count;
  uint32_t tile_log;    // log2 of its tiles
};

// Probes a pass of a circuit of several tiles may hold.  Their partials stand in
// memory during the launch, a double per tile: 256 are 1/16 of the state.  On 28
// qubits (complex128) 39 probes add 1.0 ms to a sweep of 0.7, so that cutting a
// pass at 256 adds a tenth to it.
constexpr uint32_t kBatchProbes = 256;

// Circuits [first, first + count) of one size, whose tiles are workgroups
// begin .. begin + (count << tile_log).
struct BatchGroup {
  uint32_t first, begin, tile_log;
};
constexpr uint32_t kBatchGroups = 40;  // circuits have 1 to 40 qubits
struct BatchGroups {
  uint32_t n;
  BatchGroup g[kBatchGroups];
};

// |0> in every state (buffer zeroed first).
template <typename T>
__global__ void k_batch_ones(cx<T> *__restrict__ states, const BatchCircuit *__restrict__ circ, uint64_t count) {
  const uint64_t i = blockIdx.x * (uint64_t)kThreads + threadIdx.x;
  if (i < count) states[circ[i].sv_off] = mk<T>(1, 0);
}

// Pass p of the circuits of `groups`.  V_PROBES runs register passes of lean
// ops and probes, V_FULL the others (PassDesc::batch_class says which).
template <typename T, int B, int R, int V>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(reg_pass_waves<T, B, R>()))) void k_batch(
    cx<T> *__restrict__ states, const BatchCircuit *__restrict__ circ, const BatchGroups groups, uint32_t p,
    const PassDesc *__restrict__ passes, const ROp<T> *__restrict__ rops, const TileOp *__restrict__ tops,
    const cx<double> *__restrict__ pool, double *__restrict__ partial) {
  static_assert((1 << (B - R)) == kThreads, "register passes and LDS passes share the workgroup");
  static_assert(V == V_PROBES || V == V_FULL, "the batch's two classes");
  __shared__ cx<T> lds[1 << B];
  // the LDS-pass offset table and the register passes' staged tables never
  // live at the same time: one array holds either
  __shared__ __align__(16) unsigned char aux_lds[kDiagLdsBytes > 256 * sizeof(uint64_t) ? kDiagLdsBytes
                                                                                         : 256 * sizeof(uint64_t)];
  uint64_t *hioff = reinterpret_cast<uint64_t *>(aux_lds);
  cx<double> *dlt = reinterpret_cast<cx<double> *>(aux_lds);
  __shared__ cx<T> mat[16];
  __shared__ uint32_t doff[32];
  __shared__ double red[red_doubles(kThreads / 64)];
  const uint32_t w = static_cast<uint32_t>(xcd_tile(blockIdx.x, gridDim.x));
  uint32_t g = 0;
  while (g + 1 < groups.n && w >= groups.g[g + 1].begin) ++g;
  const uint32_t tl = groups.g[g].tile_log, r = w - groups.g[g].begin;
  const BatchCircuit &c = circ[groups.g[g].first + (r >> tl)];
  const uint64_t t = r & ((1u << tl) - 1u);
  const PassDesc *pd = passes + c.pass_begin + p;
  if (pd->batch_class != (V == V_FULL ? 1u : 0u)) return;
  cx<T> *sv = states + c.sv_off;
  const ProbeSink sink{partial + pd->part_off, t, 1ull << tl};
  if constexpr (V == V_PROBES) {
    reg_tile<T, B, R, 16, V_PROBES>(sv, pd, rops, tops, pool, sink, t, lds, mat, doff, red, dlt);
  } else if (pd->kind == 2) {
    reg_tile<T, B, R, 16, V_FULL>(sv, pd, rops, tops, pool, sink, t, lds, mat, doff, red, dlt);
  } else if (pd->kind == 4) {
    const uint32_t more = pd->ncomp - tl;  // a permutation's tiles are smaller
    for (uint64_t i = 0; i < (1ull << more); ++i)
      qperm_tile<T, B - 1, kThreads>(sv, pd, tops + pd->op_begin, (t << more) + i, lds);
  } else if (pd->kind == 3) {
    probe_sweep<T, kThreads, (1 << B) / kThreads>(sv, tops + pd->op_begin, pd->nops, pd->nb, sink, t, red);
  } else {
    lds_tile<T, kThreads, B, 16>(sv, pd, tops, pool, sink, t, lds, hioff, mat, doff, red);
  }
}

}  // namespace aerhip
