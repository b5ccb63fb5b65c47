// Readout kernels of the engine: row sums of FP64 partials, marginal
// probabilities and the sampling index.  Included by engine.hip alone.
#pragma once

#include "batch.hpp"
#include "kernels.hpp"
#include "tile_pass.hpp"

namespace aerhip {

// Sums `cols` consecutive partials of each of `rows` rows, in an order fixed by
// `cols` alone.  Short rows: one thread per row, in sequence.  Others: one
// workgroup per row, whose thread t adds columns t, t + NT, ... before the
// workgroup's tree, so a row's loads are in flight together (one thread per
// row waits out a memory latency per partial).  Measured: 55 rows of 2^17
// partials 12.2 ms with one thread per row, 20 us with 1024 threads per row.
__global__ void k_sum_rows_short(const double *__restrict__ partial, uint64_t rows, uint32_t cols,
                                 double *__restrict__ out) {
  const uint64_t r = blockIdx.x * (uint64_t)kThreads + threadIdx.x;
  if (r >= rows) return;
  double s = 0;
  for (uint32_t c = 0; c < cols; ++c) s += partial[r * cols + c];
  out[r] = s;
}

template <int NT>
__global__ __launch_bounds__(NT) void k_sum_rows(const double *__restrict__ partial, uint32_t cols,
                                                 double *__restrict__ out) {
  __shared__ double red[NT / 64];
  const double *row = partial + static_cast<uint64_t>(blockIdx.x) * cols;
  double s[8] = {};
  uint32_t c = threadIdx.x;
  for (; c + 7u * NT < cols; c += 8u * NT) {
#pragma unroll
    for (int k = 0; k < 8; ++k) s[k] += row[c + static_cast<uint32_t>(k) * NT];
  }
  for (; c < cols; c += NT) s[0] += row[c];
  const double v = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
  const double t = block_sum_nt<NT>(v, red);
  if (threadIdx.x == 0) out[blockIdx.x] = t;
}

// A workgroup pays for its barriers and its tree from 32 partials per row on;
// from 8192 on a row feeds 1024 threads.
inline void sum_rows(const double *partial, uint64_t rows, uint32_t cols, double *out, hipStream_t stream) {
  if (rows == 0) return;
  if (cols < 32 || rows > (1ull << 22))
    k_sum_rows_short<<<static_cast<uint32_t>((rows + kThreads - 1) / kThreads), kThreads, 0, stream>>>(partial, rows, cols, out);
  else if (cols < 8192)
    k_sum_rows<kThreads><<<static_cast<uint32_t>(rows), kThreads, 0, stream>>>(partial, cols, out);
  else
    k_sum_rows<1024><<<static_cast<uint32_t>(rows), 1024, 0, stream>>>(partial, cols, out);
}

// The values of the probes in pass p of every circuit, each the sum of its tile
// partials: gridDim.y workgroups per circuit, a wave per probe.
__global__ __launch_bounds__(kThreads) void k_batch_sums(const BatchCircuit *__restrict__ circ, uint32_t p,
                                                      const PassDesc *__restrict__ passes,
                                                      const uint32_t *__restrict__ slots,
                                                      const double *__restrict__ partial,
                                                      double *__restrict__ values) {
  const BatchCircuit &c = circ[blockIdx.x];
  if (p >= c.pass_count) return;
  const PassDesc &pd = passes[c.pass_begin + p];
  const uint64_t tiles = 1ull << c.tile_log;
  constexpr uint32_t NW = kThreads / 64;
  for (uint32_t i = blockIdx.y * NW + (threadIdx.x >> 6); i < pd.probes; i += gridDim.y * NW) {
    const double *row = partial + pd.part_off + i * tiles;
    double s = 0;
    for (uint64_t k = threadIdx.x & 63u; k < tiles; k += 64) s += row[k];
    s = wave_sum(s);
    if ((threadIdx.x & 63u) == 0) values[slots[pd.probe_at + i]] = s;
  }
}

// Marginal probabilities, QubitVector::probabilities(qubits)
// (qubitvector.hpp:2107-2143).  Bound by the HBM read, so every wave reads runs
// of 2^low (64) consecutive amplitudes whichever qubits are measured: lanes are
// the `low` lowest qubits; a wave takes one value of the measured qubits above
// them and `len` consecutive values of the unmeasured ones (a chunk), adds up
// |psi|^2 per lane, and sums over the unmeasured lane qubits at the end.
// partial[outcome * nchunk + chunk].  12 random qubits of 29 in complex64:
// 4.50 ms when threads ran over the unmeasured qubits (a cache line per
// amplitude), 0.73 ms (5.9 TB/s) this way.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_marginal(const cx<T> *__restrict__ sv, const MarginalDesc md,
                                                       uint32_t low, uint64_t items, uint64_t len,
                                                       double *__restrict__ partial) {
  const uint32_t lane = threadIdx.x & 63u, nq = md.nq;
  const uint64_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6));
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * (kThreads / 64);
  const bool active = lane < (1u << low);
  uint64_t mask = 0;
  for (uint32_t i = 0; i < nq; ++i) mask |= 1ull << md.sorted[i];
  const uint64_t lowmask = (1ull << low) - 1ull, fixed = mask | lowmask;
  const uint32_t chunk_log = 31u - __builtin_clz(md.nchunk);
  for (uint64_t item = wave; item < items; item += nwaves) {
    const uint64_t chunk = item & (md.nchunk - 1u);
    uint64_t mh = item >> chunk_log, base = 0;  // bits of mh on the measured high qubits
    uint64_t k0 = chunk * len, idx = 0;         // bits of k0 on the unmeasured high qubits
    for (uint32_t i = 0; i < nq; ++i) {
      const uint32_t q = md.sorted[i];
      if (q < low) continue;
      base |= (mh & 1ull) << q;
      mh >>= 1;
    }
    for (uint32_t q = low; k0; ++q) {
      if ((mask >> q) & 1ull) continue;
      idx |= (k0 & 1ull) << q;
      k0 >>= 1;
    }
    double s[8] = {};  // eight short sums: less rounding than one long one
    if (active) {
      const cx<T> *p = sv + (base | lane);
      uint64_t k = 0;
      for (; k + 8 <= len; k += 8) {
        cx<T> a[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          a[u] = p[idx];
          idx = ((idx | fixed) + 1ull) & ~fixed;  // the next value of the unmeasured high qubits
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) s[u] += prob(a[u]);
      }
      for (; k < len; ++k) {
        s[0] += prob(p[idx]);
        idx = ((idx | fixed) + 1ull) & ~fixed;
      }
    }
    double acc = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    for (uint32_t b = 0; b < low; ++b)
      if (!((mask >> b) & 1ull)) acc += __shfl_xor(acc, 1 << b, 64);
    if (active && !(lane & ~mask)) {
      const uint64_t at = base | lane;
      uint64_t m = 0;
      for (uint32_t i = 0; i < nq; ++i) m |= ((at >> md.order[i]) & 1ull) << i;
      partial[m * md.nchunk + chunk] = acc;
    }
  }
}

// Sum of |psi|^2 over consecutive runs of 2^sbits amplitudes, one wave per run.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_run_sums(const cx<T> *__restrict__ sv,
                                                       uint32_t sbits, uint64_t nruns,
                                                       double *__restrict__ out) {
  const uint64_t run = blockIdx.x * (uint64_t)(kThreads / 64) + (threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63;
  if (run >= nruns) return;
  const uint64_t len = 1ull << sbits;
  const uint64_t b = run << sbits;
  double acc = 0;
  for (uint64_t j = lane; j < len; j += 64) acc += prob(sv[b + j]);
  acc = wave_sum(acc);
  if (lane == 0) out[run] = acc;
}

// The sampling index: cumulative sums in the order of the reference's
// QubitVector::sample_measure (qubitvector.hpp:2149-2228), whose index blocks
// hold 2^(n-isz) amplitudes.  Each block's runs are added one after the other
// (k_block_sums), the blocks likewise (k_prefix_blocks: upto[j] = sum up to and
// including block j), and the runs of block j on top of upto[j - 1]
// (k_prefix_runs, in place: runs[r] = sum up to and including run r).  One
// thread adds, as the order is the reference's; the values pass through LDS so
// that an addition costs its own latency and not a load's.
constexpr uint32_t kScan = 2048;

// s + v[0], s + v[0] + v[1], ... over v[0..m), in order; with `keep` the sums
// replace the values.  16 values at a time are in registers before the first
// of them is written back, so that no LDS read waits for a write.
template <bool keep>
__device__ __forceinline__ double scan_in_order(double *v, uint32_t m, double s) {
  uint32_t i = 0;
  for (; i + 16 <= m; i += 16) {
    double a[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) a[k] = v[i + k];
#pragma unroll
    for (int k = 0; k < 16; ++k) a[k] = (s += a[k]);
    if constexpr (keep) {
#pragma unroll
      for (int k = 0; k < 16; ++k) v[i + k] = a[k];
    }
  }
  for (; i < m; ++i) {
    s += v[i];
    if constexpr (keep) v[i] = s;
  }
  return s;
}

__global__ __launch_bounds__(kThreads) void k_block_sums(const double *__restrict__ runs, uint64_t rpb,
                                                        double *__restrict__ blocks) {
  __shared__ double v[kScan];
  const double *p = runs + blockIdx.x * rpb;
  double s = 0;
  for (uint64_t o = 0; o < rpb; o += kScan) {
    const uint32_t m = static_cast<uint32_t>(min(rpb - o, static_cast<uint64_t>(kScan)));
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += kThreads) v[i] = p[o + i];
    __syncthreads();
    if (threadIdx.x == 0) s = scan_in_order<false>(v, m, s);
  }
  if (threadIdx.x == 0) blocks[blockIdx.x] = s;
}

__global__ __launch_bounds__(kThreads) void k_prefix_blocks(const double *__restrict__ blocks, uint64_t nblocks,
                                                           double *__restrict__ upto) {
  __shared__ double v[kScan];
  double s = 0;
  for (uint64_t o = 0; o < nblocks; o += kScan) {
    const uint32_t m = static_cast<uint32_t>(min(nblocks - o, static_cast<uint64_t>(kScan)));
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += kThreads) v[i] = blocks[o + i];
    __syncthreads();
    if (threadIdx.x == 0) s = scan_in_order<true>(v, m, s);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += kThreads) upto[o + i] = v[i];
  }
}

__global__ __launch_bounds__(kThreads) void k_prefix_runs(double *__restrict__ runs, uint64_t rpb,
                                                         const double *__restrict__ upto) {
  __shared__ double v[kScan];
  double *p = runs + blockIdx.x * rpb;
  double s = blockIdx.x ? upto[blockIdx.x - 1] : 0.0;
  for (uint64_t o = 0; o < rpb; o += kScan) {
    const uint32_t m = static_cast<uint32_t>(min(rpb - o, static_cast<uint64_t>(kScan)));
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += kThreads) v[i] = p[o + i];
    __syncthreads();
    if (threadIdx.x == 0) s = scan_in_order<true>(v, m, s);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += kThreads) p[o + i] = v[i];
  }
}

// First i < n with rnd < sums[i] (non-decreasing, NaN from some entry on or
// nowhere), n if there is none.
__device__ __forceinline__ uint64_t first_above(const double *__restrict__ sums, uint64_t n, double rnd) {
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (rnd >= sums[mid]) lo = mid + 1;
    else hi = mid;
  }
  return lo < n && rnd < sums[lo] ? lo : n;
}

// Draws: the index block and the run by binary search in the cumulative sums,
// then the run's amplitudes one after the other in the reference's order.  A
// wave takes 16 draws: for each it loads 64 consecutive probabilities (one
// coalesced read) into LDS, then lane q adds those of draw q in sequence and
// counts how many sums stay at or below it, while the next 64 are on their way.
// 10 000 draws from 2^29 amplitudes: 514 us with the three levels walked entry
// by entry, 190 us with one draw per thread and 16 loads at a time, 37 us here.
constexpr uint32_t kDraws = 16;

template <typename T>
__global__ __launch_bounds__(64) void k_sample(const cx<T> *__restrict__ sv, uint64_t size, uint32_t isz,
                                              uint32_t sbits, const double *__restrict__ upto,
                                              const double *__restrict__ runs, const double *__restrict__ rnds,
                                              uint64_t shots, uint64_t *__restrict__ out) {
  __shared__ double v[kDraws][65];
  const uint32_t lane = threadIdx.x, q = lane & (kDraws - 1u);
  const uint64_t s = blockIdx.x * static_cast<uint64_t>(kDraws) + q;
  const uint64_t last = size - 1;
  bool done = s >= shots;
  const double rnd = done ? 0.0 : rnds[s];
  const uint64_t nblocks = 1ull << isz, loop = size >> isz;
  double p = 0;
  uint64_t sample = 0;
  if (!done) {
    const uint64_t j = first_above(upto, nblocks, rnd);
    if (j == nblocks) {  // rnd beyond the accumulated total: last amplitude
      sample = last;
      done = true;
    } else {
      p = j ? upto[j - 1] : 0.0;
      sample = j * loop;
      const uint64_t rpb = loop >> sbits;  // runs per block
      if (rpb > 1) {
        const double *r = runs + j * rpb;
        const uint64_t k = first_above(r, rpb - 1, rnd);
        if (k) p = r[k - 1];
        sample += k << sbits;
      }
    }
  }
  if (!(upto[nblocks - 1u] >= 0.0)) {
    // A NaN among the amplitudes: a window of 64 that reaches into later index
    // blocks would count it, so these draws add one amplitude after the other.
    if (!done)
      for (; sample < last; ++sample) {
        p += prob(sv[sample]);
        if (rnd < p) break;
      }
    if (lane < kDraws && s < shots) out[s] = sample;
    return;
  }
  cx<T> a[kDraws];
  auto load = [&](uint64_t from) {
#pragma unroll
    for (uint32_t d = 0; d < kDraws; ++d) {
      const uint64_t at = static_cast<uint64_t>(__shfl(static_cast<long long>(from), static_cast<int>(d), 64));
      a[d] = sv[min(at + lane, last)];
    }
  };
  load(sample);
  while (__ballot(!done)) {
#pragma unroll
    for (uint32_t d = 0; d < kDraws; ++d) v[d][lane] = prob(a[d]);
    __syncthreads();
    load(sample + 64);
    if (!done) {
      const uint32_t n = static_cast<uint32_t>(min(last - sample, static_cast<uint64_t>(64)));
      uint32_t below = 0;
#pragma unroll 16
      for (uint32_t i = 0; i < 64; ++i) {
        p += v[q][i];
        below += rnd < p ? 0u : 1u;
      }
      if (below < n) {
        sample += below;
        done = true;
      } else {
        sample += n;
        done = n < 64 || sample >= last;
      }
    }
    __syncthreads();
  }
  if (lane < kDraws && s < shots) out[s] = sample;
}

// Linear scan for small states (END < 2^isz in the reference).
template <typename T>
__global__ void k_sample_linear(const cx<T> *__restrict__ sv, uint64_t size,
                                const double *__restrict__ rnds, uint64_t shots,
                                uint64_t *__restrict__ out) {
  const uint64_t s = blockIdx.x * (uint64_t)kThreads + threadIdx.x;
  if (s >= shots) return;
  const double rnd = rnds[s];
  double p = 0;
  uint64_t sample = 0;
  for (; sample < size - 1; ++sample) {
    p += prob(sv[sample]);
    if (rnd < p) break;
  }
  out[s] = sample;
}

}  // namespace aerhip
