// Gate pass on large tiles (gfx950): the register pass for long programs of
// gates, with twice the amplitudes per thread.
//
// A pass is one read and one write of the state for as many gates as its tile
// qubits allow, so a tile of one more qubit means fewer passes, and one more
// register bit means fewer layout changes.  Both cost registers: 2^R complex128
// amplitudes are 64 VGPRs at R = 4, so ops work in place on the one copy (no
// second bank), each on a few amplitudes at a time.  Layout changes go through
// LDS one component after the other, so a tile of 2^12 complex128 amplitudes
// needs 32 KiB and the occupancy is that of the smaller tile.
//
// The op loop is an interpreter: host-computed codes name the op together with
// its register bits, and one comparison tree finds it.
//
// complex128 is bound by the FP64 units: the 30-qubit brickwork at fusion width 2
// runs 24 passes of 10.1 ms (34.4 GB each, 3.4 TB/s), 83 % of whose cycles issue
// vector instructions (3861 per wave, 3140 of them FMAs of 4x4 gates), at 119
// VGPRs and four waves per SIMD.  Register passes on 2^11 tiles take 30 passes of
// 14.1 ms for it: 425 against 244 ms a step.  At an earlier state of 269 ms, three
// waves (150 VGPRs) took 281 ms, five (96 VGPRs, spills) 390.
//
// complex64 runs its 2x2, 4x4 and 8x8 gates on MFMA, at 94 VGPRs and five waves:
// layers of SU(4) on 29 qubits 88 -> 60.5 ms (16 passes of 3.7 ms, 42 % of the
// cycles issuing vector instructions), brickwork of 2x2 gates on 27 24.8 -> 18.3.
#pragma once

#include "reg_pass.hpp"

namespace aerhip {

// Code of an op (ROp::code): group and register bits.
enum GateCode : uint32_t {
  C_NOP = 0x00,
  C_U1 = 0x10,       // + b: 2x2 gate on register bit b
  C_U2 = 0x20,       // + index of the register bits b0 < b1
  C_X = 0x30,        // + b: X on register bit b of every lane
  C_XC = 0x38,       // + b: X where the lane's predicate holds
  C_U1C = 0x40,      // + b: 2x2 gate where the predicate holds
  C_Y = 0x48,        // + b: Y where the predicate holds
  C_CXR = 0x50,      // + 4 c + t: register moves
  C_PHASE = 0x60,
  C_D1 = 0x61,
  C_DIAGF = 0x62,
  C_RELAYOUT = 0x63,
  C_DIAGK = 0x64,
  C_PROBE = 0x65,    // a run of probes
  C_U1R = 0x68,      // + b: 2x2 gate with real entries (complex128)
  C_SWAP = 0x70,     // + index of the register bits b0 < b1
  C_U3 = 0x78,       // + b: 8x8 gate on the register bits but b
};

// Index of a pair of register bits b0 < b1.
constexpr uint32_t pair_index(uint32_t b0, uint32_t b1) { return b1 * (b1 - 1) / 2 + b0; }

// The code of a register op; U2 ops come with a < b.
inline uint32_t gate_code(const ROp<double> &r, bool single) {
  switch (r.kind & ~F_ALL) {
    case Q_U1: case Q_U1X: {
      const bool real = r.u.m[1] == 0 && r.u.m[3] == 0 && r.u.m[5] == 0 && r.u.m[7] == 0;
      return (real && !single ? C_U1R : C_U1) + r.a;
    }
    case Q_U2: return C_U2 + pair_index(r.a, r.b);
    case Q_X: return (r.cl ? C_XC : C_X) + r.a;
    case Q_U1C: return C_U1C + r.a;
    case Q_Y: return C_Y + r.a;
    case Q_CXR: return C_CXR + 4 * r.a + r.b;
    case Q_PHASE: return C_PHASE;
    case Q_D1: return C_D1;
    case Q_DIAGF: return C_DIAGF;
    case Q_DIAGK: return C_DIAGK;
    case Q_PROBE: return C_PROBE;
    case Q_SWAP: return C_SWAP + pair_index(r.a, r.b);
    case Q_U3: return C_U3 + r.a;
    case Q_RELAYOUT: return C_RELAYOUT;
    default: return C_NOP;
  }
}

// (p, q) <- M (p, q), M column major (u00, u10, u01, u11).  The last FMA of
// each component writes over the amplitude it reads, so the pair needs four
// temporaries and no moves.
template <typename T>
__device__ __forceinline__ void g_u1(cx<T> &p, cx<T> &q, const cx<T> (&m)[4]) {
  T tx = -m[2].x * q.x, ty = -m[2].x * q.y, ux = -m[1].x * p.x, uy = -m[1].x * p.y;
  tx = fma_t(m[2].y, q.y, tx);
  ty = fma_t(-m[2].y, q.x, ty);
  ux = fma_t(m[1].y, p.y, ux);
  uy = fma_t(-m[1].y, p.x, uy);
  tx = fma_t(m[0].y, p.y, tx);
  ty = fma_t(-m[0].y, p.x, ty);
  ux = fma_t(m[3].y, q.y, ux);
  uy = fma_t(-m[3].y, q.x, uy);
  p.x = fma_t(m[0].x, p.x, -tx);
  p.y = fma_t(m[0].x, p.y, -ty);
  q.x = fma_t(m[3].x, q.x, -ux);
  q.y = fma_t(m[3].x, q.y, -uy);
}

template <typename T, int NR, int b>
__device__ __forceinline__ void g_u1b(Amps<T, NR> &a, const cx<T> (&u)[4]) {
#pragma unroll
  for (int k = 0; k < NR / 2; ++k) g_u1(a.v[pair_lo<b>(k)], a.v[pair_lo<b>(k) | (1 << b)], u);
}

// The same with real entries (m0, m1, m2, m3): half the work.  RY and H are
// such gates; the forward passes of a 20-qubit ansatz of RY and RZ, 16 states: 0.95 -> 0.81 ms each.
template <typename T, int NR, int b>
__device__ __forceinline__ void g_u1r(Amps<T, NR> &a, const T (&m)[4]) {
#pragma unroll
  for (int k = 0; k < NR / 2; ++k) {
    cx<T> &p = a.v[pair_lo<b>(k)], &q = a.v[pair_lo<b>(k) | (1 << b)];
    T tx = -m[2] * q.x, ty = -m[2] * q.y, ux = -m[1] * p.x, uy = -m[1] * p.y;
    asm volatile("" : "+v"(tx), "+v"(ty), "+v"(ux), "+v"(uy));  // keeps the negation in the last FMA
    p.x = fma_t(m[0], p.x, -tx);
    p.y = fma_t(m[0], p.y, -ty);
    q.x = fma_t(m[3], q.x, -ux);
    q.y = fma_t(m[3], q.y, -uy);
  }
}

// complex64 2x2 gate with MFMA: v_mfma_f32_4x4x1 runs 16 blocks of 4 x 4 (lanes
// 4k .. 4k + 3 form block k), of which the broadcast controls (16 blocks, block
// k) let all take column k of the matrix: lane 4k + i of the one register `A`
// holds entry (i, k) of the real 4x4 form.  Four accumulating issues leave the
// pair's four output components in the lane's accumulator.
template <int NR, int b>
__device__ __forceinline__ void g_u1b_mfma(Amps<float, NR> &a, float A) {
  constexpr f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  constexpr int G = 4;  // pairs whose accumulation chains interleave
#pragma unroll
  for (int g = 0; g < NR / 2; g += G) {
    f32x4 acc[G];
    // The |1> amplitude's columns come first: U3 and U2 have a real entry (0, 0),
    // whose one product then joins last and is rounded once.  20 layers of
    // brickwork on 23 qubits end 9.1e-7 of the norm off so, 9.5e-7 with |0> first
    // (register passes: 9.3e-7).
#pragma unroll
    for (int p = 0; p < G; ++p)
      acc[p] = __builtin_amdgcn_mfma_f32_4x4x1f32(A, a.v[pair_lo<b>(g + p) | (1 << b)].x, zero, 4, 2, 0);
#pragma unroll
    for (int p = 0; p < G; ++p)
      acc[p] = __builtin_amdgcn_mfma_f32_4x4x1f32(A, a.v[pair_lo<b>(g + p) | (1 << b)].y, acc[p], 4, 3, 0);
#pragma unroll
    for (int p = 0; p < G; ++p) acc[p] = __builtin_amdgcn_mfma_f32_4x4x1f32(A, a.v[pair_lo<b>(g + p)].x, acc[p], 4, 0, 0);
#pragma unroll
    for (int p = 0; p < G; ++p) acc[p] = __builtin_amdgcn_mfma_f32_4x4x1f32(A, a.v[pair_lo<b>(g + p)].y, acc[p], 4, 1, 0);
#pragma unroll
    for (int p = 0; p < G; ++p) {
      a.v[pair_lo<b>(g + p)] = mk<float>(acc[p][0], acc[p][1]);
      a.v[pair_lo<b>(g + p) | (1 << b)] = mk<float>(acc[p][2], acc[p][3]);
    }
  }
}

// complex64 4x4 gate with MFMA: the real 8x8 form in two halves of four rows,
// each a chain of eight issues per group of four amplitudes, at twice the rate
// of FMAs on the vector ALU.  Lane 4 (8h + k) + i of `A` holds entry (4h + i, k).
template <int b0, int b1, int NR, int k = 0>
__device__ __forceinline__ void g_u2_chain(const Amps<float, NR> &a, int g, float A, f32x4 (&acc)[2][2]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int j = pair_lo<b1>(pair_lo<b0>(g + q)) | (k & 2 ? 1 << b0 : 0) | (k & 4 ? 1 << b1 : 0);
    const float v = k & 1 ? a.v[j].y : a.v[j].x;
    acc[q][0] = __builtin_amdgcn_mfma_f32_4x4x1f32(A, v, acc[q][0], 4, k, 0);
    acc[q][1] = __builtin_amdgcn_mfma_f32_4x4x1f32(A, v, acc[q][1], 4, 8 + k, 0);
  }
  if constexpr (k < 7) g_u2_chain<b0, b1, NR, k + 1>(a, g, A, acc);
}

template <int NR, int b0, int b1>
__device__ __forceinline__ void g_u2_mfma(Amps<float, NR> &a, float A) {
  constexpr f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int g = 0; g < NR / 4; g += 2) {  // two groups: four chains interleave
    f32x4 acc[2][2] = {{zero, zero}, {zero, zero}};
    g_u2_chain<b0, b1, NR>(a, g, A, acc);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int j = pair_lo<b1>(pair_lo<b0>(g + q));
#pragma unroll
      for (int r = 0; r < 4; ++r)
        a.v[j | (r & 1 ? 1 << b0 : 0) | (r & 2 ? 1 << b1 : 0)] =
            mk<float>(acc[q][r >> 1][2 * (r & 1)], acc[q][r >> 1][2 * (r & 1) + 1]);
    }
  }
}

// 4x4 gate on register bits b0 (matrix bit 0) < b1, column major.
template <typename T, int NR, int b0, int b1>
__device__ __forceinline__ void g_u2(Amps<T, NR> &a, const cx<T> (&m)[16]) {
#pragma unroll
  for (int p = 0; p < NR / 4; ++p) {
    __builtin_amdgcn_sched_barrier(0);
    const int j = pair_lo<b1>(pair_lo<b0>(p));
    const int i[4] = {j, j | (1 << b0), j | (1 << b1), j | (1 << b0) | (1 << b1)};
    T tx[4], ty[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int f = r == 0 ? 1 : 0;
      tx[r] = -m[r + 4 * f].x * a.v[i[f]].x;
      ty[r] = -m[r + 4 * f].x * a.v[i[f]].y;
      tx[r] = fma_t(m[r + 4 * f].y, a.v[i[f]].y, tx[r]);
      ty[r] = fma_t(-m[r + 4 * f].y, a.v[i[f]].x, ty[r]);
#pragma unroll
      for (int c = f + 1; c < 4; ++c) {
        if (c == r) continue;
        tx[r] = fma_t(-m[r + 4 * c].x, a.v[i[c]].x, tx[r]);
        ty[r] = fma_t(-m[r + 4 * c].x, a.v[i[c]].y, ty[r]);
        tx[r] = fma_t(m[r + 4 * c].y, a.v[i[c]].y, tx[r]);
        ty[r] = fma_t(-m[r + 4 * c].y, a.v[i[c]].x, ty[r]);
      }
      tx[r] = fma_t(m[5 * r].y, a.v[i[r]].y, tx[r]);
      ty[r] = fma_t(-m[5 * r].y, a.v[i[r]].x, ty[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a.v[i[r]].x = fma_t(m[5 * r].x, a.v[i[r]].x, -tx[r]);
      a.v[i[r]].y = fma_t(m[5 * r].x, a.v[i[r]].y, -ty[r]);
    }
  }
}

// Register p (0 or 1) of those with the bits other than `omit` clear, and the
// offset of the group's amplitude i from it.
template <int omit>
constexpr int u3_base(int p) { return p << omit; }
template <int omit>
constexpr int u3_off(int i) { return (i & ((1 << omit) - 1)) | (i >> omit) << (omit + 1); }

// 8x8 gate on the register bits but `omit`, rows of m: as g_u2, a row of the
// matrix in scalar registers at a time.
template <typename T, int NR, int omit>
__device__ __forceinline__ void g_u3(Amps<T, NR> &a, const cx<T> *__restrict__ m) {
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    T tx[8], ty[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      uint64_t at = 8 * r;
      asm volatile("" : "+s"(at));  // keeps the loads of the rows apart
      const cx<T> *mr = m + at;
      cx<T> row[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) row[c] = mr[c];
      const cx<T> v = a.v[u3_base<omit>(p) | u3_off<omit>(r)];
      tx[r] = row[r].y * v.y;
      ty[r] = -row[r].y * v.x;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        if (c == r) continue;
        const cx<T> w = a.v[u3_base<omit>(p) | u3_off<omit>(c)];
        tx[r] = fma_t(-row[c].x, w.x, tx[r]);
        ty[r] = fma_t(-row[c].x, w.y, ty[r]);
        tx[r] = fma_t(row[c].y, w.y, tx[r]);
        ty[r] = fma_t(-row[c].y, w.x, ty[r]);
      }
    }
    uint64_t at = 0;
    asm volatile("" : "+s"(at));
    const cx<T> *md = m + at;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      cx<T> &v = a.v[u3_base<omit>(p) | u3_off<omit>(r)];
      const T d = md[9 * r].x;
      v.x = fma_t(d, v.x, -tx[r]);
      v.y = fma_t(d, v.y, -ty[r]);
    }
  }
}

// complex64 8x8 gate with MFMA: the real 16x16 form in four quarters of four
// rows, quarter h from lane 4k + i of A[h] = entry (4h + i, k).
template <int omit, int NR, int k = 0>
__device__ __forceinline__ void g_u3_chain(const Amps<float, NR> &a, int p, const float (&A)[4], f32x4 (&acc)[4]) {
  const cx<float> w = a.v[u3_base<omit>(p) | u3_off<omit>(k >> 1)];
  const float v = k & 1 ? w.y : w.x;
#pragma unroll
  for (int h = 0; h < 4; ++h) acc[h] = __builtin_amdgcn_mfma_f32_4x4x1f32(A[h], v, acc[h], 4, k, 0);
  if constexpr (k < 15) g_u3_chain<omit, NR, k + 1>(a, p, A, acc);
}

template <int NR, int omit>
__device__ __forceinline__ void g_u3_mfma(Amps<float, NR> &a, const float (&A)[4]) {
  constexpr f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    f32x4 acc[4] = {zero, zero, zero, zero};
    g_u3_chain<omit, NR>(a, p, A, acc);
#pragma unroll
    for (int r = 0; r < 8; ++r)
      a.v[u3_base<omit>(p) | u3_off<omit>(r)] = mk<float>(acc[r >> 1][2 * (r & 1)], acc[r >> 1][2 * (r & 1) + 1]);
  }
}

// Exchanges two components.  Written out, because as a permutation of values it
// would tie the registers of the op loop's paths in knots: the compiler then
// keeps a second copy of the amplitudes and moves between the two at every op.
__device__ __forceinline__ void g_swap(double &x, double &y) {
  double t;
  asm volatile("v_mov_b64 %2, %0\n\tv_mov_b64 %0, %1\n\tv_mov_b64 %1, %2" : "+v"(x), "+v"(y), "=&v"(t));
}
__device__ __forceinline__ void g_swap(float &x, float &y) { asm volatile("v_swap_b32 %0, %1" : "+v"(x), "+v"(y)); }
template <typename T>
__device__ __forceinline__ void g_swap(cx<T> &p, cx<T> &q) {
  g_swap(p.x, q.x);
  g_swap(p.y, q.y);
}

// a <- f a
template <typename T>
__device__ __forceinline__ void g_mul(cx<T> &a, cx<T> f) {
  T t = f.y * a.y, u = -f.y * a.x;
  asm volatile("" : "+v"(t), "+v"(u));  // keeps the negation in the last FMA
  a.x = fma_t(f.x, a.x, -t);
  a.y = fma_t(f.x, a.y, -u);
}

template <typename T, int NR, int b>
__device__ __forceinline__ void g_x(Amps<T, NR> &a) {
#pragma unroll
  for (int k = 0; k < NR / 2; ++k) {
    const int j = pair_lo<b>(k);
    g_swap(a.v[j], a.v[j | (1 << b)]);
  }
}

// Exchanges p and q in the lanes of m: six moves a pair under the execution
// mask, where selects take eight.
__device__ __forceinline__ void g_swapm(cx<double> &p, cx<double> &q, uint64_t m) {
  uint64_t e;
  double t;
  asm volatile(
      "s_mov_b64 %5, exec\n\ts_and_b64 exec, exec, %6\n\t"
      "v_mov_b64 %4, %0\n\tv_mov_b64 %0, %1\n\tv_mov_b64 %1, %4\n\t"
      "v_mov_b64 %4, %2\n\tv_mov_b64 %2, %3\n\tv_mov_b64 %3, %4\n\t"
      "s_mov_b64 exec, %5"
      : "+v"(p.x), "+v"(q.x), "+v"(p.y), "+v"(q.y), "=&v"(t), "=&s"(e)
      : "s"(m)
      : "scc");
}
__device__ __forceinline__ void g_swapm(cx<float> &p, cx<float> &q, uint64_t m) {
  uint64_t e;
  asm volatile(
      "s_mov_b64 %4, exec\n\ts_and_b64 exec, exec, %5\n\t"
      "v_swap_b32 %0, %1\n\tv_swap_b32 %2, %3\n\t"
      "s_mov_b64 exec, %4"
      : "+v"(p.x), "+v"(q.x), "+v"(p.y), "+v"(q.y), "=&s"(e)
      : "s"(m)
      : "scc");
}

// X where the predicate holds: in the lanes of m and the registers of rb.  The
// 30-qubit brickwork at fusion width 2, with 52 of them: 248.5 -> 243.2 ms.
template <typename T, int NR, int b>
__device__ __forceinline__ void g_xc(Amps<T, NR> &a, uint64_t m, uint32_t rb) {
#pragma unroll
  for (int k = 0; k < NR / 2; ++k) {
    const int j = pair_lo<b>(k);
    g_swapm(a.v[j], a.v[j | (1 << b)], (rb >> j) & 1u ? m : 0);
  }
}

template <typename T, int NR, int b>
__device__ __forceinline__ void g_yc(Amps<T, NR> &a, uint32_t tlc, const RegIdx<NR> &ri, uint32_t cl, uint32_t cvl) {
#pragma unroll
  for (int k = 0; k < NR / 2; ++k) {
    const int j = pair_lo<b>(k), jj = j | (1 << b);
    const bool on = (tlc | (ri.at(j) & cl)) == cvl;
    const cx<T> p = a.v[j], q = a.v[jj];
    a.v[j] = csel(on, mk<T>(q.y, -q.x), p);
    a.v[jj] = csel(on, mk<T>(-p.y, p.x), q);
  }
}

template <typename T, int NR, int b0, int b1>
__device__ __forceinline__ void g_swapc(Amps<T, NR> &a, uint64_t m, uint32_t rb) {
#pragma unroll
  for (int k = 0; k < NR / 4; ++k) {
    const int j = pair_lo<b1>(pair_lo<b0>(k));
    g_swapm(a.v[j | (1 << b0)], a.v[j | (1 << b1)], (rb >> j) & 1u ? m : 0);
  }
}

template <typename T, int NR, int b>
__device__ __forceinline__ void g_u1c(Amps<T, NR> &a, uint32_t tlc, const RegIdx<NR> &ri, uint32_t cl, uint32_t cvl,
                                      const cx<T> (&m)[4]) {
#pragma unroll
  for (int k = 0; k < NR / 2; ++k) {
    const int j = pair_lo<b>(k), jj = j | (1 << b);
    const bool on = (tlc | (ri.at(j) & cl)) == cvl;
    cx<T> p = a.v[j], q = a.v[jj];
    g_u1(p, q, m);
    a.v[j] = csel(on, p, a.v[j]);
    a.v[jj] = csel(on, q, a.v[jj]);
  }
}

template <typename T, int NR, int c, int t>
__device__ __forceinline__ void g_cxr(Amps<T, NR> &a) {
#pragma unroll
  for (int j = 0; j < NR; ++j)
    if (((j >> c) & 1) && !((j >> t) & 1)) g_swap(a.v[j], a.v[j | (1 << t)]);
}

// The four matrix entries of a 2x2 gate, its columns exchanged where an X is
// folded in (fx).
template <typename T>
__device__ __forceinline__ void g_load_u1(const ROp<T> &op, bool fx, cx<T> (&m)[4]) {
  const T *c0 = op.u.m + (fx ? 4 : 0), *c1 = op.u.m + (fx ? 0 : 4);
  m[0] = mk<T>(c0[0], c0[1]);
  m[1] = mk<T>(c0[2], c0[3]);
  m[2] = mk<T>(c1[0], c1[1]);
  m[3] = mk<T>(c1[2], c1[3]);
}

// Slot x of the exchange buffer, as a byte offset: x ^ ((x >> 4) & 15), so that
// consecutive lanes reach distinct banks also where the register bits are the
// low tile bits.  Linear, so it splits into a per-lane and a per-register term.
__device__ __forceinline__ uint32_t g_slot(uint32_t x) { return (x ^ ((x >> 4) & 15u)) << 3; }

// Tile index of thread `t`'s part of the layout with register tile bits rp
// (ascending): t with a zero inserted at each of them.
template <int R>
__device__ __forceinline__ uint32_t g_thread(const RLayout &lay, uint32_t t) {
#pragma unroll
  for (int r = 0; r < R; ++r) t += t & (~0u << byte_at(lay.rp, r));
  return t;
}

// The tile moves from the layout of byte offsets w0 ^ w(j) to that of r0 ^ r(j),
// w and r uniform.  complex128: one component at a time, so that the buffer
// holds half a tile.
template <typename T, int NR>
__device__ __forceinline__ void g_exchange(Amps<T, NR> &a, char *xch, uint32_t w0, const uint32_t (&w)[NR],
                                           uint32_t r0, const uint32_t (&r)[NR]) {
  asm volatile("" : "+v"(w0), "+v"(r0));  // shifted already: one XOR per address
  __syncthreads();
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int j = 0; j < NR; ++j) *reinterpret_cast<cx<T> *>(xch + (w0 ^ w[j])) = a.v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NR; ++j) a.v[j] = *reinterpret_cast<const cx<T> *>(xch + (r0 ^ r[j]));
  } else {
#pragma unroll
    for (int j = 0; j < NR; ++j) *reinterpret_cast<T *>(xch + (w0 ^ w[j])) = a.v[j].x;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NR; ++j) a.v[j].x = *reinterpret_cast<const T *>(xch + (r0 ^ r[j]));
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NR; ++j) *reinterpret_cast<T *>(xch + (w0 ^ w[j])) = a.v[j].y;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NR; ++j) a.v[j].y = *reinterpret_cast<const T *>(xch + (r0 ^ r[j]));
  }
}

// Where a gate tile's share of a probe goes: the partials hold one entry per
// 2^(B - SPLIT) amplitudes, as the other passes write them; the tile's first
// takes its sum and the others zero.
template <int SPLIT>
struct GateSink {
  double *p;
  uint64_t tile, ntiles;
  __device__ __forceinline__ void put(uint32_t slot, double v) const {
    double *e = p + ((static_cast<uint64_t>(slot) * ntiles + tile) << SPLIT);
    e[0] = v;
    if constexpr (SPLIT) e[1] = 0.0;
  }
};

template <typename T, int B, int R, bool PROBES, typename Sink>
__device__ __forceinline__ void gate_tile(cx<T> *__restrict__ sv, const PassDesc *__restrict__ pd,
                                          const ROp<T> *__restrict__ rops, const cx<double> *__restrict__ pool,
                                          uint64_t tile_id, char *xch, cx<double> *dlt, double *red,
                                          const Sink &sink) {
  static_assert(R == 4, "the op codes name four register bits");
  constexpr int TB = B - R, NT = 1 << TB, NR = 1 << R;
  const uint32_t tid = threadIdx.x;
  uint64_t base = tile_id;
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const uint32_t q = pd->spos[i];
    base = ((base >> q) << (q + 1)) | (base & ((1ull << q) - 1ull));
  }
  base = uniform64(base);
  const ROp<T> *opp = rops + pd->op_begin;
  LayoutState<NR> st;
  st.tl = g_thread<R>(opp->u.lay, tid);
  st.ri = reg_index<R>(opp->u.lay);
  const uint32_t nslot = opp->a;
  const cx<double> *dlane = pool + opp->b;
  uint2 drec = make_uint2(0u, 0u);
  uint32_t sb[256 / NT] = {};
  if (nslot) {
    drec = reinterpret_cast<const uint2 *>(dlane)[tid & 63u];
    const uint32_t *stage_back = reinterpret_cast<const uint32_t *>(dlane + 32);
#pragma unroll
    for (int j = 0; j < 256 / NT; ++j) sb[j] = stage_back[j * NT + tid];
  }
  Amps<T, NR> a;
  {
    const RegOff<NR> ro = reg_offset<R>(opp->u.lay);
    const cx<T> *p = sv + base + thread_offset<TB>(opp->u.lay, tid);
#pragma unroll
    for (int j = 0; j < NR; ++j) a.v[j] = ld_stream(p + ro.gr[j]);
  }
  if (nslot) {
    stage_diag_tables<NT>(drec, dlane, nslot, base, tid, sb, dlt);
    __syncthreads();
  }
  const uint32_t cnt = opp->extra;
  for (uint32_t i = 0; i < cnt; ++i) {
    ++opp;
    const ROp<T> &op = *opp;
    const uint32_t code = op.code;
    const bool tile_ok = (base & op.cg) == op.cvg;
    if ((code & 0xF0u) == C_U1) {
      const bool fx = tile_ok && (op.kind & ~F_ALL) == Q_U1X;
      if constexpr (sizeof(T) == 4) {
        // U X: the columns of the pair's two amplitudes change places
        const float A = op.u.mr[4 * (tid & 3u) + (((tid >> 2) & 3u) ^ (fx ? 2u : 0u))];
        switch (code) {
          case C_U1 + 0: g_u1b_mfma<NR, 0>(a, A); break;
          case C_U1 + 1: g_u1b_mfma<NR, 1>(a, A); break;
          case C_U1 + 2: g_u1b_mfma<NR, 2>(a, A); break;
          case C_U1 + 3: g_u1b_mfma<NR, 3>(a, A); break;
        }
      } else {
        cx<T> m[4];
        g_load_u1(op, fx, m);
        switch (code) {
          case C_U1 + 0: g_u1b<T, NR, 0>(a, m); break;
          case C_U1 + 1: g_u1b<T, NR, 1>(a, m); break;
          case C_U1 + 2: g_u1b<T, NR, 2>(a, m); break;
          case C_U1 + 3: g_u1b<T, NR, 3>(a, m); break;
        }
      }
      continue;
    }
    if constexpr (sizeof(T) == 8)
      if ((code & 0xF8u) == C_U1R) {
        const bool fx = tile_ok && (op.kind & ~F_ALL) == Q_U1X;
        const T *c0 = op.u.m + (fx ? 4 : 0), *c1 = op.u.m + (fx ? 0 : 4);
        const T m[4] = {c0[0], c0[2], c1[0], c1[2]};
        switch (code) {
          case C_U1R + 0: g_u1r<T, NR, 0>(a, m); break;
          case C_U1R + 1: g_u1r<T, NR, 1>(a, m); break;
          case C_U1R + 2: g_u1r<T, NR, 2>(a, m); break;
          case C_U1R + 3: g_u1r<T, NR, 3>(a, m); break;
        }
        continue;
      }
    const uint32_t cl = op.cl, cvl = op.cvl;
    if ((code & 0xF0u) == C_U2) {
      if constexpr (sizeof(T) == 4) {
        const float A = reinterpret_cast<const float *>(pool + op.extra)[tid & 63u];
        switch (code) {
          case C_U2 + pair_index(0, 1): g_u2_mfma<NR, 0, 1>(a, A); break;
          case C_U2 + pair_index(0, 2): g_u2_mfma<NR, 0, 2>(a, A); break;
          case C_U2 + pair_index(1, 2): g_u2_mfma<NR, 1, 2>(a, A); break;
          case C_U2 + pair_index(0, 3): g_u2_mfma<NR, 0, 3>(a, A); break;
          case C_U2 + pair_index(1, 3): g_u2_mfma<NR, 1, 3>(a, A); break;
          case C_U2 + pair_index(2, 3): g_u2_mfma<NR, 2, 3>(a, A); break;
        }
      } else {
        cx<T> m[16];
        const cx<T> *mp = reinterpret_cast<const cx<T> *>(pool + op.extra);
#pragma unroll
        for (int e = 0; e < 16; ++e) m[e] = mp[e];
        switch (code) {
          case C_U2 + pair_index(0, 1): g_u2<T, NR, 0, 1>(a, m); break;
          case C_U2 + pair_index(0, 2): g_u2<T, NR, 0, 2>(a, m); break;
          case C_U2 + pair_index(1, 2): g_u2<T, NR, 1, 2>(a, m); break;
          case C_U2 + pair_index(0, 3): g_u2<T, NR, 0, 3>(a, m); break;
          case C_U2 + pair_index(1, 3): g_u2<T, NR, 1, 3>(a, m); break;
          case C_U2 + pair_index(2, 3): g_u2<T, NR, 2, 3>(a, m); break;
        }
      }
      continue;
    }
    if (code == C_RELAYOUT) {
      // A CX between tile bits is a linear map of the tile index, so those that
      // come just before (or just after) cost the write addresses a shift and an
      // XOR, not the amplitudes a move.
      const uint32_t ncx = op.a;
      const uint32_t *cxw = reinterpret_cast<const uint32_t *>(op.u.rel.cx);
      for (uint32_t k = 0; k < ncx; ++k) {
        const uint32_t p = cxw[k >> 1] >> (16 * (k & 1u)), c = p & 0xFFu, t = (p >> 8) & 0xFFu;
        if (c == kNoControl) {
          st.ri.t0 ^= 1u << t;
        } else {
          auto map = [&](uint32_t x) { return x ^ (((x >> c) & 1u) << t); };
          st.tl = map(st.tl);
#pragma unroll
          for (int s = 0; s < R; ++s) st.ri.bm[s] = map(st.ri.bm[s]);
          st.ri.t0 = map(st.ri.t0);
        }
      }
      uint32_t w[NR], r[NR];
      const uint32_t w0 = g_slot(st.tl);
#pragma unroll
      for (int j = 0; j < NR; ++j) w[j] = g_slot(st.ri.at(j));
      st.tl = g_thread<R>(op.u.lay, tid);
      st.ri = reg_index<R>(op.u.lay);
      const uint32_t r0 = g_slot(st.tl);
#pragma unroll
      for (int j = 0; j < NR; ++j) r[j] = g_slot(st.ri.at(j));
      g_exchange<T, NR>(a, xch, w0, w, r0, r);
      continue;
    }
    if ((code & 0xF0u) == C_CXR) {
      switch (code) {
#define G_CASE(c, t) \
  case C_CXR + 4 * c + t: g_cxr<T, NR, c, t>(a); break;
        G_CASE(0, 1) G_CASE(0, 2) G_CASE(0, 3) G_CASE(1, 0) G_CASE(1, 2) G_CASE(1, 3)
        G_CASE(2, 0) G_CASE(2, 1) G_CASE(2, 3) G_CASE(3, 0) G_CASE(3, 1) G_CASE(3, 2)
#undef G_CASE
      }
      continue;
    }
    if (!PROBES && (code & 0xF8u) == C_U3) {
      if constexpr (sizeof(T) == 4) {
        const float *mp = reinterpret_cast<const float *>(pool + op.extra) + (tid & 63u);
        const float A[4] = {mp[0], mp[64], mp[128], mp[192]};
        switch (code) {
          case C_U3 + 0: g_u3_mfma<NR, 0>(a, A); break;
          case C_U3 + 1: g_u3_mfma<NR, 1>(a, A); break;
          case C_U3 + 2: g_u3_mfma<NR, 2>(a, A); break;
          case C_U3 + 3: g_u3_mfma<NR, 3>(a, A); break;
        }
      } else {
        const cx<T> *mp = reinterpret_cast<const cx<T> *>(pool + op.extra);
        switch (code) {
          case C_U3 + 0: g_u3<T, NR, 0>(a, mp); break;
          case C_U3 + 1: g_u3<T, NR, 1>(a, mp); break;
          case C_U3 + 2: g_u3<T, NR, 2>(a, mp); break;
          case C_U3 + 3: g_u3<T, NR, 3>(a, mp); break;
        }
      }
      continue;
    }
    if constexpr (PROBES)
      if (code == C_PROBE) {
        q_probes<T, NR, NT>(reinterpret_cast<const RProbe *>(pool + op.extra), op.a, op.b, a, st.tl, base, tid, red,
                            sink);
        continue;
      }
    if (!tile_ok) continue;  // controls fixed by the tile that do not hold
    const uint32_t tlc = st.tl & cl;
    const uint32_t rb = op.b;
    uint32_t rbits = 0;
#pragma unroll
    for (int s = 0; s < R; ++s) rbits |= st.ri.bm[s];
    const uint32_t clt = cl & ~rbits;
    const bool lane_ok = (st.tl & clt) == (cvl & clt);
    const cx<T> one = mk<T>(1, 0);
    switch (code) {
      case C_X + 0: g_x<T, NR, 0>(a); break;
      case C_X + 1: g_x<T, NR, 1>(a); break;
      case C_X + 2: g_x<T, NR, 2>(a); break;
      case C_X + 3: g_x<T, NR, 3>(a); break;
#define G_CASE(b)                                                                        \
  case C_XC + b: g_xc<T, NR, b>(a, __ballot(lane_ok), rb); break;                        \
  case C_Y + b: g_yc<T, NR, b>(a, tlc, st.ri, cl, cvl); break;                           \
  case C_U1C + b: {                                                                      \
    cx<T> m[4];                                                                          \
    g_load_u1(op, false, m);                                                             \
    g_u1c<T, NR, b>(a, tlc, st.ri, cl, cvl, m);                                          \
    break;                                                                               \
  }
      G_CASE(0) G_CASE(1) G_CASE(2) G_CASE(3)
#undef G_CASE
      case C_PHASE: {
        const cx<T> f = csel(lane_ok, mk<T>(op.u.m[0], op.u.m[1]), one);
#pragma unroll
        for (int j = 0; j < NR; ++j)
          if ((rb >> j) & 1u) {
            asm volatile("");  // keeps the branch (no if-conversion into selects)
            g_mul(a.v[j], f);
          }
        break;
      }
      case C_D1: {
        const cx<T> d0 = mk<T>(op.u.m[0], op.u.m[1]), d1 = mk<T>(op.u.m[2], op.u.m[3]);
        const uint32_t t = op.a;
        if ((rbits >> t) & 1u) {
          // target on a register bit: bit j of rb is the target's value in register j
#pragma unroll
          for (int j = 0; j < NR; ++j) {
            if ((rb >> j) & 1u) {
              asm volatile("");  // keeps the branch (no if-conversion into selects)
              g_mul(a.v[j], d1);
            } else {
              g_mul(a.v[j], d0);
            }
          }
        } else {
          const cx<T> d = csel(((st.tl >> t) & 1u) != 0, d1, d0);
#pragma unroll
          for (int j = 0; j < NR; ++j) g_mul(a.v[j], d);
        }
        break;
      }
#define G_CASE(b0, b1) \
  case C_SWAP + pair_index(b0, b1): g_swapc<T, NR, b0, b1>(a, __ballot(lane_ok), op.extra); break;
      G_CASE(0, 1) G_CASE(0, 2) G_CASE(1, 2) G_CASE(0, 3) G_CASE(1, 3) G_CASE(2, 3)
#undef G_CASE
      case C_DIAGK: {
        // one entry per lane and group of registers that share their part of the index
        const cx<double> *tab = pool + op.extra;
        const uint32_t *w = reinterpret_cast<const uint32_t *>(op.u.fq);
        uint32_t idx = 0;
#pragma unroll
        for (int d = 0; d < 8; ++d) {
          const uint32_t tb = byte_at(w, d), q = byte_at(w, 8 + d);
          if (tb < 32) idx |= ((st.tl >> tb) & 1u) << d;
          if (q < 64) idx |= static_cast<uint32_t>((base >> q) & 1ull) << d;
        }
        const uint32_t ka = op.a;
        const uint32_t *grp = reinterpret_cast<const uint32_t *>(tab + (1u << (ka & 0xFFu)));
        for (uint32_t g = 0; g < ka >> 8; ++g) {
          const uint32_t gr = grp[g];
          const cx<T> f = csel(lane_ok, to_t<T>(tab[idx | (gr >> 16)]), one);
#pragma unroll
          for (int j = 0; j < NR; ++j)
            if ((gr >> j) & 1u) {
              asm volatile("");  // keeps the branch (no if-conversion into selects)
              g_mul(a.v[j], f);
            }
        }
        break;
      }
      case C_DIAGF: {
        // the fused diagonal of Q_DIAGF: factor G L R_j, G L per lane; where the
        // lane's predicate does not hold, 0 R_j + 1, so that no register needs a
        // select (passes of a 30-qubit QFT: 8.80 -> 8.56 ms)
        const cx<double> *blk = pool + op.extra;
        uint32_t t = tid;
        asm volatile("" : "+v"(t));  // lane indices derived here, not held for the whole pass
        cx<double> g;
        const uint32_t ra = op.a;
        if (const uint32_t slot = ra >> 16) {
          const cx<double> *row = dlt + 32u * (slot - 1u);
          g = cmul(row[t & 15u], row[16u + ((t >> 4) & 15u)]);
        } else {
          g = cmul(blk[NR + (t & 15u)], blk[NR + 16 + ((t >> 4) & 15u)]);
          const cx<double> *tab = blk + NR + 32;
          for (uint32_t c = 0; c < (ra & 0xFFu); ++c, tab += 16) {
            uint32_t idx = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const uint32_t q = op.u.fq[4 * c + k];
              if (q < 64) idx |= static_cast<uint32_t>((base >> q) & 1ull) << k;
            }
            g = cmul(g, tab[idx]);
          }
        }
        const double add = lane_ok ? 0.0 : 1.0;
        g = csel(lane_ok, g, mk<double>(0, 0));
#pragma unroll
        for (int j = 0; j < NR; ++j)
          if ((rb >> j) & 1u) {
            asm volatile("");  // keeps the branch (no if-conversion into selects)
            const cx<double> r = blk[j];
            const double x = fma_t(-g.y, r.y, fma_t(g.x, r.x, add)), y = fma_t(g.y, r.x, g.x * r.y);
            g_mul(a.v[j], to_t<T>(mk<double>(x, y)));
          }
        break;
      }
      default: break;
    }
  }
  ++opp;
  if constexpr (PROBES)
    if (opp->extra) return;  // a read-only pass
  const RegOff<NR> ro = reg_offset<R>(opp->u.lay);
  cx<T> *p = sv + base + thread_offset<TB>(opp->u.lay, tid);
#pragma unroll
  for (int j = 0; j < NR; ++j) st_stream(p + ro.gr[j], a.v[j]);
}

template <typename T, int B, int R, bool PROBES>
__global__ __launch_bounds__(1 << (B - R))
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 || PROBES ? 4 : 5))) void k_gate_pass(
    cx<T> *__restrict__ sv, const PassDesc *__restrict__ pd, const ROp<T> *__restrict__ rops,
    const cx<double> *__restrict__ pool, double *__restrict__ probes, uint64_t state_stride, uint32_t pd_stride,
    uint32_t tile_log, uint32_t probes_per_state) {
  __shared__ __align__(16) char xch[8 << B];
  __shared__ double red[PROBES ? red_doubles((1 << (B - R)) / 64) : 1];
  constexpr int SPLIT = sizeof(T) == 8 ? 1 : 0;
  const StateTile st = state_tile(tile_log);
  const GateSink<SPLIT> sink{probes + ((st.b * probes_per_state * st.ntiles) << SPLIT), st.t, st.ntiles};
  gate_tile<T, B, R, PROBES>(sv + st.b * state_stride, pd + st.b * pd_stride, rops, pool, st.t, xch,
                             reinterpret_cast<cx<double> *>(aerhip_dyn_lds), red, sink);
}

}  // namespace aerhip
