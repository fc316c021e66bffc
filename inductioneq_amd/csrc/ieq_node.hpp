// Per-node stencil access of the kernels that give every thread its own nodes and read the
// neighbours through the caches.  Nodes whose row of the operator tables is the central one and
// whose central stencil lies inside the grid ("mid" nodes: all of them on periodic grids) need the
// 2 RR non-zero entries of that row, with compile-time coefficients; the others read their row
// from a table and fold the neighbours as the reference does (utils.h:91-98, 144-148).  A wave
// with a node of the second kind takes the general form for all of its lanes, and both forms are
// unrolled: their loads are independent, so a wave waits for one load latency per direction.  (A
// rolled loop over a row waits for a coefficient and a value per entry: 7 x 2 latencies at 4th order.)
#pragma once

#include "ieq_device.hpp"

namespace ieq {
namespace {

// One axis of a node: its table row and whether the unrolled central stencil applies.
struct NodeAxis {
  int i, n, row;
  bool mid;
};
template <int OPS> __device__ __forceinline__ NodeAxis node_axis(int i, int n, int periodic) {
  using O = Op<OPS>;
  constexpr int RR = O::ORDER / 2;
  NodeAxis a;
  a.i = i;
  a.n = n;
  a.row = bound_row((uint32_t)i, (uint32_t)n, O::NB, periodic);
  a.mid = a.row == O::NB && (periodic || (i >= RR && i + RR < n));
  return a;
}
// Step along the axis to the neighbour at offset k: wrapped on periodic grids; a neighbour outside a
// bounded grid is the node itself.  Without branches, so that the loads that follow stay in one run.
__device__ __forceinline__ int node_step(const NodeAxis& a, int k, int periodic) {
  const int out = periodic ? (k < 0 ? k + a.n : k - a.n) : 0;
  return (unsigned)(a.i + k) < (unsigned)a.n ? k : out;
}

// Value at a byte offset from a component's plane; I is unsigned where the plane stays below 4 GiB (one 32-bit
// register per address), long long otherwise.
template <typename R, typename I> __device__ __forceinline__ R node_ld(const R* __restrict__ f, I off) {
  return *(const R*)((const char*)f + off);
}
template <typename R, typename I> __device__ __forceinline__ void node_st(R* __restrict__ f, I off, R v) {
  *(R*)((char*)f + off) = v;
}
template <typename R> inline bool wide_plane(const Params& p) { return (long long)p.nx * p.ny * (long long)sizeof(R) >= (1LL << 32); }

// First derivative along one axis, not divided by the spacing; `at(k)` is the value k nodes away and
// T the type it is accumulated in.
template <typename T, int OPS, typename At> __device__ __forceinline__ T node_deriv_mid(At at) {
  using O = Op<OPS>;
  constexpr int C = (O::W - 1) / 2, RR = O::ORDER / 2;
  T acc = T(0);
#pragma unroll
  for (int k = -RR; k <= RR; ++k)
    if (k != 0) acc = acc + (T)O::d(O::NB, C + k) * at(k);
  return acc;
}
// A wave's own copy of the derivative table (ADJ: of the adjoint's) in LDS, written and then read by its lanes: the
// fences order the two without a workgroup barrier.
template <typename R, int OPS, bool ADJ> __device__ __forceinline__ void wave_table(R* tab) {
  using O = Op<OPS>;
  for (int i = (int)threadIdx.x & 63; i < (2 * O::NB + 1) * O::W; i += 64) tab[i] = (R)(ADJ ? O::dadj(0, i) : O::d(0, i));
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}
// The derivative for any row of the table, from a block's copy in LDS (a row differs from lane to lane: global
// loads of it cost as much as the values it weighs, and registers for it cost occupancy).
template <typename T, int OPS> struct NodeTable {
  static constexpr int W = Op<OPS>::W, C = (W - 1) / 2, ROWS = 2 * Op<OPS>::NB + 1;
  T c[ROWS][W];
  __device__ __forceinline__ void load(int tid, int nthreads) {  // a barrier must follow
    for (int i = tid; i < ROWS * W; i += nthreads) (&c[0][0])[i] = (T)Op<OPS>::d(i / W, i % W);
  }
};
template <typename T, int OPS, typename At>
__device__ __forceinline__ T node_deriv_row(const NodeTable<T, OPS>& t, const NodeAxis& a, int periodic, At at) {
  constexpr int W = NodeTable<T, OPS>::W, C = NodeTable<T, OPS>::C;
  T acc = T(0);
#pragma unroll
  for (int k = 0; k < W; ++k) acc = acc + t.c[a.row][k] * at(node_step(a, k - C, periodic));
  return acc;
}

}  // namespace
}  // namespace ieq
