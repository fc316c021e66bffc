// Reference-schedule kernels other than the stages, the curls and calc_u (ieq_node_stage.inc): SBP operators down a
// column of planes or with a thread per node, and one work-item per node for the rest.  These back the reference kernel names
// accepted by ieq_run(); the fused kernels in ieq_fused.hip replace the hot ones.
#include <algorithm>
#include <type_traits>

#include "ieq_device.hpp"
#include "ieq_generic.hpp"
#include "ieq_node.hpp"
#include "ieq_stencil.hpp"

namespace ieq {
namespace {

constexpr int BX = 64, BY = 4;

// Derivatives of one component (diff_x/y/z, SBP_operator.cl:12-51) or their M-adjoints at the nodes of a
// column (fixed x and y, the planes of a chunk): the rows and neighbour offsets along x and y are found
// once per thread, those along z are uniform in a wave.  A wave with a node near an x (y) face takes its
// general row there for all lanes.  With rows and indices looked up per node a thread spends 300 instructions:
// 192^3 FP32, 4th order, div B 63 -> 33 us, its norm 112 -> 33, projection 67 -> 38; the four fields of div B once take
// 23 us as a copy.
// I: in-plane byte offsets (ieq_node.hpp).
template <typename R, int OPS, bool ADJ, typename I> struct Column {
  using O = Op<OPS>;
  static constexpr int W = O::W, C = (W - 1) / 2;
  I o;  // in-plane byte offset of the nodes
  bool mx, my;
  R cx[W], cy[W];
  I ox[W], oy[W];
  __device__ static double coef(int row, int k) { return ADJ ? O::dadj(row, k) : O::d(row, k); }
  __device__ __forceinline__ void init(const Params& p, int ix, int iy) {
    const NodeAxis ax = node_axis<OPS>(ix, p.nx, p.periodic), ay = node_axis<OPS>(iy, p.ny, p.periodic);
    const I RB = sizeof(R);
    o = ((I)ix + (I)p.nx * (I)iy) * RB;
    mx = __all(ax.mid);
    my = __all(ay.mid);
#pragma unroll
    for (int k = 0; k < W; ++k) {
      cx[k] = (R)coef(mx ? O::NB : ax.row, k);
      cy[k] = (R)coef(my ? O::NB : ay.row, k);
      ox[k] = o + (I)node_step(ax, k - C, p.periodic) * RB;
      oy[k] = o + (I)node_step(ay, k - C, p.periodic) * (I)p.nx * RB;
    }
  }
  // MX, MY, MZ: the central row is taken along x, y, z (compile-time, so that the loads of all directions of a
  // node are one run without branches; with a branch per direction a plane waits for three load latencies).
  // f: the component's plane iz.
  template <bool MID> __device__ __forceinline__ R line(const Params& p, const R* f, const R (&c)[W], const I (&off)[W], int d) const {
    R acc = R(0);
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const double m = coef(O::NB, k);  // a literal: zero entries of the central row drop out
      if constexpr (MID) {
        if (m != 0.0) acc = acc + (R)m * node_ld(f, off[k]);
      } else {
        acc = acc + c[k] * node_ld(f, off[k]);
      }
    }
    return acc / (R)hdir(p, d);
  }
  template <bool MX> __device__ __forceinline__ R dx(const Params& p, const R* f) const { return line<MX>(p, f, cx, ox, 0); }
  template <bool MY> __device__ __forceinline__ R dy(const Params& p, const R* f) const { return line<MY>(p, f, cy, oy, 1); }
  // the central row without a wrap: fixed strides from the plane pointer
  __device__ static __forceinline__ bool inner(const Params& p, int iz) {
    constexpr int RR = O::ORDER / 2;
    return iz >= RR && iz + RR < p.nz && (p.periodic || (iz >= O::NB && iz + O::NB < p.nz));
  }
  template <bool MZ> __device__ __forceinline__ R dz(const Params& p, const R* f, int iz) const {
    const long long nxy = (long long)p.nx * p.ny;
    R acc = R(0);
    if constexpr (MZ) {
#pragma unroll
      for (int k = -C; k <= C; ++k) {
        const double m = coef(O::NB, k + C);
        if (m != 0.0) acc = acc + (R)m * node_ld(f + k * nxy, o);
      }
    } else {
      const NodeAxis az = node_axis<OPS>(iz, p.nz, p.periodic);
#pragma unroll
      for (int k = -C; k <= C; ++k) acc = acc + (R)coef(az.row, k + C) * node_ld(f + node_step(az, k, p.periodic) * nxy, o);
    }
    return acc / (R)hdir(p, 2);
  }
  template <bool MX, bool MY, bool MZ> __device__ __forceinline__ R div(const Params& p, const R* b, int iz) const {
    return dx<MX>(p, b) + dy<MY>(p, b + p.stride) + dz<MZ>(p, b + 2 * p.stride, iz);  // SBP_operator.cl:101-110
  }
  // body(mx, my, mz, iz) for the planes z0 .. z1 - 1 with the flags as compile-time constants
  template <typename Body> __device__ __forceinline__ void planes(const Params& p, int z0, int z1, Body body) const {
    using std::false_type;
    using std::true_type;
    auto march = [&](auto x, auto y) {
      for (int iz = z0; iz < z1; ++iz) {
        if (inner(p, iz)) body(x, y, true_type{}, iz);
        else body(x, y, false_type{}, iz);
      }
    };
    if (mx && my) march(true_type{}, true_type{});
    else if (my) march(false_type{}, true_type{});
    else march(false_type{}, false_type{});
  }
};

// A block of the column kernels: 256 consecutive nodes of an xy-plane of the NDRange (full lanes whatever the
// sizes) and `zc` planes; blocks in contiguous ranges per XCD, in rows of at most kRow (HIP takes fewer than 2^32
// threads in a dimension).
constexpr unsigned kRow = 1 << 22;
struct ColumnGrid {
  long long gxy;           // nodes of the NDRange in a plane
  int gx, gz, segs, zc, blocks;  // ... in x and z; runs of 256 in a plane, planes of a block, blocks
  dim3 rows() const { return blocks <= (int)kRow ? dim3((unsigned)blocks) : dim3(kRow, ((unsigned)blocks + kRow - 1) / kRow); }
};
// Planes per block, at most `most`: about 4096 blocks, so that the chip is full and a thread still has a few planes to
// share its rows between.
ColumnGrid column_grid(const uint32_t g[3], long long most) {
  ColumnGrid c;
  c.gxy = (long long)g[0] * g[1];
  c.gx = (int)g[0];
  c.gz = (int)g[2];
  c.segs = (int)((c.gxy + 255) / 256);
  c.zc = (int)std::max(1LL, std::min(most, (long long)c.segs * c.gz / 4096));
  c.blocks = c.segs * ((c.gz + c.zc - 1) / c.zc);
  return c;
}
#define IEQ_COLUMN_PREAMBLE(OFF)                                                                              \
  const int linear = (int)(blockIdx.y * kRow + blockIdx.x);                                                   \
  if (linear >= cg.blocks) return;                                                                            \
  const int tile = xcd_tile(linear, cg.blocks), ch = tile / cg.segs;                                          \
  using P = std::conditional_t<std::is_same_v<I, unsigned>, uint32_t, uint64_t>;                              \
  const P jt = (P)(tile - ch * cg.segs) * 256 + threadIdx.x, gx = (P)cg.gx;                                   \
  if (jt >= (P)cg.gxy) return;                                                                                \
  const int ix = (int)(jt % gx) + (OFF), iy = (int)(jt / gx) + (OFF);                                         \
  const int z0 = ch * cg.zc + (OFF), z1 = min(z0 + cg.zc, cg.gz + (OFF));                                     \
  const long long S = p.stride, nxy = (long long)p.nx * p.ny;                                                 \
  (void)S; (void)nxy;

#define IEQ_NODE_PREAMBLE(OFF)                                            \
  uint32_t ix = blockIdx.x * BX + threadIdx.x, iy = blockIdx.y * BY + threadIdx.y, iz = blockIdx.z; \
  if (ix >= g.x || iy >= g.y) return;                                     \
  ix += (OFF); iy += (OFF); iz += (OFF);                                  \
  const long long idx = lin(p, ix, iy, iz);                               \
  const long long S = p.stride;                                           \
  (void)S; (void)idx;

struct Range { uint32_t x, y, z; };

template <typename R> __device__ inline void set_time(const Range& g, R* time, double c, double dt, uint32_t ix, uint32_t iy, uint32_t iz) {
  if (ix == 0 && iy == 0 && iz == 0 && c >= 0) time[1] = time[0] + (R)c * (R)dt;
}

// 2R "b" stage: X = X + a*D; O = X + b*D  (kernel_time_integrator.cl:642-660)
template <typename R>
__global__ __launch_bounds__(BX* BY) void k_update_2r(Params p, Range g, R* X, R* O, const R* D, R a, R b, R* time, double tc) {
  IEQ_NODE_PREAMBLE(0)
  for (int c = 0; c < 3; ++c) {
    R x = X[c * S + idx] + a * D[c * S + idx];
    X[c * S + idx] = x;
    O[c * S + idx] = x + b * D[c * S + idx];
  }
  set_time(g, time, tc, p.dt, ix, iy, iz);
}

// 2N "b" stage: X = X + b*D (kernel_time_integrator.cl:1036-1057)
template <typename R>
__global__ __launch_bounds__(BX* BY) void k_update_2n(Params p, Range g, R* X, const R* D, R b, R* time, double tc) {
  IEQ_NODE_PREAMBLE(0)
  for (int c = 0; c < 3; ++c) X[c * S + idx] = X[c * S + idx] + b * D[c * S + idx];
  set_time(g, time, tc, p.dt, ix, iy, iz);
}

// SSPRK104_06 (kernel_time_integrator.cl:458-477)
template <typename R>
__global__ __launch_bounds__(BX* BY) void k_ssprk104_06(Params p, Range g, const R* b1, R* b2, R* b3, R* time) {
  IEQ_NODE_PREAMBLE(0)
  for (int c = 0; c < 3; ++c) {
    R x1 = b1[c * S + idx], x2 = b2[c * S + idx];
    b3[c * S + idx] = R(0.04) * x1 + R(0.36) * x2;
    b2[c * S + idx] = R(0.60) * x1 + R(0.40) * x2;
  }
  if (ix == 0 && iy == 0 && iz == 0) time[1] = time[0] + (R)(p.dt / 3.0);
}

// time-only kernels: mode 0 sets time[1] = time[0] + c*DT; mode 1 is calc_time_* (time[0] += DT).
template <typename R> __global__ void k_time(R* time, double c, double dt, int mode) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    if (mode == 1) {
      time[0] = time[0] + (R)dt;
      time[1] = time[0];
    } else {
      time[1] = time[0] + (R)(c * dt);
    }
  }
}

// init_b / init_u / init_rho / analytical_b (kernel_init.cl:3-48)
template <typename R> __global__ __launch_bounds__(BX* BY) void k_init(Params p, Range g, R* f, int which, const R* time) {
  IEQ_NODE_PREAMBLE(0)
  if (which == 0) st3(f, S, idx, b_analytical<R>(p, ix, iy, iz, R(0)));
  else if (which == 1) st3(f, S, idx, u_analytical<R>(p, ix, iy, iz, R(0)));
  else if (which == 2) f[idx] = R(1);
  else st3(f, S, idx, b_analytical<R>(p, ix, iy, iz, time[0]));
}

template <typename R, int OPS, typename I> __global__ __launch_bounds__(256) void k_div_column(Params p, ColumnGrid cg, const R* b, R* out, int off) {
  IEQ_COLUMN_PREAMBLE(off)
  Column<R, OPS, false, I> c;
  c.init(p, ix, iy);
  c.planes(p, z0, z1, [&](auto x, auto y, auto z, int iz) {
    node_st(out + iz * nxy, c.o, c.template div<x.value, y.value, z.value>(p, b + iz * nxy, iz));
  });
}

// The curl down a column: FP32 of 2nd order on bounded grids (gen_curl).
template <typename R, int OPS> __global__ __launch_bounds__(256) void k_curl_column(Params p, ColumnGrid cg, const R* b, R* out) {
  using I = unsigned;
  IEQ_COLUMN_PREAMBLE(0)
  Column<R, OPS, false, I> c;
  c.init(p, ix, iy);
  c.planes(p, z0, z1, [&](auto x, auto y, auto z, int iz) {  // SBP_operator.cl:126-135
    const R *bx = b + iz * nxy, *by = bx + S, *bz = by + S;
    R* f = out + iz * nxy;
    node_st(f, c.o, c.template dy<y.value>(p, bz) - c.template dz<z.value>(p, by, iz));
    node_st(f + S, c.o, c.template dz<z.value>(p, bx, iz) - c.template dx<x.value>(p, bz));
    node_st(f + 2 * S, c.o, c.template dx<x.value>(p, by) - c.template dy<y.value>(p, bx));
  });
}

template <typename R, int OPS, typename I> __global__ __launch_bounds__(256) void k_grad_column(Params p, ColumnGrid cg, const R* f, R* out) {
  IEQ_COLUMN_PREAMBLE(0)
  Column<R, OPS, false, I> c;
  c.init(p, ix, iy);
  c.planes(p, z0, z1, [&](auto x, auto y, auto z, int iz) {
    const R* fz = f + iz * nxy;
    R* o = out + iz * nxy;
    node_st(o, c.o, c.template dx<x.value>(p, fz));
    node_st(o + S, c.o, c.template dy<y.value>(p, fz));
    node_st(o + 2 * S, c.o, c.template dz<z.value>(p, fz, iz));
  });
}

// The derivatives along x, y and z of fx, fy and fz (a node's plane of a component each) with a thread per node: rows of
// the table from LDS where a wave has a boundary row.
template <typename R, int OPS, bool ADJ, int D, bool MID, typename I>
__device__ __forceinline__ R line_deriv(const Params& p, const NodeAxis& A, const R* f, I o, R* tab) {
  using O = Op<OPS>;
  constexpr int W = O::W, C = (W - 1) / 2, NB = O::NB;
  const long long nxy = (long long)p.nx * p.ny;
  const bool mid = MID || (D == 2 ? A.mid : (bool)__all(A.mid));
  if (D != 2 && !mid) wave_table<R, OPS, ADJ>(tab);
  R acc = R(0);
  auto at = [&](int step) {
    return D == 2 ? node_ld(f + (long long)step * nxy, o) : node_ld(f, o + (D == 0 ? (I)step : (I)step * (I)p.nx) * (I)sizeof(R));
  };
  if (mid) {
#pragma unroll
    for (int k = -C; k <= C; ++k) {
      const double m = ADJ ? O::dadj(NB, C + k) : O::d(NB, C + k);
      if (m != 0.0) acc = acc + (R)m * at(node_step(A, k, p.periodic));
    }
  } else {
#pragma unroll
    for (int k = -C; k <= C; ++k)
      acc = acc + (D != 2 ? tab[A.row * W + C + k] : (R)(ADJ ? O::dadj(A.row, C + k) : O::d(A.row, C + k))) * at(node_step(A, k, p.periodic));
  }
  return acc / (R)hdir(p, D);
}
template <typename R, int OPS, bool ADJ, typename I>
__device__ __forceinline__ V3<R> line_derivs(const Params& p, int ix, int iy, int iz, const R* fx, const R* fy, const R* fz, I o, R* tab) {
  const int per = p.periodic;
  const NodeAxis ax = node_axis<OPS>(ix, p.nx, per), ay = node_axis<OPS>(iy, p.ny, per), az = node_axis<OPS>(iz, p.nz, per);
  if (per || (az.mid && __all(ax.mid && ay.mid)))
    return mk(line_deriv<R, OPS, ADJ, 0, true>(p, ax, fx, o, tab), line_deriv<R, OPS, ADJ, 1, true>(p, ay, fy, o, tab),
              line_deriv<R, OPS, ADJ, 2, true>(p, az, fz, o, tab));
  if constexpr (sizeof(R) == 4 && Op<OPS>::ORDER == 2) {  // short rows: all loads in one run before the table is needed
    constexpr int W = Op<OPS>::W, C = (W - 1) / 2;
    const long long nxy = (long long)p.nx * p.ny;
    R vx[W], vy[W], vz[W], sx = R(0), sy = R(0), sz = R(0);
#pragma unroll
    for (int k = 0; k < W; ++k) {
      vx[k] = node_ld(fx, o + (I)node_step(ax, k - C, per) * (I)sizeof(R));
      vy[k] = node_ld(fy, o + (I)node_step(ay, k - C, per) * (I)p.nx * (I)sizeof(R));
      vz[k] = node_ld(fz + (long long)node_step(az, k - C, per) * nxy, o);
    }
    wave_table<R, OPS, ADJ>(tab);
#pragma unroll
    for (int k = 0; k < W; ++k) {
      sx = sx + tab[ax.row * W + k] * vx[k];
      sy = sy + tab[ay.row * W + k] * vy[k];
      sz = sz + (R)(ADJ ? Op<OPS>::dadj(az.row, k) : Op<OPS>::d(az.row, k)) * vz[k];
    }
    return mk(sx / (R)p.dx, sy / (R)p.dy, sz / (R)p.dz);
  }
  return mk(line_deriv<R, OPS, ADJ, 0, false>(p, ax, fx, o, tab), line_deriv<R, OPS, ADJ, 1, false>(p, ay, fy, o, tab),
            line_deriv<R, OPS, ADJ, 2, false>(p, az, fz, o, tab));
}
#define IEQ_RUN_PREAMBLE(OFF)                                                                                \
  using O = Op<OPS>;                                                                                          \
  __shared__ R tabs[4][(2 * O::NB + 1) * O::W];                                                               \
  R* tab = tabs[__builtin_amdgcn_readfirstlane(threadIdx.x / 64)];                                            \
  const int linear = (int)(blockIdx.y * kRow + blockIdx.x);                                                   \
  if (linear >= cg.blocks) return;                                                                            \
  const int tile = xcd_tile(linear, cg.blocks), zt = tile / cg.segs;                                          \
  using P = std::conditional_t<std::is_same_v<I, unsigned>, uint32_t, uint64_t>;                              \
  const P jt = (P)(tile - zt * cg.segs) * 256 + threadIdx.x, gx = (P)cg.gx, j = min(jt, (P)cg.gxy - 1);       \
  const int ix = (int)(j % gx) + (OFF), iy = (int)(j / gx) + (OFF), iz = zt + (OFF);                          \
  const long long S = p.stride, nxy = (long long)p.nx * p.ny;                                                 \
  const I o = ((I)ix + (I)p.nx * (I)iy) * (I)sizeof(R);                                                       \
  (void)S;
template <typename R, int OPS, typename I> __global__ __launch_bounds__(256) void k_div(Params p, ColumnGrid cg, const R* b, R* out, int off) {
  IEQ_RUN_PREAMBLE(off)
  const R* f = b + iz * nxy;
  const V3<R> d = line_derivs<R, OPS, false>(p, ix, iy, iz, f, f + S, f + 2 * S, o, tab);
  if (jt < (P)cg.gxy) node_st(out + iz * nxy, o, d.x + d.y + d.z);
}
template <typename R, int OPS, typename I> __global__ __launch_bounds__(256) void k_grad(Params p, ColumnGrid cg, const R* f, R* out) {
  IEQ_RUN_PREAMBLE(0)
  const R* fz = f + iz * nxy;
  const V3<R> d = line_derivs<R, OPS, false>(p, ix, iy, iz, fz, fz, fz, o, tab);
  R* q = out + iz * nxy;
  if (jt < (P)cg.gxy) {
    node_st(q, o, d.x);
    node_st(q + S, o, d.y);
    node_st(q + 2 * S, o, d.z);
  }
}
// Partial sums of the squared SBP norm of div B (calc_div + norm2_S, kernel_operator.cl:98-155): the
// divergence in REAL as calc_div stores it, weights, squares and sums in double, of a component below 2 GiB (its
// caller's limit).  One partial per block, at
// most kNormBlocks of them: runs of a plane beyond that many are walked with a stride.
constexpr int kNormBlocks = 1024;
template <typename R, int OPS> __global__ __launch_bounds__(256) void k_div_norm(Params p, int segs, int zc, const R* b, double* part) {
  using O = Op<OPS>;
  const int nxy = p.nx * p.ny, tile = xcd_tile(blockIdx.x, gridDim.x), ch = tile / segs;
  const int z0 = ch * zc, z1 = min(z0 + zc, p.nz);
  double acc = 0.0;
  for (int j = (tile - ch * segs) * 256 + (int)threadIdx.x; j < nxy; j += segs * 256) {
    const int ix = j % p.nx, iy = j / p.nx;
    Column<R, OPS, false, unsigned> c;
    c.init(p, ix, iy);
    const double fxy = (p.dx / O::minv(bound_row(ix, p.nx, O::NB, p.periodic))) * (p.dy / O::minv(bound_row(iy, p.ny, O::NB, p.periodic)));
    c.planes(p, z0, z1, [&](auto x, auto y, auto z, int iz) {
      const double d = (double)c.template div<x.value, y.value, z.value>(p, b + (long long)iz * nxy, iz);
      acc += fxy * (p.dz / O::minv(bound_row(iz, p.nz, O::NB, p.periodic))) * (d * d);
    });
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  __shared__ double sm[4];
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) part[tile] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
}
// out[0] = sum of n partials in a fixed order.
__global__ __launch_bounds__(256) void k_sum(const double* part, int n, double* out) {
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) acc += part[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  __shared__ double sm[4];
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[0] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
}

// -Laplacian of kernel_div_cleaning.cl:11-56 on the range offset by BNODES.
template <typename R, int OPS> __device__ inline R lap_node(const Params& p, const R* f, uint32_t ix, uint32_t iy, uint32_t iz) {
  using O = Op<OPS>;
  int nbl = p.laplace == 0 ? O::LNB0 : p.laplace == 1 ? O::LNB1 : O::LNB2;
  int wl = p.laplace == 0 ? O::LW0 : p.laplace == 1 ? O::LW1 : O::LW2;
  int c = (wl - 1) / 2;
  int bx = bound_row(ix, p.nx, nbl, p.periodic), by = bound_row(iy, p.ny, nbl, p.periodic), bz = bound_row(iz, p.nz, nbl, p.periodic);
  R dx2 = (R)p.dx * (R)p.dx, dy2 = (R)p.dy * (R)p.dy, dz2 = (R)p.dz * (R)p.dz;
  R val = R(0);
  for (int i = 0; i < wl; ++i) {
    R cx, cy, cz;
    if (p.laplace == 0) { cx = (R)O::lap0(bx, i); cy = (R)O::lap0(by, i); cz = (R)O::lap0(bz, i); }
    else if (p.laplace == 1) { cx = (R)O::lap1(bx, i); cy = (R)O::lap1(by, i); cz = (R)O::lap1(bz, i); }
    else { cx = (R)O::lap2(bx, i); cy = (R)O::lap2(by, i); cz = (R)O::lap2(bz, i); }
    val = val + cx * f[at_dir(p, ix, iy, iz, 0, i - c)] / dx2 + cy * f[at_dir(p, ix, iy, iz, 1, i - c)] / dy2 +
          cz * f[at_dir(p, ix, iy, iz, 2, i - c)] / dz2;
  }
  return val;
}

template <typename R, int OPS> __global__ __launch_bounds__(BX* BY) void k_lap(Params p, Range g, const R* f, R* out) {
  IEQ_NODE_PREAMBLE(p.bnodes)
  out[idx] = lap_node<R, OPS>(p, f, ix, iy, iz);
}

// projector_divcleaning (kernel_div_cleaning.cl:96-109): B +/- grad(phi), .xyz only
template <typename R, int OPS, bool ADJ, typename I> __global__ __launch_bounds__(256) void k_proj(Params p, ColumnGrid cg, R* b, const R* phi) {
  IEQ_RUN_PREAMBLE(0)
  const R* f = phi + iz * nxy;
  R* q = b + iz * nxy;
  const R vx = node_ld(q, o), vy = node_ld(q + S, o), vz = node_ld(q + 2 * S, o);
  const V3<R> d = line_derivs<R, OPS, ADJ>(p, ix, iy, iz, f, f, f, o, tab);
  const R sgn = ADJ ? R(-1) : R(1);
  if (jt < (P)cg.gxy) {
    node_st(q, o, vx + sgn * d.x);
    node_st(q + S, o, vy + sgn * d.y);
    node_st(q + 2 * S, o, vz + sgn * d.z);
  }
}

template <typename R, int OPS, bool ADJ, typename I> __global__ __launch_bounds__(256) void k_proj_column(Params p, ColumnGrid cg, R* b, const R* phi) {
  IEQ_COLUMN_PREAMBLE(0)
  const R sgn = ADJ ? R(-1) : R(1);
  Column<R, OPS, ADJ, I> c;
  c.init(p, ix, iy);
  c.planes(p, z0, z1, [&](auto x, auto y, auto z, int iz) {
    const R* f = phi + iz * nxy;
    R *bx = b + iz * nxy, *by = bx + S, *bz = by + S;
    const R vx = node_ld(bx, c.o), vy = node_ld(by, c.o), vz = node_ld(bz, c.o);
    const R dx = c.template dx<x.value>(p, f), dy = c.template dy<y.value>(p, f), dz = c.template dz<z.value>(p, f, iz);
    node_st(bx, c.o, vx + sgn * dx);
    node_st(by, c.o, vy + sgn * dy);
    node_st(bz, c.o, vz + sgn * dz);
  });
}

// calc_axpy (x = a x + y) / calc_xpay (x = x + a y), kernel_CG.cl:8-30
template <typename R> __global__ __launch_bounds__(BX* BY) void k_axpy(Params p, Range g, R* x, const R* y, const R* a, int xpay) {
  IEQ_NODE_PREAMBLE(p.bnodes)
  R av = a[0];
  x[idx] = xpay ? x[idx] + av * y[idx] : av * x[idx] + y[idx];
}

// Group reductions: output[g] = sum over the W_SIZE nodes of group g of
//   which 0: fac*|B|^2 (norm2), 1: fac*|B1-B2|^2 (norm2_diff), 2: fac*s^2 (norm2_S), 3: a*b (dot_product)
// with fac the SBP norm weight prod_d dx_d / M_INV[row_d] (kernel_operator.cl:11-137), accumulated in
// double.
template <typename R, int OPS>
__global__ __launch_bounds__(256) void k_group_reduce(Params p, const R* a, const R* b, R* out, int which, long long wsize,
                                                      long long nnodes) {
  using O = Op<OPS>;
  __shared__ double part[256];
  const long long g0 = (long long)blockIdx.x * wsize;
  double acc = 0.0;
  const long long S = p.stride;
  const long long nxy = (long long)p.nx * p.ny;
  for (long long l = threadIdx.x; l < wsize; l += blockDim.x) {
    long long gid = g0 + l;
    if (gid >= nnodes) continue;  // padding nodes hold zeros
    // every product formed in double (FP32 programs widen the nodal values first); only the group
    // partial is rounded to REAL, as the reference's output array is REAL
    double v;
    if (which == 3) {
      v = (double)a[gid] * (double)b[gid];
    } else {
      uint32_t iz = (uint32_t)(gid / nxy), iy = (uint32_t)((gid - iz * nxy) / p.nx), ix = (uint32_t)(gid - iy * p.nx - iz * nxy);
      const double fac = (p.dx / O::minv(bound_row(ix, p.nx, O::NB, p.periodic))) *
                         (p.dy / O::minv(bound_row(iy, p.ny, O::NB, p.periodic))) *
                         (p.dz / O::minv(bound_row(iz, p.nz, O::NB, p.periodic)));
      double q;
      if (which == 0) {
        const double fx = a[gid], fy = a[S + gid], fz = a[2 * S + gid];
        q = fx * fx + fy * fy + fz * fz;
      } else if (which == 1) {
        const double fx = (double)a[gid] - (double)b[gid], fy = (double)a[S + gid] - (double)b[S + gid],
                     fz = (double)a[2 * S + gid] - (double)b[2 * S + gid];
        q = fx * fx + fy * fy + fz * fz;
      } else {
        const double f = a[gid];
        q = f * f;
      }
      v = fac * q;
    }
    acc += v;
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = (R)part[0];
}

// AoS REAL4 <-> SoA conversion (the reference host layout <-> this library's).
template <typename R> __global__ void k_aos_to_soa(const R* aos, R* soa, long long n, long long stride) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  soa[i] = aos[4 * i];
  soa[stride + i] = aos[4 * i + 1];
  soa[2 * stride + i] = aos[4 * i + 2];
}
template <typename R> __global__ void k_soa_to_aos(const R* soa, R* aos, long long n, long long stride) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  aos[4 * i] = soa[i];
  aos[4 * i + 1] = soa[stride + i];
  aos[4 * i + 2] = soa[2 * stride + i];
  aos[4 * i + 3] = R(0);
}

dim3 grid_of(Range g) { return dim3((g.x + BX - 1) / BX, (g.y + BY - 1) / BY, g.z); }

}  // namespace

// ----------------------------------------------------------------------------------
// Host launchers (dispatch the operator set at run time).

#define IEQ_OPS_SWITCH(ops, CALL) \
  switch (ops) {                  \
    case 0: { constexpr int OPS = 0; CALL; } break; \
    case 1: { constexpr int OPS = 1; CALL; } break; \
    case 2: { constexpr int OPS = 2; CALL; } break; \
    case 3: { constexpr int OPS = 3; CALL; } break; \
    case 4: { constexpr int OPS = 4; CALL; } break; \
    default: { constexpr int OPS = 5; CALL; } break; \
  }

// Whether the column kernels run an operator, or a thread per node.  A column finds the rows of a thread's nodes once and
// runs whole planes without a branch, but holds the rows in registers, and on a wave that touches a face takes general
// rows for all its lanes.  Columns / thread per node, us: FP32 bounded, div: 4th order 192^3 33 / 49, 256^3 62 / 109; 6th
// extended 1000 x 8 x 200 42 / 21, 500 x 500 x 8 49 / 27; FP64 div: 2nd order 192^3 35 / 42, 4th 1000 x 8 x 200 36 / 19; 6th 128^3 56 / 33,
// 256^3 482 / 254; projection, 6th extended, 1000 x 8 x 200 127 / 38.  Below 1.8 M nodes they are alike or the thread wins.
template <typename R, int OPS> constexpr bool has_columns() { return sizeof(R) == 4 || Op<OPS>::W <= 7; }
bool columns_pay(const Params& p) { return std::min(p.ny, p.nz) >= 32 && (long long)p.nx * p.ny * p.nz >= 1800000; }

#define IEQ_COLUMN_SWITCH(R, p, ops, g, COLUMN, NODE)                \
  const bool wide = wide_plane<R>(p), columns = columns_pay(p);      \
  IEQ_OPS_SWITCH(ops, {                                              \
    bool done = false;                                               \
    if constexpr (has_columns<R, OPS>()) {                           \
      if (columns) {                                                 \
        const ColumnGrid cg = column_grid(g, 16);                    \
        if (wide) { using I = long long; COLUMN; }                   \
        else { using I = unsigned; COLUMN; }                         \
        done = true;                                                 \
      }                                                              \
    }                                                                \
    const ColumnGrid cg = column_grid(g, 1);                         \
    if (!done && wide) { using I = long long; NODE; }                \
    else if (!done) { using I = unsigned; NODE; }                    \
  })

template <typename R>
void gen_update_2r(const Params& p, hipStream_t s, const uint32_t g[3], R* X, R* O, const R* D, R a, R b, R* time, double tc) {
  Range r{g[0], g[1], g[2]};
  k_update_2r<R><<<grid_of(r), dim3(BX, BY), 0, s>>>(p, r, X, O, D, a, b, time, tc);
}

template <typename R>
void gen_update_2n(const Params& p, hipStream_t s, const uint32_t g[3], R* X, const R* D, R b, R* time, double tc) {
  Range r{g[0], g[1], g[2]};
  k_update_2n<R><<<grid_of(r), dim3(BX, BY), 0, s>>>(p, r, X, D, b, time, tc);
}

template <typename R> void gen_ssprk104_06(const Params& p, hipStream_t s, const uint32_t g[3], const R* b1, R* b2, R* b3, R* time) {
  Range r{g[0], g[1], g[2]};
  k_ssprk104_06<R><<<grid_of(r), dim3(BX, BY), 0, s>>>(p, r, b1, b2, b3, time);
}

template <typename R> void gen_time(hipStream_t s, R* time, double c, double dt, int mode) {
  k_time<R><<<1, 64, 0, s>>>(time, c, dt, mode);
}

template <typename R> void gen_init(const Params& p, hipStream_t s, const uint32_t g[3], R* f, int which, const R* time) {
  Range r{g[0], g[1], g[2]};
  k_init<R><<<grid_of(r), dim3(BX, BY), 0, s>>>(p, r, f, which, time);
}

template <typename R> void gen_div(const Params& p, int ops, hipStream_t s, const uint32_t g[3], const R* b, R* out, int off) {
  IEQ_COLUMN_SWITCH(R, p, ops, g, (k_div_column<R, OPS, I><<<cg.rows(), 256, 0, s>>>(p, cg, b, out, off)),
                    (k_div<R, OPS, I><<<cg.rows(), 256, 0, s>>>(p, cg, b, out, off)))
}

template <typename R> void gen_div_norm2(const Params& p, int ops, hipStream_t s, const R* b, double* part, double* out) {
  const long long runs = ((long long)p.nx * p.ny + 255) / 256;
  const int segs = (int)std::min<long long>(runs, kNormBlocks), most = kNormBlocks / segs, zc = (p.nz + most - 1) / most;
  const int nb = segs * ((p.nz + zc - 1) / zc);
  IEQ_OPS_SWITCH(ops, (k_div_norm<R, OPS><<<nb, 256, 0, s>>>(p, segs, zc, b, part)))
  k_sum<<<1, 256, 0, s>>>(part, nb, out);
}

// calc_curl as columns where they beat k_node_pre_flat, us: FP32 bounded 2nd order 160^3 24 / 26, 192^3 37 / 40, 200^3 42 / 46,
// 256^3 120 / 111; 2nd extended 192^3 42 / 48, 200^3 45 / 52, 256^3 151 / 136.
template <typename R> bool gen_curl(const Params& p, int ops, hipStream_t s, const uint32_t g[3], const R* b, R* out) {
  if (sizeof(R) != 4 || p.periodic || !columns_pay(p) || (long long)p.nx * p.ny * p.nz > 12000000 || (ops != 0 && ops != 3)) return false;
  const ColumnGrid cg = column_grid(g, 16);
  if (ops == 0) k_curl_column<float, 0><<<cg.rows(), 256, 0, s>>>(p, cg, (const float*)b, (float*)out);
  else k_curl_column<float, 3><<<cg.rows(), 256, 0, s>>>(p, cg, (const float*)b, (float*)out);
  return true;
}

template <typename R> void gen_grad(const Params& p, int ops, hipStream_t s, const uint32_t g[3], const R* f, R* out) {
  IEQ_COLUMN_SWITCH(R, p, ops, g, (k_grad_column<R, OPS, I><<<cg.rows(), 256, 0, s>>>(p, cg, f, out)),
                    (k_grad<R, OPS, I><<<cg.rows(), 256, 0, s>>>(p, cg, f, out)))
}

template <typename R> void gen_lap(const Params& p, int ops, hipStream_t s, const uint32_t g[3], const R* f, R* out) {
  Range r{g[0], g[1], g[2]};
  IEQ_OPS_SWITCH(ops, (k_lap<R, OPS><<<grid_of(r), dim3(BX, BY), 0, s>>>(p, r, f, out)))
}

template <typename R> void gen_proj(const Params& p, int ops, hipStream_t s, const uint32_t g[3], R* b, const R* phi) {
  if (p.laplace == 2) {
    IEQ_COLUMN_SWITCH(R, p, ops, g, (k_proj_column<R, OPS, true, I><<<cg.rows(), 256, 0, s>>>(p, cg, b, phi)),
                      (k_proj<R, OPS, true, I><<<cg.rows(), 256, 0, s>>>(p, cg, b, phi)))
  } else {
    IEQ_COLUMN_SWITCH(R, p, ops, g, (k_proj_column<R, OPS, false, I><<<cg.rows(), 256, 0, s>>>(p, cg, b, phi)),
                      (k_proj<R, OPS, false, I><<<cg.rows(), 256, 0, s>>>(p, cg, b, phi)))
  }
}

template <typename R> void gen_axpy(const Params& p, hipStream_t s, const uint32_t g[3], R* x, const R* y, const R* a, int xpay) {
  Range r{g[0], g[1], g[2]};
  k_axpy<R><<<grid_of(r), dim3(BX, BY), 0, s>>>(p, r, x, y, a, xpay);
}

template <typename R>
void gen_group_reduce(const Params& p, int ops, hipStream_t s, const R* a, const R* b, R* out, int which, long long wsize,
                      long long ngroups, long long nnodes) {
  IEQ_OPS_SWITCH(ops, (k_group_reduce<R, OPS><<<(unsigned)ngroups, 256, 0, s>>>(p, a, b, out, which, wsize, nnodes)))
}

template <typename R> void gen_aos_to_soa(hipStream_t s, const R* aos, R* soa, long long n, long long stride) {
  if (n > 0) k_aos_to_soa<R><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(aos, soa, n, stride);
}
template <typename R> void gen_soa_to_aos(hipStream_t s, const R* soa, R* aos, long long n, long long stride) {
  if (n > 0) k_soa_to_aos<R><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(soa, aos, n, stride);
}

#define IEQ_INSTANTIATE(R)                                                                                                   \
  template void gen_update_2r<R>(const Params&, hipStream_t, const uint32_t*, R*, R*, const R*, R, R, R*, double);           \
  template void gen_update_2n<R>(const Params&, hipStream_t, const uint32_t*, R*, const R*, R, R*, double);                  \
  template void gen_ssprk104_06<R>(const Params&, hipStream_t, const uint32_t*, const R*, R*, R*, R*);                        \
  template void gen_time<R>(hipStream_t, R*, double, double, int);                                                           \
  template void gen_init<R>(const Params&, hipStream_t, const uint32_t*, R*, int, const R*);                                 \
  template void gen_div<R>(const Params&, int, hipStream_t, const uint32_t*, const R*, R*, int);                             \
  template void gen_div_norm2<R>(const Params&, int, hipStream_t, const R*, double*, double*);                              \
  template bool gen_curl<R>(const Params&, int, hipStream_t, const uint32_t*, const R*, R*);                                 \
  template void gen_grad<R>(const Params&, int, hipStream_t, const uint32_t*, const R*, R*);                                 \
  template void gen_lap<R>(const Params&, int, hipStream_t, const uint32_t*, const R*, R*);                                  \
  template void gen_proj<R>(const Params&, int, hipStream_t, const uint32_t*, R*, const R*);                                 \
  template void gen_axpy<R>(const Params&, hipStream_t, const uint32_t*, R*, const R*, const R*, int);                       \
  template void gen_group_reduce<R>(const Params&, int, hipStream_t, const R*, const R*, R*, int, long long, long long,      \
                                    long long);                                                                              \
  template void gen_aos_to_soa<R>(hipStream_t, const R*, R*, long long, long long);                                         \
  template void gen_soa_to_aos<R>(hipStream_t, const R*, R*, long long, long long);

IEQ_INSTANTIATE(double)
IEQ_INSTANTIATE(float)

}  // namespace ieq
