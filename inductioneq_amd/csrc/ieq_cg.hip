// Conjugate-gradient divergence cleaning with device-side alpha/beta.
//
// Restates the host loop of matlab/+divergence_cleaning/clean_div_CG.m:31-86
// (calc_div_divcleaning -> r; repeat { u = beta u + r; q = -Lap u; alpha = rr/(u.q);
// phi += alpha u; r -= alpha q; rr = r.r } while rr > thr^2 and it < max; projection)
// as two kernels per iteration with all scalars kept on the device:
//   k_cg_lap     rr = r.r (sum of the previous update's partials), the stop test,
//                u' = beta*u + r (beta = rr/old, old = 1 at start), q = -Lap u' on the
//                BNODES interior, partial u'.q  (u' goes to the other direction register)
//   k_cg_update  alpha = rr / u'.q (sum of the Laplacian's partials), phi += alpha u',
//                r -= alpha q, partial r.r
// Dot products accumulate in FP64 whatever the field precision: every block writes its
// partial, and every block of the next kernel sums all partials in the same fixed order, so
// all blocks agree on alpha (beta) bit for bit and the result is deterministic.  rr of
// iteration i is kept in slot i % 2 of the device state, so the block that records it never
// overwrites the value the other blocks of the same launch read.  Once the stop test holds,
// every kernel returns immediately, so any number of iterations can be enqueued without a
// host round trip and the result equals stopping exactly at convergence.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "ieq_cg.hpp"
#include "ieq_device.hpp"
#include "ieq_generic.hpp"
#include "ieq_stencil.hpp"

namespace ieq {

struct CgState {
  double rr, old, alpha, rr0;
  double tol2;       // stop when rr <= tol2 ...
  double rel2;       // ... or rr <= rel2 * rr0 (rel2 = 0: absolute test only)
  double rrs[2];     // r.r of iteration i in slot i % 2 (slot 1 starts at 1: old of iteration 0)
  int it, max_it, done, pad;
};

namespace {

constexpr int kBlk = 256;
constexpr int kAhead = 6;              // iterations the host launches ahead of the device (one takes 10 us or more, the host 6 us to launch it)
constexpr long long kNodeLap = 150000;  // interior nodes up to which the Laplacian runs with a thread per node
constexpr int kLapRows = 32;  // table rows held in LDS by k_cg_lap (2 * NUM_BOUNDS + 1 of the Laplacian)

// Deterministic block reduction of one double (wave64 shuffles, then LDS).
__device__ inline double block_sum(double v, double* smem) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int tid = threadIdx.y * blockDim.x + threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int nw = (blockDim.x * blockDim.y + 63) >> 6;
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  double t = 0.0;
  if (wid == 0) {
    t = lane < nw ? smem[lane] : 0.0;
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  }
  __syncthreads();
  return t;  // valid in wave 0
}

// This thread's share of a sum of partials, four loads in flight.
__device__ inline double own_partials(const double* part, unsigned int n) {
  double v = 0.0;
  const int tid = threadIdx.y * blockDim.x + threadIdx.x, nt = blockDim.x * blockDim.y;
  for (unsigned int i = tid; i < n; i += 4 * nt) {
    double x[4];
#pragma unroll
    for (unsigned int k = 0; k < 4; ++k) x[k] = part[min(i + k * nt, n - 1)];
#pragma unroll
    for (unsigned int k = 0; k < 4; ++k) v += i + k * nt < n ? x[k] : 0.0;
  }
  return v;
}
__device__ inline double sum_partials(const double* part, unsigned int n, double* smem) {
  return block_sum(own_partials(part, n), smem);
}

// The block's sum of v, returned to every thread (smem: at least 17 doubles).
__device__ inline double block_sum_all(double v, double* smem) {
  const double t = block_sum(v, smem);
  if (threadIdx.x == 0 && threadIdx.y == 0) smem[16] = t;
  __syncthreads();
  const double all = smem[16];
  __syncthreads();
  return all;
}

constexpr int kMaxHW = 7;
template <typename R> struct LapArgs {
  int nx, ny, nz, off;  // grid and BNODES
  int zc;               // planes per block
  int nbl, wl;          // table rows per side, width
  const double* tab;    // (2nbl+1) x wl, device copy
  double idx2, idy2, idz2;
  R cz[2 * kMaxHW + 1];  // central row of the table / dz^2, as REAL, offsets -hw .. hw
};

// The iteration's rr from the previous update's partials (the initial residual's for iteration 0), the
// stop test and beta = rr / old (clean_div_CG.m:45-48), the same in every block; false once stopped.  The
// host follows `progress` (host memory): iteration + 1, negative once stopped.  own: this thread's share of the
// partials.
__device__ inline bool cg_direction(CgState* st, double own, int iter, int* progress, double* red, double& beta) {
  const double rr = block_sum_all(own, red);
  const double old = st->rrs[(iter + 1) & 1];
  const bool go = rr > st->tol2 && (st->rel2 <= 0.0 || rr > st->rel2 * st->rr0) && iter < st->max_it;
  if (threadIdx.x == 0 && threadIdx.y == 0 && blockIdx.x == 0) {
    st->rr = rr;
    st->old = old;
    st->it = iter;
    if (go) st->rrs[iter & 1] = rr;
    else st->done = 1;
    __hip_atomic_store(progress, go ? iter + 1 : -(iter + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  beta = rr / old;
  return go;
}

// Fused direction update and Laplacian on [off, n-off)^3:
//   u' = beta u + r (beta = rr/old),  q = -Lap u',  partial u'.q
// u' is written to a second buffer (neighbouring blocks still read u), so the direction
// registers alternate between iterations.  Outside the interior u and r are 0 (never
// written), so u' is 0 there as in the reference, where calc_axpy runs on the interior
// only; neighbours outside the grid count as 0 (their coefficients are 0).
// z-march: u' of the own column's z-stencil lives in a register window, one xy-plane plus
// halo at a time in LDS (double-buffered).  Loads are issued PD planes ahead of their use:
// they always target a valid node (coordinates clamped into the grid) and land in raw
// (u, r) registers; the masking and beta u + r happen only when a plane is used, so no
// load is waited for before it is needed.  The per-plane barrier orders LDS traffic only.
// The halo cells are numbered along the halo and thread i loads cell i (y rows first, so a
// wave reads whole rows), one (u, r) pair per thread and plane instead of one pair for an x
// cell and one for a y cell that most threads do not have.
// What bounds it is the sum of LDS reads, L1 accesses and FMAs of a plane, not its latency (tiles
// from 64 x 4 to 64 x 16 measure the same), so the z row comes from scalar registers except on
// boundary planes and the centre from the window: 16 LDS reads a node and plane instead of 27
// (192^3 FP32, half-width 4: 37.8 -> 33.5 us; its four fields once take 23 us as a copy).  Stepping phi here, where
// u is at hand, spares the update a field but costs more than it saves (192^3, an iteration: FP32 63.4 -> 67.0 us,
// FP64 122.9 -> 134.3).  A second plane in flight gives nothing.
// Tiles are handed out per XCD in contiguous ranges (x fastest, then y, then z-chunk), so
// the halo rows of y-neighbours are read through one L2.
template <typename R, int HW, int TY, int PD, int TX>
__global__ __launch_bounds__(TX * TY) void k_cg_lap(LapArgs<R> a, const R* __restrict__ u, const R* __restrict__ r,
                                                    R* __restrict__ un, R* __restrict__ q, CgState* st,
                                                    const double* rr_part, unsigned int n_rr, double* part, int iter,
                                                    int* progress) {
  constexpr int LX = TX + 2 * HW, LY = TY + 2 * HW, Q = 2 * HW + 1, NT = TX * TY;
  constexpr int NYH = 2 * HW * TX, NHALO = NYH + 2 * HW * TY, NH = (NHALO + NT - 1) / NT;  // halo cells, per thread
  __shared__ R s[2][LY * LX];
  __shared__ double red[17];
  if (st->done) return;
  double beta_d;
  if (!cg_direction(st, own_partials(rr_part, n_rr), iter, progress, red, beta_d)) return;
  const R beta = (R)beta_d;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = tx + TX * ty;
  const int gx = a.nx - 2 * a.off, gy = a.ny - 2 * a.off, gz = a.nz - 2 * a.off;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ntx = (gx + TX - 1) / TX, nty = (gy + TY - 1) / TY;
  const int bx = tile % ntx, by = (tile / ntx) % nty, bz = tile / (ntx * nty);
  const int x0 = a.off + bx * TX, y0 = a.off + by * TY, x = x0 + tx, y = y0 + ty;
  const bool active = (x - a.off) < gx && (y - a.off) < gy;
  const unsigned RB = sizeof(R);
  const unsigned plb = (unsigned)(a.nx * a.ny) * RB;
  auto cl = [](int v, int n) { return v < 0 ? 0 : (v >= n ? n - 1 : v); };
  auto inb = [](int v, int n) { return (unsigned)v < (unsigned)n; };
  // In-plane byte offsets (clamped) and in-grid masks of the column and of this thread's halo cells; a
  // thread without one re-reads a fixed node, so the memory counter is the same on every path.
  const unsigned oc = (unsigned)(cl(x, a.nx) + a.nx * cl(y, a.ny)) * RB;
  const bool colin = inb(x, a.nx) && inb(y, a.ny);
  unsigned oh[NH];
  int lh[NH];  // LDS index of the cell, -1: none
  bool mh[NH];
#pragma unroll
  for (int k = 0; k < NH; ++k) {
    const int h = tid + k * NT, hx = h - NYH;
    int lx, ly;
    if (h < NYH) {
      const int row = h / TX;
      lx = h % TX;
      ly = row < HW ? row - HW : TY + row - HW;
    } else {
      const int col = hx % (2 * HW);
      lx = col < HW ? col - HW : TX + col - HW;
      ly = hx / (2 * HW);
    }
    lh[k] = h < NHALO ? (ly + HW) * LX + lx + HW : -1;
    mh[k] = inb(x0 + lx, a.nx) && inb(y0 + ly, a.ny);
    oh[k] = h < NHALO ? (unsigned)(cl(x0 + lx, a.nx) + a.nx * cl(y0 + ly, a.ny)) * RB : 0u;
  }
  // per-thread x/y rows
  R cx[Q], cy[Q];
  {
    const int rx = bound_row((uint32_t)x, (uint32_t)a.nx, a.nbl, 0), ry = bound_row((uint32_t)y, (uint32_t)a.ny, a.nbl, 0);
    const int c0 = (a.wl - 1) / 2;
    double tcx[Q], tcy[Q];  // unconditional loads (clamped column), masked below
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const int j = min(max(c0 - HW + k, 0), a.wl - 1);
      tcx[k] = a.tab[rx * a.wl + j];
      tcy[k] = a.tab[ry * a.wl + j];
    }
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const int j = c0 - HW + k;
      cx[k] = (j >= 0 && j < a.wl) ? (R)(tcx[k] * a.idx2) : R(0);
      cy[k] = (j >= 0 && j < a.wl) ? (R)(tcy[k] * a.idy2) : R(0);
    }
  }
  // z rows of the table, scaled by 1/dz^2 and rounded to REAL once (uniform per plane)
  __shared__ R sz[kLapRows][Q];
  {
    const int rows = 2 * a.nbl + 1, c0 = (a.wl - 1) / 2;
    for (int i = tid; i < rows * Q; i += NT) {
      const int row = i / Q, k = i % Q, j = c0 - HW + k;
      sz[row][k] = (j >= 0 && j < a.wl) ? (R)(a.tab[row * a.wl + j] * a.idz2) : R(0);
    }
  }
  double dot = 0.0;
  const int z0 = a.off + bz * a.zc;
  const int zn = min(a.zc, gz - bz * a.zc);
  // u' from raw values (0 outside the grid)
  auto dir = [&](R uu, R rr, bool in) { return in ? beta * uu + rr : R(0); };
  // Raw loads ride in NS = PD+1 register slots that rotate with the plane index: the
  // column value of plane z0+HW+1+m and the halo of plane z0+m sit in slot m % NS.  The
  // z-loop is unrolled NS times so every slot index is a compile-time constant: a register
  // with a load in flight is never copied (a copy would wait for the load).
  constexpr int NS = PD + 1;
  static_assert(NS >= 2 && NS <= 4, "1 <= PD <= 3");
  R w[Q];                          // u' of the column, planes z-HW .. z+HW
  R lu[NS], lr[NS];                // raw column values
  R hu[NS][NH], hrw[NS][NH];       // raw halo values
  auto load_col = [&](R& uu, R& rr, int zz) {
    const unsigned o = oc + (unsigned)cl(zz, a.nz) * plb;
    uu = ldo(u, o);
    rr = ldo(r, o);
  };
  auto load_halo = [&](R* uu, R* rr, int zz) {  // unconditional: every path issues 2*NH loads
    const unsigned pz = (unsigned)cl(zz, a.nz) * plb;
#pragma unroll
    for (int k = 0; k < NH; ++k) {
      uu[k] = ldo(u, oh[k] + pz);
      rr[k] = ldo(r, oh[k] + pz);
    }
  };
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    R uu, rr;
    load_col(uu, rr, z0 - HW + j);
    w[j] = dir(uu, rr, colin && inb(z0 - HW + j, a.nz));
  }
  // first PD planes in flight, in the order the z-loop issues them (halo, then column); the
  // scheduling barriers keep that order, which the memory-counter waits in the loop rely on
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int m = 0; m < PD; ++m) {
    load_halo(hu[m], hrw[m], z0 + m);
    load_col(lu[m], lr[m], z0 + HW + 1 + m);
    __builtin_amdgcn_sched_barrier(0);
  }
  auto body = [&](auto slot, int zi) {
    constexpr int S = decltype(slot)::value, SN = (S + PD) % NS;
    const int z = z0 + zi;
    R* sp = s[zi & 1];
    sp[(ty + HW) * LX + tx + HW] = w[HW];
#pragma unroll
    for (int k = 0; k < NH; ++k)
      if (lh[k] >= 0) sp[lh[k]] = dir(hu[S][k], hrw[S][k], mh[k]);
    // loads PD planes ahead (halo first), in flight across PD barriers and computes; past the
    // chunk they read a clamped plane and are never used
    load_halo(hu[SN], hrw[SN], z + PD);
    load_col(lu[SN], lr[SN], z + HW + 1 + PD);
    lds_barrier();
    if (active && zi < zn) {
      const int rz = bound_row((uint32_t)z, (uint32_t)a.nz, a.nbl, 0);
      const R *sx = sp + (ty + HW) * LX + tx, *sy = sp + ty * LX + tx + HW;
      auto apply = [&](auto zrow) {
        R acc = R(0);
#pragma unroll
        for (int k = 0; k < Q; ++k)
          acc = acc + cx[k] * (k == HW ? w[HW] : sx[k]) + cy[k] * (k == HW ? w[HW] : sy[k * LX]) + zrow(k) * w[k];
        return acc;
      };
      const R acc = rz == a.nbl ? apply([&](int k) { return a.cz[k]; }) : apply([&](int k) { return sz[rz][k]; });
      const unsigned o = oc + (unsigned)z * plb;
      sto(un, o, w[HW]);
      sto(q, o, acc);
      dot += (double)w[HW] * (double)acc;
    }
    // advance: the window takes plane z+HW+1 (slot S, issued PD iterations ago)
#pragma unroll
    for (int j = 0; j < Q - 1; ++j) w[j] = w[j + 1];
    w[Q - 1] = dir(lu[S], lr[S], colin && inb(z + HW + 1, a.nz));
  };
  // Whole groups of NS planes (the host makes the chunk a multiple of NS; a shorter last
  // chunk runs its trailing planes without output), so every path issues the same loads.
  for (int zb = 0; zb < zn; zb += NS) {
    body(std::integral_constant<int, 0>{}, zb);
    body(std::integral_constant<int, 1 % NS>{}, zb + 1);
    if constexpr (NS > 2) body(std::integral_constant<int, 2 % NS>{}, zb + 2);
    if constexpr (NS > 3) body(std::integral_constant<int, 3 % NS>{}, zb + 3);
  }
  const double bs = block_sum(dot, red);
  if (tx == 0 && ty == 0) part[tile] = bs;
}

// The same with a thread per node, for grids with too few tiles to fill the chip: a block takes 64
// consecutive nodes of an interior xy-plane, three of its waves the stencil along one direction each and
// the fourth the node itself.  All loads are in flight while the partials are summed.  40^3 FP64,
// half-width 4: 7.0 us, where the z-march takes 22 us in 15 workgroups.
template <typename R, int HW>
__global__ __launch_bounds__(256) void k_cg_lap_node(LapArgs<R> a, const R* __restrict__ u, const R* __restrict__ r, R* __restrict__ un,
                                                     R* __restrict__ q, CgState* st, const double* rr_part, unsigned int n_rr,
                                                     double* part, int iter, int* progress) {
  constexpr int Q = 2 * HW + 1;
  __shared__ double red[17];
  __shared__ R sum[3][64];
  const int done = st->done;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int gx = a.nx - 2 * a.off, gxy = gx * (a.ny - 2 * a.off), segs = (gxy + 63) / 64;
  const int tile = xcd_tile(blockIdx.x, gridDim.x), zt = tile / segs, jt = (tile - zt * segs) * 64 + lane, j = min(jt, gxy - 1);
  const int i3[3] = {a.off + j % gx, a.off + j / gx, a.off + zt}, n3[3] = {a.nx, a.ny, a.nz};
  const int nxy = a.nx * a.ny, st3[3] = {1, a.nx, nxy};
  const unsigned o = (unsigned)(i3[0] + a.nx * i3[1] + nxy * i3[2]) * (unsigned)sizeof(R);
  const int d = wave < 3 ? wave : 0, i = wave == 0 ? i3[0] : wave == 1 ? i3[1] : i3[2], n = n3[d];
  R uu[Q], rr[Q];
  double tc[Q];
  if (wave < 3) {
#pragma unroll
    for (int k = -HW; k <= HW; ++k) {  // outside the grid: the node itself, with a zero below
      const unsigned ok = o + (unsigned)((unsigned)(i + k) < (unsigned)n ? k * st3[d] : 0) * (unsigned)sizeof(R);
      uu[k + HW] = ldo(u, ok);
      rr[k + HW] = ldo(r, ok);
    }
    const double* row = a.tab + bound_row((uint32_t)i, (uint32_t)n, a.nbl, 0) * a.wl + (a.wl - 1) / 2 - HW;  // wl = Q
#pragma unroll
    for (int k = 0; k < Q; ++k) tc[k] = row[k];
  } else {
    uu[HW] = ldo(u, o);
    rr[HW] = ldo(r, o);
  }
  const double own = own_partials(rr_part, n_rr);
  if (done) return;
  double beta_d;
  if (!cg_direction(st, own, iter, progress, red, beta_d)) return;
  const R beta = (R)beta_d;
  if (wave < 3) {
    const double ih2 = d == 0 ? a.idx2 : d == 1 ? a.idy2 : a.idz2;
    R acc = R(0);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const R v = (unsigned)(i + k - HW) < (unsigned)n ? beta * uu[k] + rr[k] : R(0);
      acc = acc + (R)(tc[k] * ih2) * v;
    }
    sum[d][lane] = acc;
  }
  __syncthreads();
  if (wave < 3) return;
  const R w = beta * uu[HW] + rr[HW], acc = (sum[0][lane] + sum[1][lane]) + sum[2][lane];
  double dot = 0.0;
  if (jt < gxy) {
    sto(un, o, w);
    sto(q, o, acc);
    dot = (double)w * (double)acc;
  }
  for (int k = 32; k > 0; k >>= 1) dot += __shfl_xor(dot, k, 64);
  if (lane == 0) part[tile] = dot;
}

// One workgroup, after the last enqueued iteration when the stop test never held: rr of the
// final update and the iteration count (what the next Laplacian launch would record).
__global__ __launch_bounds__(256) void k_cg_finish(const double* rr_part, unsigned int n, CgState* st, int iter) {
  __shared__ double red[16];
  if (st->done) return;
  const double rr = sum_partials(rr_part, n, red);
  if (threadIdx.x == 0) {
    st->old = st->rrs[(iter + 1) & 1];
    st->rr = rr;
    st->it = iter;
    st->done = 1;
  }
}

// Every block sums the Laplacian's u'.q partials in the same order (alpha = rr / u'.q).  The
// reductions run inside the bulk kernels: a "last block finishes" scheme would need a
// device-scope fence in every block, which on gfx950 writes back and invalidates the L2 of
// its XCD.
template <typename R>
__global__ __launch_bounds__(kBlk) void k_cg_update(R* __restrict__ phi, const R* __restrict__ u, R* __restrict__ r,
                                                    const R* __restrict__ q, long long n, CgState* st,
                                                    const double* uq_part, unsigned int n_uq, double* part, int iter) {
  __shared__ double red[17];
  // The first element's loads go out with those of the state and the partials (40^3 FP64: with the partials four at a time 4.4 -> 3.7 us).
  const int done = st->done;
  const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x, step = (long long)gridDim.x * blockDim.x;
  const bool in = i0 < n;
  const long long at = in ? i0 : 0;
  const R p0 = phi[at], u0 = u[at], r0 = r[at], q0 = q[at];
  __builtin_amdgcn_sched_barrier(0);
  const double rr = st->rrs[iter & 1], own = own_partials(uq_part, n_uq);
  if (done) return;
  const double alpha_d = rr / block_sum_all(own, red);
  if (threadIdx.x == 0 && blockIdx.x == 0) st->alpha = alpha_d;
  const R alpha = (R)alpha_d;
  double acc = 0.0;
  if (in) {
    phi[i0] = p0 + alpha * u0;
    const R rn = r0 + (-alpha) * q0;
    r[i0] = rn;
    acc = (double)rn * (double)rn;
  }
  for (long long i = i0 + step; i < n; i += step) {
    phi[i] = phi[i] + alpha * u[i];
    const R rn = r[i] + (-alpha) * q[i];
    r[i] = rn;
    acc += (double)rn * (double)rn;
  }
  const double bs = block_sum(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// r.r partials of the initial residual.
template <typename R>
__global__ __launch_bounds__(kBlk) void k_cg_init(const R* __restrict__ r, long long n, double* part) {
  __shared__ double red[16];
  double acc = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    acc += (double)r[i] * (double)r[i];
  const double bs = block_sum(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// State initialisation from the partials of k_cg_init.
__global__ __launch_bounds__(256) void k_cg_init_state(const double* part, unsigned int n, CgState* st, double tol2,
                                                       double rel2, int max_it) {
  __shared__ double red[16];
  const double rr = sum_partials(part, n, red);
  if (threadIdx.x == 0) {
    st->rr = rr;
    st->rr0 = rr;
    st->old = 1.0;  // clean_div_CG.m:43
    st->rrs[0] = 0.0;
    st->rrs[1] = 1.0;  // old of iteration 0
    st->alpha = 0.0;
    st->it = 0;
    st->max_it = max_it;
    st->tol2 = tol2;
    st->rel2 = rel2;
    st->done = (rr > tol2 && (rel2 <= 0.0 || rr > rel2 * rr) && max_it > 0) ? 0 : 1;
  }
}

constexpr int kLapPD = 1;  // planes of the Laplacian's z-march in flight per thread
// Shape of a Laplacian tile (TX x TY threads) for stencil half-width hw: 32 x 16 up to hw = 5 (half-width 4,
// FP64 / FP32: 192^3 65.6 / 36.0 us, 128^3 and 96^3 22.7 / 15.2 us; 64 x 8 68.0 / 35.9 and 24.5 / 17.6 us; 64 x 16
// spills), 64 x 8 for the wider stencils.
constexpr int lap_ty(int hw) { return hw <= 5 ? 16 : 8; }
constexpr int lap_tx(int hw) { return hw <= 5 ? 32 : 64; }

// Launch of one iteration's Laplacian; zc = 0: a thread per node.
template <typename R, int HW>
void launch_lap(const LapArgs<R>& a, unsigned int blocks, const R* u, const R* r, R* un, R* q, CgState* st, const double* rr_part,
                unsigned int n_rr, double* part, int iter, int* progress, hipStream_t s) {
  constexpr int TX = lap_tx(HW), TY = lap_ty(HW);
  if (a.zc == 0) k_cg_lap_node<R, HW><<<blocks, 256, 0, s>>>(a, u, r, un, q, st, rr_part, n_rr, part, iter, progress);
  else k_cg_lap<R, HW, TY, kLapPD, TX><<<blocks, dim3(TX, TY), 0, s>>>(a, u, r, un, q, st, rr_part, n_rr, part, iter, progress);
}

// Planes per z-chunk: the smallest chunk whose grid fits in one round of resident
// workgroups (so no partial second round), at least 8 planes, rounded up to the kernel's
// group of PD+1 planes.
template <typename R, int HW, int TY> int lap_zc(int gx, int gy, int gz) {
  constexpr int TX = lap_tx(HW);
  int dev = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_cg_lap<R, HW, TY, kLapPD, TX>, TX * TY, 0) != hipSuccess ||
      cus <= 0 || per_cu <= 0)
    return 16;
  const long long xy = (long long)((gx + TX - 1) / TX) * ((gy + TY - 1) / TY);
  const long long resident = (long long)cus * per_cu;
  const long long chunks = std::max(1LL, resident / std::max(1LL, xy));
  const int ns = kLapPD + 1;  // the kernel's z-loop advances in groups of ns planes
  const int zc = std::max(8, (int)((gz + chunks - 1) / chunks));
  return (zc + ns - 1) / ns * ns;
}

}  // namespace

struct CgWork {
  void* buf = nullptr;  // r, u, q, u' (num_nodes each) + partials + state + table
  size_t bytes = 0;
  struct Host {         // pinned
    CgState st;
    double norm2;
    int progress;
  }* host = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
};

void cg_release(CgWork* w) {
  if (!w) return;
  if (w->buf) (void)hipFree(w->buf);
  if (w->host) (void)hipHostFree(w->host);
  if (w->e0) (void)hipEventDestroy(w->e0);
  if (w->e1) (void)hipEventDestroy(w->e1);
  delete w;
}

template <typename R>
int cg_run_t(const Params& p, const ieq_program_info& info, const double* host_tab, int nbl, int wl, hipStream_t s, CgWork** work,
             R* b, R* phi, double abs_thr, double rel_tol, int max_it, ieq_cg_result* res, std::string& err) {
  const long long n = info.num_nodes;
  const int hw = (wl - 1) / 2;
  if (hw < 1 || hw > kMaxHW || info.periodic || 2 * nbl + 1 > kLapRows || !offsets_fit(p.nx, p.ny, p.nz, sizeof(R)))
    return 1;  // not covered by the fused loop
  const int TX = lap_tx(hw), TY = lap_ty(hw);
  const int gx = p.nx - 2 * p.bnodes, gy = p.ny - 2 * p.bnodes, gz = p.nz - 2 * p.bnodes;
  // A thread per node up to kNodeLap interior nodes, the z-march beyond, where its tiles fill more of the chip
  // and it loads a node once instead of once per stencil point.  An iteration, node / z-march, FP32 and FP64:
  // half-width 4: 40^3 11.6 / 18.6 and 12.4 / 21.9 us, 56^3 19.2 / 20.2 and 21.1 / 23.2, 64^3 24.0 / 21.3 and
  // 27.3 / 24.2, 96^3 55.8 / 24.7 and 67.8 / 29.3; half-width 1: 40^3 10.4 / 14.1 and 10.7 / 16.1, 56^3
  // 16.5 / 15.2 and 17.5 / 17.2.
  int zc = 0;
  if (const char* e = getenv("IEQ_LAP_ZC")) zc = std::max(0, atoi(e));
  else if ((long long)gx * gy * gz > kNodeLap) switch (hw) {
    case 1: zc = lap_zc<R, 1, lap_ty(1)>(gx, gy, gz); break;
    case 2: zc = lap_zc<R, 2, lap_ty(2)>(gx, gy, gz); break;
    case 3: zc = lap_zc<R, 3, lap_ty(3)>(gx, gy, gz); break;
    case 4: zc = lap_zc<R, 4, lap_ty(4)>(gx, gy, gz); break;
    case 5: zc = lap_zc<R, 5, lap_ty(5)>(gx, gy, gz); break;
    case 6: zc = lap_zc<R, 6, lap_ty(6)>(gx, gy, gz); break;
    default: zc = lap_zc<R, 7, lap_ty(7)>(gx, gy, gz); break;
  }
  const unsigned int lap_blocks = zc > 0 ? (unsigned)(((gx + TX - 1) / TX) * ((gy + TY - 1) / TY) * ((gz + zc - 1) / zc))
                                         : (unsigned)((gx * gy + 63) / 64 * gz);
  const unsigned int vec_blocks = (unsigned)std::min<long long>(1024, (n + kBlk - 1) / kBlk);
  const size_t fbytes = ((size_t)info.stride * sizeof(R) + 255) / 256 * 256;
  // u'.q partials, then r.r partials (later the 1024 of the final divergence norm)
  const size_t part_bytes = ((size_t)(lap_blocks + 1024) * sizeof(double) + 255) / 256 * 256;
  const size_t tab_bytes = (size_t)(2 * nbl + 1) * wl * sizeof(double);
  const size_t need = 4 * fbytes + part_bytes + 512 + tab_bytes;
  if (!*work) *work = new CgWork();
  CgWork* w = *work;
  if (!w->host && hipHostMalloc(&w->host, sizeof(CgWork::Host)) != hipSuccess) return w->host = nullptr, err = "hipHostMalloc failed", -4;
  if (!w->e0 && hipEventCreate(&w->e0) != hipSuccess) return w->e0 = nullptr, err = "event creation failed", -4;
  if (!w->e1 && hipEventCreate(&w->e1) != hipSuccess) return w->e1 = nullptr, err = "event creation failed", -4;
  const bool fresh = w->bytes < need;
  if (fresh) {
    if (w->buf) (void)hipFree(w->buf);
    w->buf = nullptr;
    w->bytes = 0;
    if (hipMalloc(&w->buf, need) != hipSuccess) return w->buf = nullptr, err = "hipMalloc failed", -4;
    w->bytes = need;
  }
  char* base = (char*)w->buf;
  R* r = (R*)base;
  R* ub[2] = {(R*)(base + fbytes), (R*)(base + 3 * fbytes)};  // direction registers, alternating
  R* q = (R*)(base + 2 * fbytes);
  CgState* st = (CgState*)(base + 4 * fbytes);
  double* norm2 = (double*)((char*)st + 256);
  double* tab = (double*)((char*)st + 512);
  double* part_uq = tab + (2 * nbl + 1) * wl;
  double* part_rr = part_uq + lap_blocks;
  // The Laplacian writes interior nodes only, so u' and q stay 0 outside from call to call.  The first
  // direction (u of iteration 0) and the result start from 0 everywhere, and so does r outside the interior
  // (an alpha that is not finite has left a NaN there).
  if ((fresh && (hipMemsetAsync(base, 0, 4 * fbytes, s) != hipSuccess ||
                 hipMemcpyAsync(tab, host_tab, tab_bytes, hipMemcpyHostToDevice, s) != hipSuccess)) ||
      hipMemsetAsync(r, 0, 2 * fbytes, s) != hipSuccess || hipMemsetAsync(phi, 0, (size_t)info.stride * sizeof(R), s) != hipSuccess ||
      hipMemsetAsync(st, 0, sizeof(CgState), s) != hipSuccess)
    return err = "CG set-up failed", -4;

  (void)hipEventRecord(w->e0, s);
  // r = div B on the interior (calc_div_divcleaning, kernel_div_cleaning.cl:60-70)
  const uint32_t g_dc[3] = {(uint32_t)gx, (uint32_t)gy, (uint32_t)gz};
  gen_div<R>(p, info.opset, s, g_dc, b, r, p.bnodes);
  k_cg_init<R><<<vec_blocks, kBlk, 0, s>>>(r, n, part_rr);
  k_cg_init_state<<<1, 256, 0, s>>>(part_rr, vec_blocks, st, abs_thr * abs_thr, rel_tol * rel_tol, max_it);

  LapArgs<R> la{};
  la.nx = p.nx;
  la.ny = p.ny;
  la.nz = p.nz;
  la.off = p.bnodes;
  la.nbl = nbl;
  la.wl = wl;
  la.tab = tab;
  la.idx2 = 1.0 / (p.dx * p.dx);
  la.idy2 = 1.0 / (p.dy * p.dy);
  la.idz2 = 1.0 / (p.dz * p.dz);
  for (int k = 0; k <= 2 * hw; ++k) la.cz[k] = (R)(host_tab[nbl * wl + (wl - 1) / 2 - hw + k] * la.idz2);
  la.zc = zc;
  // The host stays kAhead iterations in front of the one the device has reached, so the device never waits for
  // it and few launches are left over (they return at once) when the stop test holds.
  volatile int* progress = &w->host->progress;
  *progress = 0;
  int launched = 0;
  // Nothing of a call that fails is left in flight (the workspace is the program's) or in the last error.
  auto failed = [&](hipError_t e) {
    (void)hipStreamSynchronize(s);
    (void)hipGetLastError();
    return err = std::string("CG kernel launch or state read failed: ") + hipGetErrorString(e), -4;
  };
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return failed(e);
  while (launched < max_it && *progress >= 0) {
    for (unsigned spin = 1; launched - *progress >= kAhead && *progress >= 0; ++spin) {
      if (spin % 4096) continue;
      const int before = *progress;
      e = hipStreamQuery(s);
      (void)hipGetLastError();  // of the query: every launch so far has been looked at
      if (e == hipErrorNotReady) continue;
      if (e != hipSuccess) return failed(e);
      if (*progress == before) break;  // everything launched has ended without a further iteration: stopped at once
    }
    if (launched - *progress >= kAhead) break;
    const int it = launched++;
    const R* u = ub[it & 1];
    R* un = ub[(it + 1) & 1];
    int* pr = &w->host->progress;
    switch (hw) {
      case 1: launch_lap<R, 1>(la, lap_blocks, u, r, un, q, st, part_rr, vec_blocks, part_uq, it, pr, s); break;
      case 2: launch_lap<R, 2>(la, lap_blocks, u, r, un, q, st, part_rr, vec_blocks, part_uq, it, pr, s); break;
      case 3: launch_lap<R, 3>(la, lap_blocks, u, r, un, q, st, part_rr, vec_blocks, part_uq, it, pr, s); break;
      case 4: launch_lap<R, 4>(la, lap_blocks, u, r, un, q, st, part_rr, vec_blocks, part_uq, it, pr, s); break;
      case 5: launch_lap<R, 5>(la, lap_blocks, u, r, un, q, st, part_rr, vec_blocks, part_uq, it, pr, s); break;
      case 6: launch_lap<R, 6>(la, lap_blocks, u, r, un, q, st, part_rr, vec_blocks, part_uq, it, pr, s); break;
      default: launch_lap<R, 7>(la, lap_blocks, u, r, un, q, st, part_rr, vec_blocks, part_uq, it, pr, s); break;
    }
    k_cg_update<R><<<vec_blocks, kBlk, 0, s>>>(phi, un, r, q, n, st, part_uq, lap_blocks, part_rr, it);
    if ((e = hipGetLastError()) != hipSuccess) return failed(e);
  }
  k_cg_finish<<<1, 256, 0, s>>>(part_rr, vec_blocks, st, launched);  // no-op once the stop test held
  (void)hipEventRecord(w->e1, s);
  // projection over the whole grid and the final divergence norm (clean_div_CG.m:78-86)
  const uint32_t g_full[3] = {(uint32_t)p.nx, (uint32_t)p.ny, (uint32_t)p.nz};
  gen_proj<R>(p, info.opset, s, g_full, b, phi);
  gen_div_norm2<R>(p, info.opset, s, b, part_rr, norm2);
  if ((e = hipGetLastError()) != hipSuccess ||
      (e = hipMemcpyAsync(&w->host->st, st, sizeof(CgState), hipMemcpyDeviceToHost, s)) != hipSuccess ||
      (e = hipMemcpyAsync(&w->host->norm2, norm2, sizeof(double), hipMemcpyDeviceToHost, s)) != hipSuccess ||
      (e = hipStreamSynchronize(s)) != hipSuccess)
    return failed(e);
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, w->e0, w->e1);
  const CgState& hst = w->host->st;
  res->iterations = hst.it;
  res->residual_norm = std::sqrt(hst.rr);
  res->divergence_norm_initial = std::sqrt(hst.rr0);
  res->divergence_norm_final = std::sqrt(std::max(w->host->norm2, 0.0));
  res->seconds = ms * 1e-3;
  return 0;
}

template int cg_run_t<double>(const Params&, const ieq_program_info&, const double*, int, int, hipStream_t, CgWork**, double*,
                              double*, double, double, int, ieq_cg_result*, std::string&);
template int cg_run_t<float>(const Params&, const ieq_program_info&, const double*, int, int, hipStream_t, CgWork**, float*,
                             float*, double, double, int, ieq_cg_result*, std::string&);

}  // namespace ieq
