// EMF and RK stage of the fused periodic path with a workgroup per TX x TY x TZ brick of nodes: every value
// a brick needs is loaded at once, the planes' x/y stencils go through LDS after a single barrier and the
// z stencils through the registers of the thread that owns the column.
//
// The z-marching kernels (ieq_fused_tiles.hpp) read a node once, but take a global load's latency and a
// barrier for each of the TZ + 2 RR planes of a chunk, and on grids that give a workgroup only a few planes
// this chain, not bandwidth or arithmetic, is their time.
// A brick's time is the sum of its phases (instructions, LDS reads, L1 accesses), since on such a grid the workgroups run them
// together; hence plane offsets found once, without branches (taken from wrap() per load, 1000 of a wave's 1900
// instructions were scalar: 96^3 FP32, half-width 3, EMF 9.7 -> 7.4 us, stage 15.6 -> 13.0).  The march's two take 11 and 16.6.
#pragma once

#include "ieq_stencil.hpp"

namespace ieq {
namespace {

// Component base pointers of a field in scalar registers of their own; without it the compiler adds the
// component's offset to every lane's address.
template <typename R> struct Bases {
  R* c[3];
  __device__ __forceinline__ Bases(R* f, long long S) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      c[k] = f + k * S;
      asm("" : "+s"(c[k]));
    }
  }
};

template <typename R, int RR, int TX, int TY, int TZ> struct Brick {
  static constexpr int NT = TX * TY, LX = TX + 2 * RR, LY = TY + 2 * RR, Q = 2 * RR + 1, N = TZ + 2 * RR;
  static constexpr int NYH = 2 * RR * TX, NXH = 2 * RR * TY, NH = NYH + NXH;  // halo cells of a plane: y rows, x columns
  static_assert(NH <= NT, "one halo cell per thread and plane");

  int tx, ty, z0, lh;     // lh: LDS index of the halo cell in a plane
  bool active, has_h, hx;  // output column in the grid; this thread has a halo cell; it lies beside the tile in x
  unsigned col, halo;     // in-plane byte offsets of the column and of the halo cell
  unsigned pz[N];         // byte offsets of the planes z0 - RR .. z0 + TZ + RR - 1 (uniform)

  // `v` lies at most a tile and a half-width outside [0, n)
  __device__ static __forceinline__ int at(int v, int n, bool once) {
    if (!once) return wrap(v, n);
    v = v < 0 ? v + n : v;
    return v >= n ? v - n : v;
  }
  __device__ __forceinline__ Brick(int nx, int ny, int nz) {
    tx = threadIdx.x;
    ty = threadIdx.y;
    int x0, y0;
    tile_origin<TY, TX>(xcd_tile(blockIdx.x, gridDim.x), nx, ny, TZ, x0, y0, z0);
    active = x0 + tx < nx && y0 + ty < ny;
    const int tid = tx + TX * ty, h = min(tid, NH - 1), c = h - NYH;
    has_h = tid < NH;
    hx = h >= NYH;
    const int row = h / TX, cc = c % (2 * RR);
    const int lx = hx ? (cc < RR ? cc - RR : TX + cc - RR) : h % TX;
    const int ly = hx ? c / (2 * RR) : (row < RR ? row - RR : TY + row - RR);
    lh = (ly + RR) * LX + lx + RR;
    const bool once = nx >= LX && ny >= LY && nz >= N;
    col = (unsigned)(at(x0 + tx, nx, once) + nx * at(y0 + ty, ny, once)) * (unsigned)sizeof(R);
    halo = (unsigned)(at(x0 + lx, nx, once) + nx * at(y0 + ly, ny, once)) * (unsigned)sizeof(R);
    const unsigned plb = (unsigned)(nx * ny) * (unsigned)sizeof(R);
    if (once) {
#pragma unroll
      for (int j = 0; j < N; ++j) pz[j] = (unsigned)at(z0 - RR + j, nz, true) * plb;
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) pz[j] = (unsigned)wrap(z0 - RR + j, nz) * plb;
    }
  }
  // derivative along x / y at the own node of an LDS plane
  __device__ __forceinline__ R dx(const StencilCoef<R>& c, const R (*s)[LX]) const {
    R v[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) v[k] = s[ty + RR][tx + k];
    return deriv<R, RR>(c, v);
  }
  __device__ __forceinline__ R dy(const StencilCoef<R>& c, const R (*s)[LX]) const {
    R v[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) v[k] = s[ty + k][tx + RR];
    return deriv<R, RR>(c, v);
  }
};

// E = (curl_D B / rho) x B
template <typename R, int RR, int TX, int TY, int TZ> __global__ __launch_bounds__(TX * TY) void k_brick_emf(FArgs<R> a) {
  using G = Brick<R, RR, TX, TY, TZ>;
  __shared__ R s[TZ][3][G::LY][G::LX];
  const G g(a.nx, a.ny, a.nz);
  const long long S = a.S;
  const unsigned hs = g.halo + (g.hx ? (unsigned)(S * sizeof(R)) : 0u);
  const Bases<const R> Y(a.Y, S);
  const Bases<R> E(a.Eout, S);
  R q[3][G::N], h[TZ][2];
#pragma unroll
  for (int t = 0; t < TZ; ++t) {
#pragma unroll
    for (int c = 0; c < 3; ++c) q[c][RR + t] = ldo(Y.c[c], g.col + g.pz[RR + t]);
    h[t][0] = ldo(Y.c[0], hs + g.pz[RR + t]);  // B_y beside the tile in x, B_x in y
    h[t][1] = ldo(Y.c[2], g.halo + g.pz[RR + t]);
  }
#pragma unroll
  for (int j = 0; j < RR; ++j)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      q[c][RR - 1 - j] = ldo(Y.c[c], g.col + g.pz[RR - 1 - j]);
      q[c][RR + TZ + j] = ldo(Y.c[c], g.col + g.pz[RR + TZ + j]);
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < TZ; ++t) {
#pragma unroll
    for (int c = 0; c < 3; ++c) s[t][c][g.ty + RR][g.tx + RR] = q[c][RR + t];
    if (g.has_h) {
      (&s[t][g.hx ? 1 : 0][0][0])[g.lh] = h[t][0];
      (&s[t][2][0][0])[g.lh] = h[t][1];
    }
  }
  lds_barrier();
  const R irho = R(1) / a.rho;
#pragma unroll
  for (int t = 0; t < TZ; ++t) {
    const R dxBy = g.dx(a.c, s[t][1]) * a.inv_h[0], dxBz = g.dx(a.c, s[t][2]) * a.inv_h[0];
    const R dyBx = g.dy(a.c, s[t][0]) * a.inv_h[1], dyBz = g.dy(a.c, s[t][2]) * a.inv_h[1];
    const R dzBx = deriv<R, RR>(a.c, &q[0][t]) * a.inv_h[2], dzBy = deriv<R, RR>(a.c, &q[1][t]) * a.inv_h[2];
    // J = curl B / rho  (SBP_operator.cl:126-135, kernel_time_integrator.cl:147)
    const R Jx = (dyBz - dzBy) * irho, Jy = (dzBx - dxBz) * irho, Jz = (dxBy - dyBx) * irho;
    const R Bx = q[0][RR + t], By = q[1][RR + t], Bz = q[2][RR + t];
    if (g.active && g.z0 + t < a.nz) {
      const unsigned o = g.col + g.pz[RR + t];
      sto(E.c[0], o, Jy * Bz - Jz * By);
      sto(E.c[1], o, Jz * Bx - Jx * Bz);
      sto(E.c[2], o, Jx * By - Jy * Bx);
    }
  }
}

// RHS = convection - curl E + dissipation, then the RK update (MODE as in stage_tile of ieq_fused_tiles.hpp,
// and its order of operations).
template <typename R, int RR, int TX, int TY, int TZ, bool HALL, bool HOD, bool CONV, bool ADJ, int MODE>
__global__ __launch_bounds__(TX * TY) void k_brick_stage(FArgs<R> a) {
  using G = Brick<R, RR, TX, TY, TZ>;
  static_assert(!ADJ || MODE == 0, "the transposed stages use mode 0");
  constexpr int Q = G::Q;
  constexpr bool STB = HOD || CONV;                                  // B enters by its stencils
  __shared__ R sB[STB ? TZ : 1][STB ? 3 : 1][STB ? G::LY : 1][G::LX];
  __shared__ R sE[HALL ? TZ : 1][HALL ? 3 : 1][HALL ? G::LY : 1][G::LX];
  const G g(a.nx, a.ny, a.nz);
  const long long S = a.S;
  const R* Pp = MODE == 1 ? a.b2 : (a.P ? a.P : a.Y);  // an absent operand is read from Y and not used
  const R* Qp = a.Q ? a.Q : a.Y;
  const R* Gp = a.G ? a.G : a.Y;
  const unsigned hs = g.halo + (g.hx ? (unsigned)(S * sizeof(R)) : 0u);
  const Bases<const R> Y(a.Y, S), E(HALL ? a.E : a.Y, S), P(Pp, S), Qb(Qp, S), Gb(Gp, S);
  const Bases<R> out(a.out, S), b2(MODE == 1 ? a.b2 : a.out, S);
  R qb[3][G::N], qe[3][G::N], hb[TZ][3], he[TZ][2], pw[TZ][9];
#pragma unroll
  for (int t = 0; t < TZ; ++t) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      qb[c][RR + t] = ldo(Y.c[c], g.col + g.pz[RR + t]);
      if constexpr (STB) hb[t][c] = ldo(Y.c[c], g.halo + g.pz[RR + t]);
      if constexpr (HALL) qe[c][RR + t] = ldo(E.c[c], g.col + g.pz[RR + t]);
    }
    if constexpr (HALL) {
      he[t][0] = ldo(E.c[0], hs + g.pz[RR + t]);  // E_y beside the tile in x, E_x in y
      he[t][1] = ldo(E.c[2], g.halo + g.pz[RR + t]);
    }
  }
#pragma unroll
  for (int j = 0; j < 2 * RR; ++j) {
    const int jp = j < RR ? j : TZ + j;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if constexpr (STB) qb[c][jp] = ldo(Y.c[c], g.col + g.pz[jp]);
      if constexpr (HALL) {
        if (c < 2) qe[c][jp] = ldo(E.c[c], g.col + g.pz[jp]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < TZ; ++t)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if constexpr (MODE != 3) pw[t][c] = ldo(P.c[c], g.col + g.pz[RR + t]);
      if constexpr (MODE == 0) pw[t][3 + c] = ldo(Qb.c[c], g.col + g.pz[RR + t]);
      if constexpr (ADJ) pw[t][6 + c] = ldo(Gb.c[c], g.col + g.pz[RR + t]);
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < TZ; ++t) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if constexpr (STB) {
        sB[t][c][g.ty + RR][g.tx + RR] = qb[c][RR + t];
        if (g.has_h) (&sB[t][c][0][0])[g.lh] = hb[t][c];
      }
      if constexpr (HALL) sE[t][c][g.ty + RR][g.tx + RR] = qe[c][RR + t];
    }
    if constexpr (HALL) {
      if (g.has_h) {
        (&sE[t][g.hx ? 1 : 0][0][0])[g.lh] = he[t][0];
        (&sE[t][2][0][0])[g.lh] = he[t][1];
      }
    }
  }
  lds_barrier();
#pragma unroll
  for (int t = 0; t < TZ; ++t) {
    R r[3] = {R(0), R(0), R(0)}, hod[3];
    // rows of B along x and y: the convection derivative and the dissipation sum
    //   convection: sum_d (2/dx_d) 0.5 ([ZERO] u (D_d B)_d - u_d (D_d B))
    if constexpr (STB) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        R h = R(0);
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          R v[Q];
#pragma unroll
          for (int k = 0; k < Q; ++k)
            v[k] = k == RR ? qb[c][RR + t] : d == 0 ? sB[t][c][g.ty + RR][g.tx + k] : sB[t][c][g.ty + k][g.tx + RR];
          if constexpr (CONV) {
            const R der = deriv<R, RR>(a.c, v);
            const R f = a.two_h[d] * R(0.5);
            r[c] = r[c] - f * (a.u[d] * der);
            if constexpr (ADJ) {
              if (a.src_adj) r[d] = r[d] + f * (a.u[c] * der);
            }
            if (c == d && a.src_zero && !(ADJ && a.src_adj)) {
#pragma unroll
              for (int e = 0; e < 3; ++e) r[e] = r[e] + f * (a.u[e] * der);
            }
          }
          if constexpr (HOD) h = d == 0 ? hodsum<R, RR>(a.c, v) : h + hodsum<R, RR>(a.c, v);
        }
        if constexpr (HOD) hod[c] = h;
      }
    }
    if constexpr (HALL) {  // -curl_D E, x/y terms
      const R dxEy = g.dx(a.c, sE[t][1]), dxEz = g.dx(a.c, sE[t][2]);
      const R dyEx = g.dy(a.c, sE[t][0]), dyEz = g.dy(a.c, sE[t][2]);
      r[0] = r[0] + a.inv_h[1] * (-dyEz);
      r[1] = r[1] + a.inv_h[0] * dxEz;
      r[2] = r[2] + (a.inv_h[0] * (-dxEy) + a.inv_h[1] * dyEx);
    }
    if constexpr (HOD) {
#pragma unroll
      for (int c = 0; c < 3; ++c) r[c] = r[c] + hod[c];
    }
    if constexpr (CONV) {
      const R f = a.two_h[2] * R(0.5);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const R der = deriv<R, RR>(a.c, &qb[c][t]);
        r[c] = r[c] - f * (a.u[2] * der);
        if constexpr (ADJ) {
          if (a.src_adj) r[2] = r[2] + f * (a.u[c] * der);
        }
        if (c == 2 && a.src_zero && !(ADJ && a.src_adj)) {
#pragma unroll
          for (int e = 0; e < 3; ++e) r[e] = r[e] + f * (a.u[e] * der);
        }
      }
    }
    if constexpr (HALL) {
      r[0] = r[0] + a.inv_h[2] * deriv<R, RR>(a.c, &qe[1][t]);
      r[1] = r[1] + a.inv_h[2] * (-deriv<R, RR>(a.c, &qe[0][t]));
    }
    if constexpr (HOD) {
#pragma unroll
      for (int c = 0; c < 3; ++c) r[c] = r[c] + hodsum<R, RR>(a.c, &qb[c][t]);
    }
    if constexpr (ADJ) {
      if (a.G) {
#pragma unroll
        for (int c = 0; c < 3; ++c) r[c] = r[c] - pw[t][6 + c];
      }
    }
    if (g.active && g.z0 + t < a.nz) {
      const unsigned oc = g.col + g.pz[RR + t];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const R y = qb[c][RR + t];
        if constexpr (MODE == 1) {
          const R v = a.cP * pw[t][c] + a.cD * r[c];
          sto(b2.c[c], oc, v);
          sto(out.c[c], oc, y + a.cQ * v);
        } else {
          R o = a.cD * r[c];
          if constexpr (ADJ) o = a.cY * y + o;
          if constexpr (MODE != 3) {
            if (a.Q) o = a.cQ * (MODE == 0 ? pw[t][3 + c] : y) + o;
          }
          if (MODE == 2 || a.P) o = a.cP * (MODE == 3 ? y : pw[t][c]) + o;
          sto(out.c[c], oc, o);
        }
      }
    }
  }
}

}  // namespace
}  // namespace ieq
