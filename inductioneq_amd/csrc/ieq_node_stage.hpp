// Reference-schedule kernels with a thread per node: one RK stage (out = cP*P + cQ*Q + cD*DB(Y),
// kernel_time_integrator.cl:9-31), every option of the program, any NDRange; and what precedes it,
// curl B / rho and the velocity at the stage time.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ieq {

struct Params;

// The stage time.  time[1] holds it, unless `set`: then it is time[0] + add, and the kernel also stores
// it in time[1] (the listed time kernel that comes before, without a launch of its own).
template <typename R> struct NodeTime {
  R* time = nullptr;
  int set = 0;
  R add = R(0);
};

// Enqueue one stage on the nodes [0, g) of the grid (P or Q null: absent), with curl B / rho in J (read by
// programs with the Hall term) and the velocity field u.  With b1 non-null also the second half of a 2N
// stage: b1 = Y + cB * out (b1 a field of its own, because neighbours still read Y).
template <typename R>
hipError_t node_stage(const Params& p, int ops, hipStream_t s, const uint32_t g[3], R* out, const R* P, R cP, const R* Q, R cQ,
                      const R* Y, R cD, const R* J, const R* u, const NodeTime<R>& t, R* b1 = nullptr, R cB = R(0));

// Enqueue J = curl B / rho (J non-null; calc_curlB_rho_*, kernel_time_integrator.cl:136-208; rho null: curl B)
// and u = u_analytical at the stage time (u non-null; calc_u_*, :84-134) on the nodes [0, g).
template <typename R>
hipError_t node_pre(const Params& p, int ops, hipStream_t s, const uint32_t g[3], const R* b, R* J, const R* rho, R* u,
                    const NodeTime<R>& t);

}  // namespace ieq
