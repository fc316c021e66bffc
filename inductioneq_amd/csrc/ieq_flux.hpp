// Flux-differencing convection sums shared by the tiled and the per-node stage kernels.
#pragma once

#include "ieq_device.hpp"

namespace ieq {
namespace {

// The flux-differencing convection along d with one row of the operator table, sum_k c_k
// f(B_m, u_m, B_k, u_k) for the two-point flux f of induction_Eq_volume.cl:13-165: f is bilinear in
// the node and neighbour values and every row of a first-derivative operator sums to zero, so the sum
// follows from four weighted neighbour sums for every choice of the three flux forms (one pass over
// the neighbours, twelve accumulators).
template <typename R> struct FluxSums {
  V3<R> sb, su, sbu, sub;  // sum c_k B_k, sum c_k u_k, sum c_k B_k,d u_k, sum c_k u_k,d B_k
  __device__ void init() { sb = su = sbu = sub = zero3<R>(); }
  __device__ void add(R c, int d, V3<R> Bk, V3<R> uk) {
    sb = sb + c * Bk;
    su = su + c * uk;
    sbu = sbu + (c * cmp(Bk, d)) * uk;
    sub = sub + (c * cmp(uk, d)) * Bk;
  }
  __device__ V3<R> conv(const Params& p, int d, V3<R> Bm, V3<R> um) const {
    const R bmd = cmp(Bm, d), umd = cmp(um, d), sbd = cmp(sb, d), sud = cmp(su, d);
    V3<R> f1, f2, f3;
    switch (p.form_uibj) {  // CENTRAL, SPLIT, PRODUCT
      case 0: f1 = R(0.5) * sbu; break;
      case 1: f1 = R(0.25) * ((bmd * su + sbd * um) + sbu); break;
      default: f1 = R(0.5) * (sbd * um + bmd * su); break;
    }
    switch (p.form_source) {  // ZERO, CENTRAL, SPLIT
      case 0: f2 = zero3<R>(); break;
      case 1: f2 = (R(0.5) * sbd) * um; break;
      default: f2 = R(0.25) * ((sbd * um + sbu) - bmd * su); break;
    }
    switch (p.form_ujbi) {  // CENTRAL, SPLIT, PRODUCT
      case 0: f3 = R(0.5) * sub; break;
      case 1: f3 = R(0.25) * ((umd * sb + sud * Bm) + sub); break;
      default: f3 = R(0.5) * (umd * sb + sud * Bm); break;
    }
    return (f1 - f2) - f3;
  }
};

}  // namespace
}  // namespace ieq
