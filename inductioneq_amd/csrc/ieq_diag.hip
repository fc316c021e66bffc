// FP64 diagnostics of a vector field for either REAL type: the SBP-norm energy (norm2,
// kernel_operator.cl:11-44), the norm of the SBP divergence (calc_div + norm2_S,
// kernel_operator.cl:98-155) and the error against the testcase's analytic field
// (analytical_b + norm2_diff, kernel_init.cl:36-48, kernel_operator.cl:50-92), evaluated in
// one pass with every product and sum in double.  The blocks split the grid by its sizes alone;
// each block writes one partial triple and a second one-block kernel adds the partials in a
// fixed order, so the result is deterministic and independent of the caller.
#include <mutex>

#include "ieq_device.hpp"
#include "ieq_diag.hpp"
#include "ieq_node.hpp"

namespace ieq {
namespace {

// Partial sums of ieq_diagnostics_noalloc: kDiagBlocks triples (24 KiB), one copy per GPU, held
// until the process ends.  Host code never passes this name to a kernel or a copy: it uses the
// device address that diag_scratch() looked up for the current device.
__device__ __align__(256) double scratch[3 * kDiagBlocks];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

// Work split of the partial pass: a block takes a run of 256 consecutive nodes of an xy-plane (so the
// lanes are full whatever nx is) and `zc` planes of it; `segs` runs times `chunks` z-chunks make at most
// kDiagBlocks blocks.  A plane of more than kDiagBlocks runs is walked with a stride.
struct DiagSplit {
  int segs, chunks, zc;
};
__host__ __device__ inline DiagSplit diag_split(const Params& p) {
  const long long nseg = ((long long)p.nx * p.ny + kDiagThreads - 1) / kDiagThreads;
  DiagSplit s;
  s.segs = (int)(nseg < kDiagBlocks ? nseg : kDiagBlocks);
  const int most = kDiagBlocks / s.segs;
  s.zc = (p.nz + most - 1) / most;
  s.chunks = (p.nz + s.zc - 1) / s.zc;
  return s;
}

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Bound by FP64 instruction issue (about 280 instructions per node with an analytic field) and by the
// latency of one plane's loads at three waves per SIMD; the node's x and y neighbours are the same for
// every plane of the chunk, so their rows are found once per thread, and the z row is uniform in a wave.
// 128^3 FP32, 4th order, with an analytic field: 31 us, against 72 us with a 64-bit division and rolled
// table rows per node.  TC is the testcase whose analytic field the error is taken against (-1: none):
// with all of them in one kernel the code of the other seven holds 235 registers (44 us).  Numbers of a plane's
// nodes are P: 64 bits, and then the program's testcase (kAnyCase), only where 32 do not hold them.
constexpr int kAnyCase = -2;
template <typename R, int OPS, int TC, typename P>
__global__ __launch_bounds__(kDiagThreads) void k_diag(Params p, DiagSplit sp, const R* b, double t, double* part) {
  using O = Op<OPS>;
  const P nxy = (P)p.nx * p.ny;
  const int per = p.periodic;
  const long long S = p.stride;
  const double ih[3] = {1.0 / p.dx, 1.0 / p.dy, 1.0 / p.dz};
  const int seg0 = (int)blockIdx.x % sp.segs, z0 = ((int)blockIdx.x / sp.segs) * sp.zc, z1 = min(z0 + sp.zc, p.nz);
  if (TC != kAnyCase) p.testcase = TC;
  const bool analytic = TC >= 0 || (TC == kAnyCase && p.testcase >= 0);
  const double st = analytic ? sin(t) : 0.0, ct = analytic ? cos(t) : 0.0;
  __shared__ NodeTable<double, OPS> tab;
  tab.load(threadIdx.x, kDiagThreads);
  __syncthreads();
  double acc[3] = {0.0, 0.0, 0.0};
  for (P j = seg0 * kDiagThreads + (int)threadIdx.x; j < nxy; j += sp.segs * kDiagThreads) {
    const int iy = (int)(j / p.nx), ix = (int)(j - (P)iy * p.nx);
    const NodeAxis ax = node_axis<OPS>(ix, p.nx, per), ay = node_axis<OPS>(iy, p.ny, per);
    const bool mxy = __all(ax.mid && ay.mid);
    const double fxy = (p.dx / O::minv(ax.row)) * (p.dy / O::minv(ay.row));
    for (int iz = z0; iz < z1; ++iz) {
      asm volatile("" ::: "memory");  // the table stays in LDS instead of in registers across the planes
      const NodeAxis az = node_axis<OPS>(iz, p.nz, per);
      const R* f = b + (long long)iz * nxy;  // plane iz
      const R *fx = f, *fy = f + S, *fz = f + 2 * S;
      const double bx = (double)fx[j], by = (double)fy[j], bz = (double)fz[j];
      const double fac = fxy * (p.dz / O::minv(az.row));
      acc[0] += fac * (bx * bx + by * by + bz * bz);
      // one branch for the three directions: the loads of either form are all in flight together
      double dx, dy, dz;
      if (mxy && az.mid) {
        dx = node_deriv_mid<double, OPS>([&](int k) { return (double)fx[j + node_step(ax, k, per)]; });
        dy = node_deriv_mid<double, OPS>([&](int k) { return (double)fy[j + (P)p.nx * node_step(ay, k, per)]; });
        dz = node_deriv_mid<double, OPS>([&](int k) { return (double)fz[j + (long long)nxy * node_step(az, k, per)]; });
      } else {
        dx = node_deriv_row<double, OPS>(tab, ax, per, [&](int st) { return (double)fx[j + st]; });
        dy = node_deriv_row<double, OPS>(tab, ay, per, [&](int st) { return (double)fy[j + (P)p.nx * st]; });
        dz = node_deriv_row<double, OPS>(tab, az, per, [&](int st) { return (double)fz[j + (long long)nxy * st]; });
      }
      const double dv = dx * ih[0] + dy * ih[1] + dz * ih[2];
      acc[1] += fac * (dv * dv);
      if (analytic) {
        const V3<double> a = b_analytical<double>(p, ix, iy, iz, t, st, ct);
        const double ex = bx - a.x, ey = by - a.y, ez = bz - a.z;
        acc[2] += fac * (ex * ex + ey * ey + ez * ez);
      }
    }
  }
  __shared__ double sm[3][kDiagThreads / 64];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double v = wave_sum(acc[c]);
    if ((threadIdx.x & 63) == 0) sm[c][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double s = 0.0;
    for (int w = 0; w < kDiagThreads / 64; ++w) s += sm[threadIdx.x][w];
    part[blockIdx.x * 3 + threadIdx.x] = s;
  }
}

// out = (energy, divergence norm, error norm) from nblk partial triples, summed in a fixed order by one
// workgroup (three lanes adding 1024 triples one after the other took 107 us); the error norm is NaN
// without an analytic field.
__global__ __launch_bounds__(kDiagThreads) void k_diag_sum(const double* part, int nblk, int analytic, double* out) {
  __shared__ double sm[3][kDiagThreads / 64];
  double acc[3] = {0.0, 0.0, 0.0};
  for (int k = threadIdx.x; k < nblk; k += kDiagThreads)
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[c] += part[k * 3 + c];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double v = wave_sum(acc[c]);
    if ((threadIdx.x & 63) == 0) sm[c][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  if (threadIdx.x >= 3) return;
  double s = 0.0;
  for (int w = 0; w < kDiagThreads / 64; ++w) s += sm[threadIdx.x][w];
  out[threadIdx.x] = threadIdx.x == 0 ? s : (threadIdx.x == 2 && !analytic) ? __longlong_as_double(0x7ff8000000000000LL)
                                                                            : sqrt(fmax(s, 0.0));
}

template <typename R, int OPS> const void* diag_kernel_t(int tc, bool wide) {
  if (wide) return reinterpret_cast<const void*>(&k_diag<R, OPS, kAnyCase, long long>);
  switch (tc) {
    case TC_ROTATION_2D: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_ROTATION_2D, int>);
    case TC_ROTATION_3D: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_ROTATION_3D, int>);
    case TC_HALL_PERIODIC: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_HALL_PERIODIC, int>);
    case TC_HALL_TRAVELLING_WAVE: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_HALL_TRAVELLING_WAVE, int>);
    case TC_CONFINED_DOMAIN: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_CONFINED_DOMAIN, int>);
    case TC_ALFVEN_PERIODIC_2D: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_ALFVEN_PERIODIC_2D, int>);
    case TC_GAUSSIAN_ROTATION_3D: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_GAUSSIAN_ROTATION_3D, int>);
    case TC_UNIFORM_FLOW: return reinterpret_cast<const void*>(&k_diag<R, OPS, TC_UNIFORM_FLOW, int>);
    default: return reinterpret_cast<const void*>(&k_diag<R, OPS, -1, int>);
  }
}
template <typename R> const void* diag_kernel(int ops, int tc, bool wide) {
  switch (ops) {
    case 0: return diag_kernel_t<R, 0>(tc, wide);
    case 1: return diag_kernel_t<R, 1>(tc, wide);
    case 2: return diag_kernel_t<R, 2>(tc, wide);
    case 3: return diag_kernel_t<R, 3>(tc, wide);
    case 4: return diag_kernel_t<R, 4>(tc, wide);
    default: return diag_kernel_t<R, 5>(tc, wide);
  }
}

}  // namespace

int diag_blocks(const Params& p) {
  const DiagSplit s = diag_split(p);
  return s.segs * s.chunks;
}

template <typename R>
hipError_t diag_launch(const Params& p, int ops, hipStream_t s, const R* b, double t, int analytic, double* part,
                       double* out_dev) {
  const DiagSplit sp = diag_split(p);
  const int nblk = sp.segs * sp.chunks;
  Params q = p;
  if (!analytic) q.testcase = -1;
  const void* k = diag_kernel<R>(ops, q.testcase, (long long)p.nx * p.ny >= (1LL << 30));
  DiagSplit split = sp;
  void* kargs[5] = {(void*)&q, (void*)&split, (void*)&b, (void*)&t, (void*)&part};
  const hipError_t e = hipLaunchKernel(k, dim3(nblk), dim3(kDiagThreads), kargs, 0, s);
  if (e != hipSuccess) return e;
  k_diag_sum<<<1, kDiagThreads, 0, s>>>(part, nblk, analytic, out_dev);
  return hipGetLastError();
}

hipError_t diag_scratch(double** ptr) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[dev] = (double*)p;
  }
  *ptr = g_scratch_ptr[dev];
  return hipSuccess;
}

template hipError_t diag_launch<double>(const Params&, int, hipStream_t, const double*, double, int, double*, double*);
template hipError_t diag_launch<float>(const Params&, int, hipStream_t, const float*, double, int, double*, double*);

}  // namespace ieq
