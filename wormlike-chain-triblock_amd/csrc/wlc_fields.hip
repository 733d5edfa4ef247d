// Whole-field kernels of the handle: the contour sum of the density (SCFT_Density_FE.f90:97-118),
// phi, and the copies between the caller's dense fields and the padded layout.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "wlc_fields.h"

namespace wlc {

// One thread per x pair keeps its sum over the contour points of a run in registers: rho is read
// and written once per run instead of once per point, and a sweep of small slices needs some 15
// launches and events instead of one of each per point (an event between two kernels of a stream
// costs about 5.5 us, of 31 us per contour step at 24^3 / Lmax 6).  The harmonic loop is unrolled so that
// many independent loads are in flight; the sums run in harmonic and contour order.
__global__ void __launch_bounds__(256) k_density_run(Geom g, DensityRun r) {
  const int nxy2 = (g.nx * g.ny) >> 1;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nxy2) return;
  const long long at = (long long)blockIdx.y * g.zs + 2 * e;
  const long long hs = g.hs;
  const int part = blockIdx.z;
  const int t0 = (int)((long long)part * r.n / r.parts), t1 = (int)((long long)(part + 1) * r.n / r.parts);
  if (t0 == t1) return;
  double2* p = reinterpret_cast<double2*>(r.rho + part * r.pstride + at);
  double2 acc = *p;
  for (int k = t0; k < t1; ++k) {
    const int t = r.step > 0 ? k : r.n - 1 - k;
    const double* q = r.q + t * r.stride + at;
    const double* qs = r.qs + t * r.stride + at;
    const double w = r.w[t];
    double2 s = make_double2(0.0, 0.0);
#pragma unroll 8
    for (int i = 0; i < r.lim; ++i) {
      const double2 a = *reinterpret_cast<const double2*>(q + i * hs);
      const double2 b = *reinterpret_cast<const double2*>(qs + i * hs);
      s.x = __builtin_fma(a.x, b.x, s.x);
      s.y = __builtin_fma(a.y, b.y, s.y);
    }
    acc.x = __builtin_fma(w, s.x, acc.x);
    acc.y = __builtin_fma(w, s.y, acc.y);
  }
  *p = acc;
}

int density_parts(const Geom& g) {
  // 512 workgroups (two per CU) per launch where the grid alone has fewer
  const long long wg = (long long)g.nz * ((g.nx * g.ny / 2 + 255) / 256);
  return (int)std::min<long long>(16, std::max<long long>(1, 512 / wg));
}

hipError_t launch_density_run(const Geom& g, const DensityRun& r, hipStream_t st) {
  if (r.n <= 0 || r.lim <= 0) return hipSuccess;
  const dim3 grid((g.nx * g.ny / 2 + 255) / 256, g.nz, r.parts);
  hipLaunchKernelGGL(k_density_run, grid, dim3(256), 0, st, g, r);
  return hipGetLastError();
}

__global__ void k_sum_parts(double* rho, long long n, int parts, long long pstride) {
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    double s = rho[e];
    for (int p = 1; p < parts; ++p) s += rho[p * pstride + e];
    rho[e] = s;
  }
}

hipError_t launch_sum_parts(double* rho, long long n, int parts, long long pstride, hipStream_t st) {
  if (parts <= 1) return hipSuccess;
  const int blocks = (int)std::min<long long>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_sum_parts, dim3(blocks), dim3(256), 0, st, rho, n, parts, pstride);
  return hipGetLastError();
}

// grid (blocks over the nx ny plane, nz x fields)
__global__ void k_scatter_fields(Geom g, const double* __restrict__ dense, double* __restrict__ padded) {
  const int nxy = g.nx * g.ny;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nxy) return;
  const long long f = blockIdx.y / g.nz, z = blockIdx.y % g.nz;
  padded[f * g.hs + z * g.zs + e] = dense[(long long)blockIdx.y * nxy + e];
}

hipError_t launch_scatter_fields(const Geom& g, const double* dense, int nf, double* padded, hipStream_t st) {
  const dim3 grid((g.nx * g.ny + 255) / 256, g.nz * nf);
  hipLaunchKernelGGL(k_scatter_fields, grid, dim3(256), 0, st, g, dense, padded);
  return hipGetLastError();
}

__global__ void k_phi_dense(Geom g, const double* __restrict__ rho, double V, const double* __restrict__ totden,
                            double* __restrict__ phi, double* __restrict__ bad) {
  const int nxy = g.nx * g.ny;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nxy) return;
  const long long f = blockIdx.y / g.nz, z = blockIdx.y % g.nz;
  const double v = rho[f * g.hs + z * g.zs + e] * (V / *totden);
  phi[(long long)blockIdx.y * nxy + e] = v;
  if (!isfinite(v)) *bad = 1.0;
}

hipError_t launch_phi_dense(const Geom& g, const double* rho, int nblk, double V, const double* totden,
                            double* phi, double* bad, hipStream_t st) {
  const dim3 grid((g.nx * g.ny + 255) / 256, g.nz * nblk);
  hipLaunchKernelGGL(k_phi_dense, grid, dim3(256), 0, st, g, rho, V, totden, phi, bad);
  return hipGetLastError();
}

}  // namespace wlc
