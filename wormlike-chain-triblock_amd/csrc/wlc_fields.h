// Launches on whole fields: contour runs of the density sum, dense <-> padded fields (internal).
#pragma once
#include "wlc_kernels.h"

namespace wlc {

// rho[part] += sum over the contour points t of the run of w[t] sum_{i < lim} q_i(t) q*_i(t):
// n points whose slices lie `stride` doubles apart (q, qs at the first), weights w[t] in device
// memory, taken in order (step = +1) or from the last (step = -1).  The run is cut into `parts`
// consecutive pieces, each with its own accumulator (pstride doubles apart).
struct DensityRun {
  const double *q, *qs;
  long long stride;
  int n, lim, step;
  const double* w;
  double* rho;
  int parts;
  long long pstride;
};
hipError_t launch_density_run(const Geom& g, const DensityRun& r, hipStream_t st);
// accumulators of one run that give the GPU enough workgroups on this grid (1..16)
int density_parts(const Geom& g);
// rho[0] += rho[1] + ... in order (n doubles each, pstride apart)
hipError_t launch_sum_parts(double* rho, long long n, int parts, long long pstride, hipStream_t st);

// dense [nf][nz][ny][nx] -> padded fields
hipError_t launch_scatter_fields(const Geom& g, const double* dense, int nf, double* padded, hipStream_t st);
// phi_b = V rho_b / totden (totden on the device), written dense; *bad = 1 when a value is not
// finite (the caller clears it)
hipError_t launch_phi_dense(const Geom& g, const double* rho, int nblk, double V, const double* totden,
                            double* phi, double* bad, hipStream_t st);

}  // namespace wlc
