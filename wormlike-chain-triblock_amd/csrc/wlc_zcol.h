// Launch shape of the column z solve (wlc_zcol.hip), shared by host and device.
#pragma once
#include "wlc_kernels.h"

namespace wlc {

// z axes the kernel takes (the two-factor plans of wlc_dft.h up to 54)
inline bool zcol_nz(int nz) {
  return nz == 8 || nz == 12 || nz == 16 || nz == 18 || nz == 24 || nz == 32 || nz == 36 || nz == 48 || nz == 54;
}

// log2 of the kx columns of a workgroup: 4 to nz = 16, else 2
__host__ __device__ constexpr int zcol_log2_cols(int nz) { return nz <= 16 ? 2 : 1; }

// one workgroup per column group, the 4-kx tiles rounded up to the 8 XCDs
inline unsigned zcol_grid(const Geom& g) {
  return (unsigned)((g.nt * g.ny + 7) / 8 * 8 * (kKxTile >> zcol_log2_cols(g.nz)));
}
// four waves per 64 points of the columns
inline int zcol_threads(int nz) { return 256 * (((nz << zcol_log2_cols(nz)) + 63) / 64); }
inline size_t zcol_lds_bytes(int nz, int M) { return sizeof(double2) * (size_t)M * (nz << zcol_log2_cols(nz)); }

}  // namespace wlc
