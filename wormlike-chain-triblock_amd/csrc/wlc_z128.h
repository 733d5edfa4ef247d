// Launch shape of the three-part nz = 128 z solve (wlc_z128.hip), shared by host and device.
#pragma once
#include "wlc_kernels.h"

namespace wlc {

constexpr int kZ128MinL = 5;     // Lmax 5-8
constexpr int kZ128Threads = 768;
constexpr int kZ128Chains = 13;  // chains that cross from one part to the next (|m| <= 6)
constexpr int kZ128Frame = 98;   // of a (column, half): (cq, sq), one free, (ct, st) and gk of 64 points

// one workgroup per CU (LDS admits no second one) goes through the column pairs of its XCD's
// tiles; fewer where there are fewer pairs
inline unsigned z128_grid(const Geom& g) {
  const unsigned per_xcd = 2u * (unsigned)((g.nt * g.ny + 7) / 8);
  return 8u * (per_xcd < 32u ? per_xcd : 32u);
}
// eight rows of 64 points per wave, the crossing chains of four (column, half), the twiddles,
// the frames
inline size_t z128_lds_bytes() { return sizeof(double2) * (12 * 512 + 4 * kZ128Chains * 64 + 128 + 4 * kZ128Frame); }

}  // namespace wlc
