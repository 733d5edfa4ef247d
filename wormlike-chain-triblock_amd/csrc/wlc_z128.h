// Launch shape of the three-part nz = 128 z solve (wlc_z128.hip), shared by host and device.
#pragma once
#include "wlc_kernels.h"

namespace wlc {

constexpr int kZ128MinL = 5;     // Lmax 5-8
constexpr int kZ128Threads = 768;
constexpr int kZ128Chains = 13;  // chains that cross from one part to the next (|m| <= 6)
constexpr int kZ128Frame = 98;   // of a (column, half): (cq, sq), one free, (ct, st) and gk of 64 points

constexpr int kZ128Rows = 8 * 72;  // a wave's LDS: eight harmonics
// LDS of a (column, half): the crossing chains, which share the first part's rows, and the rows of
// the other two parts
constexpr int kZ128Col = kZ128Chains * 64 + 2 * kZ128Rows;
static_assert(kZ128Chains * 64 >= kZ128Rows, "the chains' rows hold the first part's");

// one workgroup per CU (LDS admits no second one) goes through the column pairs of its XCD's
// tiles; fewer where there are fewer pairs
inline unsigned z128_grid(const Geom& g) {
  const unsigned per_xcd = 2u * (unsigned)((g.nt * g.ny + 7) / 8);
  return 8u * (per_xcd < 32u ? per_xcd : 32u);
}
// the rows of the three parts of four (column, half), the twiddles, the frames
inline size_t z128_lds_bytes() { return sizeof(double2) * (4 * kZ128Col + 192 + 4 * kZ128Frame); }

}  // namespace wlc
