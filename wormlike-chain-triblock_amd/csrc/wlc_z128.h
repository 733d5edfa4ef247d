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

// Where a kernel of two degree parts that takes one column to a workgroup (k_zsolve128s) is the
// faster one: on grids of at most one column per CU, and with the FP32 spectrum, where half the
// bytes leave the three-part kernel less to hide, at Lmax 5 and 6 on any.  Per launch, two parts /
// three parts, on 24 x 16 (208 columns): Lmax 5 26.1 / 29.2 us, Lmax 6 31.6 / 35.4, with the FP32
// spectrum Lmax 5 21.8 / 26.2, 6 27.2 / 31.6, 7 37.3 / 41.3, 8 42.1 / 52.5; on 24 x 24 (312): 32.6 /
// 30.6, 41.7 / 37.2, 27.3 / 26.7, 35.5 / 33.2, 48.2 / 42.4, 73.5 / 54.2.  Pairs of concurrent sweeps
// (the three-part kernel leaves no room beside it on a CU), FP32, Lmax 5: 32^2 8.08 / 8.36 ms, 48^2
// 18.2 / 19.3, 64^2 28.0 / 28.7, 96^2 81.8 / 82.9, 128^2 49.4 / 49.8; Lmax 6: 32^2 11.0 / 11.2, 48^2
// 25.1 / 25.5, 96^2 110.2 / 111.7, 128^2 67.6 / 67.0.  With the FP64 spectrum of Lmax 7 and 8 it has
// no advantage (24 x 16: whole columns 55.2 and 83.4, three parts 45.4 and 58.8).
inline bool z128_two_parts(const Geom& g, int L) {
  return L <= 6 ? g.spec32 || g.nxh * g.ny <= 256 : g.spec32 && g.nxh * g.ny <= 256;
}

// one workgroup per CU (LDS admits no second one) goes through the column pairs of its XCD's
// tiles; fewer where there are fewer pairs
inline unsigned z128_grid(const Geom& g) {
  const unsigned per_xcd = 2u * (unsigned)((g.nt * g.ny + 7) / 8);
  return 8u * (per_xcd < 32u ? per_xcd : 32u);
}
// the rows of the three parts of four (column, half), the twiddles, the frames
inline size_t z128_lds_bytes() { return sizeof(double2) * (4 * kZ128Col + 192 + 4 * kZ128Frame); }

}  // namespace wlc
