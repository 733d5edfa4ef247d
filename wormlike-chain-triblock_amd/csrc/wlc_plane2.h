// Launch shape of the two-pass plane kernels (wlc_plane2.hip), shared by host and device.
#pragma once
#include "wlc_dft.h"

namespace wlc {
namespace p2 {

constexpr int kMaxThreads = 384;
constexpr int kItems = 4;  // x pairs of two rows per lane in the right-hand side

// A plane of nx x ny points, both axes of a two-factor plan n = R T.
//   row role     T(nx) lanes per row pair, whole row pairs per wave (ppw of them)
//   column role  lane c + h jy: column c of h = nx/2, jy < T(ny)
struct Shape {
  int pairs, h, stride, ppw, waves;
};
__host__ __device__ constexpr Shape shape_of(int nx, int ny) {
  Shape s{};
  s.pairs = ny / 2;
  s.h = nx / 2;
  // complex slots between row pairs: 5 past a multiple of 16 the lanes of a pass (T slots of each
  // of several pairs) fall on distinct banks for T = 4 and nearly so for 6 and 8
  s.stride = nx + ((5 - nx) & 15);
  const int tx = two_pass(nx).T, ty = two_pass(ny).T;
  int most = 64 / tx;
  if (most > 64 * kItems / s.h) most = 64 * kItems / s.h;
  const int wx = (s.pairs + most - 1) / most, wy = (s.h * ty + 63) / 64;
  s.waves = wx > wy ? wx : wy;
  s.ppw = (s.pairs + s.waves - 1) / s.waves;
  return s;
}
// the plane, columns kx = 0 and nx/2 of the spectrum, the twiddles of both axes
inline size_t lds_bytes(int nx, int ny) {
  const Shape s = shape_of(nx, ny);
  return sizeof(double2) * (size_t)(s.pairs * s.stride + 2 * ny + nx + ny);
}
inline bool takes(int nx, int ny) { return two_pass(nx).R > 0 && two_pass(ny).R > 0; }

// kind 0: A, 1: C, 2: fused C + A
const void* kernel(int nx, int ny, int kind, bool batch);

}  // namespace p2
}  // namespace wlc
