// Radix-6 and radix-9 register DFTs and the two-factor plans of short axes (device code shared
// by the column z solve and the two-pass plane kernels).
#pragma once
#include "wlc_device.h"

namespace wlc {

// X[k] = sum_n x[n] exp(DIR 2 pi i n k / 6): two DFT-3 and one radix-2 step
template <int DIR>
struct Dft<6, DIR> {
  __device__ __forceinline__ static void run(double2* v) {
    double2 e[3] = {v[0], v[2], v[4]};
    double2 o[3] = {v[1], v[3], v[5]};
    Dft<3, DIR>::run(e);
    Dft<3, DIR>::run(o);
    const double s = 0.86602540378443864676;  // sqrt(3)/2
    // W6 = (1/2, DIR s), W6^2 = (-1/2, DIR s)
    const double2 o1 = make_double2(0.5 * o[1].x - DIR * s * o[1].y, 0.5 * o[1].y + DIR * s * o[1].x);
    const double2 o2 = make_double2(-0.5 * o[2].x - DIR * s * o[2].y, -0.5 * o[2].y + DIR * s * o[2].x);
    v[0] = cadd(e[0], o[0]);
    v[3] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);
    v[4] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);
    v[5] = csub(e[2], o2);
  }
};

// X[k] = sum_n x[n] exp(DIR 2 pi i n k / 9): 3 x 3 four-step (n = a + 3 b, k = c + 3 d)
template <int DIR>
struct Dft<9, DIR> {
  __device__ __forceinline__ static double2 rot(double2 a, double c, double s) {
    return make_double2(c * a.x - DIR * s * a.y, c * a.y + DIR * s * a.x);
  }
  __device__ __forceinline__ static void run(double2* v) {
    double2 t0[3] = {v[0], v[3], v[6]};
    double2 t1[3] = {v[1], v[4], v[7]};
    double2 t2[3] = {v[2], v[5], v[8]};
    Dft<3, DIR>::run(t0);
    Dft<3, DIR>::run(t1);
    Dft<3, DIR>::run(t2);
    // cos, sin of 2 pi k / 9 for k = 1, 2, 4
    const double c1 = 0.76604444311897803520, s1 = 0.64278760968653932632;
    const double c2 = 0.17364817766693034885, s2 = 0.98480775301220805937;
    const double c4 = -0.93969262078590838405, s4 = 0.34202014332566873304;
    t1[1] = rot(t1[1], c1, s1);
    t1[2] = rot(t1[2], c2, s2);
    t2[1] = rot(t2[1], c2, s2);
    t2[2] = rot(t2[2], c4, s4);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double2 w[3] = {t0[c], t1[c], t2[c]};
      Dft<3, DIR>::run(w);
      v[c] = w[0];
      v[c + 3] = w[1];
      v[c + 6] = w[2];
    }
  }
};

// n = R T: the two radices of an axis transformed in two register passes; R = 0: no such plan
struct TwoPass {
  int R, T;
};
__host__ __device__ constexpr TwoPass two_pass(int n) {
  return n == 8    ? TwoPass{4, 2}
         : n == 12 ? TwoPass{3, 4}
         : n == 16 ? TwoPass{4, 4}
         : n == 18 ? TwoPass{3, 6}
         : n == 24 ? TwoPass{6, 4}
         : n == 32 ? TwoPass{8, 4}
         : n == 36 ? TwoPass{6, 6}
         : n == 48 ? TwoPass{6, 8}
         : n == 54 ? TwoPass{9, 6}
         : n == 64 ? TwoPass{8, 8}
         : n == 72 ? TwoPass{9, 8}
                   : TwoPass{0, 0};
}

}  // namespace wlc
