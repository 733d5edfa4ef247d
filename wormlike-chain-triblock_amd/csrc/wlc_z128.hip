// Kernel B of the propagator step at nz = 128, Lmax 5-8 (compiled once per L with -DWLC_L=<L>): z
// pass of the forward FFT, k-aligned solve of G(k) q = P(k) (the per-k G^-1 apply of
// wormlike_MDE_2dcomp_mod.f90:395-409), inverse z pass.
//
// Two columns of 81 harmonics are 332 KB: they fill the registers of a CU, so what bounds a kernel
// here is how much runs at the same time.  One workgroup of twelve waves holds a column pair: a
// wave has one column, one half of kz (the even or the odd ones, a 64-point transform after one
// radix-2 step) and one of three degree parts, at most 32 harmonics, which leaves three waves per
// SIMD.  (The kernel it replaces at Lmax 8 keeps all harmonics of a half column in one wave, one
// wave per SIMD, and issues in a third of its cycles.)  Rotations stay within a degree and so
// within a wave; the tridiagonal chains are handed from part to part through LDS.  The workgroup
// goes through its pairs in a loop and asks for the next pair while it transforms this one back,
// in the registers that its harmonics leave, eight harmonics of each part at a time.  A pair, not
// a column: 32-byte pieces of the tiles move at the full rate (a bare copy of the spectrum in
// place 594 us, in 16-byte pieces 863 to 1279).  Per launch on 128^3: Lmax 8 1853 -> 1085 us (of
// them 565 for the bare copy), with the FP32 spectrum 1537 -> 875; Lmax 7 1275 -> 818, Lmax 6
// 820 -> 594.
#include <hip/hip_runtime.h>

#include "wlc_device.h"
#include "wlc_z128.h"

#ifndef WLC_L
#error "compile with -DWLC_L=<Lmax>"
#endif

#define WLC_CAT2(a, b) a##b
#define WLC_CAT(a, b) WLC_CAT2(a, b)

namespace wlc {
namespace WLC_CAT(z128_l_, WLC_L) {

constexpr int kL = WLC_L;
// degrees of the three parts: 0..kLA, kLA+1..kLB, kLB+1..L (at Lmax 8: 25, 24 and 32 harmonics)
constexpr int kLA = kL >= 7 ? 4 : 3;
constexpr int kLB = kL >= 7 ? 6 : (kL == 6 ? 5 : 4);
template <int PART>
struct Share;
template <>
struct Share<0> : SolverPart<kL, 0, kLA> {
  static constexpr int L0 = 0, L1 = kLA;
};
template <>
struct Share<1> : SolverPart<kL, kLA + 1, kLB> {
  static constexpr int L0 = kLA + 1, L1 = kLB;
};
template <>
struct Share<2> : SolverPart<kL, kLB + 1, kL> {
  static constexpr int L0 = kLB + 1, L1 = kL;
};
constexpr int imax(int a, int b) { return a > b ? a : b; }
constexpr int kNV = imax(Share<0>::NH, imax(Share<1>::NH, Share<2>::NH));
constexpr int kRounds = (kNV + 7) / 8;  // eight harmonics of every part per round
static_assert(kZ128Chains >= 2 * kLB + 1, "crossing chains fit the exchange rows");

// z rotation of degree l (v[B + m + l])
template <int l, int B, int N>
__device__ __forceinline__ void zr_degree(double2 (&v)[N], double ca, double sa) {
  double cm = ca, sm = sa;
#pragma unroll
  for (int m = 1; m <= l; ++m) {
    if (m > 1) {
      const double c2 = cm * ca - sm * sa;
      sm = sm * ca + cm * sa;
      cm = c2;
    }
    const double2 vp = v[B + l + m], vn = v[B + l - m];
    const double zp = kZsign[l * l + l + m] * sm, zn = kZsign[l * l + l - m] * sm;
    v[B + l + m] = make_double2(cm * vp.x + zp * vn.x, cm * vp.y + zp * vn.y);
    v[B + l - m] = make_double2(cm * vn.x + zn * vp.x, cm * vn.y + zn * vp.y);
  }
}
// y rotation by pi/2 of degree l, or its transpose: it maps m < 0 and m >= 0 to themselves, and
// one real half of one of the two at a time needs the fewest registers beside the harmonics
template <int l, int B, bool TR, int N>
__device__ __forceinline__ void yh_degree(double2 (&v)[N]) {
#pragma unroll
  for (int im = 0; im < 2; ++im) {
    int e = yh_off(l);
#pragma unroll
    for (int pos = 0; pos < 2; ++pos) {
      double o[2 * l + 1];
#pragma unroll
      for (int m = (pos ? 0 : -l); m <= (pos ? l : -1); ++m) o[m + l] = 0.0;
#pragma unroll
      for (int m = (pos ? 0 : -l); m <= (pos ? l : -1); ++m)
#pragma unroll
        for (int mp = (pos ? 0 : -l); mp <= (pos ? l : -1); ++mp)
          if (yh_pat(l, m, mp)) {
            const double c = kYh[e++];
            const double2 x = v[B + l + (TR ? m : mp)];
            o[(TR ? mp : m) + l] += c * (im ? x.y : x.x);
          }
#pragma unroll
      for (int m = (pos ? 0 : -l); m <= (pos ? l : -1); ++m) {
        if (im) v[B + l + m].y = o[m + l];
        else v[B + l + m].x = o[m + l];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}
// (cq, sq) at f[0], (ct, st) of this lane's kz at f[2 + lane], read where they are used
template <int PART, bool TO, int l = Share<PART>::L0, int N>
__device__ __forceinline__ void rotate(double2 (&v)[N], const double2* f, int lane) {
  if constexpr (l <= Share<PART>::L1) {
    if constexpr (l > 0) {
      constexpr int B = l * l - Share<PART>::B0;
      {
        const double2 r = TO ? f[0] : f[2 + lane];
        if (!TO) yh_degree<l, B, false>(v);
        zr_degree<l, B>(v, r.x, TO ? r.y : -r.y);
      }
      if (TO) yh_degree<l, B, false>(v);
      else yh_degree<l, B, true>(v);
      {
        const double2 r = TO ? f[2 + lane] : f[0];
        zr_degree<l, B>(v, r.x, TO ? r.y : -r.y);
        if (TO) yh_degree<l, B, true>(v);
      }
    }
    rotate<PART, TO, l + 1>(v, f, lane);
  }
}

// The tridiagonal chains (l, m), l = |m|..L, run through the parts: forward elimination hands
// g(m) of a part's last degree on in x[m], back substitution hands y(m) of its first degree down.
// Forward elimination of a part; the last part goes on to its back substitution.
template <int PART, int N>
__device__ __forceinline__ void chains_up(double2 (&v)[N], double cdelta, double dslam, double gk, double2* x) {
  using P = Share<PART>;
#pragma unroll
  for (int a = 0; a <= P::L1; ++a) {
    double rb[kL + 1];
    P::template pivots<P::L1>(rb, a, cdelta, dslam, gk);
    const int lf = a > P::L0 ? a : P::L0;  // first degree of the chain in this part
#pragma unroll
    for (int sgn = 0; sgn < (a == 0 ? 1 : 2); ++sgn) {
      const int m = sgn ? -a : a;
      double2 g = make_double2(0.0, 0.0);
      if (a < P::L0) g = x[(m + kLB) * 64];
#pragma unroll
      for (int l = lf; l <= P::L1; ++l) {
        const double2 vl = v[P::at(l, m)];
        if (l > a) {
          const double mu = gk * kTri[(l - 1) * (l - 1) + (l - 1) + m] * rb[l - 1];
          g = make_double2(vl.x + mu * g.y, vl.y - mu * g.x);
        } else {
          g = vl;
        }
        v[P::at(l, m)] = g;
      }
      if constexpr (P::L1 < kL) {
        x[(m + kLB) * 64] = g;
      } else {
        double2 y = make_double2(g.x * rb[kL], g.y * rb[kL]);
        v[P::at(kL, m)] = y;
#pragma unroll
        for (int l = kL - 1; l >= lf; --l) {
          const double bb = gk * kTri[l * l + l + m];
          const double2 gl = v[P::at(l, m)];
          y = make_double2((gl.x + bb * y.y) * rb[l], (gl.y - bb * y.x) * rb[l]);
          v[P::at(l, m)] = y;
        }
        if (a < P::L0) x[(m + kLB) * 64] = y;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <int PART, int N>
__device__ __forceinline__ void chains_down(double2 (&v)[N], double cdelta, double dslam, double gk, double2* x) {
  using P = Share<PART>;
#pragma unroll
  for (int a = 0; a <= P::L1; ++a) {
    double rb[kL + 1];
    P::template pivots<P::L1>(rb, a, cdelta, dslam, gk);
    const int lf = a > P::L0 ? a : P::L0;
#pragma unroll
    for (int sgn = 0; sgn < (a == 0 ? 1 : 2); ++sgn) {
      const int m = sgn ? -a : a;
      double2 y = x[(m + kLB) * 64];
#pragma unroll
      for (int l = P::L1; l >= lf; --l) {
        const double bb = gk * kTri[l * l + l + m];
        const double2 gl = v[P::at(l, m)];
        y = make_double2((gl.x + bb * y.y) * rb[l], (gl.y - bb * y.x) * rb[l]);
        v[P::at(l, m)] = y;
      }
      if (a < P::L0) x[(m + kLB) * 64] = y;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// orders LDS accesses of one wave, and keeps the scheduler from moving work across
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  __builtin_amdgcn_sched_barrier(0);
}

// A wave's LDS rows hold 64 points of eight harmonics, 72 places apart.  Natural order: point z at
// place z.  Between the two radix-8 passes: element m of row k at 9 k + m, the order in which the
// solve takes the points (lane 8 k + m).  All three ways of going over them meet every bank equally
// often and differ from a lane's first place by constants, which cost no registers (with places that
// were turned by the row instead, Lmax 8 took 1201 us, not 1098).
__device__ __forceinline__ int place(int q, int z) { return 72 * q + z; }
__device__ __forceinline__ int slot(int q, int k, int m) { return 72 * q + 9 * k + m; }
__device__ __forceinline__ int point(int q, int lane) { return slot(q, lane >> 3, lane & 7); }

// The column pairs of a workgroup.  The tiles are dealt to the XCDs and the pairs of an XCD's
// tiles to its workgroups in turn, so the two pairs of a tile, which share cache lines, are at
// work at the same time on one XCD.
template <class S>
struct Pairs {
  S* spec;
  int ny, nt, nxh, n, step, xcd;
  int ky, kx0;  // of the pair at hand; ky < 0: no more
  long long istride;
  __device__ __forceinline__ Pairs(const Geom& g, void* sp)
      : spec(reinterpret_cast<S*>(sp)), ny(g.ny), nt(g.nt), nxh(g.nxh), n(blockIdx.x >> 3),
        step(gridDim.x >> 3), xcd(blockIdx.x & 7), istride(spec_index(1, 0, 0, 0, g.ny, g.nt, 128)) {
    find();
  }
  __device__ __forceinline__ void find() {
    for (;; n += step) {
      const int tl = (n >> 1) * 8 + xcd;
      ky = -1;
      if (tl >= nt * ny) return;
      kx0 = (tl % nt) * kKxTile + 2 * (n & 1);
      if (kx0 >= nxh) continue;  // padding columns
      ky = tl / nt;
      return;
    }
  }
  __device__ __forceinline__ void next() {
    n += step;
    find();
  }
  // element (harmonic 0, z, column c) of the pair
  __device__ __forceinline__ S* at(int z, int c) const { return spec + spec_index(0, ky, kx0, z, ny, nt, 128) + c; }
};

template <int N>
__device__ __forceinline__ void clear8(double2 (&v)[N], int b0) {
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (b0 + q < N) v[b0 + q] = make_double2(0.0, 0.0);
}

template <int PART, class S>
__device__ __forceinline__ void column_pairs(const Geom& g, const SolveArgs& a, double2* lds) {
  using P = Share<PART>;
  constexpr int NH = P::NH;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wc = (wv >> 1) & 1, wh = wv & 1;  // this wave's column and half
  // rows of (column, half): kZ128Col (2 c + h); those of part 0 are the chains' rows too, during
  // the solve
  double2* rows = lds + (PART == 0 ? 0 : kZ128Chains * 64 + kZ128Rows * (PART - 1));
  double2* own = rows + kZ128Col * (2 * wc + wh);
  double2* chain = lds + kZ128Col * (2 * wc + wh);
  const double2* tw = lds + 4 * kZ128Col;  // exp(-2 pi i t / 128)
  const double2* tw64 = tw + 128;          // exp(-2 pi i j n / 64) at 8 n + j
  double2* frame = lds + 4 * kZ128Col + 192 + (2 * wc + wh) * kZ128Frame;
  Pairs<S> w(g, a.spec);
  double2 v[NH];
  if (w.ky >= 0 && w.kx0 + (int)(threadIdx.x & 1) < w.nxh) {
    const S* src = w.at((threadIdx.x & 255) >> 1, threadIdx.x & 1) + P::B0 * w.istride;
#pragma unroll
    for (int i = 0; i < NH; ++i) v[i] = spec_ld(src + i * w.istride);
  } else {
#pragma unroll
    for (int i = 0; i < NH; ++i) v[i] = make_double2(0.0, 0.0);
  }
#pragma unroll 1
  while (w.ky >= 0) {
    const bool real = w.kx0 + wc < w.nxh;
    const bool act = a.solve && real;
    // (places, addresses and pivot terms are worked out again where they are used: the registers
    // hold harmonics)
    double cdelta = a.cdelta, dslam = a.dslam;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid), "+s"(cdelta), "+s"(dslam));
    {
      const int lane = tid & 63;
      if (PART == 0 && real) {
        const int hq = lane >> 3, j = lane & 7;
        // lane = 8 k1 + k2 holds kz = 2 (k1 + 8 k2) + half
        const KFrame kf(signed_k(w.kx0 + wc, g.nx) * a.kfac[0], signed_k(w.ky, g.ny) * a.kfac[1],
                        signed_k(2 * (hq + 8 * j) + wh, 128) * a.kfac[2], a.sigma, a.ds);
        if (lane == 0) frame[0] = make_double2(kf.cq, kf.sq);
        frame[2 + lane] = make_double2(kf.ct, kf.st);
        reinterpret_cast<double*>(frame + 66)[lane] = kf.gk;
      }
#pragma unroll
      for (int k = 0; k < kRounds; ++k) {
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, hq = lane >> 3, j = lane & 7;
        const int tz = (tid & 255) >> 1, tc = tid & 1, tm = tz & 63;
        __syncthreads();  // the rows are free (first round of all: the twiddles are in LDS)
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (8 * k + q < NH) rows[kZ128Col * (2 * tc + (tz >> 6)) + place(q, tm)] = v[8 * k + q];
        __syncthreads();
        double2 u[8];
        if (8 * k < NH && real) {
          // radix-2 step: the even kz have x(m) + x(m + 64), the odd ones (x(m) - x(m + 64)) W128^m
          const double2 *lo = rows + kZ128Col * (2 * wc), *hi = lo + kZ128Col;
          if (wh == 0) {
#pragma unroll
            for (int r = 0; r < 8; ++r) u[r] = cadd(lo[place(hq, j + 8 * r)], hi[place(hq, j + 8 * r)]);
          } else {
#pragma unroll
            for (int r = 0; r < 8; ++r)
              u[r] = twiddle<-1>(csub(lo[place(hq, j + 8 * r)], hi[place(hq, j + 8 * r)]), tw[j + 8 * r]);
          }
        }
        __syncthreads();  // both halves have read the rows
        if (8 * k < NH && real) {
          Dft<8, -1>::run(u);
#pragma unroll
          for (int n = 1; n < 8; ++n) u[n] = twiddle<-1>(u[n], tw64[8 * n + j]);
#pragma unroll
          for (int n = 0; n < 8; ++n) own[slot(hq, n, j)] = u[n];
          wave_sync();
#pragma unroll
          for (int m = 0; m < 8; ++m) u[m] = own[slot(hq, j, m)];
          Dft<8, -1>::run(u);
#pragma unroll
          for (int m = 0; m < 8; ++m) own[slot(hq, j, m)] = u[m];
          wave_sync();
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (8 * k + q < NH) v[8 * k + q] = own[point(q, lane)];
        } else {
          clear8(v, 8 * k);  // (nothing is kept across the round: registers)
        }
      }
      double2* x = chain + lane;
      const double* gk = reinterpret_cast<const double*>(frame + 66) + lane;
      if (act) rotate<PART, true>(v, frame, lane);
      if (PART == 0 && act) chains_up<0>(v, cdelta, dslam, *gk, x);
      __syncthreads();
      if (PART == 1 && act) chains_up<1>(v, cdelta, dslam, *gk, x);
      __syncthreads();
      if (PART == 2 && act) chains_up<2>(v, cdelta, dslam, *gk, x);
      __syncthreads();
      if (PART == 1 && act) chains_down<1>(v, cdelta, dslam, *gk, x);
      if (PART == 2 && act) rotate<2, false>(v, frame, lane);
      __syncthreads();
      if (PART == 0 && act) chains_down<0>(v, cdelta, dslam, *gk, x);
      if (PART != 2 && act) rotate<PART, false>(v, frame, lane);
    }
    S* dst0 = w.at(0, 0) + P::B0 * w.istride;
    const int ncol = w.nxh - w.kx0;  // real columns (1 or more)
    w.next();
    const S* src0 = w.at(0, 0) + P::B0 * w.istride;
    const int nload = w.ky >= 0 ? w.nxh - w.kx0 : 0;  // of the next pair
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
      asm volatile("" : "+v"(tid));
      const int lane = tid & 63, hq = lane >> 3, j = lane & 7;
      const int tz = (tid & 255) >> 1, tc = tid & 1, tm = tz & 63;
      const bool io = tc < ncol, load = tc < nload;
      S* dst = dst0 + (4 * tz + tc);
      const S* src = src0 + (4 * tz + tc);
      double2 u[8];
      if (8 * k < NH && real) {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (8 * k + q < NH) own[point(q, lane)] = v[8 * k + q];
        wave_sync();
      }
      // the next pair's harmonics take the registers of the round before
      if (k > 0 && load) {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (8 * (k - 1) + q < NH) v[8 * (k - 1) + q] = spec_ld(src + (8 * (k - 1) + q) * w.istride);
      } else if (k > 0) {
        clear8(v, 8 * (k - 1));
      }
      if (8 * k < NH && real) {
#pragma unroll
        for (int m = 0; m < 8; ++m) u[m] = own[slot(hq, j, m)];
        Dft<8, +1>::run(u);
#pragma unroll
        for (int m = 1; m < 8; ++m) u[m] = twiddle<+1>(u[m], tw64[8 * m + j]);
#pragma unroll
        for (int m = 0; m < 8; ++m) own[slot(hq, j, m)] = u[m];
        wave_sync();
#pragma unroll
        for (int n = 0; n < 8; ++n) u[n] = own[slot(hq, n, j)];
        Dft<8, +1>::run(u);
        if (wh) {
#pragma unroll
          for (int r = 0; r < 8; ++r) u[r] = twiddle<+1>(u[r], tw[j + 8 * r]);
        }
        wave_sync();
#pragma unroll
        for (int r = 0; r < 8; ++r) own[place(hq, j + 8 * r)] = u[r];
      }
      __syncthreads();
      if (k + 1 == kRounds && load) {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (8 * k + q < NH) v[8 * k + q] = spec_ld(src + (8 * k + q) * w.istride);
      } else if (k + 1 == kRounds) {
        clear8(v, 8 * k);
      }
      if (io) {
        const double2 *even = rows + kZ128Col * (2 * tc), *odd = even + kZ128Col;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          if (8 * k + q < NH) {
            const double2 e = even[place(q, tm)], o = odd[place(q, tm)];
            spec_st(dst + (8 * k + q) * w.istride, tz < 64 ? cadd(e, o) : csub(e, o));
          }
        }
      }
      if (k + 1 < kRounds) __syncthreads();  // the rows have been read
    }
  }
}

template <class S>
__device__ __forceinline__ void k_z128_body(const Geom& g, const SolveArgs& a) {
  extern __shared__ double2 lds[];
  if (threadIdx.x < 128) lds[4 * kZ128Col + threadIdx.x] = g.az.tw[threadIdx.x];
  else if (threadIdx.x < 192)
    lds[4 * kZ128Col + threadIdx.x] = g.az.tw[2 * ((threadIdx.x & 63) >> 3) * (threadIdx.x & 7)];
  // wave 4 part + 2 column + half: every SIMD gets one wave of each part
  const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  if (part == 0) column_pairs<0, S>(g, a, lds);
  else if (part == 1) column_pairs<1, S>(g, a, lds);
  else column_pairs<2, S>(g, a, lds);
}

template <class S>
__global__ void __launch_bounds__(kZ128Threads, 3) k_z128(Geom g, SolveArgs a) {
  k_z128_body<S>(g, a);
}

// the same for one instance of a batch per blockIdx.z
template <class S>
__global__ void __launch_bounds__(kZ128Threads, 3) k_z128_b(const ZJob* __restrict__ jobs) {
  const ZJob& j = jobs[blockIdx.z];
  if (j.skip && *j.skip) return;
  k_z128_body<S>(j.g, j.a);
}

}  // namespace z128_l_<L>

using namespace WLC_CAT(z128_l_, WLC_L);

const void* WLC_CAT(z128_kernel_L, WLC_L)(bool spec32, bool batch) {
  if (spec32) {
#if WLC_L >= 7
    return batch ? (const void*)k_z128_b<float2> : (const void*)k_z128<float2>;
#else
    return nullptr;  // runs in two parts (z128_two_parts)
#endif
  }
  return batch ? (const void*)k_z128_b<double2> : (const void*)k_z128<double2>;
}

}  // namespace wlc
