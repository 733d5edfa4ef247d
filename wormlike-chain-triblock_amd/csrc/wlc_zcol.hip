// Kernel B of the propagator step for short z axes (nz of a two-factor plan, nz <= 54), for
// one Lmax (compiled once per L with -DWLC_L=<L>): z pass of the forward FFT, k-aligned solve
// of G(k) q = P(k) (the per-k G^-1 apply of wormlike_MDE_2dcomp_mod.f90:395-409), inverse z
// pass.
//
// These grids leave most of the GPU idle (24^3: 312 columns for 1024 SIMDs), so a launch takes
// as long as one workgroup's chain of dependent phases.  The work of a group of columns is
// therefore spread over a workgroup phase by phase, with all its harmonics in LDS between the
// phases: transforms by (harmonic, butterfly), rotations into and out of the k frame by degree
// (four waves, degrees dealt to equal numbers of harmonics), the tridiagonal chains by |m|
// (four waves again).  The loads of the first radix pass and the stores of the last go straight
// between HBM and registers.  The transform is two register passes (n = R T), both in place, so
// kz index k1 + R k2 sits in row k1 (T slots) during the solve and nothing is reordered.
// Per launch in one kernel trace, against the half-tile kernel it replaces (all harmonics of half a
// column in the registers of one wave): 24^3 / Lmax 6 17.0 -> 12.8 us (of which 2.2 are launch and 2.4
// the first loads), Lmax 4 10.6 -> 8.6, 32^3 / Lmax 4 15.6 -> 12.7, 48^3 / Lmax 6 46.6 -> 40.7, but 48^3 /
// Lmax 4 21.9 -> 24.7 and Lmax 5 28.7 -> 31.3 (its 624 groups are a second round of 512, a fifth full);
// against the generic kernel, 36^3 / Lmax 4 28.9 -> 14.1, 54^3 / Lmax 4 64.7 -> 28.3.  It is bound by the
// latency of its phases.  Where it is not taken: zcol_groups in wlc_dispatch.cpp.
#include <hip/hip_runtime.h>

#include "wlc_dft.h"
#include "wlc_zcol.h"

#ifndef WLC_L
#error "compile with -DWLC_L=<Lmax>"
#endif

#define WLC_CAT2(a, b) a##b
#define WLC_CAT(a, b) WLC_CAT2(a, b)

namespace wlc {
namespace WLC_CAT(zcol_l_, WLC_L) {

constexpr int kL = WLC_L;
constexpr int kM = (kL + 1) * (kL + 1);
constexpr int kParts = 4;
// waves per SIMD the registers are held to: 4 (two eight-wave workgroups of 48-point columns on a
// CU) while a rotation of degree L fits 128 registers; above that LDS admits fewer workgroups anyway
constexpr int kWaves = kL >= 8 ? 2 : (kL == 7 ? 3 : 4);

// degrees (weight 2l + 1) and chains (|m| = a: weight L + 1 or 2 (L + 1 - a)) dealt to the four
// waves, heaviest first to the lightest wave
struct Deal {
  int deg[kL + 1] = {}, chain[kL + 1] = {};
};
constexpr Deal deal() {
  Deal d{};
  for (int what = 0; what < 2; ++what) {
    int load[kParts] = {};
    bool used[kL + 1] = {};
    for (int n = 0; n <= kL; ++n) {
      int best = -1, bw = -1;
      for (int x = 0; x <= kL; ++x) {
        const int w = what == 0 ? 2 * x + 1 : (x ? 2 : 1) * (kL + 1 - x);
        if (!used[x] && w > bw) {
          best = x;
          bw = w;
        }
      }
      int p = 0;
      for (int q = 1; q < kParts; ++q)
        if (load[q] < load[p]) p = q;
      used[best] = true;
      load[p] += bw;
      (what == 0 ? d.deg : d.chain)[best] = p;
    }
  }
  return d;
}
constexpr Deal kDeal = deal();

// harmonics of degree l of one point (stride np in LDS) into or out of the k frame, in place
template <int l, bool TO>
__device__ __forceinline__ void rotate_degree(double2* at, int np, const KFrame& f) {
  if constexpr (l > 0) {
    using P = SolverPart<kL, l, l>;
    double2 v[2 * l + 1];
#pragma unroll
    for (int m = 0; m < 2 * l + 1; ++m) v[m] = at[(l * l + m) * np];
    if (TO) P::to_frame(v, f);
    else P::from_frame(v, f);
#pragma unroll
    for (int m = 0; m < 2 * l + 1; ++m) at[(l * l + m) * np] = v[m];
  }
}

template <int PART, bool TO, int l = 0>
__device__ __forceinline__ void rotate_part(double2* at, int np, const KFrame& f) {
  if constexpr (l <= kL) {
    if constexpr (kDeal.deg[l] == PART) rotate_degree<l, TO>(at, np, f);
    rotate_part<PART, TO, l + 1>(at, np, f);
  }
}

// the chains (l, +-a), l = a..L, of one point: Thomas solve with real pivots
template <int a>
__device__ __forceinline__ void solve_chain(double2* at, int np, double cdelta, double dslam, double gk) {
  double rb[kL + 1];
  SolverPart<kL, 0, kL>::template pivots<kL>(rb, a, cdelta, dslam, gk);
#pragma unroll
  for (int sgn = 0; sgn < (a == 0 ? 1 : 2); ++sgn) {
    const int m = sgn ? -a : a;
    double2 g[kL + 1];
#pragma unroll
    for (int l = a; l <= kL; ++l) g[l] = at[(l * l + l + m) * np];
#pragma unroll
    for (int l = a + 1; l <= kL; ++l) {
      const double mu = gk * kTri[(l - 1) * (l - 1) + (l - 1) + m] * rb[l - 1];
      g[l] = make_double2(g[l].x + mu * g[l - 1].y, g[l].y - mu * g[l - 1].x);
    }
    double2 y = make_double2(g[kL].x * rb[kL], g[kL].y * rb[kL]);
    at[(kL * kL + kL + m) * np] = y;
#pragma unroll
    for (int l = kL - 1; l >= a; --l) {
      const double bb = gk * kTri[l * l + l + m];
      y = make_double2((g[l].x + bb * y.y) * rb[l], (g[l].y - bb * y.x) * rb[l]);
      at[(l * l + l + m) * np] = y;
    }
  }
}

template <int PART, int a = 0>
__device__ __forceinline__ void chains_part(double2* at, int np, double cdelta, double dslam, double gk) {
  if constexpr (a <= kL) {
    if constexpr (kDeal.chain[a] == PART) solve_chain<a>(at, np, cdelta, dslam, gk);
    chains_part<PART, a + 1>(at, np, cdelta, dslam, gk);
  }
}

// One workgroup's columns: element (harmonic i, z, column c) of the spectrum at
// p[i istride + 4 z + c]; column c is real when c < nc.  In LDS harmonic i holds R rows of T
// slots of 1 << lc columns: element m of row k at slot_of(k, m).  The rows are a power of two
// of 16-byte units apart when T is, so the lanes of a pass over the rows would meet on one
// bank group; the order within a row is turned by the row (48^3 / Lmax 6 47.0 -> 40.6 us).
struct Cols {
  double2* p;
  unsigned istride;
  int lc, nc, np;
};

template <int T>
__device__ __forceinline__ int turn(int k, int lc) {
  if constexpr (T == 2 || T == 4 || T == 8) {
    // rows per 16 units: 1 << sh
    constexpr int lt = T == 8 ? 3 : (T == 4 ? 2 : 1);
    const int sh = 4 - lt - lc > 0 ? 4 - lt - lc : 0;
    return (k >> sh) & (T - 1);
  }
  return 0;
}
template <int T>
__device__ __forceinline__ int slot_of(int k, int m, int lc) {
  return T * k + (m ^ turn<T>(k, lc));
}

// forward pass 1: DFT-R over z = j + T r, twiddle, from HBM into LDS
template <int R, int T>
__device__ __forceinline__ void pass_in(double2* lds, const Cols& w, const double2* __restrict__ tw) {
  constexpr int U = R <= 4 ? 4 : 2;  // butterflies in flight per thread
  const int total = (kM * T) << w.lc, nthr = blockDim.x;
  for (int base = threadIdx.x; base < total; base += U * nthr) {
    double2 u[U][R];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int idx = base + q * nthr;
      const int c = idx & ((1 << w.lc) - 1), r = idx >> w.lc;
      const int i = r / T, j = r - i * T;
      const bool ok = idx < total && c < w.nc;
      const double2* src = w.p + (unsigned(i) * w.istride + unsigned(kKxTile * j + c));
#pragma unroll
      for (int k = 0; k < R; ++k) u[q][k] = ok ? spec_ld(src + kKxTile * T * k) : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int idx = base + q * nthr;
      if (idx < total) {
        const int c = idx & ((1 << w.lc) - 1), r = idx >> w.lc;
        const int i = r / T, j = r - i * T;
        Dft<R, -1>::run(u[q]);
#pragma unroll
        for (int k = 1; k < R; ++k) u[q][k] = twiddle<-1>(u[q][k], tw[j * k]);
#pragma unroll
        for (int k = 0; k < R; ++k) lds[i * w.np + (slot_of<T>(k, j, w.lc) << w.lc) + c] = u[q][k];
      }
    }
  }
}

// forward pass 2 (DIR = -1: DFT-T over row k1) and inverse pass 1 (DIR = +1: the same, then the
// twiddle), in place in LDS
template <int R, int T, int DIR>
__device__ __forceinline__ void pass_mid(double2* lds, const Cols& w, const double2* __restrict__ tw) {
  constexpr int U = 2;
  const int total = (kM * R) << w.lc, nthr = blockDim.x;
  for (int base = threadIdx.x; base < total; base += U * nthr) {
    double2 u[U][T];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int idx = base + q * nthr;
      const int c = idx & ((1 << w.lc) - 1), r = idx >> w.lc;
      const int i = r / R, k1 = r - i * R;
      if (idx < total) {
#pragma unroll
        for (int m = 0; m < T; ++m) u[q][m] = lds[i * w.np + (slot_of<T>(k1, m, w.lc) << w.lc) + c];
      }
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int idx = base + q * nthr;
      const int c = idx & ((1 << w.lc) - 1), r = idx >> w.lc;
      const int i = r / R, k1 = r - i * R;
      if (idx < total) {
        Dft<T, DIR>::run(u[q]);
        if (DIR > 0) {
#pragma unroll
          for (int m = 1; m < T; ++m) u[q][m] = twiddle<+1>(u[q][m], tw[k1 * m]);
        }
#pragma unroll
        for (int m = 0; m < T; ++m) lds[i * w.np + (slot_of<T>(k1, m, w.lc) << w.lc) + c] = u[q][m];
      }
    }
  }
}

// inverse pass 2: DFT-R over the rows, from LDS to HBM
template <int R, int T>
__device__ __forceinline__ void pass_out(const double2* lds, const Cols& w) {
  constexpr int U = 2;
  const int total = (kM * T) << w.lc, nthr = blockDim.x;
  for (int base = threadIdx.x; base < total; base += U * nthr) {
    double2 u[U][R];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int idx = base + q * nthr;
      const int c = idx & ((1 << w.lc) - 1), r = idx >> w.lc;
      const int i = r / T, j = r - i * T;
      if (idx < total) {
#pragma unroll
        for (int k = 0; k < R; ++k) u[q][k] = lds[i * w.np + (slot_of<T>(k, j, w.lc) << w.lc) + c];
      }
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int idx = base + q * nthr;
      const int c = idx & ((1 << w.lc) - 1), r = idx >> w.lc;
      const int i = r / T, j = r - i * T;
      if (idx < total && c < w.nc) {
        Dft<R, +1>::run(u[q]);
        double2* dst = w.p + (unsigned(i) * w.istride + unsigned(kKxTile * j + c));
#pragma unroll
        for (int k = 0; k < R; ++k) spec_st(dst + kKxTile * T * k, u[q][k]);
      }
    }
  }
}

__device__ __forceinline__ int turn_of(int T, int k, int lc) {
  return T == 2 ? turn<2>(k, lc) : T == 4 ? turn<4>(k, lc) : T == 8 ? turn<8>(k, lc) : 0;
}

template <int NZ>
__device__ __forceinline__ void transform_in(double2* lds, const Cols& w, const double2* __restrict__ tw) {
  constexpr int R = two_pass(NZ).R, T = two_pass(NZ).T;
  pass_in<R, T>(lds, w, tw);
  __syncthreads();
  pass_mid<R, T, -1>(lds, w, tw);
}
template <int NZ>
__device__ __forceinline__ void transform_out(double2* lds, const Cols& w, const double2* __restrict__ tw) {
  constexpr int R = two_pass(NZ).R, T = two_pass(NZ).T;
  pass_mid<R, T, +1>(lds, w, tw);
  __syncthreads();
  pass_out<R, T>(lds, w);
}

#define WLC_EACH_NZ(X) X(8) X(12) X(16) X(18) X(24) X(32) X(36) X(48) X(54)

__device__ __forceinline__ void k_zcol_body(const Geom& g, const SolveArgs& a) {
  extern __shared__ double2 lds[];
  const int nz = g.nz, ny = g.ny, nt = g.nt;
  const int lc = zcol_log2_cols(nz), sub = kKxTile >> lc;  // column groups per 4-kx tile
  // the groups of a tile run back to back on one XCD: they write parts of the same cache lines,
  // and from two L2s those go out as partial lines (36^3 / Lmax 4: 22 us a launch, not 13)
  const int b = blockIdx.x, t = b >> 3;
  const int grp = t % sub, tl = (t / sub) * 8 + (b & 7);
  if (tl >= nt * ny) return;  // (uniform)
  const int t4 = tl % nt, ky = tl / nt;
  const int kx0 = t4 * kKxTile + (grp << lc);
  Cols w;
  w.lc = lc;
  w.nc = min(1 << lc, g.nxh - kx0);
  if (w.nc <= 0) return;  // padding columns only (uniform)
  w.np = nz << lc;
  w.istride = (unsigned)spec_index(1, 0, 0, 0, ny, nt, nz);
  w.p = a.spec + spec_index(0, ky, kx0, 0, ny, nt, nz);
  const double2* tw = g.az.tw;
  int R = 1, T = 1;
  switch (nz) {
#define X(N)                          \
  case N:                             \
    R = two_pass(N).R;                \
    T = two_pass(N).T;                \
    transform_in<N>(lds, w, tw);      \
    break;
    WLC_EACH_NZ(X)
#undef X
  }
  if (a.solve) {
    const int wv = threadIdx.x >> 6, part = wv & (kParts - 1);
    const int pt = (wv / kParts) * 64 + (threadIdx.x & 63);
    const int c = pt & ((1 << lc) - 1), slot = pt >> lc;
    const bool act = pt < w.np && c < w.nc;
    const int k1 = slot / T, kz = k1 + R * ((slot - k1 * T) ^ turn_of(T, k1, lc));
    const KFrame f(signed_k(kx0 + c, g.nx) * a.kfac[0], signed_k(ky, ny) * a.kfac[1],
                   signed_k(act ? kz : 0, nz) * a.kfac[2], a.sigma, a.ds);
    double2* at = lds + pt;
    __syncthreads();
    if (act) {
      if (part == 0) rotate_part<0, true>(at, w.np, f);
      else if (part == 1) rotate_part<1, true>(at, w.np, f);
      else if (part == 2) rotate_part<2, true>(at, w.np, f);
      else rotate_part<3, true>(at, w.np, f);
    }
    __syncthreads();
    if (act) {
      if (part == 0) chains_part<0>(at, w.np, a.cdelta, a.dslam, f.gk);
      else if (part == 1) chains_part<1>(at, w.np, a.cdelta, a.dslam, f.gk);
      else if (part == 2) chains_part<2>(at, w.np, a.cdelta, a.dslam, f.gk);
      else chains_part<3>(at, w.np, a.cdelta, a.dslam, f.gk);
    }
    __syncthreads();
    if (act) {
      if (part == 0) rotate_part<0, false>(at, w.np, f);
      else if (part == 1) rotate_part<1, false>(at, w.np, f);
      else if (part == 2) rotate_part<2, false>(at, w.np, f);
      else rotate_part<3, false>(at, w.np, f);
    }
  }
  __syncthreads();
  switch (nz) {
#define X(N)                          \
  case N: transform_out<N>(lds, w, tw); break;
    WLC_EACH_NZ(X)
#undef X
  }
}

__global__ void __launch_bounds__(512, kWaves) k_zcol(Geom g, SolveArgs a) {
  k_zcol_body(g, a);
}

// the same for one instance of a batch per blockIdx.z
__global__ void __launch_bounds__(512, kWaves) k_zcol_b(const ZJob* __restrict__ jobs) {
  const ZJob& j = jobs[blockIdx.z];
  if (j.skip && *j.skip) return;
  k_zcol_body(j.g, j.a);
}

}  // namespace zcol_l_<L>

using namespace WLC_CAT(zcol_l_, WLC_L);

const void* WLC_CAT(zcol_kernel_L, WLC_L)(bool batch) {
  return batch ? (const void*)k_zcol_b : (const void*)k_zcol;
}

}  // namespace wlc
