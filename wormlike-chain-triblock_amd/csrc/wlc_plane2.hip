// Plane kernels of the propagator step for edges of a two-factor plan n = R T (8 .. 72; 64 x 64
// planes have their own), any pair of them: per (harmonic, z-plane) the BDF right-hand side
// (wormlike_MDE_2dcomp_mod.f90:325-343, 484-502, 584-608; junction padding :697-806) with the
// x (R2C, two real rows per complex transform) and y passes of the forward FFT (A), the inverse y
// and x (C2R) passes with 1/N and the store of q(s) (C, :433-455), and C of one step fused with A
// of the next.
//
// A transform is two register passes of radix R and T through LDS.  Both work in place (the second
// reads the rows the first leaves), so a y transform needs one workgroup barrier between them, an
// x transform only wave synchronisation, since the T lanes of a row pair belong to one wave; the
// real rows stand in the order y = r / T + R (r % T) in between, which only the addresses of the
// right-hand side and the unpacking see.  At these sizes a launch is as long as one plane's chain of
// dependent phases, so everything the plane reads (spectrum, twiddles, history, w) is asked for at
// the start and the twiddles are kept in LDS.
#include <hip/hip_runtime.h>

#include "wlc_plane2.h"

namespace wlc {
namespace p2 {
namespace {

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// block -> (z-plane, harmonic): XCD k takes the z-planes [k nz/8, (k+1) nz/8) of every harmonic
// when nz is a multiple of 8 (w stays in its L2; the planes sharing a spectrum cache line run back
// to back on one XCD), else a contiguous range of (harmonic, z)
__device__ __forceinline__ void plane_of_block(int nz, int& z, int& i) {
  const int nb = gridDim.x, b = blockIdx.x;
  if ((nz & 7) == 0) {
    const int zr = nz >> 3, t = b >> 3;
    i = t / zr;
    z = (b & 7) * zr + (t - i * zr);
    return;
  }
  const int q = nb >> 3;
  const int logical = (b < (q << 3)) ? ((b & 7) * q + (b >> 3)) : b;
  i = logical / nz;
  z = logical - i * nz;
}

// one point of the BDF right-hand side in a fixed rounding sequence (fused and unfused kernels
// give the same bits)
__device__ __forceinline__ double bdf_rhs(double q1, double q2, double q3, double w, const RhsArgs& a) {
  const double t = __builtin_fma(a.a[2], q3, __builtin_fma(a.a[1], q2, a.a[0] * q1));
  const double u = __builtin_fma(a.b[2], q3, __builtin_fma(a.b[1], q2, a.b[0] * q1));
  return __builtin_fma(-(a.ds * w), u, t);
}

// The plane in LDS.  Row pair b owns the slots b stride ..: in the x layout its rows 2b and 2b + 1
// are the real and imaginary parts of x = 0 .. nx - 1, in the y layout row slot r = 2b + o, column
// c < h is at o h + c; column 0 holds X(kx = 0) + i X(kx = h).
struct Plane {
  double2 *buf, *col, *tx, *ty;  // plane, columns kx = 0 and h (ny each), twiddles
  Shape s;
  int nx, ny;
  __device__ __forceinline__ double2& row(int r, int c) const {
    return buf[(r >> 1) * s.stride + (r & 1) * s.h + c];
  }
};

// workgroup-uniform base of spectrum plane (i, z) and 32-bit offsets
struct SpecPlane {
  double2* p;
  unsigned rs, ts;
  __device__ __forceinline__ SpecPlane(double2* spec, const Geom& g, int i, int z)
      : p(spec + spec_index(i, 0, 0, z, g.ny, g.nt, g.nz)),
        rs(unsigned(g.nt) * unsigned(g.nz) * kKxTile),
        ts(unsigned(g.nz) * kKxTile) {}
  __device__ __forceinline__ double2* at(int ky, int kx) const {
    return p + (unsigned(ky) * rs + unsigned(kx >> 2) * ts + unsigned(kx & 3));
  }
};

// what a plane reads before its first transform, in flight
template <int R>
struct Start {
  double2 v[R];  // spectrum column c = tid % h at ky = jy + T r (c > 0)
};

// the spectrum (R, T of the y axis), then columns 0 and h and the twiddles into LDS; the caller's
// own loads are issued by `more` before anything is waited for, and a barrier follows
template <int RMAX, class F>
__device__ __forceinline__ void start(Start<RMAX>& st, const Plane& pl, int R, int T, const double2* spec, const Geom& g,
                                      int i, int z, bool inv, F&& more) {
  const int tid = threadIdx.x, nthr = blockDim.x;
  const SpecPlane sp(const_cast<double2*>(spec), g, i, z);
  if (inv) {
    const int jy = tid / pl.s.h, c = tid - jy * pl.s.h;
    if (jy < T && c) {
#pragma unroll
      for (int r = 0; r < RMAX; ++r)
        if (r < R) st.v[r] = spec_ld(sp.at(jy + T * r, c));
    }
  }
  // at most two rounds: ny <= 72 and at least one wave
  double2 c0[2], ch[2], t0[3];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int ky = tid + q * nthr;
    if (inv && ky < pl.ny) {
      c0[q] = spec_ld(sp.at(ky, 0));
      ch[q] = spec_ld(sp.at(ky, pl.s.h));
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int e = tid + q * nthr;
    if (e < pl.nx + pl.ny) t0[q] = e < pl.nx ? g.ax.tw[e] : g.ay.tw[e - pl.nx];
  }
  more();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int ky = tid + q * nthr;
    if (inv && ky < pl.ny) {
      pl.col[ky] = c0[q];
      pl.col[pl.ny + ky] = ch[q];
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int e = tid + q * nthr;
    if (e < pl.nx + pl.ny) pl.tx[e] = t0[q];  // ty follows tx
  }
  __syncthreads();
}

// Inverse y transform of the spectrum plane into the y layout (unscaled).  Columns kx = 0 and h
// enter as H0 + i Hh with H(ky) = (X(ky) + conj X(-ky)) / 2: the inverse of H is the real part of
// the inverse of X, what a C2R transform keeps of those columns.
template <int NY, int RMAX>
__device__ __forceinline__ void y_inverse(const Plane& pl, const Start<RMAX>& st) {
  constexpr int R = two_pass(NY).R, T = two_pass(NY).T;
  const int jy = threadIdx.x / pl.s.h, c = threadIdx.x - jy * pl.s.h;
  const double2* tw = pl.ty;
  if (jy < T) {
    double2 v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = st.v[r];
    if (c == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int ky = jy + T * r, kn = ky ? NY - ky : 0;
        const double2 a = pl.col[ky], an = pl.col[kn], b = pl.col[NY + ky], bn = pl.col[NY + kn];
        const double2 h0 = make_double2(0.5 * (a.x + an.x), 0.5 * (a.y - an.y));
        const double2 h1 = make_double2(0.5 * (b.x + bn.x), 0.5 * (b.y - bn.y));
        v[r] = make_double2(h0.x - h1.y, h0.y + h1.x);
      }
    }
    Dft<R, +1>::run(v);
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = twiddle<+1>(v[k], tw[jy * k]);
#pragma unroll
    for (int k = 0; k < R; ++k) pl.row(T * k + jy, c) = v[k];
  }
  __syncthreads();
  if (jy < T) {
#pragma unroll
    for (int q = 0; q < (R + T - 1) / T; ++q) {
      const int k1 = jy + q * T;
      if (R % T == 0 || k1 < R) {
        double2 v[T];
#pragma unroll
        for (int m = 0; m < T; ++m) v[m] = pl.row(T * k1 + m, c);
        Dft<T, +1>::run(v);
#pragma unroll
        for (int m = 0; m < T; ++m) pl.row(T * k1 + m, c) = v[m];
      }
    }
  }
  __syncthreads();
}

// real row at row slot r
template <int NY>
__device__ __forceinline__ int real_row(int r) {
  constexpr int R = two_pass(NY).R, T = two_pass(NY).T;
  return r / T + R * (r % T);
}

// Inverse x transform of the row pairs (C2R, one complex transform each) from the y layout into
// the x layout; the Hermitian extension Z_k = A_k + i B_k, Z_{n-k} = conj A_k + i conj B_k is
// formed while loading.
template <int NX>
__device__ __forceinline__ void x_inverse(const Plane& pl) {
  const double2* tw = pl.tx;
  constexpr int R = two_pass(NX).R, T = two_pass(NX).T, H = NX / 2, Q = (R + T - 1) / T;
  const int lane = threadIdx.x & 63, lb = lane / T, j = lane - lb * T;
  const int b = (threadIdx.x >> 6) * pl.s.ppw + lb;
  const bool act = lb < pl.s.ppw && b < pl.s.pairs;
  double2* at = pl.buf + b * pl.s.stride;
  double2 v[R];
  if (act) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int k = j + T * r;
      const bool lo = k < H;
      const int kk = k > H ? NX - k : (lo ? k : 0);  // k = H: packed column 0
      const double2 A = at[kk], B = at[H + kk];
      v[r] = lo ? make_double2(A.x - B.y, A.y + B.x) : make_double2(A.x + B.y, B.x - A.y);
      if (kk == 0) v[r] = lo ? make_double2(A.x, B.x) : make_double2(A.y, B.y);
    }
    Dft<R, +1>::run(v);
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = twiddle<+1>(v[k], tw[j * k]);
  }
  wave_lds_sync();  // the pair's y-layout slots have been read
  if (act) {
#pragma unroll
    for (int k = 0; k < R; ++k) at[T * k + j] = v[k];
  }
  wave_lds_sync();
  double2 u[Q][T];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k1 = j + q * T;
    if (act && (R % T == 0 || k1 < R)) {
#pragma unroll
      for (int m = 0; m < T; ++m) u[q][m] = at[T * k1 + m];
      Dft<T, +1>::run(u[q]);
    }
  }
  wave_lds_sync();
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k1 = j + q * T;
    if (act && (R % T == 0 || k1 < R)) {
#pragma unroll
      for (int m = 0; m < T; ++m) at[k1 + R * m] = u[q][m];
    }
  }
  wave_lds_sync();
}

// Forward x transform of the row pairs, in place: Z_k ends at slot T (k % R) + k / R.
template <int NX>
__device__ __forceinline__ void x_forward(const Plane& pl) {
  const double2* tw = pl.tx;
  constexpr int R = two_pass(NX).R, T = two_pass(NX).T, Q = (R + T - 1) / T;
  const int lane = threadIdx.x & 63, lb = lane / T, j = lane - lb * T;
  const int b = (threadIdx.x >> 6) * pl.s.ppw + lb;
  const bool act = lb < pl.s.ppw && b < pl.s.pairs;
  double2* at = pl.buf + b * pl.s.stride;
  if (act) {
    double2 v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = at[j + T * r];
    Dft<R, -1>::run(v);
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = twiddle<-1>(v[k], tw[j * k]);
#pragma unroll
    for (int k = 0; k < R; ++k) at[T * k + j] = v[k];
  }
  wave_lds_sync();
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k1 = j + q * T;
    if (act && (R % T == 0 || k1 < R)) {
      double2 u[T];
#pragma unroll
      for (int m = 0; m < T; ++m) u[m] = at[T * k1 + m];
      Dft<T, -1>::run(u);
#pragma unroll
      for (int m = 0; m < T; ++m) at[T * k1 + m] = u[m];
    }
  }
}

template <int NX>
__device__ __forceinline__ int x_slot(int k) {
  constexpr int R = two_pass(NX).R, T = two_pass(NX).T;
  return T * (k % R) + k / R;
}

// Unpack of the row pairs (A_k = (Z_k + conj Z_{n-k}) / 2 the even row slot, B_k = (Z_k -
// conj Z_{n-k}) / 2i the odd one), forward y transform, store of the spectrum plane; pk and pn are
// the slots of Z_c and Z_{n-c} (c = 0: of Z_0 and Z_h, the real values of the packed column).
template <int NY>
__device__ __forceinline__ void y_forward(const Plane& pl, int pk, int pn, double2* spec, const Geom& g, int i, int z) {
  constexpr int R = two_pass(NY).R, T = two_pass(NY).T, Q = (R + T - 1) / T;
  static_assert(T % 2 == 0, "a thread unpacks whole row pairs");
  const int jy = threadIdx.x / pl.s.h, c = threadIdx.x - jy * pl.s.h;
  const double2* tw = pl.ty;
  double2* col = pl.col;
  __syncthreads();
  double2 u[Q][T];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k1 = jy + q * T;
    if (jy < T && (R % T == 0 || k1 < R)) {
#pragma unroll
      for (int m = 0; m < T; m += 2) {
        const double2* at = pl.buf + ((T * k1 + m) >> 1) * pl.s.stride;
        const double2 zk = at[pk], zn = at[pn];
        u[q][m] = c ? make_double2(0.5 * (zk.x + zn.x), 0.5 * (zk.y - zn.y)) : make_double2(zk.x, zn.x);
        u[q][m + 1] = c ? make_double2(0.5 * (zk.y + zn.y), -0.5 * (zk.x - zn.x)) : make_double2(zk.y, zn.y);
      }
      Dft<T, -1>::run(u[q]);
#pragma unroll
      for (int m = 1; m < T; ++m) u[q][m] = twiddle<-1>(u[q][m], tw[k1 * m]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k1 = jy + q * T;
    if (jy < T && (R % T == 0 || k1 < R)) {
#pragma unroll
      for (int m = 0; m < T; ++m) pl.row(T * k1 + m, c) = u[q][m];
    }
  }
  __syncthreads();
  const SpecPlane sp(spec, g, i, z);
  if (jy < T) {
    double2 v[R];
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = pl.row(T * k + jy, c);
    Dft<R, -1>::run(v);
#pragma unroll
    for (int p = 0; p < R; ++p) {
      if (c) spec_st(sp.at(jy + T * p, c), v[p]);
      else col[jy + T * p] = v[p];
    }
  }
  __syncthreads();
  for (int ky = threadIdx.x; ky < NY; ky += blockDim.x) {
    // P = X0 + i Xh, both Hermitian along ky: X0 = (P + conj P(-ky)) / 2, Xh = (P - conj P(-ky)) / 2i
    const double2 p = col[ky], n = col[ky ? NY - ky : 0];
    spec_st(sp.at(ky, 0), make_double2(0.5 * (p.x + n.x), 0.5 * (p.y - n.y)));
    spec_st(sp.at(ky, pl.s.h), make_double2(0.5 * (p.y + n.y), -0.5 * (p.x - n.x)));
  }
}

#define WLC_EACH_EDGE(X) X(8) X(12) X(16) X(18) X(24) X(32) X(36) X(48) X(54) X(64) X(72)

// NX, NY = 0: the edge is a run-time value and picks its transform by a uniform switch
template <int NY, int RMAX>
__device__ __forceinline__ void y_inverse_any(const Plane& pl, const Start<RMAX>& st) {
  if constexpr (NY > 0) y_inverse<NY>(pl, st);
  else switch (pl.ny) {
#define X(N) case N: y_inverse<N>(pl, st); break;
    WLC_EACH_EDGE(X)
#undef X
  }
}
template <int NX>
__device__ __forceinline__ void x_inverse_any(const Plane& pl) {
  if constexpr (NX > 0) x_inverse<NX>(pl);
  else switch (pl.nx) {
#define X(N) case N: x_inverse<N>(pl); break;
    WLC_EACH_EDGE(X)
#undef X
  }
}
template <int NX, int NY>
__device__ __forceinline__ void forward_any(const Plane& pl, double2* spec, const Geom& g, int i, int z) {
  const int c = threadIdx.x % pl.s.h, cn = c ? pl.nx - c : pl.s.h;
  int pk = 0, pn = 0;
  if constexpr (NX > 0) {
    x_forward<NX>(pl);
    pk = x_slot<NX>(c);
    pn = x_slot<NX>(cn);
  } else switch (pl.nx) {
#define X(N)                   \
  case N:                      \
    x_forward<N>(pl);          \
    pk = x_slot<N>(c);         \
    pn = x_slot<N>(cn);        \
    break;
    WLC_EACH_EDGE(X)
#undef X
  }
  if constexpr (NY > 0) y_forward<NY>(pl, pk, pn, spec, g, i, z);
  else switch (pl.ny) {
#define X(N) case N: y_forward<N>(pl, pk, pn, spec, g, i, z); break;
    WLC_EACH_EDGE(X)
#undef X
  }
}
// a / b for 0 <= a < 2^20, 0 < b <= 256 (the quotient's distance to the next integer is at least
// 1 / 2b, far above the error of the reciprocal)
__device__ __forceinline__ int quot(int a, int b) { return (int)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)b)); }

template <int NY>
__device__ __forceinline__ int real_row_any(const Plane& pl, int r) {
  if constexpr (NY > 0) return real_row<NY>(r);
  const TwoPass p = two_pass(pl.ny);
  const int k = quot(r, p.T);
  return k + p.R * (r - k * p.T);
}

template <int NX, int NY>
__device__ __forceinline__ Plane plane_of(double2* lds, const Geom& g) {
  Plane pl;
  pl.buf = lds;
  pl.nx = NX ? NX : g.nx;
  pl.ny = NY ? NY : g.ny;
  if constexpr (NX > 0) {
    constexpr Shape s = shape_of(NX, NY);
    pl.s = s;
  } else {
    pl.s.pairs = g.ny / 2;
    pl.s.h = g.nx / 2;
    pl.s.stride = g.nx + ((5 - g.nx) & 15);
    pl.s.waves = blockDim.x >> 6;
    pl.s.ppw = quot(pl.s.pairs + pl.s.waves - 1, pl.s.waves);
  }
  pl.col = lds + pl.s.pairs * pl.s.stride;
  pl.tx = pl.col + 2 * pl.ny;
  pl.ty = pl.tx + pl.nx;
  return pl;
}

// Real rows: lane items m = 0 .. kItems - 1 of a wave, item lane + 64 m = (row pair, x pair) of the
// wave's row pairs; 16-byte accesses of rows 2b and 2b + 1 at x, x + 1.
template <int NX, int NY>
struct Items {
  // at most kItems, exactly as many as a compile-time shape needs
  static constexpr int N = NX > 0 ? (shape_of(NX > 0 ? NX : 8, NY > 0 ? NY : 8).ppw * (NX / 2) + 63) / 64 : kItems;
  int at[N];       // LDS slot of x (row pair's x layout), -1: no item
  int o0[N], o1[N];  // offsets of the rows in a z-plane
  __device__ __forceinline__ Items() {}
  __device__ __forceinline__ void set(const Plane& pl) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int m = 0; m < N; ++m) {
      const int e = lane + 64 * m, lb = NX > 0 ? e / pl.s.h : quot(e, pl.s.h), xp = e - lb * pl.s.h;
      const int b = wv * pl.s.ppw + lb;
      const bool in = lb < pl.s.ppw && b < pl.s.pairs;
      at[m] = in ? b * pl.s.stride + 2 * xp : -1;
      o0[m] = in ? real_row_any<NY>(pl, 2 * b) * pl.nx + 2 * xp : 0;
      o1[m] = in ? real_row_any<NY>(pl, 2 * b + 1) * pl.nx + 2 * xp : 0;
    }
  }
};

// the operands of the right-hand side that do not depend on this launch
template <int N>
struct Hist {
  double2 a0[N], a1[N], b0[N], b1[N], w0[N], w1[N];
};

__device__ __forceinline__ double2 ld2(const double* p) { return *reinterpret_cast<const double2*>(p); }

// history slices 1 and 2 (a zero plane is read from the zero field) and w, all loads issued here
template <int NX, int NY>
__device__ __forceinline__ void load_hist(Hist<Items<NX, NY>::N>& hv, const Items<NX, NY>& it, const Geom& g,
                                          const RhsArgs& a, int i, long long plane) {
  const double* h1 = i < a.hM[1] ? a.h[1] + i * g.hs + plane : a.zero + plane;
  const double* h2 = i < a.hM[2] ? a.h[2] + i * g.hs + plane : a.zero + plane;
  const double* w = a.w + plane;
#pragma unroll
  for (int m = 0; m < Items<NX, NY>::N; ++m)
    if (it.at[m] >= 0) {
      hv.a0[m] = ld2(h1 + it.o0[m]);
      hv.a1[m] = ld2(h1 + it.o1[m]);
      hv.b0[m] = ld2(h2 + it.o0[m]);
      hv.b1[m] = ld2(h2 + it.o1[m]);
      hv.w0[m] = ld2(w + it.o0[m]);
      hv.w1[m] = ld2(w + it.o1[m]);
    }
}

// right-hand side of one item into the x layout
template <int N>
__device__ __forceinline__ void put_rhs(double2* buf, int at, int m, double2 q0, double2 q1, const Hist<N>& hv,
                                        const RhsArgs& a) {
  buf[at] = make_double2(bdf_rhs(q0.x, hv.a0[m].x, hv.b0[m].x, hv.w0[m].x, a),
                         bdf_rhs(q1.x, hv.a1[m].x, hv.b1[m].x, hv.w1[m].x, a));
  buf[at + 1] = make_double2(bdf_rhs(q0.y, hv.a0[m].y, hv.b0[m].y, hv.w0[m].y, a),
                             bdf_rhs(q1.y, hv.a1[m].y, hv.b1[m].y, hv.w1[m].y, a));
}

// radices of the y axis, and registers for its first
template <int NY>
struct YPlan {
  static constexpr int RMAX = NY > 0 ? two_pass(NY > 0 ? NY : 8).R : 9;
};

// A: right-hand side from the history slices, forward x and y passes
template <int NX, int NY>
__device__ __forceinline__ void k_rhs_body(const Geom& g, const RhsArgs& a) {
  extern __shared__ double2 lds[];
  int z, i;
  plane_of_block(g.nz, z, i);
  const long long plane = (long long)z * g.zs;
  const Plane pl = plane_of<NX, NY>(lds, g);
  const TwoPass py = two_pass(pl.ny);
  Start<YPlan<NY>::RMAX> st;
  Items<NX, NY> it;
  Hist<Items<NX, NY>::N> hv;
  start(st, pl, py.R, py.T, a.spec, g, i, z, false, [&] {
    it.set(pl);
    load_hist<NX, NY>(hv, it, g, a, i, plane);
  });
  const double* h0 = i < a.hM[0] ? a.h[0] + i * g.hs + plane : a.zero + plane;
#pragma unroll
  for (int m = 0; m < Items<NX, NY>::N; ++m)
    if (it.at[m] >= 0) put_rhs(lds, it.at[m], m, ld2(h0 + it.o0[m]), ld2(h0 + it.o1[m]), hv, a);
  wave_lds_sync();
  forward_any<NX, NY>(pl, a.spec, g, i, z);
}

// C: inverse y and x passes, 1/N, store of q(s)
template <int NX, int NY>
__device__ __forceinline__ void k_inv_body(const Geom& g, const InvArgs& c) {
  extern __shared__ double2 lds[];
  int z, i;
  plane_of_block(g.nz, z, i);
  const Plane pl = plane_of<NX, NY>(lds, g);
  const TwoPass py = two_pass(pl.ny);
  Start<YPlan<NY>::RMAX> st;
  Items<NX, NY> it;
  start(st, pl, py.R, py.T, c.spec, g, i, z, true, [&] { it.set(pl); });
  y_inverse_any<NY>(pl, st);
  x_inverse_any<NX>(pl);
  double* out = c.out + i * g.hs + (long long)z * g.zs;
#pragma unroll
  for (int m = 0; m < Items<NX, NY>::N; ++m)
    if (it.at[m] >= 0) {
      const double2 z0 = lds[it.at[m]], z1 = lds[it.at[m] + 1];
      *reinterpret_cast<double2*>(out + it.o0[m]) = make_double2(z0.x * c.scale, z1.x * c.scale);
      *reinterpret_cast<double2*>(out + it.o1[m]) = make_double2(z0.y * c.scale, z1.y * c.scale);
    }
}

// C of step s fused with A of the next: harmonic i < M(s) is inverted and stored and stays in LDS
// as the newest history plane (zero beyond: a junction that grows the basis); for i < M(next) the
// right-hand side is formed in place and transformed into the same spectrum plane.
template <int NX, int NY>
__device__ __forceinline__ void k_inv_rhs_body(const Geom& g, const InvArgs& c, const RhsArgs& a) {
  extern __shared__ double2 lds[];
  int z, i;
  plane_of_block(g.nz, z, i);
  const long long plane = (long long)z * g.zs;
  const Plane pl = plane_of<NX, NY>(lds, g);
  const TwoPass py = two_pass(pl.ny);
  const bool inv = i < c.M, rhs = i < a.M;
  Start<YPlan<NY>::RMAX> st;
  Items<NX, NY> it;
  Hist<Items<NX, NY>::N> hv;
  start(st, pl, py.R, py.T, c.spec, g, i, z, inv, [&] {
    it.set(pl);
    if (rhs) load_hist<NX, NY>(hv, it, g, a, i, plane);
  });
  if (inv) {
    y_inverse_any<NY>(pl, st);
    x_inverse_any<NX>(pl);
  }
  double* out = c.out + i * g.hs + plane;
#pragma unroll
  for (int m = 0; m < Items<NX, NY>::N; ++m)
    if (it.at[m] >= 0) {
      double2 q0 = make_double2(0.0, 0.0), q1 = q0;
      if (inv) {
        const double2 z0 = lds[it.at[m]], z1 = lds[it.at[m] + 1];
        q0 = make_double2(z0.x * c.scale, z1.x * c.scale);
        q1 = make_double2(z0.y * c.scale, z1.y * c.scale);
        *reinterpret_cast<double2*>(out + it.o0[m]) = q0;
        *reinterpret_cast<double2*>(out + it.o1[m]) = q1;
      }
      if (rhs) put_rhs(lds, it.at[m], m, q0, q1, hv, a);
    }
  if (!rhs) return;
  wave_lds_sync();
  forward_any<NX, NY>(pl, a.spec, g, i, z);
}

// run-time edges: two waves per SIMD (220 registers); held to three they spill (36 x 54, Lmax 4
// 41 -> 57 us)
#define WLC_BOUNDS(NX, NY) __launch_bounds__(NX > 0 ? 64 * shape_of(NX > 0 ? NX : 8, NY > 0 ? NY : 8).waves : kMaxThreads, NX > 0 ? 1 : 2)

template <int NX, int NY>
__global__ void WLC_BOUNDS(NX, NY) k2_rhs(Geom g, RhsArgs a) {
  k_rhs_body<NX, NY>(g, a);
}
template <int NX, int NY>
__global__ void WLC_BOUNDS(NX, NY) k2_inv(Geom g, InvArgs c) {
  k_inv_body<NX, NY>(g, c);
}
template <int NX, int NY>
__global__ void WLC_BOUNDS(NX, NY) k2_inv_rhs(Geom g, InvArgs c, RhsArgs a) {
  k_inv_rhs_body<NX, NY>(g, c, a);
}

// the same for one instance of a batch per blockIdx.z
template <int NX, int NY>
__global__ void WLC_BOUNDS(NX, NY) k2_rhs_b(const PlaneJob* __restrict__ jobs) {
  const PlaneJob& j = jobs[blockIdx.z];
  if (j.skip && *j.skip) return;
  k_rhs_body<NX, NY>(j.g, j.a);
}
template <int NX, int NY>
__global__ void WLC_BOUNDS(NX, NY) k2_inv_b(const PlaneJob* __restrict__ jobs) {
  const PlaneJob& j = jobs[blockIdx.z];
  if (j.skip && *j.skip) return;
  k_inv_body<NX, NY>(j.g, j.c);
}
template <int NX, int NY>
__global__ void WLC_BOUNDS(NX, NY) k2_inv_rhs_b(const PlaneJob* __restrict__ jobs) {
  const PlaneJob& j = jobs[blockIdx.z];
  if (j.skip && *j.skip) return;
  k_inv_rhs_body<NX, NY>(j.g, j.c, j.a);
}

template <int NX, int NY>
const void* pick(int kind, bool batch) {
  if (kind == 0) return batch ? (const void*)k2_rhs_b<NX, NY> : (const void*)k2_rhs<NX, NY>;
  if (kind == 1) return batch ? (const void*)k2_inv_b<NX, NY> : (const void*)k2_inv<NX, NY>;
  return batch ? (const void*)k2_inv_rhs_b<NX, NY> : (const void*)k2_inv_rhs<NX, NY>;
}

}  // namespace

const void* kernel(int nx, int ny, int kind, bool batch) {
  // 48 x 48 (the batching workload) with compile-time edges, any other pair without
  if (nx == 48 && ny == 48) return pick<48, 48>(kind, batch);
  return pick<0, 0>(kind, batch);
}

}  // namespace p2
}  // namespace wlc
