// Warm-start network for the SCFT fields: a 3D convolutional U-Net trained and run with
// hand-written kernels.  The reference has no counterpart (it starts every SCFT from the
// hand-built fields of init_w, init_array_2dcomp_mod.f90:843-1065); this network proposes
// initial fields from a seed field and the instance's parameters, and plain SCFT from them
// still decides the converged state.
//
// Layout: activations channels-last [B][D][H][W][C] with C a multiple of 16, stored as
// bfloat16 where a convolution reads them; gradients and master weights FP32.  Convolutions are
// 3x3x3, zero padding 1, stride 1, weights [Cout][27][Cin] (tap t = 9 kz + 3 ky + kx).  Every
// convolution (forward, gradient with respect to the input, gradient with respect to the weights)
// is an implicit GEMM on the bf16 matrix cores (FP32 accumulation):
//   forward   M = Cout, N = voxels, K = 27 Cin
//   input     the forward kernel on the output gradient with the flipped, transposed kernel
//             W'[ci][26 - t][co] = W[co][t][ci]
//   weights   M = Cout, N = Cin per tap, K = voxels, split over voxel chunks whose partial
//             sums are added in a fixed order (deterministic)
// Architecture (levels n, n/2, n/4, n/8; base 32 channels):
//   e0: conv 16->32, conv 32->32 (skip s0) | pool | e1: 32->64, 64->64 (s1) | pool |
//   e2: 64->128, 128->128 (s2) | pool | bottleneck 128->128 | up, concat s2 -> conv 256->64 |
//   up, concat s1 -> conv 128->32 | up, concat s0 -> conv 64->32 | conv 32->16 (output)
// ReLU after every convolution but the last; 2x2x2 average pooling; nearest 2x upsampling.
// Input channels: 3 seed fields and 8 broadcast scalars (11, padded to 16); output: the
// first 3 of 16 channels (the others have zero weights and no loss).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/wlc_mde.h"
#include "wlc_host.h"

namespace wlc {
namespace nn {

typedef unsigned short bf16;
typedef short bf16x4 __attribute__((__vector_size__(4 * sizeof(short))));
typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// round to nearest even (finite inputs)
__host__ __device__ inline bf16 f2bf(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__host__ __device__ inline float bf2f(bf16 h) {
  uint32_t u = (uint32_t)h << 16;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

struct Vol {
  int B, D, H, W;
  __host__ __device__ long long voxels() const { return (long long)B * D * H * W; }
};

// neighbour of voxel v at tap t (zero padding: -1 outside)
__device__ __forceinline__ long long neighbour(const Vol& g, long long v, int t) {
  const int x = (int)(v % g.W);
  long long r = v / g.W;
  const int y = (int)(r % g.H);
  r /= g.H;
  const int z = (int)(r % g.D);
  const long long b = r / g.D;
  const int zz = z + t / 9 - 1, yy = y + (t / 3) % 3 - 1, xx = x + t % 3 - 1;
  if (zz < 0 || zz >= g.D || yy < 0 || yy >= g.H || xx < 0 || xx >= g.W) return -1;
  return ((b * g.D + zz) * g.H + yy) * g.W + xx;
}

// The weights in the order the matrix cores read them: K input channels (KI = 32 of them per step
// when K is a multiple of 32, else 16), N output channels; one step of 16 output channels is a
// run of 64 lanes x KI / 4 values, lane l holding the channels KI/4 (l / 16) .. of output
// channel l % 16.
__host__ __device__ inline size_t packed_at(int K, int N, int t, int k, int n) {
  if (K % 32 == 0)
    return ((((size_t)t * (K / 32) + k / 32) * (N / 16) + n / 16) * 64 + n % 16 + 16 * ((k % 32) / 8)) * 8 + k % 8;
  return ((((size_t)t * (K / 16) + k / 16) * (N / 16) + n / 16) * 64 + n % 16 + 16 * ((k % 16) / 4)) * 4 + k % 4;
}

typedef unsigned short us4 __attribute__((ext_vector_type(4)));

// What a convolution does with four consecutive output channels co .. co + 3 of voxel v.
struct EpiF32 {  // Y = sum + bias
  float* Y;
  const float* bias;
  int C;
  __device__ __forceinline__ void operator()(int v, int co, f32x4 s) const {
    if (bias) s += *reinterpret_cast<const f32x4*>(bias + co);
    *reinterpret_cast<f32x4*>(Y + (size_t)v * C + co) = s;
  }
};
struct EpiOut {  // the network's output: the first 3 channels
  float* Y;
  const float* bias;
  __device__ __forceinline__ void operator()(int v, int co, f32x4 s) const {
    if (co) return;
    s += *reinterpret_cast<const f32x4*>(bias);
    Y[(size_t)v * 3] = s[0];
    Y[(size_t)v * 3 + 1] = s[1];
    Y[(size_t)v * 3 + 2] = s[2];
  }
};
// bf16(relu(sum + bias)) into channels off .. of a tensor of Ct channels, or (up) into those of
// the eight voxels of the next finer grid it is upsampled to
template <bool UP>
struct EpiAct {
  bf16* a;
  const float* bias;
  int Ct, off;
  Vol g;
  __device__ __forceinline__ void operator()(int v, int co, f32x4 s) const {
    s += *reinterpret_cast<const f32x4*>(bias + co);
    us4 h;
#pragma unroll
    for (int r = 0; r < 4; ++r) h[r] = f2bf(s[r] < 0.f ? 0.f : s[r]);
    if constexpr (!UP) {
      *reinterpret_cast<us4*>(a + (size_t)v * Ct + off + co) = h;
    } else {
      const int x = v % g.W;
      int q = v / g.W;
      const int y = q % g.H;
      q /= g.H;  // b D + z
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const size_t f = ((size_t)(2 * q + (d >> 2)) * 2 * g.H + 2 * y + ((d >> 1) & 1)) * 2 * g.W + 2 * x + (d & 1);
        *reinterpret_cast<us4*>(a + f * Ct + off + co) = h;
      }
    }
  }
};
// gradient of a pre-activation: the sum where the activation is positive (not where it is NaN),
// FP32 and bf16
struct EpiMask {
  const bf16* act;
  float* dy;
  bf16* dyb;
  int C;
  __device__ __forceinline__ void operator()(int v, int co, f32x4 s) const {
    const size_t at = (size_t)v * C + co;
    const us4 m = *reinterpret_cast<const us4*>(act + at);
    us4 h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = bf2f(m[r]) > 0.f ? s[r] : 0.f;
      h[r] = f2bf(s[r]);
    }
    *reinterpret_cast<f32x4*>(dy + at) = s;
    *reinterpret_cast<us4*>(dyb + at) = h;
  }
};

// sum_{t, ci} W[co][t][ci] X[nbr(v, t)][ci] (zero outside the grid) for 16 MT voxels x 16 NT
// output channels per wave, four waves (64 MT voxels) per workgroup.  Matrix-core step: A the
// packed weights (16 output channels x KI), B the KI channels of 16 voxels; lane l receives the
// sums of output channels 4 (l / 16) .. + 3 of voxel l % 16, so the epilogue stores 8 or 16 bytes.
// A voxel outside the grid is read from a zero row: a tap's neighbour is one bit of a mask per
// voxel and an address select, every load is unconditional, and the operands of the next D steps
// are in flight.  The steps run in the order tap, then channel.
// The first version loaded each step's operands one step ahead, the weights through LDS with a
// barrier per step (64^3: 32 -> 32 channels 57 us, 64 -> 32 130 us, 16^3: 128 -> 128 49 us).
template <int MT, int NT, int KI, int D, class Epi>
__global__ void __launch_bounds__(256) k_conv(const bf16* __restrict__ X, const bf16* __restrict__ Wp,
                                              const bf16* __restrict__ zrow, Vol g, int Cin, int Cout, Epi epi) {
  constexpr int CPL = KI / 4;  // channels per lane and step
  typedef short frag __attribute__((ext_vector_type(CPL)));
  const int lane = threadIdx.x & 63, row = lane & 15, kq = lane >> 4;
  const int V = (int)g.voxels();
  const int vb = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (16 * MT);
  const int co0 = blockIdx.y * 16 * NT;
  const bf16* xb[MT];
  unsigned mask[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int v = vb + 16 * m + row;
    const int x = v % g.W, q = v / g.W, y = q % g.H, z = (q / g.H) % g.D;
    const unsigned mx = (x > 0 ? 1u : 0u) | 2u | (x + 1 < g.W ? 4u : 0u);
    const unsigned my = (y > 0 ? 1u : 0u) | 2u | (y + 1 < g.H ? 4u : 0u);
    const unsigned mz = (z > 0 ? 1u : 0u) | 2u | (z + 1 < g.D ? 4u : 0u);
    unsigned b = 0;
#pragma unroll
    for (int t = 0; t < 9; ++t)
      b |= ((my >> (t / 3)) & 1u) && ((mx >> (t % 3)) & 1u) ? 1u << t : 0u;
    mask[m] = v < V ? ((mz & 1u) ? b : 0u) | (b << 9) | ((mz & 4u) ? b << 18 : 0u) : 0u;
    xb[m] = X + (size_t)v * Cin + CPL * kq;
  }
  const int nch = Cin / KI, K = 27 * nch;
  const bf16* wp = Wp + ((size_t)(co0 / 16) * 64 + lane) * CPL;
  const size_t wstep = (size_t)(Cout / 16) * 64 * CPL;
  const bf16* zr = zrow + CPL * kq;
  // the step loaded next: tap, channel, offset of the tap's neighbour
  int lt = 0, lc = 0;
  long long shift = (long long)(-g.H * g.W - g.W - 1) * Cin;
  frag a[D][NT], b[D][MT];
  auto load = [&](int d) {
#pragma unroll
    for (int j = 0; j < NT; ++j) a[d][j] = *reinterpret_cast<const frag*>(wp + j * 64 * CPL);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const bf16* p = (mask[m] >> lt) & 1u ? xb[m] + shift + lc : zr;
      b[d][m] = *reinterpret_cast<const frag*>(p);
    }
    wp += wstep;
    lc += KI;
    if (lc == Cin) {
      lc = 0;
      ++lt;
      const int dz = lt / 9 - 1, dy = (lt / 3) % 3 - 1, dx = lt % 3 - 1;
      shift = (long long)((dz * g.H + dy) * g.W + dx) * Cin;
    }
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  static_assert(27 % D == 0, "K is a multiple of D");
#pragma unroll
  for (int d = 0; d < D; ++d) load(d);
  for (int ks = 0; ks < K; ks += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if constexpr (KI == 32)
            acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[d][j]),
                                                                __builtin_bit_cast(bf16x8, b[d][m]), acc[m][j], 0, 0, 0);
          else
            acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4, a[d][j]),
                                                                  __builtin_bit_cast(bf16x4, b[d][m]), acc[m][j], 0, 0, 0);
        }
      if (ks + d + D < K) load(d);
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int v = vb + 16 * m + row;
    if (v >= V) continue;
#pragma unroll
    for (int j = 0; j < NT; ++j) epi(v, co0 + 16 * j + 4 * kq, acc[m][j]);
  }
}

// One layer's weight and bias gradient.  All layers go through each kernel below in one launch
// (their inputs are all there once the gradient has run down the network): a layer of the coarse
// grids alone fills a fraction of the GPU.  first[k] is the layer's first workgroup in launch k.
struct GradJob {
  const bf16 *X, *dYb;  // input and output gradient, channels-last
  const float* dYf;
  bf16 *xt, *dyt;       // transposed: [C][V]
  float *part, *bpart, *dW, *db;
  Vol g;
  int V, cin, cout;
  int mc, nc;           // 16-channel tiles per wave: output, input
  int chunk, nch;       // voxels per chunk, chunks
  int nbp, bchunk;      // bias parts, voxels of each
  int first[6];
};
enum { kTrX = 0, kTrY = 1, kDw = 2, kSum = 3, kBias = 4, kBiasEnd = 5 };
constexpr int kMaxJobs = 11;
struct GradJobs {
  GradJob j[kMaxJobs];
  int n;
};

// the job of workgroup b of launch k (uniform); b becomes its own count
__device__ __forceinline__ const GradJob& job_of(const GradJobs* __restrict__ J, int k, int& b) {
  int i = 0;
  for (int t = 1; t < J->n; ++t)
    if (b >= J->j[t].first[k]) i = t;
  b -= J->j[i].first[k];
  return J->j[i];
}

// xt[c][v] = X[v][c], dyt[c][v] = dYb[v][c] (bf16), 32 x 32 tiles through LDS
__global__ void __launch_bounds__(256) k_transpose(const GradJobs* __restrict__ J, int which) {
  __shared__ bf16 tile[32][33];
  int b = blockIdx.x;
  const GradJob& q = job_of(J, which, b);
  const bf16* in = which == kTrX ? q.X : q.dYb;
  bf16* out = which == kTrX ? q.xt : q.dyt;
  const int V = q.V, C = which == kTrX ? q.cin : q.cout;
  const int nc = (C + 31) / 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int v0 = (b / nc) * 32, c0 = (b % nc) * 32;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int v = v0 + ty + 8 * r, c = c0 + tx;
    if (v < V && c < C) tile[ty + 8 * r][tx] = in[(size_t)v * C + c];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = c0 + ty + 8 * r, v = v0 + tx;
    if (v < V && c < C) out[(size_t)c * V + v] = tile[tx][ty + 8 * r];
  }
}

// part[chunk][co][t][ci] = sum_{v in chunk} dY[v][co] X[nbr(v, t)][ci] from the transposed
// operands: the voxels are the reduction index, so lane l's eight consecutive voxels 8 (l / 16) ..
// of a 32-voxel step are one 16-byte load of a channel row.  Needs W % 8 == 0 (eight consecutive
// voxels lie in one x row: their tap neighbours are the same run shifted by dx, read as the
// aligned run and one element of its left or right neighbour run) and V, chunk multiples of 32.
// One wave per (dz, dy), 16 MC output channels, 16 NC input channels and voxel chunk: its three
// taps dx = -1, 0, 1 share the output gradient's and the input's run.
template <int MC, int NC>
__device__ __forceinline__ void dw_wave(const GradJob& q, int idx) {
  const int lane = threadIdx.x, row = lane & 15, kq = lane >> 4;
  const Vol g = q.g;
  const int V = q.V, Cin = q.cin, Cout = q.cout, nci = Cin / (16 * NC);
  const int ch = idx % q.nch;
  idx /= q.nch;
  const int t3 = idx % 9;
  idx /= 9;
  const int ci0 = (idx % nci) * 16 * NC, co0 = (idx / nci) * 16 * MC;
  const int dz = t3 / 3 - 1, dy = t3 % 3 - 1;
  const int vb0 = ch * q.chunk, ve = min(vb0 + q.chunk, V);
  const int rowshift = (dz * g.H + dy) * g.W;
  const s16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const bf16* dyr = q.dyt + (size_t)(co0 + row) * V;
  const bf16* xr = q.xt + (size_t)(ci0 + row) * V + rowshift;
  f32x4 acc[3][MC][NC];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int i = 0; i < MC; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j) acc[d][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  s16x8 an[MC], cn[NC];
  short ln[NC], rn[NC];
  auto load = [&](int vb) {
    const int v = vb + 8 * kq;  // this lane's eight voxels v .. v + 7: one x-row run
    const int x = v % g.W, r1 = v / g.W, y = r1 % g.H, z = (r1 / g.H) % g.D;
    const bool ok = (unsigned)(z + dz) < (unsigned)g.D && (unsigned)(y + dy) < (unsigned)g.H;
    const bool lok = ok && x > 0, rok = ok && x + 8 < g.W;
#pragma unroll
    for (int i = 0; i < MC; ++i) an[i] = *reinterpret_cast<const s16x8*>(dyr + (size_t)(16 * i) * V + v);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const bf16* p = xr + (size_t)(16 * j) * V + v;
      cn[j] = ok ? *reinterpret_cast<const s16x8*>(p) : zero;
      ln[j] = lok ? (short)p[-1] : (short)0;
      rn[j] = rok ? (short)p[8] : (short)0;
    }
  };
  if (vb0 < ve) load(vb0);
  for (int vb = vb0; vb < ve; vb += 32) {
    s16x8 a[MC], c[NC];
    short l[NC], r[NC];
#pragma unroll
    for (int i = 0; i < MC; ++i) a[i] = an[i];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      c[j] = cn[j];
      l[j] = ln[j];
      r[j] = rn[j];
    }
    if (vb + 32 < ve) load(vb + 32);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const s16x8 bl = s16x8{l[j], c[j][0], c[j][1], c[j][2], c[j][3], c[j][4], c[j][5], c[j][6]};
      const s16x8 br = s16x8{c[j][1], c[j][2], c[j][3], c[j][4], c[j][5], c[j][6], c[j][7], r[j]};
#pragma unroll
      for (int i = 0; i < MC; ++i) {
        const bf16x8 av = __builtin_bit_cast(bf16x8, a[i]);
        acc[0][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, bl), acc[0][i][j], 0, 0, 0);
        acc[1][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, c[j]), acc[1][i][j], 0, 0, 0);
        acc[2][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, br), acc[2][i][j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int i = 0; i < MC; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          q.part[(((size_t)ch * Cout + co0 + 16 * i + 4 * kq + r) * 27 + 3 * t3 + d) * Cin + ci0 + 16 * j + row] =
              acc[d][i][j][r];
}

__global__ void __launch_bounds__(64) k_conv_dw_t(const GradJobs* __restrict__ J) {
  int b = blockIdx.x;
  const GradJob& q = job_of(J, kDw, b);
  if (q.mc == 2) {
    if (q.nc == 2) dw_wave<2, 2>(q, b);
    else dw_wave<2, 1>(q, b);
  } else {
    if (q.nc == 2) dw_wave<1, 2>(q, b);
    else dw_wave<1, 1>(q, b);
  }
}

// part[chunk][co][t][ci] = sum_{v in chunk} dY[v][co] X[nbr(v, t)][ci] on the channels-last
// operands, element by element (grids whose x edge is not a multiple of 8, i.e. the coarsest
// levels of small grids): one wave per (tap, 16 co, 16 ci) and voxel chunk; lane l holds
// A[co = l % 16][v = 4 (l / 16) + j] and B[v = 4 (l / 16) + j][ci = l % 16]
__global__ void __launch_bounds__(64) k_conv_dw(const bf16* __restrict__ dY, const bf16* __restrict__ X,
                                                float* __restrict__ part, Vol g, int Cin, int Cout,
                                                long long chunk) {
  const int l = threadIdx.x, row = l & 15, kq = l >> 4;
  const int nci = Cin / 16;
  int idx = blockIdx.x;
  const int t = idx % 27;
  idx /= 27;
  const int ci0 = (idx % nci) * 16, co0 = (idx / nci) * 16;
  const long long V = g.voxels();
  const long long vb0 = (long long)blockIdx.y * chunk;
  const long long ve = vb0 + chunk < V ? vb0 + chunk : V;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (long long vb = vb0; vb < ve; vb += 16) {
    bf16x4 a, b;
    for (int j = 0; j < 4; ++j) {
      const long long vv = vb + 4 * kq + j;
      const bool ok = vv < ve;
      a[j] = ok ? (short)dY[vv * Cout + co0 + row] : (short)0;
      const long long nb = ok ? neighbour(g, vv, t) : -1;
      b[j] = nb >= 0 ? (short)X[nb * Cin + ci0 + row] : (short)0;
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  }
  for (int r = 0; r < 4; ++r)
    part[(((long long)blockIdx.y * Cout + co0 + 4 * kq + r) * 27 + t) * Cin + ci0 + row] = acc[r];
}

// dW[i] = sum_c part[c][i], chunks in order
__global__ void __launch_bounds__(256) k_sum_chunks(const GradJobs* __restrict__ J) {
  int b = blockIdx.x;
  const GradJob& q = job_of(J, kSum, b);
  const long long n = (long long)q.cout * 27 * q.cin;
  const long long i = b * 256LL + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
#pragma unroll 8
  for (int c = 0; c < q.nch; ++c) s += q.part[(long long)c * n + i];
  q.dW[i] = s;
}

// bpart[p][c] = sum of dY[v][c] over the voxels of part p (FP32): the 256 threads are
// 256 / C voxel lanes x C channels (C <= 256), so each pass reads 256 / C whole voxel rows;
// every lane keeps four partial sums (independent loads in flight), and the sums are added
// in a fixed order (deterministic)
__global__ void __launch_bounds__(256) k_bias_partial(const GradJobs* __restrict__ J) {
  __shared__ float red[256];
  int b = blockIdx.x;
  const GradJob& q = job_of(J, kBias, b);
  const float* __restrict__ dY = q.dYf;
  const int C = q.cout, nr = 256 / C, c = threadIdx.x % C, r = threadIdx.x / C;
  const int v0 = b * q.bchunk, v1 = min(v0 + q.bchunk, q.V);
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (r < nr) {
    int v = v0 + r;
    for (; v + 3 * nr < v1; v += 4 * nr) {
      s0 += dY[(size_t)v * C + c];
      s1 += dY[(size_t)(v + nr) * C + c];
      s2 += dY[(size_t)(v + 2 * nr) * C + c];
      s3 += dY[(size_t)(v + 3 * nr) * C + c];
    }
    for (; v < v1; v += nr) s0 += dY[(size_t)v * C + c];
  }
  red[threadIdx.x] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (threadIdx.x < C) {
    float t = 0.f;
    for (int k = 0; k < nr; ++k) t += red[k * C + c];
    q.bpart[(size_t)b * C + c] = t;
  }
}

// db[c] = sum over the parts of bpart[p][c]: one workgroup per channel, each thread adds
// the parts t, t + 256, ... in order, then a tree in shared memory (fixed order)
__global__ void __launch_bounds__(256) k_bias_final(const GradJobs* __restrict__ J) {
  __shared__ float red[256];
  int c = blockIdx.x;
  const GradJob& q = job_of(J, kBiasEnd, c);
  float s = 0.f;
  for (int p = threadIdx.x; p < q.nbp; p += 256) s += q.bpart[(size_t)p * q.cout + c];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) q.db[c] = red[0];
}

// where a weight goes in the packed copies: fwd of the layer's own kernel, bwd of the flipped,
// transposed one
struct PackLayer {
  long long woff;
  int cin, cout;
};
struct PackTable {
  PackLayer l[11];
  int n;
};
__device__ __forceinline__ void pack_weight(const PackTable& T, bf16* fwd, bf16* bwd, long long i, bf16 h) {
  int k = 0;
  for (int t = 1; t < T.n; ++t)
    if (i >= T.l[t].woff) k = t;
  const int cin = T.l[k].cin, cout = T.l[k].cout;
  const long long j = i - T.l[k].woff;
  if (j >= (long long)cout * 27 * cin) return;  // a bias
  const int ci = (int)(j % cin), r = (int)(j / cin), t = r % 27, co = r / 27;
  fwd[T.l[k].woff + packed_at(cin, cout, t, ci, co)] = h;
  bwd[T.l[k].woff + packed_at(cout, cin, 26 - t, co, ci)] = h;
}
__global__ void k_pack(const float* __restrict__ p, PackTable T, bf16* __restrict__ fwd, bf16* __restrict__ bwd,
                       long long n) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n) pack_weight(T, fwd, bwd, i, f2bf(p[i]));
}

// input [V][11] -> bf16 [V][16], the last five zero
__global__ void k_input(const float* __restrict__ x, bf16* __restrict__ o, long long V) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= V * 16) return;
  const long long v = i >> 4;
  const int c = (int)(i & 15);
  o[i] = c < 11 ? f2bf(x[v * 11 + c]) : (bf16)0;
}

// 2x2x2 average pooling of channels [off, off + C) of a tensor of Ct (bf16 in and out)
__global__ void k_pool(const bf16* __restrict__ x, bf16* __restrict__ o, Vol go, int C, int Ct, int off) {
  const long long n = go.voxels() * (C / 4);
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = 4 * (int)(i % (C / 4));
  long long v = i / (C / 4);
  const long long vo = v;
  const int X = (int)(v % go.W);
  v /= go.W;
  const int Y = (int)(v % go.H);
  v /= go.H;  // b D + Z
  const int Wi = 2 * go.W, Hi = 2 * go.H;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const size_t f = ((size_t)(2 * v + (d >> 2)) * Hi + 2 * Y + ((d >> 1) & 1)) * Wi + 2 * X + (d & 1);
    const us4 h = *reinterpret_cast<const us4*>(x + f * Ct + off + c);
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] += bf2f(h[r]);
  }
  us4 h;
#pragma unroll
  for (int r = 0; r < 4; ++r) h[r] = f2bf(s[r] * 0.125f);
  *reinterpret_cast<us4*>(o + vo * C + c) = h;
}

// gradient of a pre-activation whose activation was upsampled into channels [0, C) of the Ct of
// the next finer grid: the sum of the eight fine gradients where the activation (read at the first
// of its eight copies) is positive
__global__ void k_up_back(const float* __restrict__ dfine, const bf16* __restrict__ act, float* __restrict__ dy,
                          bf16* __restrict__ dyb, Vol gc, int C, int Ct) {
  const long long n = gc.voxels() * (C / 4);
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = 4 * (int)(i % (C / 4));
  long long v = i / (C / 4);
  const long long vo = v;
  const int X = (int)(v % gc.W);
  v /= gc.W;
  const int Y = (int)(v % gc.H);
  v /= gc.H;
  const int Wf = 2 * gc.W, Hf = 2 * gc.H;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  us4 m = {0, 0, 0, 0};
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const size_t f = ((size_t)(2 * v + (d >> 2)) * Hf + 2 * Y + ((d >> 1) & 1)) * Wf + 2 * X + (d & 1);
    s += *reinterpret_cast<const f32x4*>(dfine + f * Ct + c);
    if (d == 0) m = *reinterpret_cast<const us4*>(act + f * Ct + c);
  }
  us4 h;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    s[r] = bf2f(m[r]) > 0.f ? s[r] : 0.f;
    h[r] = f2bf(s[r]);
  }
  *reinterpret_cast<f32x4*>(dy + vo * C + c) = s;
  *reinterpret_cast<us4*>(dyb + vo * C + c) = h;
}

// gradient of a pre-activation whose activation is the skip half [off, off + C) of a concatenated
// tensor of Ct channels and was pooled: the skip's gradient plus an eighth of the pooled one,
// where the activation is positive
__global__ void k_skip_back(const float* __restrict__ dcat, const float* __restrict__ dpool,
                            const bf16* __restrict__ act, float* __restrict__ dy, bf16* __restrict__ dyb, Vol g, int C,
                            int Ct, int off) {
  const long long n = g.voxels() * (C / 4);
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = 4 * (int)(i % (C / 4));
  const long long v = i / (C / 4);
  const int X = (int)(v % g.W);
  long long r1 = v / g.W;
  const int Y = (int)(r1 % g.H);
  r1 /= g.H;  // b D + z
  const long long vc = ((r1 / 2) * (g.H / 2) + Y / 2) * (g.W / 2) + X / 2;
  f32x4 s = *reinterpret_cast<const f32x4*>(dcat + v * Ct + off + c);
  const f32x4 p = *reinterpret_cast<const f32x4*>(dpool + vc * C + c);
  const us4 m = *reinterpret_cast<const us4*>(act + v * Ct + off + c);
  us4 h;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    s[r] += p[r] * 0.125f;
    s[r] = bf2f(m[r]) > 0.f ? s[r] : 0.f;
    h[r] = f2bf(s[r]);
  }
  *reinterpret_cast<f32x4*>(dy + v * C + c) = s;
  *reinterpret_cast<us4*>(dyb + v * C + c) = h;
}

// loss partials: sum over the nout channels of (y - t)^2 and the gradient 2 (y - t) / count, FP32
// and bf16, of the C channels of the output convolution (zero on the padding)
__global__ void __launch_bounds__(256) k_mse(const float* __restrict__ y, const float* __restrict__ t,
                                             float* __restrict__ dy, bf16* __restrict__ dyb,
                                             float* __restrict__ part, long long V, int C, int nout,
                                             float inv_count) {
  __shared__ float red[256];
  float s = 0.f;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < V * C; i += (long long)gridDim.x * 256) {
    const long long v = i / C;
    const int c = (int)(i - v * C);
    float g = 0.f;
    if (c < nout) {
      const float d = y[v * nout + c] - t[v * nout + c];
      s += d * d;
      g = 2.f * d * inv_count;
    }
    dy[i] = g;
    dyb[i] = f2bf(g);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Adam on FP32 master weights with the packed bf16 copies for the matrix cores; `mask` zeroes the
// padding entries (kept exactly zero)
__global__ void k_adam(float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
                       const float* __restrict__ g, PackTable T, bf16* __restrict__ fwd, bf16* __restrict__ bwd,
                       const unsigned char* __restrict__ mask, long long n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  float pi = 0.f;
  if (mask[i]) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
  p[i] = pi;
  pack_weight(T, fwd, bwd, i, f2bf(pi));
}

inline unsigned blocks(long long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

struct Layer {
  int cin, cout;          // padded channel counts (multiples of 16)
  int cin_real, cout_real;
  int level;              // grid n >> level
  int relu;
  long long woff, boff;   // offsets of W [cout][27][cin] and b [cout] in the flat parameters
};

// the network: 11 convolutions (see the file header)
std::vector<Layer> architecture() {
  const int L[11][6] = {
      // cin, cout, cin_real, cout_real, level, relu
      {16, 32, 11, 32, 0, 1}, {32, 32, 32, 32, 0, 1},    // e0
      {32, 64, 32, 64, 1, 1}, {64, 64, 64, 64, 1, 1},    // e1
      {64, 128, 64, 128, 2, 1}, {128, 128, 128, 128, 2, 1},  // e2
      {128, 128, 128, 128, 3, 1},                          // bottleneck
      {256, 64, 256, 64, 2, 1},                            // d2
      {128, 32, 128, 32, 1, 1},                            // d1
      {64, 32, 64, 32, 0, 1},                              // d0
      {32, 16, 32, 3, 0, 0},                               // output
  };
  std::vector<Layer> out;
  long long off = 0;
  for (auto& r : L) {
    Layer l{r[0], r[1], r[2], r[3], r[4], r[5], 0, 0};
    l.woff = off;
    off += (long long)l.cout * 27 * l.cin;
    l.boff = off;
    off += l.cout;
    out.push_back(l);
  }
  return out;
}

// normal deviates by Marsaglia's polar method, in the order and with the roundings of
// std::normal_distribution<float> on the same engine.  That one's uniform numbers take two long double
// logarithms each, and with them the creation of a network took 77 to 133 ms, depending on the
// address that its code was linked to; 21 ms with these.
class Normals {
 public:
  explicit Normals(unsigned long long seed) : rng_(seed) {}
  float operator()() {
    if (have_) {
      have_ = false;
      return kept_;
    }
    float x, y, r2;
    do {
      x = 2.f * uniform() - 1.f;
      y = 2.f * uniform() - 1.f;
      r2 = x * x + y * y;
    } while (r2 > 1.f || r2 == 0.f);
    const float scale = std::sqrt(-2.f * std::log(r2) / r2);
    kept_ = x * scale;
    have_ = true;
    return y * scale;
  }

 private:
  float uniform() {  // [0, 1): a draw that rounds up to 1 becomes the number below it
    const float u = (float)rng_() * 0x1p-64f;
    return u < 1.f ? u : 1.f - 0x1p-24f;
  }
  std::mt19937_64 rng_;
  float kept_ = 0.f;
  bool have_ = false;
};

}  // namespace nn
}  // namespace wlc

using namespace wlc::nn;

struct wlc_unet {
  int device = 0;
  hipStream_t st = nullptr;
  int n = 0, B = 0;       // 0: no buffers (a resize failed)
  std::vector<Layer> layers;
  PackTable pack{};
  long long np = 0;       // flat parameter count (padded)
  float *p = nullptr, *m = nullptr, *v = nullptr, *g = nullptr;
  bf16 *wf = nullptr, *wb = nullptr;  // packed bf16 weights of the convolutions and of their adjoints
  bf16* zrow = nullptr;               // a row of zeros (a voxel outside the grid)
  unsigned char* mask = nullptr;
  float* lpart = nullptr;
  int adam_t = 0;
  // activations (bf16): cN holds the concatenation [upsampled, skip] of level N, pN the pooled skip
  // of level N - 1
  bf16 *x0 = nullptr, *a0a = nullptr, *p1 = nullptr, *a1a = nullptr, *p2 = nullptr, *a2a = nullptr, *p3 = nullptr,
       *c2 = nullptr, *c1 = nullptr, *c0 = nullptr, *d0 = nullptr;
  // gradients (FP32) of the concatenations and the pooled tensors
  float *gp1 = nullptr, *gp2 = nullptr, *gp3 = nullptr, *gc2 = nullptr, *gc1 = nullptr, *gc0 = nullptr;
  float* y = nullptr;     // output [V][3]
  float* dy[11] = {};     // gradients of the pre-activations
  bf16* dyb[11] = {};     // bf16 copies (matrix-core operand)
  float *xin = nullptr, *target = nullptr;
  std::vector<GradJob> jobs;          // weight gradients in one launch per kernel ...
  std::vector<GradJob> odd;           // ... and of the layers whose x edge is no multiple of 8
  GradJobs *djobs = nullptr, *dall = nullptr;
  unsigned grid[6] = {};              // workgroups of each launch
  std::vector<void*> allocs;  // parameters and optimiser state
  std::vector<void*> acts;    // activations, gradients and scratch of the current grid and batch
  Vol vol(int level) const { return Vol{B, n >> level, n >> level, n >> level}; }
};

namespace {

int ufail(int code, const std::string& m) { return wlc::host_fail(code, m); }

#define UCHK(call)                                                                          \
  do {                                                                                      \
    hipError_t e_ = (call);                                                                 \
    if (e_ != hipSuccess) return ufail(WLC_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

template <class T>
int ualloc(std::vector<void*>& list, T** ptr, long long count) {
  void* q = nullptr;
  if (hipMalloc(&q, sizeof(T) * (size_t)std::max<long long>(count, 1)) != hipSuccess)
    return ufail(WLC_ENOMEM, "device allocation failed (warm-start network)");
  list.push_back(q);
  if (hipMemset(q, 0, sizeof(T) * (size_t)std::max<long long>(count, 1)) != hipSuccess)
    return ufail(WLC_EHIP, "device initialisation failed (warm-start network)");
  *ptr = static_cast<T*>(q);
  return WLC_OK;
}

void free_acts(wlc_unet* u) {
  for (void* q : u->acts) (void)hipFree(q);
  u->acts.clear();
  u->n = u->B = 0;
}

void unet_free(wlc_unet* u) {
  if (!u) return;
  (void)hipSetDevice(u->device);
  if (u->st) (void)hipStreamSynchronize(u->st);
  free_acts(u);
  for (void* q : u->allocs) (void)hipFree(q);
  if (u->st) (void)hipStreamDestroy(u->st);
  delete u;
}

// partial sums of the bias gradient (at most; about 256 voxels each)
constexpr int kBiasParts = 1024;
// voxel chunks of the weight-gradient reduction: 2048 voxels each (one wave's 64 steps), at most 128
constexpr int kChunkVoxels = 2048, kMaxChunks = 128;

// the transposed kernel takes the layer (else the element-wise one)
bool grad_rows(const Vol& g) { return g.W % 8 == 0 && g.voxels() % 32 == 0; }

// sizes of a layer's gradient job (the pointers are the caller's)
GradJob grad_job(const Vol& g, int cin, int cout) {
  GradJob q{};
  q.g = g;
  q.V = (int)g.voxels();
  q.cin = cin;
  q.cout = cout;
  q.mc = cout % 32 == 0 ? 2 : 1;
  q.nc = cin % 32 == 0 ? 2 : 1;
  const int step = 32;
  const int want = std::max(kChunkVoxels, (q.V + kMaxChunks - 1) / kMaxChunks);
  q.chunk = (std::min(want, q.V) + step - 1) / step * step;
  q.nch = (q.V + q.chunk - 1) / q.chunk;
  q.nbp = (int)std::min<long long>(kBiasParts, std::max<long long>(1, q.V / 256));
  q.bchunk = (q.V + q.nbp - 1) / q.nbp;
  return q;
}
long long part_floats(const GradJob& q) { return (long long)q.nch * q.cout * 27 * q.cin; }

// first workgroups of every job in every launch, and the launches' sizes
void place_jobs(std::vector<GradJob>& rows, unsigned grid[6]) {
  for (int k = 0; k < 6; ++k) {
    long long b = 0;
    for (GradJob& q : rows) {
      q.first[k] = (int)b;
      const long long v32 = (q.V + 31) / 32;
      switch (k) {
        case kTrX: b += v32 * ((q.cin + 31) / 32); break;
        case kTrY: b += v32 * ((q.cout + 31) / 32); break;
        case kDw: b += 9LL * q.nch * (q.cout / (16 * q.mc)) * (q.cin / (16 * q.nc)); break;
        case kSum: b += ((long long)q.cout * 27 * q.cin + 255) / 256; break;
        case kBias: b += q.nbp; break;
        case kBiasEnd: b += q.cout; break;
      }
    }
    grid[k] = (unsigned)b;
  }
}

// weight and bias gradients: `jobs` (device: every layer, with the first workgroups of the sum and
// bias launches) and `rows` (device: those of the transposed kernel), odd the element-wise layers
int launch_grads(hipStream_t st, const GradJobs* all, const GradJobs* rows, bool any_rows,
                 const std::vector<GradJob>& odd, const unsigned grid[6]) {
  if (any_rows) {
    hipLaunchKernelGGL(k_transpose, dim3(grid[kTrX]), dim3(256), 0, st, rows, (int)kTrX);
    hipLaunchKernelGGL(k_transpose, dim3(grid[kTrY]), dim3(256), 0, st, rows, (int)kTrY);
    hipLaunchKernelGGL(k_conv_dw_t, dim3(grid[kDw]), dim3(64), 0, st, rows);
  }
  for (const GradJob& q : odd)
    hipLaunchKernelGGL(k_conv_dw, dim3(27 * (q.cout / 16) * (q.cin / 16), q.nch), dim3(64), 0, st, q.dYb, q.X, q.part,
                       q.g, q.cin, q.cout, (long long)q.chunk);
  hipLaunchKernelGGL(k_sum_chunks, dim3(grid[kSum]), dim3(256), 0, st, all);
  hipLaunchKernelGGL(k_bias_partial, dim3(grid[kBias]), dim3(256), 0, st, all);
  hipLaunchKernelGGL(k_bias_final, dim3(grid[kBiasEnd]), dim3(256), 0, st, all);
  UCHK(hipGetLastError());
  return WLC_OK;
}

// places of the activation, gradient and scratch buffers of u's grid edge and batch from `base`
// on, the gradient jobs of all layers into `all`; the bytes they take
size_t lay_acts(wlc_unet* u, uintptr_t base, std::vector<GradJob>& all) {
  size_t bytes = 0;
  auto take = [&](auto*& ptr, long long count) {
    ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(base + bytes);
    bytes += (sizeof(*ptr) * (size_t)std::max<long long>(count, 1) + 255) / 256 * 256;
  };
#define UA(ptr, cnt) take(ptr, cnt)
  const long long V0 = u->vol(0).voxels(), V1 = u->vol(1).voxels(), V2 = u->vol(2).voxels(), V3 = u->vol(3).voxels();
  UA(u->lpart, 256);
  UA(u->x0, V0 * 16); UA(u->a0a, V0 * 32); UA(u->p1, V1 * 32); UA(u->a1a, V1 * 64);
  UA(u->p2, V2 * 64); UA(u->a2a, V2 * 128); UA(u->p3, V3 * 128);
  UA(u->c2, V2 * 256); UA(u->c1, V1 * 128); UA(u->c0, V0 * 64); UA(u->d0, V0 * 32);
  UA(u->gp1, V1 * 32); UA(u->gp2, V2 * 64); UA(u->gp3, V3 * 128);
  UA(u->gc2, V2 * 256); UA(u->gc1, V1 * 128); UA(u->gc0, V0 * 64);
  UA(u->y, V0 * 3); UA(u->xin, V0 * 11); UA(u->target, V0 * 3);
  const bf16* X[11] = {u->x0, u->a0a, u->p1, u->a1a, u->p2, u->a2a, u->p3, u->c2, u->c1, u->c0, u->d0};
  all.clear();
  for (int li = 0; li < 11; ++li) {
    const Layer& l = u->layers[li];
    const Vol g = u->vol(l.level);
    const long long V = g.voxels();
    UA(u->dy[li], V * l.cout); UA(u->dyb[li], V * l.cout);
    GradJob q = grad_job(g, l.cin, l.cout);
    q.X = X[li];
    q.dYb = u->dyb[li];
    q.dYf = u->dy[li];
    q.dW = u->g + l.woff;
    q.db = u->g + l.boff;
    UA(q.part, part_floats(q));
    UA(q.bpart, (long long)q.nbp * l.cout);
    if (grad_rows(g)) {
      UA(q.xt, V * l.cin);
      UA(q.dyt, V * l.cout);
    }
    all.push_back(q);
  }
  UA(u->djobs, 1); UA(u->dall, 1);
#undef UA
  return bytes;
}

// activation, gradient and scratch buffers for grid edge n and batch B: one allocation for all of
// them, cleared at once (a hundred of them one by one took 50 ms), its size learned from a copy of
// the network.  Both sizes need not fit at once, so the old buffers go first; without new ones the
// network has none (n = B = 0) and refuses to run until a resize succeeds.
int alloc_acts(wlc_unet* u, int n, int B) {
  free_acts(u);
  std::vector<GradJob> all;
  wlc_unet dry = *u;
  dry.n = n;
  dry.B = B;
  const size_t bytes = lay_acts(&dry, 0, all);
  char* block = nullptr;
  if (const int rc = ualloc(u->acts, &block, (long long)bytes)) {
    free_acts(u);
    return rc;
  }
  u->n = n;
  u->B = B;
  lay_acts(u, reinterpret_cast<uintptr_t>(block), all);
  u->jobs.clear();
  u->odd.clear();
  // launches 0 .. 2 run over the layers of the transposed kernel, 3 .. 5 over all of them
  for (const GradJob& q : all) (grad_rows(q.g) ? u->jobs : u->odd).push_back(q);
  unsigned gr[6] = {}, ga[6] = {};
  place_jobs(u->jobs, gr);
  place_jobs(all, ga);
  for (int k = 0; k < 6; ++k) u->grid[k] = k <= kDw ? gr[k] : ga[k];
  GradJobs t{};
  t.n = (int)u->jobs.size();
  std::copy(u->jobs.begin(), u->jobs.end(), t.j);
  hipError_t e = hipMemcpy(u->djobs, &t, sizeof(t), hipMemcpyHostToDevice);
  t.n = (int)all.size();
  std::copy(all.begin(), all.end(), t.j);
  if (e == hipSuccess) e = hipMemcpy(u->dall, &t, sizeof(t), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    free_acts(u);
    return ufail(WLC_EHIP, "job table upload failed");
  }
  return WLC_OK;
}

// launches shared by the network and the convolution test entry point (stream st)

// a convolution (adjoint: of packed flipped weights) of X with cin channels into cout (multiples
// of 16).  Tile: the largest of 64 x 64, 64 x 32, 32 x 32, 16 x 32 and 16 x 16 voxels x output
// channels per wave that divides cout and leaves a wave for every SIMD (1024); the smaller the
// tile, the more steps in flight, since there the chain of steps is what takes the time (see
// k_conv for the times of the tile this replaced)
template <class Epi>
int launch_conv(hipStream_t st, const bf16* X, const bf16* Wp, const bf16* zrow, Vol g, int cin, int cout,
                const Epi& epi) {
  const long long V = g.voxels();
  const int nt = cout / 16;
#define CONV(MT, NT, KI, D) \
  hipLaunchKernelGGL((k_conv<MT, NT, KI, D, Epi>), dim3(blocks(V, 64 * (MT)), nt / (NT)), dim3(256), 0, st, X, Wp, zrow, g, cin, cout, epi)
#define CONV_K(MT, NT, D) do { if (cin % 32 == 0) CONV(MT, NT, 32, D); else CONV(MT, NT, 16, D); } while (0)
  auto waves = [&](int mt, int nn) { return (V + 16 * mt - 1) / (16 * mt) * (nt / nn); };
  if (nt % 4 == 0 && waves(4, 4) >= 1024) CONV_K(4, 4, 3);
  else if (nt % 2 == 0 && waves(4, 2) >= 1024) CONV_K(4, 2, 3);
  else if (nt % 2 == 0 && waves(2, 2) >= 1024) CONV_K(2, 2, 3);
  else if (nt % 2 == 0 && waves(1, 2) >= 1024) CONV_K(1, 2, 9);
  else if (waves(4, 1) >= 1024) CONV_K(4, 1, 3);
  else CONV_K(1, 1, 9);
#undef CONV_K
#undef CONV
  UCHK(hipGetLastError());
  return WLC_OK;
}

template <class Epi>
int conv(wlc_unet* u, int li, const bf16* X, const Epi& epi) {
  const Layer& l = u->layers[li];
  return launch_conv(u->st, X, u->wf + l.woff, u->zrow, u->vol(l.level), l.cin, l.cout, epi);
}
// gradient with respect to the input of layer li
template <class Epi>
int conv_back(wlc_unet* u, int li, const Epi& epi) {
  const Layer& l = u->layers[li];
  return launch_conv(u->st, u->dyb[li], u->wb + l.woff, u->zrow, u->vol(l.level), l.cout, l.cin, epi);
}

int forward(wlc_unet* u) {
  const Vol g0 = u->vol(0), g1 = u->vol(1), g2 = u->vol(2), g3 = u->vol(3);
  auto act = [&](int li, bf16* a, int Ct, int off) {
    return EpiAct<false>{a, u->p + u->layers[li].boff, Ct, off, u->vol(u->layers[li].level)};
  };
  auto up = [&](int li, bf16* a, int Ct) {
    return EpiAct<true>{a, u->p + u->layers[li].boff, Ct, 0, u->vol(u->layers[li].level)};
  };
  auto pool = [&](const bf16* x, bf16* o, const Vol& go, int C) {
    hipLaunchKernelGGL(k_pool, dim3(blocks(go.voxels() * (C / 4))), dim3(256), 0, u->st, x, o, go, C, 2 * C, C);
  };
  int rc;
  if ((rc = conv(u, 0, u->x0, act(0, u->a0a, 32, 0)))) return rc;
  if ((rc = conv(u, 1, u->a0a, act(1, u->c0, 64, 32)))) return rc;
  pool(u->c0, u->p1, g1, 32);
  if ((rc = conv(u, 2, u->p1, act(2, u->a1a, 64, 0)))) return rc;
  if ((rc = conv(u, 3, u->a1a, act(3, u->c1, 128, 64)))) return rc;
  pool(u->c1, u->p2, g2, 64);
  if ((rc = conv(u, 4, u->p2, act(4, u->a2a, 128, 0)))) return rc;
  if ((rc = conv(u, 5, u->a2a, act(5, u->c2, 256, 128)))) return rc;
  pool(u->c2, u->p3, g3, 128);
  if ((rc = conv(u, 6, u->p3, up(6, u->c2, 256)))) return rc;
  if ((rc = conv(u, 7, u->c2, up(7, u->c1, 128)))) return rc;
  if ((rc = conv(u, 8, u->c1, up(8, u->c0, 64)))) return rc;
  if ((rc = conv(u, 9, u->c0, act(9, u->d0, 32, 0)))) return rc;
  if ((rc = conv(u, 10, u->d0, EpiOut{u->y, u->p + u->layers[10].boff}))) return rc;
  UCHK(hipGetLastError());
  return WLC_OK;
}

// gradients of all parameters for the loss mse(y, target); *loss on the host
int backward(wlc_unet* u, float* loss) {
  const Vol g0 = u->vol(0), g1 = u->vol(1), g2 = u->vol(2), g3 = u->vol(3);
  const long long V0 = g0.voxels();
  int rc;
  auto mask = [&](int li, const bf16* a) { return EpiMask{a, u->dy[li], u->dyb[li], u->layers[li].cout}; };
  auto f32 = [&](float* q, int C) { return EpiF32{q, nullptr, C}; };
  auto up_back = [&](int li, const float* gc, const bf16* c, const Vol& g, int C, int Ct) {
    hipLaunchKernelGGL(k_up_back, dim3(blocks(g.voxels() * (C / 4))), dim3(256), 0, u->st, gc, c, u->dy[li], u->dyb[li],
                       g, C, Ct);
  };
  auto skip_back = [&](int li, const float* gc, const float* gp, const bf16* c, const Vol& g, int C) {
    hipLaunchKernelGGL(k_skip_back, dim3(blocks(g.voxels() * (C / 4))), dim3(256), 0, u->st, gc, gp, c, u->dy[li],
                       u->dyb[li], g, C, 2 * C, C);
  };
  hipLaunchKernelGGL(k_mse, dim3(256), dim3(256), 0, u->st, u->y, u->target, u->dy[10], u->dyb[10], u->lpart, V0, 16, 3,
                     1.0f / (float)(V0 * 3));
  if ((rc = conv_back(u, 10, mask(9, u->d0)))) return rc;
  if ((rc = conv_back(u, 9, f32(u->gc0, 64)))) return rc;
  up_back(8, u->gc0, u->c0, g1, 32, 64);
  if ((rc = conv_back(u, 8, f32(u->gc1, 128)))) return rc;
  up_back(7, u->gc1, u->c1, g2, 64, 128);
  if ((rc = conv_back(u, 7, f32(u->gc2, 256)))) return rc;
  up_back(6, u->gc2, u->c2, g3, 128, 256);
  if ((rc = conv_back(u, 6, f32(u->gp3, 128)))) return rc;
  skip_back(5, u->gc2, u->gp3, u->c2, g2, 128);
  if ((rc = conv_back(u, 5, mask(4, u->a2a)))) return rc;
  if ((rc = conv_back(u, 4, f32(u->gp2, 64)))) return rc;
  skip_back(3, u->gc1, u->gp2, u->c1, g1, 64);
  if ((rc = conv_back(u, 3, mask(2, u->a1a)))) return rc;
  if ((rc = conv_back(u, 2, f32(u->gp1, 32)))) return rc;
  skip_back(1, u->gc0, u->gp1, u->c0, g0, 32);
  if ((rc = conv_back(u, 1, mask(0, u->a0a)))) return rc;
  if ((rc = launch_grads(u->st, u->dall, u->djobs, !u->jobs.empty(), u->odd, u->grid))) return rc;
  float lp[256];
  UCHK(hipMemcpyAsync(lp, u->lpart, sizeof(lp), hipMemcpyDeviceToHost, u->st));
  UCHK(hipStreamSynchronize(u->st));
  double s = 0.0;
  for (float x : lp) s += x;
  if (loss) *loss = (float)(s / (double)(V0 * 3));
  return WLC_OK;
}

// input [B][n^3][11] (host FP32), converted on the device; targets [B][n^3][3].  The caller waits
// for the stream before it returns (the host arrays are read until then).
int upload(wlc_unet* u, const float* x, const float* t) {
  if (!u->B) return ufail(WLC_ESTATE, "the network has no buffers: its last resize failed");
  const long long V = u->vol(0).voxels();
  UCHK(hipMemcpyAsync(u->xin, x, sizeof(float) * (size_t)V * 11, hipMemcpyHostToDevice, u->st));
  hipLaunchKernelGGL(k_input, dim3(blocks(V * 16)), dim3(256), 0, u->st, u->xin, u->x0, V);
  if (t) UCHK(hipMemcpyAsync(u->target, t, sizeof(float) * (size_t)V * 3, hipMemcpyHostToDevice, u->st));
  UCHK(hipGetLastError());
  return WLC_OK;
}

// the packed bf16 weights from the master copy
int repack(wlc_unet* u) {
  hipLaunchKernelGGL(k_pack, dim3(blocks(u->np)), dim3(256), 0, u->st, u->p, u->pack, u->wf, u->wb, u->np);
  UCHK(hipGetLastError());
  UCHK(hipStreamSynchronize(u->st));
  return WLC_OK;
}

}  // namespace

extern "C" {

int wlc_unet_create(int n, int batch, unsigned long long seed, wlc_unet** out) {
  if (!out) return ufail(WLC_EINVAL, "out is NULL");
  *out = nullptr;
  if (n < 8 || n % 8 || batch < 1) return ufail(WLC_EINVAL, "grid edge must be a multiple of 8 and batch >= 1");
  if ((long long)batch * n * n * n * 256 >= (1LL << 31))
    return ufail(WLC_EINVAL, "batch x grid too large (the kernels index an activation tensor with 32 bits)");
  wlc_unet* u = new wlc_unet();
  if (hipGetDevice(&u->device) != hipSuccess || hipStreamCreateWithFlags(&u->st, hipStreamNonBlocking) != hipSuccess) {
    delete u;
    return ufail(WLC_EHIP, "no HIP device / stream");
  }
  u->layers = architecture();
  const Layer& last = u->layers.back();
  u->np = last.boff + last.cout;
  int rc;
#define UA(ptr, cnt) if ((rc = ualloc(u->allocs, &(ptr), (cnt)))) { unet_free(u); return rc; }
  UA(u->p, u->np); UA(u->m, u->np); UA(u->v, u->np); UA(u->g, u->np); UA(u->mask, u->np);
  UA(u->wf, u->np); UA(u->wb, u->np); UA(u->zrow, 64);
#undef UA
  u->pack.n = (int)u->layers.size();
  for (size_t li = 0; li < u->layers.size(); ++li)
    u->pack.l[li] = PackLayer{u->layers[li].woff, u->layers[li].cin, u->layers[li].cout};
  if ((rc = alloc_acts(u, n, batch))) {
    unet_free(u);
    return rc;
  }
  // He-normal weights over the real fan-in, zero biases, zero padding entries; the output
  // layer starts small
  std::vector<float> hp((size_t)u->np, 0.f);
  std::vector<unsigned char> hm((size_t)u->np, 0);
  Normals normal(seed);
  for (size_t li = 0; li < u->layers.size(); ++li) {
    const Layer& l = u->layers[li];
    const float sd = std::sqrt(2.f / (27.f * l.cin_real)) * (li + 1 == u->layers.size() ? 0.1f : 1.f);
    for (int co = 0; co < l.cout; ++co)
      for (int t = 0; t < 27; ++t)
        for (int ci = 0; ci < l.cin; ++ci) {
          const long long i = l.woff + ((long long)co * 27 + t) * l.cin + ci;
          const bool real = co < l.cout_real && ci < l.cin_real;
          const float w = normal();
          hp[i] = real ? sd * w : 0.f;
          hm[i] = real ? 1 : 0;
        }
    for (int co = 0; co < l.cout; ++co) hm[l.boff + co] = co < l.cout_real ? 1 : 0;
  }
  if (hipMemcpy(u->p, hp.data(), sizeof(float) * hp.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(u->mask, hm.data(), hm.size(), hipMemcpyHostToDevice) != hipSuccess) {
    unet_free(u);
    return ufail(WLC_EHIP, "parameter upload failed");
  }
  if ((rc = repack(u))) {
    unet_free(u);
    return rc;
  }
  *out = u;
  return WLC_OK;
}

void wlc_unet_destroy(wlc_unet* u) { unet_free(u); }

int wlc_unet_resize(wlc_unet* u, int n, int batch) {
  if (!u) return ufail(WLC_EINVAL, "NULL network");
  if (n < 8 || n % 8 || batch < 1) return ufail(WLC_EINVAL, "grid edge must be a multiple of 8 and batch >= 1");
  if ((long long)batch * n * n * n * 256 >= (1LL << 31))
    return ufail(WLC_EINVAL, "batch x grid too large (the kernels index an activation tensor with 32 bits)");
  UCHK(hipSetDevice(u->device));
  UCHK(hipStreamSynchronize(u->st));
  return alloc_acts(u, n, batch);
}

long long wlc_unet_num_params(const wlc_unet* u, int padded) {
  if (!u) return WLC_EINVAL;
  if (padded) return u->np;
  long long n = 0;
  for (const Layer& l : u->layers) n += (long long)l.cout_real * 27 * l.cin_real + l.cout_real;
  return n;
}

int wlc_unet_layer(const wlc_unet* u, int i, int* info) {
  if (!u || !info || i < 0 || i >= (int)u->layers.size()) return ufail(WLC_EINVAL, "bad layer");
  const Layer& l = u->layers[i];
  info[0] = l.cin; info[1] = l.cout; info[2] = l.cin_real; info[3] = l.cout_real;
  info[4] = l.level; info[5] = l.relu; info[6] = (int)l.woff; info[7] = (int)l.boff;
  return WLC_OK;
}

int wlc_unet_forward(wlc_unet* u, const float* x, float* y) {
  if (!u || !x) return ufail(WLC_EINVAL, "NULL argument");
  UCHK(hipSetDevice(u->device));
  int rc = upload(u, x, nullptr);
  if (rc || (rc = forward(u))) return rc;
  if (y)
    UCHK(hipMemcpyAsync(y, u->y, sizeof(float) * 3 * (size_t)u->vol(0).voxels(), hipMemcpyDeviceToHost, u->st));
  UCHK(hipStreamSynchronize(u->st));
  return WLC_OK;
}

int wlc_unet_gradients(wlc_unet* u, const float* x, const float* t, float* loss) {
  if (!u || !x || !t) return ufail(WLC_EINVAL, "NULL argument");
  UCHK(hipSetDevice(u->device));
  int rc = upload(u, x, t);
  if (rc || (rc = forward(u)) || (rc = backward(u, loss))) return rc;
  return WLC_OK;
}

int wlc_unet_adam(wlc_unet* u, float lr) {
  if (!u) return ufail(WLC_EINVAL, "NULL argument");
  UCHK(hipSetDevice(u->device));
  u->adam_t += 1;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - std::pow(b1, (float)u->adam_t), c2 = 1.f - std::pow(b2, (float)u->adam_t);
  hipLaunchKernelGGL(k_adam, dim3(blocks(u->np)), dim3(256), 0, u->st, u->p, u->m, u->v, u->g, u->pack,
                     u->wf, u->wb, u->mask, u->np, lr, b1, b2, eps, c1, c2);
  UCHK(hipGetLastError());
  UCHK(hipStreamSynchronize(u->st));
  return WLC_OK;
}

int wlc_unet_train_step(wlc_unet* u, const float* x, const float* t, float lr, float* loss) {
  int rc = wlc_unet_gradients(u, x, t, loss);
  if (rc) return rc;
  return wlc_unet_adam(u, lr);
}

// flat parameters / gradients (padded layout: per layer W [cout][27][cin] then b [cout])
int wlc_unet_get(wlc_unet* u, int which, float* out) {
  if (!u || !out || which < 0 || which > 1) return ufail(WLC_EINVAL, "bad arguments");
  UCHK(hipSetDevice(u->device));
  UCHK(hipStreamSynchronize(u->st));
  UCHK(hipMemcpy(out, which == 0 ? u->p : u->g, sizeof(float) * (size_t)u->np, hipMemcpyDeviceToHost));
  return WLC_OK;
}

int wlc_unet_set_params(wlc_unet* u, const float* in) {
  if (!u || !in) return ufail(WLC_EINVAL, "NULL argument");
  UCHK(hipSetDevice(u->device));
  UCHK(hipMemcpy(u->p, in, sizeof(float) * (size_t)u->np, hipMemcpyHostToDevice));
  return repack(u);
}

// Test hook: one convolution and its gradients on host arrays (x [V][cin], w [cout][27][cin],
// b [cout], dy [V][cout], all rounded to bf16 where the matrix cores read them, as in the
// network): y = conv(x), dx, dw, db.  cin, cout multiples of 16.
int wlc_test_conv3d(int B, int D, int H, int W, int cin, int cout, const float* x, const float* w,
                    const float* b, const float* dy, float* y, float* dx, float* dw, float* db) {
  if (cin % 16 || cout % 16 || cin > 256 || cout > 256 || B < 1 || D < 1 || H < 1 || W < 1 || !x || !w || !b ||
      !dy || !y || !dx || !dw || !db)
    return ufail(WLC_EINVAL, "bad arguments");
  const Vol g{B, D, H, W};
  const long long V = g.voxels(), nw = (long long)cout * 27 * cin;
  if (V * std::max(cin, cout) >= (1LL << 31)) return ufail(WLC_EINVAL, "tensor too large");
  std::vector<bf16> hx((size_t)(V * cin)), hdy((size_t)(V * cout));
  for (size_t i = 0; i < hx.size(); ++i) hx[i] = f2bf(x[i]);
  for (size_t i = 0; i < hdy.size(); ++i) hdy[i] = f2bf(dy[i]);
  GradJob q = grad_job(g, cin, cout);
  bf16 *dX = nullptr, *dDY = nullptr, *dF = nullptr, *dBk = nullptr, *dZ = nullptr;
  float *dW = nullptr, *dB = nullptr, *dYo = nullptr, *dDX = nullptr, *dDYf = nullptr;
  GradJobs* dJ = nullptr;
  hipError_t e = hipSuccess;
  auto M = [&](void** p, size_t bytes) { if (e == hipSuccess) e = hipMalloc(p, bytes); };
  M((void**)&dX, sizeof(bf16) * hx.size()); M((void**)&dDY, sizeof(bf16) * hdy.size());
  M((void**)&dF, sizeof(bf16) * nw); M((void**)&dBk, sizeof(bf16) * nw); M((void**)&dZ, 128);
  M((void**)&dW, sizeof(float) * nw); M((void**)&dB, sizeof(float) * cout); M((void**)&dYo, sizeof(float) * V * cout);
  M((void**)&dDX, sizeof(float) * V * cin); M((void**)&dDYf, sizeof(float) * V * cout); M((void**)&dJ, sizeof(GradJobs));
  M((void**)&q.xt, sizeof(bf16) * hx.size()); M((void**)&q.dyt, sizeof(bf16) * hdy.size());
  M((void**)&q.part, sizeof(float) * part_floats(q)); M((void**)&q.bpart, sizeof(float) * q.nbp * cout);
  M((void**)&q.dW, sizeof(float) * nw); M((void**)&q.db, sizeof(float) * cout);
  if (e == hipSuccess) e = hipMemcpy(dX, hx.data(), sizeof(bf16) * hx.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dW, w, sizeof(float) * nw, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dDY, hdy.data(), sizeof(bf16) * hdy.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dB, b, sizeof(float) * cout, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dDYf, dy, sizeof(float) * V * cout, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(dZ, 0, 128);
  q.X = dX;
  q.dYb = dDY;
  q.dYf = dDYf;
  std::vector<GradJob> one{q};
  unsigned grid[6];
  place_jobs(one, grid);
  GradJobs J{};
  J.n = 1;
  J.j[0] = one[0];
  if (e == hipSuccess) e = hipMemcpy(dJ, &J, sizeof(J), hipMemcpyHostToDevice);
  int rc = WLC_OK;
  if (e == hipSuccess) {
    PackTable T{};
    T.n = 1;
    T.l[0] = PackLayer{0, cin, cout};
    hipLaunchKernelGGL(k_pack, dim3(blocks(nw)), dim3(256), 0, nullptr, dW, T, dF, dBk, nw);
    rc = launch_conv(nullptr, dX, dF, dZ, g, cin, cout, EpiF32{dYo, dB, cout});
    const bool rows = grad_rows(g);
    if (!rc) rc = launch_grads(nullptr, dJ, dJ, rows, rows ? std::vector<GradJob>{} : one, grid);
    if (!rc) rc = launch_conv(nullptr, dDY, dBk, dZ, g, cout, cin, EpiF32{dDX, nullptr, cin});
    if (!rc) e = hipGetLastError();
  }
  if (!rc && e == hipSuccess) e = hipDeviceSynchronize();
  if (!rc && e == hipSuccess) e = hipMemcpy(y, dYo, sizeof(float) * V * cout, hipMemcpyDeviceToHost);
  if (!rc && e == hipSuccess) e = hipMemcpy(dx, dDX, sizeof(float) * V * cin, hipMemcpyDeviceToHost);
  if (!rc && e == hipSuccess) e = hipMemcpy(dw, q.dW, sizeof(float) * nw, hipMemcpyDeviceToHost);
  if (!rc && e == hipSuccess) e = hipMemcpy(db, q.db, sizeof(float) * cout, hipMemcpyDeviceToHost);
  for (void* p : {(void*)dX, (void*)dDY, (void*)dF, (void*)dBk, (void*)dZ, (void*)dW, (void*)dB, (void*)dYo, (void*)dDX,
                  (void*)dDYf, (void*)dJ, (void*)q.xt, (void*)q.dyt, (void*)q.part, (void*)q.bpart, (void*)q.dW,
                  (void*)q.db})
    if (p) (void)hipFree(p);
  if (rc) return rc;
  if (e != hipSuccess) return ufail(WLC_EHIP, std::string("test conv3d: ") + hipGetErrorString(e));
  return WLC_OK;
}

}  // extern "C"
