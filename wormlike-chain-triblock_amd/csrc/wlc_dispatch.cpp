// Host dispatch of the per-Lmax kernel-B translation units (wlc_zsolve.hip is
// compiled once per L = 0..8) and of the orientation-table uploads.
#include <hip/hip_runtime.h>

#include "wlc_kernels.h"
#include "wlc_z128.h"
#include "wlc_zcol.h"

namespace wlc {

#define WLC_DECL(L)                                                                          \
  hipError_t zsolve_launch_L##L(const Geom&, const SolveArgs&, hipStream_t);                 \
  hipError_t zsolve_batch_L##L(const ZJob&, const ZJob*, int, hipStream_t);                 \
  LaunchKey zsolve_key_L##L(const Geom&, const SolveArgs&);                                  \
  hipError_t test_solve_L##L(int, const double*, double, double, double, double, double2*,   \
                             hipStream_t);                                                   \
  const void* zcol_kernel_L##L(bool);

WLC_DECL(0) WLC_DECL(1) WLC_DECL(2) WLC_DECL(3) WLC_DECL(4) WLC_DECL(5) WLC_DECL(6) WLC_DECL(7) WLC_DECL(8)
#undef WLC_DECL
const void* z128_kernel_L5(bool, bool);
const void* z128_kernel_L6(bool, bool);
const void* z128_kernel_L7(bool, bool);
const void* z128_kernel_L8(bool, bool);

namespace {
// Column groups up to which the column kernel is the faster one for short z axes.  It spreads the
// harmonics of a group over a workgroup: with one to four of them most of its threads idle, which
// costs nothing while the groups fit the GPU together and the most where they take many rounds, and
// there the generic kernel's thread per k-point is faster.  Per launch, generic / column kernel:
// Lmax 0, 48^2 x 48 (624 groups) 10.1 / 10.0 us, 72 x 54 x 48 (1008) 10.5 / 12.6, 128^2 x 48 19.7 /
// 31.5, 54^2 x 24 (756) 8.1 / 7.3, 64^2 x 24 (1088) 8.1 / 9.2, 108 x 72 x 8 (1080) and on 7.5 / 9.2;
// Lmax 1, 48^2 x 36 13.7 / 12.5, 64^2 x 36 16.3 / 16.8, 128^2 x 48 32.2 / 44.2.  The generic
// transform of 18 and 54 has the most radix-3 passes: Lmax 1, 64^2 x 54 20.9 / 18.4, 108 x 72 x 54
// (2016) 24.8 / 26.4; 96^2 x 18 (2352) 16.5 / 16.7, 128^2 x 18 22.3 / 22.0.  At Lmax 2 the column
// kernel is behind only with very many groups: 128^2 x 8 (2176) 15.8 / 17.2; where the two sweeps
// run at once, its LDS beside the planes' of 96^2 and 128^2 costs more than it gains: pair of sweeps
// of 60 steps on 96^2 x 48 (2400) 12.7 / 13.3 ms, of 160 on 128^2 x 48 (4224) 38.9 / 40.4, of 80 on
// 128^2 x 36 16.2 / 16.7, but 96^2 x 36 11.0 / 10.8.  Above that nowhere, but at Lmax 7 nz = 48 has a
// kernel of its own for many columns (k_zsolve48 in wlc_zsolve.hip).
unsigned zcol_groups(int nz, int L) {
  const bool slow3 = nz == 18 || nz == 54, wide = nz == 36 || nz == 48;
  if (L == 0) return wide ? 640 : 1024;
  if (L == 1) return slow3 ? (nz == 18 ? 3072 : 1536) : 1024;
  if (L == 7 && nz == 48) return 960;
  if (L == 2) return nz == 8 || nz == 48 ? 2048 : nz == 36 ? 4096 : ~0u;
  return ~0u;
}

// short z axes with the FP64 spectrum take the column kernel unless the generic kernel or its
// degree split (1) is asked for; with the FP32 spectrum the generic ones: another order of the same
// operations rounds some stored values the other way, which moves phi by up to 1e-7 of itself after
// 40 to 100 steps, and that mode keeps its results.  It costs time: 24^3 / Lmax 6 41.9 us a launch
// against 15.2 with the FP64 spectrum, 32^3 / Lmax 4 25.7 against 15.1 (launches timed by events).
bool use_zcol(const Geom& g, const SolveArgs& a) {
  if (!zcol_nz(g.nz) || g.spec32 || a.generic || a.split < 2 || a.M != (a.L + 1) * (a.L + 1)) return false;
  const int cols = 1 << zcol_log2_cols(g.nz);
  return unsigned((g.nxh + cols - 1) / cols * g.ny) <= zcol_groups(g.nz, a.L);
}

// nz = 128 with a degree split asked for: the three-part kernel where there are columns for it
bool use_z128(const Geom& g, const SolveArgs& a) {
  return g.nz == 128 && a.L >= kZ128MinL && !a.generic && a.split && !z128_two_parts(g, a.L) &&
         a.M == (a.L + 1) * (a.L + 1);
}

const void* zcol_kernel(const SolveArgs& a, bool batch) {
  switch (a.L) {
#define WLC_CASE(L) \
  case L: return zcol_kernel_L##L(batch);
    WLC_CASE(0) WLC_CASE(1) WLC_CASE(2) WLC_CASE(3) WLC_CASE(4) WLC_CASE(5) WLC_CASE(6) WLC_CASE(7) WLC_CASE(8)
#undef WLC_CASE
  }
  return nullptr;
}
const void* z128_kernel(const Geom& g, const SolveArgs& a, bool batch) {
  switch (a.L) {
#define WLC_CASE(L) \
  case L: return z128_kernel_L##L(g.spec32 != 0, batch);
    WLC_CASE(5) WLC_CASE(6) WLC_CASE(7) WLC_CASE(8)
#undef WLC_CASE
  }
  return nullptr;
}

bool own_file(const Geom& g, const SolveArgs& a) { return use_zcol(g, a) || use_z128(g, a); }

LaunchKey own_key(const Geom& g, const SolveArgs& a, bool batch) {
  if (use_z128(g, a))
    return LaunchKey{z128_kernel(g, a, batch), z128_grid(g), 1u, (unsigned)kZ128Threads, z128_lds_bytes()};
  return LaunchKey{zcol_kernel(a, batch), zcol_grid(g), 1u, (unsigned)zcol_threads(g.nz),
                   zcol_lds_bytes(g.nz, a.M)};
}

hipError_t own_launch(const Geom& g, const SolveArgs& a, const ZJob* jobs, int n, hipStream_t st) {
  const LaunchKey key = own_key(g, a, jobs != nullptr);
  if (!key.k) return hipErrorInvalidValue;
  if (key.lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(key.k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)key.lds);
    if (e != hipSuccess) return e;
  }
  Geom gg = g;
  SolveArgs aa = a;
  const ZJob* jp = jobs;
  void* one[] = {&gg, &aa};
  void* many[] = {&jp};
  return hipLaunchKernel(key.k, dim3(key.gx, 1, n), dim3(key.threads), jobs ? many : one, key.lds, st);
}
}  // namespace

hipError_t launch_zsolve(const Geom& g, const SolveArgs& a, hipStream_t st) {
  if (own_file(g, a)) return own_launch(g, a, nullptr, 1, st);
  switch (a.L) {
#define WLC_CASE(L) \
  case L: return zsolve_launch_L##L(g, a, st);
    WLC_CASE(0) WLC_CASE(1) WLC_CASE(2) WLC_CASE(3) WLC_CASE(4) WLC_CASE(5) WLC_CASE(6) WLC_CASE(7) WLC_CASE(8)
#undef WLC_CASE
  }
  return hipErrorInvalidValue;
}

hipError_t launch_zsolve_batch(const ZJob& rep, const ZJob* jobs, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  if (own_file(rep.g, rep.a)) return own_launch(rep.g, rep.a, jobs, n, st);
  switch (rep.a.L) {
#define WLC_CASE(L) \
  case L: return zsolve_batch_L##L(rep, jobs, n, st);
    WLC_CASE(0) WLC_CASE(1) WLC_CASE(2) WLC_CASE(3) WLC_CASE(4) WLC_CASE(5) WLC_CASE(6) WLC_CASE(7) WLC_CASE(8)
#undef WLC_CASE
  }
  return hipErrorInvalidValue;
}

LaunchKey zsolve_key(const Geom& g, const SolveArgs& a) {
  if (own_file(g, a)) return own_key(g, a, false);
  switch (a.L) {
#define WLC_CASE(L) \
  case L: return zsolve_key_L##L(g, a);
    WLC_CASE(0) WLC_CASE(1) WLC_CASE(2) WLC_CASE(3) WLC_CASE(4) WLC_CASE(5) WLC_CASE(6) WLC_CASE(7) WLC_CASE(8)
#undef WLC_CASE
  }
  return LaunchKey{nullptr, 0, 0, 0, 0};
}

hipError_t launch_test_solve(int L, int nk, const double* kvec, double cdelta, double sigma,
                             double ds, double dslam, double2* v, hipStream_t st) {
  switch (L) {
#define WLC_CASE(LL) \
  case LL: return test_solve_L##LL(nk, kvec, cdelta, sigma, ds, dslam, v, st);
    WLC_CASE(0) WLC_CASE(1) WLC_CASE(2) WLC_CASE(3) WLC_CASE(4) WLC_CASE(5) WLC_CASE(6) WLC_CASE(7) WLC_CASE(8)
#undef WLC_CASE
  }
  return hipErrorInvalidValue;
}

namespace {
#define WLC_TABLE_QUAL static constexpr
#include "wlc_tables.inc"
#undef WLC_TABLE_QUAL
}  // namespace

// The device code carries the orientation tables as compile-time constants; check
// them against the ones the host set-up code derives now.
hipError_t upload_orientation_tables(const OrientTables& t) {
  for (int i = 0; i < kMaxM; ++i)
    if (kZsign[i] != t.zsign[i] || kTri[i] != t.tri_e[i]) return hipErrorInvalidValue;
  const int ny = t.yh_off[kMaxL + 1];
  if (ny != (int)(sizeof(kYh) / sizeof(kYh[0]))) return hipErrorInvalidValue;
  for (int i = 0; i < ny; ++i)
    if (kYh[i] != t.yh[i]) return hipErrorInvalidValue;
  return hipSuccess;
}

}  // namespace wlc
