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
// short z axes with the FP64 spectrum take the column kernel unless the generic kernel or its
// degree split (1) is asked for; with the FP32 spectrum the generic ones, as before the column
// kernel: another order of the same operations rounds some stored values the other way, which
// moves phi by up to 1e-7 of itself after 40 to 100 steps
bool use_zcol(const Geom& g, const SolveArgs& a) {
  return zcol_nz(g.nz) && !g.spec32 && !a.generic && a.split >= 2 && a.M == (a.L + 1) * (a.L + 1);
}

// nz = 128 with a degree split asked for: the three-part kernel
bool use_z128(const Geom& g, const SolveArgs& a) {
  return g.nz == 128 && a.L >= kZ128MinL && !a.generic && a.split && a.M == (a.L + 1) * (a.L + 1);
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
