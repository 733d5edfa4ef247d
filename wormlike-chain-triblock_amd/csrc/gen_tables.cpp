// Build-time generator of the compiled-in tables.
//   gen_tables wlc_tables.inc wlc_twiddles.inc
// wlc_tables.inc: the orientation tables of the k-aligned solve (z-rotation pair signs, packed
// pi/2 y-rotation, rotated-frame tridiagonal couplings) as compile-time constants for the device
// code.  They are produced by the same host code (build_orientation_tables) that the library
// re-runs at handle creation to check the compiled-in values.
// wlc_twiddles.inc: the FFT twiddles of every grid edge the library accepts (make_axis_plan),
// one device array, for the step entry point that neither allocates nor uploads anything.
#include <cstdio>
#include <string>

#include "wlc_internal.h"

int main(int argc, char** argv) {
  wlc::OrientTables t;
  std::string err = wlc::build_orientation_tables(wlc::kMaxL, &t);
  if (!err.empty()) {
    std::fprintf(stderr, "gen_tables: %s\n", err.c_str());
    return 1;
  }
  FILE* f = argc > 1 ? std::fopen(argv[1], "w") : stdout;
  if (!f) return 1;
  std::fprintf(f, "// Generated by gen_tables.cpp (build_orientation_tables, Lmax %d); do not edit.\n", wlc::kMaxL);
  std::fprintf(f, "#define WLC_TABLE_LMAX %d\n", wlc::kMaxL);
  std::fprintf(f, "WLC_TABLE_QUAL double kZsign[%d] = {", wlc::kMaxM);
  for (int i = 0; i < wlc::kMaxM; ++i) std::fprintf(f, "%s%.1f", i ? ", " : "", t.zsign[i]);
  std::fprintf(f, "};\n");
  const int ny = t.yh_off[wlc::kMaxL + 1];
  std::fprintf(f, "WLC_TABLE_QUAL double kYh[%d] = {\n", ny);
  for (int i = 0; i < ny; ++i) std::fprintf(f, "    %.17g,\n", t.yh[i]);
  std::fprintf(f, "};\n");
  std::fprintf(f, "WLC_TABLE_QUAL double kTri[%d] = {\n", wlc::kMaxM);
  for (int i = 0; i < wlc::kMaxM; ++i) std::fprintf(f, "    %.17g,\n", t.tri_e[i]);
  std::fprintf(f, "};\n");
  if (f != stdout) std::fclose(f);
  if (argc < 3) return 0;
  f = std::fopen(argv[2], "w");
  if (!f) return 1;
  std::string edges, offs, vals;
  int total = 0;
  for (int n = 2; n <= 256; n += 2) {
    wlc::AxisPlan pl;
    if (!wlc::make_axis_plan(n, &pl).empty()) continue;
    edges += std::to_string(n) + ", ";
    offs += std::to_string(total) + ", ";
    total += n;
    char b[64];
    for (int k = 0; k < 2 * n; ++k) {
      std::snprintf(b, sizeof b, "%a,%c", pl.tw[k], k % 4 == 3 ? '\n' : ' ');
      vals += b;
    }
    vals += "\n";
  }
  std::fprintf(f, "// Generated by gen_tables.cpp (make_axis_plan); do not edit.\n");
  std::fprintf(f, "const int kTwEdge[] = {%s};\nconst int kTwOff[] = {%s};\n", edges.c_str(), offs.c_str());
  std::fprintf(f, "__device__ __align__(16) double kTwiddles[%d] = {\n%s};\n", 2 * total, vals.c_str());
  std::fclose(f);
  return 0;
}
