// march_rules.cpp -- the tiling of the two-step kernel against what the kernel
// assumes, for extents from degenerate to huge (built and run by
// tests/test_march_rules.py).  Prints, for the extents given as arguments, whether
// the automatic choice takes the two-step kernel.
#include <cstdio>
#include <cstdlib>

#include "config_rules.hpp"

static int failures = 0;
static void check(bool ok, const char* what, int nx, int ny, int nz, int columns) {
  if (ok) return;
  std::printf("FAIL %s at %d x %d x %d, %d columns\n", what, nx, ny, nz, columns);
  ++failures;
}

// (columns, interior, side) of D3Q19 and D3Q27 in FP32 and in FP64, without and with
// force tables
static const int kernels[8][3] = {
    {2560, 2048, 0}, {2508, 2048, 264}, {1704, 1024, 0}, {1672, 1024, 264},
    {1280, 512, 0},  {1228, 512, 264},  {852, 512, 0},   {820, 512, 264}};

int main(int argc, char** argv) {
  if (argc == 9) {  // nx ny nz columns interior side line limit
    int v[8];
    for (int k = 1; k < 8; ++k) v[k] = std::atoi(argv[k]);
    const lbm::MarchShape m = lbm::march_shape(v[1], v[2], v[3], v[4], v[5], v[6], 256, v[7]);
    std::printf("%d\n", (int)lbm::march_pays(m, (double)v[1] * v[2] * v[3], v[5],
                                             std::atof(argv[8])));
    return 0;
  }
  const int extents[] = {1,   2,   3,   7,    8,    9,    31,   32,   33,    64,     96,
                         130, 161, 256, 257,  263,  264,  265,  511,  512,   513,    1000,
                         1025, 2047, 2048, 2049, 2561, 8193, 65537, 1000003};
  int shapes = 0;
  for (const auto& k : kernels)
    for (int nx : {1, 2, 3, 17, 256, 1000})
      for (int ny : extents)
        for (int nz : extents) {
          if ((double)ny * nz * 4.0 >= 4294967296.0) continue;
          const lbm::MarchShape m = lbm::march_shape(nx, ny, nz, k[0], k[1], k[2], 256, 32);
          if (m.ranges == 0) continue;
          ++shapes;
          auto ok = [&](bool c, const char* what) { check(c, what, nx, ny, nz, k[0]); };
          const long long pitch = m.tiles_z == 1 ? m.tz : m.tz + 2;
          ok(m.ty >= 1 && m.tz >= 1 && m.ranges >= 1 && m.ranges <= nx, "positive");
          ok((long long)m.ty * m.tiles_y >= ny && (long long)m.ty * (m.tiles_y - 1) < ny, "rows");
          ok((long long)m.tz * m.tiles_z >= nz && (long long)m.tz * (m.tiles_z - 1) < nz, "places");
          ok((m.ty + 2) * pitch <= k[0], "columns in LDS");
          ok((long long)m.ty * m.tz <= k[1], "columns in registers");
          ok(m.ty + 1 < 32768 && pitch <= 32767, "packed column index");
          if (k[2]) ok(m.ty + 2 <= k[2] && pitch <= k[2], "force tables");
          ok((long long)m.tiles_y * m.tiles_z * m.ranges < (1ll << 31), "grid");
        }
  std::printf("%d shapes, %d failures\n", shapes, failures);
  return failures != 0 || shapes < 2000;
}
