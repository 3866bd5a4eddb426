// tile_rules.cpp -- the tiling of the multi-step 2D kernel against what the kernel
// assumes, for extents from degenerate to huge (built and run by
// tests/test_tile_rules.py).
#include <cstdio>

#include "config_rules.hpp"

int main() {
  const int extents[] = {1,  2,  3,   4,   5,   7,   8,   15,  16,   17,   24,   31,    32,
                         33, 56, 63,  64,  65,  127, 128, 129, 192,  255,  320,  511,   512,
                         513, 777, 1024, 2047, 2048, 4096, 8193, 65537, 1000003};
  const int rows[3][2] = {{71, 17}, {142, 35}, {284, 71}};  // FP64, FP32, FP16
  int shapes = 0, failures = 0;
  for (int type = 0; type < 3; ++type)
    for (int exact = 0; exact < 2; ++exact)
      for (int nx : extents)
        for (int ny : extents) {
          const lbm::TileShape m = lbm::tile_shape(nx, ny, rows[type], type == 0, exact);
          if (m.steps == 0) continue;
          ++shapes;
          const int halo = m.steps - 1, width = m.wide ? 64 : 16;
          const bool whole_x = m.tx == nx, whole_y = m.ty == ny;
          const bool ok = m.steps >= 2 && m.tx >= 1 && m.ty >= 1 && m.tx <= nx && m.ty <= ny &&
                          m.tx + (whole_x ? 0 : 2 * halo) <= rows[type][m.wide] &&
                          m.ty + (whole_y ? 0 : 2 * halo) <= width &&
                          (whole_x || halo <= nx) && (whole_y || halo <= ny);
          if (!ok) {
            std::printf("FAIL %d x %d type %d exact %d: %d %d x %d, %d steps\n", nx, ny, type,
                        exact, m.wide, m.tx, m.ty, m.steps);
            ++failures;
          }
        }
  std::printf("%d shapes, %d failures\n", shapes, failures);
  return failures != 0 || shapes < 1000;
}
