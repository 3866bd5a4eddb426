// step_choice.cpp -- prints what the automatic choice takes for one domain (built and run
// by tests/test_step_choice.py):
//   tile nx ny rows16 rows64 fp64 exact                          -> wide steps
//   march nx ny nz columns interior side line limit              -> taken
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "config_rules.hpp"

int main(int argc, char** argv) {
  if (argc == 8 && !std::strcmp(argv[1], "tile")) {
    int v[6];
    for (int k = 0; k < 6; ++k) v[k] = std::atoi(argv[2 + k]);
    const int rows[2] = {v[2], v[3]};
    const lbm::TileShape m = lbm::tile_shape(v[0], v[1], rows, v[4], v[5]);
    std::printf("%d %d\n", m.wide, m.steps);
    return 0;
  }
  if (argc == 10 && !std::strcmp(argv[1], "march")) {
    int v[7];
    for (int k = 0; k < 7; ++k) v[k] = std::atoi(argv[2 + k]);
    const lbm::MarchShape m = lbm::march_shape(v[0], v[1], v[2], v[3], v[4], v[5], 256, v[6]);
    std::printf("%d\n", (int)lbm::march_pays(m, (double)v[0] * v[1] * v[2], v[4],
                                             std::atof(argv[9])));
    return 0;
  }
  return 2;
}
