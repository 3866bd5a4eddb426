// step_mixed_d3q27.hip -- FP32-compute instantiations for D3Q27 with shifted FP16 and
// FP64 storage: a unit of their own, since D3Q27's are the longest of the build.  Built
// with FMA contraction.
#include "instantiate.hpp"

namespace lbm {

void register_step_mixed_d3q27(Registry& r) {
  register_combo<Lattice<LatticeType::D3Q27>, _Float16, float, true, 8, 4, 2>(r, TYPE_F16, TYPE_F32);
  register_combo<Lattice<LatticeType::D3Q27>, double, float, true, 2>(r, TYPE_F64, TYPE_F32);
}

}  // namespace lbm
