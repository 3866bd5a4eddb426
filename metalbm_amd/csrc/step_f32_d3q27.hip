// step_f32_d3q27.hip -- FP32-compute instantiations for D3Q27 with FP32 storage
// (shifted f - w and unshifted).  Built with FMA contraction.
#include "instantiate.hpp"

namespace lbm {

void register_step_f32_d3q27(Registry& r) {
  register_combo<Lattice<LatticeType::D3Q27>, float, float, false, 4, 2>(r, TYPE_F32, TYPE_F32);
  register_combo<Lattice<LatticeType::D3Q27>, float, float, true, 4, 2>(r, TYPE_F32, TYPE_F32);
}

}  // namespace lbm
