// instantiate.hpp -- instantiates and registers the fused step kernels for
// one compute type.  Included by exactly one translation unit per compute
// type, so each type can be built with its own floating-point contraction
// mode (FP64: off, for reference-order parity; FP32: fused).
#pragma once

#include <algorithm>

#include "fused_march.hpp"
#include "fused_step.hpp"
#include "fused_step_vec.hpp"
#include "fused_tile.hpp"
#include "registry.hpp"

namespace lbm {

template <class L, class S, class C, int FS, int EQ, bool SH, int CO>
hipError_t launch_step(const StepArgs& a, int fsx, int block, int grid,
                       hipStream_t st) {
  if constexpr (CO == (int)CollisionType::BGK) {
    if (a.nt_loads)
      hipLaunchKernelGGL((k_bgk<L, S, C, FS, EQ, SH, 256, true>), dim3(grid),
                         dim3(block), 0, st, a, fsx);
    else
      hipLaunchKernelGGL((k_bgk<L, S, C, FS, EQ, SH, 256, false>), dim3(grid),
                         dim3(block), 0, st, a, fsx);
  }
  else {
    constexpr bool REF = std::is_same_v<C, double> && !SH;
    constexpr bool FLAT = L::dimQ <= 9;
    auto whole = [&](auto mode, size_t lds = 0) {
      hipLaunchKernelGGL((k_elbm<L, S, C, FS, EQ, SH, 256, decltype(mode)::value>), dim3(grid),
                         dim3(block), lds, st, a, fsx);
    };
    // the listed cells, or without a list every cell
    auto listed = [&](auto mode) {
      const int blocks =
          a.defer.cells ? a.defer.shards * kDeferBlocks : (int)(((long long)a.N + 255) / 256);
      hipLaunchKernelGGL((k_elbm<L, S, C, FS, EQ, SH, 256, decltype(mode)::value>), dim3(blocks),
                         dim3(256), 0, st, a, fsx);
    };
    if (a.alpha_mode == 0) {
      if constexpr (REF) {
        whole(std::integral_constant<int, 6>{});
      } else {
        if (a.defer.cells) whole(std::integral_constant<int, 0>{});
        if constexpr (FLAT) {
          if (a.defer.cells) listed(std::integral_constant<int, 5>{});
          else whole(std::integral_constant<int, 6>{});
        } else {
          listed(std::integral_constant<int, 5>{});
        }
      }
    } else if (a.alpha_mode == 3) {
      if (FLAT || a.defer.cells) whole(std::integral_constant<int, 4>{});
      if constexpr (!FLAT) listed(std::integral_constant<int, 7>{});
    } else {
      if (a.alpha_mode == 2) {
        whole(std::integral_constant<int, 2>{});
      } else if constexpr (MlpShape<L>::NIN > 0) {
        // The learned solver stages the network in LDS (dynamic shared memory).
        using M = MfmaLayout<MlpShape<L>::NIN, MlpShape<L>::H1, MlpShape<L>::H2>;
        whole(std::integral_constant<int, 1>{}, M::BYTES);
      } else {
        return hipErrorInvalidValue;
      }
      listed(std::integral_constant<int, FLAT ? 3 : 7>{});
    }
  }
  return hipGetLastError();
}

template <class L, class S, class C, int FS, int EQ, bool SH, int V>
hipError_t launch_step_vec(const StepArgs& a, int fsx, int block, int grid,
                           hipStream_t st) {
  (void)block;
  hipLaunchKernelGGL((k_bgk_vec<L, S, C, FS, EQ, SH, V>), dim3(grid), dim3(64 * kVecWaves),
                     0, st, a, fsx);
  return hipGetLastError();
}

template <class L, class S, class C, int FS, int EQ, bool SH, bool SIDE>
hipError_t launch_march(const StepArgs& a, const MarchTiling& m, hipStream_t st) {
  hipLaunchKernelGGL((k_bgk_march<L, S, C, FS, EQ, SH, SIDE>),
                     dim3(m.tiles_y * m.tiles_z * m.ranges), dim3(kMarchThreads), 0, st, a, m);
  return hipGetLastError();
}
template <class L, class S, class C, int FS, int EQ, bool SH>
MarchKernel march_kernel() {
  MarchKernel k;
  k.launch[0] = &launch_march<L, S, C, FS, EQ, SH, false>;
  k.columns[0] = kMarchColumns<L, S, C, false>;
  if constexpr (FS != SRC_ZERO) {
    k.launch[1] = &launch_march<L, S, C, FS, EQ, SH, true>;
    k.columns[1] = kMarchColumns<L, S, C, true>;
  } else {  // no source: the force does not enter the step
    k.launch[1] = k.launch[0];
    k.columns[1] = k.columns[0];
  }
  k.interior = kMarchUnits<L, S> * kMarchThreads;
  k.side = kMarchSide;
  return k;
}

template <class L, class S, class C, int FS, int EQ, bool SH, int W>
hipError_t launch_tile(const StepArgs& a, const Tile2D& m, int fsx, hipStream_t st) {
  hipLaunchKernelGGL((k_bgk_tile<L, S, C, FS, EQ, SH, W>), dim3(m.tiles_x * m.tiles_y),
                     dim3(kTileThreads), 0, st, a, m, fsx);
  return hipGetLastError();
}

template <class L, class S, class C, bool SH, int... Vs>
void register_combo(Registry& r, int storage, int compute) {
  auto add_eq = [&](auto eqc) {
    constexpr int EQ = decltype(eqc)::value;
    auto add_fs = [&](auto fsc) {
      constexpr int FS = decltype(fsc)::value;
      r.add({(int)L::Type, (int)CollisionType::BGK, FS, EQ, storage, compute, SH, 0},
            &launch_step<L, S, C, FS, EQ, SH, (int)CollisionType::BGK>);
      // FP64 arithmetic on D3Q27 gains without a source only (192^3 a step: 615 ->
      // 504 us; with Guo's 616 -> 844, with the product equilibrium 608 -> 868: its
      // registers spill).
      constexpr bool HEAVY = std::is_same_v<C, double> && L::dimQ > 19 &&
                             (FS != SRC_ZERO || EQ != (int)EquilibriumType::TruncationMa3);
      if constexpr (L::dimD == 3 && kSeveralSteps<L, S, C> && !HEAVY)
        r.add({(int)L::Type, (int)CollisionType::BGK, FS, EQ, storage, compute, SH, 0},
              march_kernel<L, S, C, FS, EQ, SH>());
      if constexpr (L::dimD == 2 && kSeveralSteps<L, S, C>)
        r.add({(int)L::Type, (int)CollisionType::BGK, FS, EQ, storage, compute, SH, 0},
              TileKernel{{&launch_tile<L, S, C, FS, EQ, SH, 16>,
                          &launch_tile<L, S, C, FS, EQ, SH, 64>},
                         {kTileRows<L, S, 16>, kTileRows<L, S, 64>}});
      r.add({(int)L::Type, (int)CollisionType::ELBM, FS, EQ, storage, compute, SH, 0},
            &launch_step<L, S, C, FS, EQ, SH, (int)CollisionType::ELBM>);
      (r.add({(int)L::Type, (int)CollisionType::BGK, FS, EQ, storage, compute, SH, Vs},
             &launch_step_vec<L, S, C, FS, EQ, SH, Vs>), ...);
    };
    add_fs(std::integral_constant<int, SRC_ZERO>{});
    add_fs(std::integral_constant<int, SRC_GUO>{});
    add_fs(std::integral_constant<int, SRC_EDM>{});
  };
  add_eq(std::integral_constant<int, (int)EquilibriumType::TruncationMa3>{});
  // There is no Exact equilibrium for D3Q19 (Equilibrium.h:36-126).
  if constexpr (L::Type != LatticeType::D3Q19)
    add_eq(std::integral_constant<int, (int)EquilibriumType::Exact>{});
}

}  // namespace lbm
