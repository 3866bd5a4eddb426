// config_rules.hpp -- host-side rules of the C ABI with no HIP dependency:
// configuration validation and the kernel-shape choice.  Included by
// capi.hip; the host sanitizer build (tests/test_sanitizers.py) compiles it
// for the CPU on its own.
#pragma once

#include <cmath>
#include <string>

#include "../../include/metalbm_amd.h"

namespace lbm {

// LBM_OK, or LBM_E_INVALID with the reason in why.  The reference takes its
// configuration from compile-time constants and has no run-time check.
inline int validate_config(const lbm_config* c, std::string& why) {
  const int lat = c->lattice;
  if (lat != LBM_D2Q9 && lat != LBM_D3Q19 && lat != LBM_D3Q27) {
    why = "lattice must be D2Q9 (3), D3Q19 (9) or D3Q27 (10)";
    return LBM_E_INVALID;
  }
  if (c->collision != LBM_BGK && c->collision != LBM_ELBM) {
    why = "collision must be BGK (1) or ELBM (2)";
    return LBM_E_INVALID;
  }
  if (c->forcing_scheme < LBM_FS_NONE || c->forcing_scheme > LBM_FS_EDM) {
    why = "forcing_scheme must be None (1), Guo (2), ShanChen (3) or EDM (4)";
    return LBM_E_INVALID;
  }
  if (c->force != LBM_FORCE_NONE && (c->force < LBM_FORCE_CONSTANT ||
                                      c->force > LBM_FORCE_TURBULENT_2D)) {
    why = "force must be None (0), Constant (4), Sinusoidal (5), Kolmogorov (6), "
          "ConstantShell (7), EnergyRemoval (8) or Turbulent2D (9)";
    return LBM_E_INVALID;
  }
  if ((c->force == LBM_FORCE_CONSTANT_SHELL || c->force == LBM_FORCE_TURBULENT_2D) &&
      (c->force_kmin < 0 || c->force_kmax < c->force_kmin)) {
    why = "spectral force shell needs 0 <= force_kmin <= force_kmax";
    return LBM_E_INVALID;
  }
  if ((c->force == LBM_FORCE_ENERGY_REMOVAL || c->force == LBM_FORCE_TURBULENT_2D) &&
      (c->removal_kmin < 0 || c->removal_kmax < c->removal_kmin)) {
    why = "energy removal shell needs 0 <= removal_kmin <= removal_kmax";
    return LBM_E_INVALID;
  }
  if (c->equilibrium != LBM_EQ_MA3 && c->equilibrium != LBM_EQ_EXACT) {
    why = "equilibrium must be TruncationMa3 (3) or Exact (1)";
    return LBM_E_INVALID;
  }
  if (c->equilibrium == LBM_EQ_EXACT && lat == LBM_D3Q19) {
    why = "there is no Exact equilibrium for D3Q19";
    return LBM_E_INVALID;
  }
  if (c->nx <= 0 || c->ny <= 0 || c->nz <= 0) {
    why = "nx, ny, nz must be positive";
    return LBM_E_INVALID;
  }
  if (lat == LBM_D2Q9 && c->nz != 1) {
    why = "nz must be 1 for D2Q9";
    return LBM_E_INVALID;
  }
  const double cells = (double)c->nx * c->ny * c->nz;
  if (cells >= 2147483648.0) {
    why = "nx*ny*nz must be below 2^31";
    return LBM_E_INVALID;
  }
  if (!(c->tau > 0.0) || !std::isfinite(c->tau)) {
    why = "tau must be positive and finite";
    return LBM_E_INVALID;
  }
  const int D = lat == LBM_D2Q9 ? 2 : 3;
  if (c->force == LBM_FORCE_SINUSOIDAL)
    for (int d = 0; d < D; ++d)
      if (c->wavelength[d] == 0.0) {
        why = "Sinusoidal force needs nonzero wavelength in every dimension";
        return LBM_E_INVALID;
      }
  if (c->force == LBM_FORCE_KOLMOGOROV && c->wavelength[0] == 0.0) {
    why = "Kolmogorov force needs a nonzero wavelength[0]";
    return LBM_E_INVALID;
  }
  if (c->storage < LBM_F64 || c->storage > LBM_F16 || c->compute < LBM_F64 ||
      c->compute > LBM_F32) {
    why = "storage must be F64/F32/F16 and compute F64/F32";
    return LBM_E_INVALID;
  }
  if (c->storage == LBM_F16 && !c->shifted) {
    why = "F16 storage requires shifted populations (f - w)";
    return LBM_E_INVALID;
  }
  if (c->compute == LBM_F64 && c->storage != LBM_F64) {
    why = "F64 compute requires F64 storage";
    return LBM_E_INVALID;
  }
  if (c->compute == LBM_F32 && c->storage == LBM_F64 && !c->shifted) {
    why = "F32 compute with F64 storage requires shifted populations";
    return LBM_E_INVALID;
  }
  if (c->kernel < LBM_KERNEL_AUTO || c->kernel > LBM_KERNEL_VECTOR) {
    why = "kernel must be AUTO (0), CELL (1) or VECTOR (2)";
    return LBM_E_INVALID;
  }
  if (c->kernel == LBM_KERNEL_VECTOR && c->collision != LBM_BGK) {
    why = "the vector kernel implements BGK only";
    return LBM_E_INVALID;
  }
  if (c->collision == LBM_ELBM && c->alpha_mode != LBM_ALPHA_NEWTON &&
      c->alpha_mode != LBM_ALPHA_LEARNED && c->alpha_mode != LBM_ALPHA_WARM_RESIDUAL &&
      c->alpha_mode != LBM_ALPHA_NEWTON_RESIDUAL) {
    why = "alpha_mode must be NEWTON (0), LEARNED (1), WARM_RESIDUAL (2) or NEWTON_RESIDUAL (3)";
    return LBM_E_INVALID;
  }
  if (c->collision == LBM_ELBM && c->alpha_mode == LBM_ALPHA_LEARNED &&
      lat == LBM_D3Q19) {
    why = "learned alpha is defined for D2Q9 and D3Q27 (tensor moment basis)";
    return LBM_E_INVALID;
  }
  if (c->collision == LBM_ELBM && c->alpha_mode != LBM_ALPHA_NEWTON &&
      !(c->residual_tol > 0.0)) {
    why = "residual_tol must be positive";
    return LBM_E_INVALID;
  }
  return LBM_OK;
}

// Workgroup size of the one-cell-per-lane kernel for a contiguous extent nk:
// one tile per row up to 256 cells, else the largest of 256/192/128 dividing
// the row, else 256.
inline int pick_block(int nk) {
  if (nk <= 256) return ((nk + 63) / 64) * 64;
  for (int b : {256, 192, 128})
    if (nk % b == 0) return b;
  return 256;
}

// Cells per lane V of the vector kernel for a validated configuration, or 0
// for one cell per lane.  instantiated(V) tells whether the vector kernel of
// this configuration exists with that V.
template <class F>
int pick_vector_width(const lbm_config* cfg, F&& instantiated) {
  const int D = cfg->lattice == LBM_D2Q9 ? 2 : 3;
  const int nk = D == 3 ? cfg->nz : cfg->ny;
  const int elem = cfg->storage == LBM_F64 ? 8 : (cfg->storage == LBM_F32 ? 4 : 2);
  // LBM_KERNEL_AUTO takes the vector kernel only where it measured faster
  // than one cell per lane (MI355X, 100-step runs): D3Q19 with FP32 storage
  // at 256^3 (+2%) and FP64 storage with FP32 compute (D3Q27 384^3, +2%).
  // One cell per lane won for D3Q19 FP64 (+12%), D3Q27 FP16 (+10%) and FP32
  // (+4%) storage, and D2Q9 128^2 FP64 (+48%): more wavefronts in flight.
  const bool vector_preferred =
      (cfg->lattice == LBM_D3Q19 && cfg->storage == LBM_F32) ||
      (cfg->storage == LBM_F64 && cfg->compute == LBM_F32);
  if (cfg->collision != LBM_BGK ||
      !(cfg->kernel == LBM_KERNEL_VECTOR ||
        (cfg->kernel == LBM_KERNEL_AUTO && vector_preferred)))
    return 0;
  // Vector width V, in this order (measured on D3Q27 384^3 rows):
  //  1. 16-byte lanes (V sizeof(S) = 16) even if the last 64-lane segment
  //     of a row is partial (FP32 V=4 split 64 + 32 lanes: +3% over V=2);
  //  2. else the widest V whose 64-lane segments tile the row (FP16 V=2,
  //     three full segments: 37.2k MLUPS, V=4 split 64 + 32: 31.8k);
  //  3. else the widest V dividing the row.
  // FP16 V=8 only for D2Q9: 27 x 8 (19 x 8) population values alone fill a
  // wavefront's registers (one wavefront per SIMD, 23.8k MLUPS).
  static const int cands[3][3] = {{2, 0, 0}, {4, 2, 0}, {8, 4, 2}};
  static const int cands_f16_3d[3] = {4, 2, 0};
  const int* cand = (cfg->storage == LBM_F16 && D == 3) ? cands_f16_3d : cands[cfg->storage];
  for (int k = 0; k < 3; ++k) {
    const int V = cand[k];
    if (V != 0 && V * elem == 16 && nk % V == 0 && instantiated(V)) return V;
  }
  for (int k = 0; k < 3; ++k) {
    const int V = cand[k];
    if (V != 0 && nk % (64 * V) == 0 && instantiated(V)) return V;
  }
  for (int k = 0; k < 3; ++k) {
    const int V = cand[k];
    if (V != 0 && nk % V == 0 && instantiated(V)) return V;
  }
  return 0;
}

// Tiling of the two-step kernel: tiles of ty x tz columns and a split of the x
// extent into ranges, for a kernel that holds `columns` columns with the rim and
// `interior` without, force tables of `side` rows or places (0: none needed),
// `slots` workgroups running at once and `line` values to a cache line.  cost
// estimates the time of a launch in units of one pass over the lattice: the
// writes, the reads (rows of the rim, whole lines at the ends of split rows, two
// planes for each range) and a fixed time per plane (a least-squares fit over 15
// shapes of eight configurations gives it as 0.35 to 1.2 of the time that
// `interior` columns take; residuals of 4 to 12 %), over the share of the slots
// that is busy.
// ranges == 0: nothing fits.
struct MarchShape {
  int ty = 0, tz = 0, tiles_y = 0, tiles_z = 0, ranges = 0;
  double cost = 0.0;
};
inline MarchShape march_shape(int nx, int ny, int nz, int columns, int interior, int side,
                              int slots, int line) {
  MarchShape best;
  // splits of the rows from the longest parts that fit, down to about a line
  const int first = (nz + interior - 1) / interior;
  for (int parts = first; parts <= (nz + 31) / 32 && parts < first + 64; ++parts) {
    const int tz = (nz + parts - 1) / parts, kz = (nz + tz - 1) / tz;
    const int pitch = kz == 1 ? tz : tz + 2;
    if (tz > interior || 3 * pitch > columns || (side && pitch > side) || pitch > 32767) continue;
    int ty = columns / pitch - 2;
    if (ty > interior / tz) ty = interior / tz;
    if (side && ty > side - 2) ty = side - 2;
    if (ty > ny) ty = ny;
    if (ty < 1) continue;
    int ky = (ny + ty - 1) / ty;
    ty = (ny + ky - 1) / ky;
    ky = (ny + ty - 1) / ty;
    const long long tiles = (long long)ky * kz;
    const double lines = (double)((tz + line - 1) / line);
    const double rows = (double)(ty + 2) * ky / ny * (kz == 1 ? 1.0 : (lines + 2.0) / lines);
    for (int r = 1; r <= nx; ++r) {
      const long long rounds = (tiles * r + slots - 1) / slots;
      if (r > 1 && rounds > 32) break;
      const int len = (nx + r - 1) / r;
      const double busy = (double)tiles * nx / ((double)rounds * slots * len);
      const double fixed = 0.75 * interior * (double)tiles / ((double)ny * nz);
      const double cost = (1.0 + (rows + fixed) * (len + 2) / len) / busy;
      if (best.ranges == 0 || cost < best.cost) best = MarchShape{ty, tz, ky, kz, r, cost};
    }
  }
  return best;
}

// Whether that tiling beats two one-step launches, from 15 to 21 shapes of at least
// 2^18 cells under 19 combinations of lattice, equilibrium, source, force and number
// format.  Below the limits the two-step kernel took 0.13 to 1.00 of the one-step
// kernel's time; above them up to 1.5 of it: the more a collision computes (a
// product equilibrium with a source, the exact-difference source's second
// equilibrium, FP64), the less the rim's second collision may cost.  D3Q19's
// one-step kernel is slow on small domains (64^3: 19.2 us a step, two-step 13.0;
// D3Q27: 12.6 and 12.7).  Tiles that fill less than half of the kernel's columns (2048 x
// 16 x 16) leave lanes idle.
inline double march_limit(bool fp64, bool q27, bool exact, bool source, bool difference) {
  if (fp64) return 4.9;
  if (exact && source) return 3.9;
  if (q27) return 6.1;
  return difference ? 5.3 : 13.0;
}
inline bool march_pays(const MarchShape& m, double cells, int interior, double limit) {
  return m.ranges > 0 && cells >= 262144.0 && 2 * m.ty * m.tz >= interior && m.cost <= limit;
}

// Tiling of the multi-step 2D kernel: rows of 16 cells (wide 0) or of 64 with the
// halo, tx x ty cells without it, up to `steps` steps in a launch (0: one step at a
// time is faster).  rows: rows of each width that a workgroup holds.  From 14 sizes
// from 32^2 to 2048^2 (a launch costs 2.5 us, a step 4.1 to 4.9 us with it on the
// small ones), five steps to a launch were the best of 3, 4, 5 and 7; time over the
// one-step kernel's, Ma3 with the Guo source in FP64 / FP32 / FP16, then the product
// equilibrium with the exact-difference source:
//   16-cell rows, 8 x 8 tiles, up to 256 of them (128^2: 0.46 / 0.32 / 0.34, 0.44 to
//   0.49), taller ones up to 24 x 8 (192^2: 0.57 / 0.36 / 0.37, 0.58 to 0.60); at 256^2
//   64-cell rows are the better ones (0.68 / 0.43 / 0.44 against 0.79 / 0.44 / 0.48);
//   64-cell rows: the tile whose row passes (eight wavefronts, 512 workgroups at once,
//   the rows shrinking with the steps) and launches cost least per step: 320^2, 8 rows:
//   0.56 / 0.41 / 0.40; 512^2, 16 rows: 0.81 / 0.55 / 0.78; 2048^2, all rows: 0.72 /
//   0.42 / 0.61, in FP64 with three steps (five: 0.79).  On domains of more than 512
//   tiles of 8 rows the product equilibrium gains in FP64 only (0.58 to 0.92; FP32
//   0.76 to 1.15, FP16 1.0 to 1.3).  (FP16 without its conversions' products takes
//   another 2 to 12 % less with Ma3.)
// Tiles narrower than half a row leave lanes idle.
struct TileShape {
  int wide = 0, steps = 0, tx = 0, ty = 0;
};
inline TileShape tile_shape(int nx, int ny, const int (&rows)[2], bool fp64, bool exact) {
  auto fit = [&](int wide, int steps, int tx) {
    TileShape m;
    const int halo = steps - 1, width = wide ? 64 : 16;
    m.wide = wide;
    m.ty = ny <= width ? ny : width - 2 * halo;
    m.tx = tx >= nx || halo > nx ? nx : tx;
    if (m.tx + (m.tx == nx ? 0 : 2 * halo) <= rows[wide] && 2 * m.ty >= width - 2 * halo)
      m.steps = steps;
    return m;
  };
  auto groups = [&](const TileShape& m) {
    return (long long)((nx + m.tx - 1) / m.tx) * ((ny + m.ty - 1) / m.ty);
  };
  if ((long long)nx * ny <= 49152)
    for (int tx : {8, 16, 24}) {
      const TileShape m = fit(0, 5, tx);
      if (m.steps && groups(m) <= 256) return m;
    }
  if (exact && !fp64 && groups(fit(1, 5, 8)) > 512) return TileShape{};
  TileShape best;
  double least = 0.0;
  for (int steps = 5; steps >= (fp64 ? 3 : 5); steps -= 2)
    for (int tx : {8, 16, 24, 32, rows[1] - 2 * (steps - 1)}) {
      const TileShape m = fit(1, steps, tx);
      if (!m.steps) continue;
      int passes = 0;
      for (int t = 1; t <= steps; ++t)
        passes += (m.tx + (m.tx == nx ? 0 : 2 * (steps - t)) + 7) / 8;
      // a launch takes as long as 2.5 row passes in FP64, 5 in FP32
      const double cost =
          ((double)((groups(m) + 511) / 512) * passes + (fp64 ? 2.5 : 5.0)) / steps;
      if (best.steps && cost >= least) continue;
      best = m;
      least = cost;
    }
  return best;
}

// Launches of at most `per` steps each for `steps` steps: as many, modulo two, as steps,
// so that the populations end in the lattice that one launch a step would leave them in.
inline int launches_of(int steps, int per) {
  const int n = steps / per + (steps % per != 0);
  return n + ((steps - n) & 1);
}
// Steps of the next of `launches` launches with `steps` left.
inline int steps_of_next(int steps, int launches) {
  return steps / launches + (steps % launches != 0);
}

}  // namespace lbm
