// fused_tile.hpp -- several BGK steps of a 2D lattice in one launch.
//
// A step of a small lattice is a launch and little else (D2Q9 128^2: 3.4 us a step,
// 2.5 of them the launch), and one of a large lattice runs at what the memory streams
// (2048^2 FP32: 55 us).  A workgroup takes a tile with a halo through several steps
// in LDS: the first one pulls from memory, the halo shrinks by a cell a step, and the
// last one stores.  Tiles recompute each other's halos.
//
// The populations stay in place, one copy of them: even steps read a cell's own
// slots and write the result of population i into the slot of the opposite one, odd
// steps read those at the neighbours that they come from and write to the neighbours
// that they go to.  Either way a cell writes the slots that it has read and nobody
// else touches, so one barrier a step is enough, and each parity (and the first and
// the last step) is compiled for itself.  A lane keeps its place in the rows, so that
// its memory offsets, its LDS neighbours and forces along y are found once.
//
// Rounding is that of one step at a time, to the bit: every step goes through the
// storage type and the one-step kernels' collision.
//
// Measured, microseconds a step, one-step kernel -> this one: 128^2 FP64 3.4 -> 1.8, FP32
// and FP16 3.7 -> 1.2 (one handle, a hundred steps a call: launch, load and the dependent
// instructions of one wavefront a SIMD; four handles on streams of their own overlap, 1.1
// and 0.6 each); 2048^2 FP32 55 -> 22, FP64 113 -> 74, FP16 34 -> 21: bound by the vector
// instructions (five steps with a force field in FP32, 149 us: 87 % of the issue slots, a
// quarter of the work in halos; with the parities chosen at run time it took 12 % longer).
#pragma once

#include "fused_step.hpp"

namespace lbm {

// Threads, LDS (two workgroups to a CU) and the rows of W cells that it holds.
constexpr int kTileThreads = 512, kTileLds = 81920;
template <class L, class S, int W>
constexpr int kTileRows = kTileLds / (L::dimQ * int(sizeof(S)) * W);

// W: cells in a row of the tile with its halo, a power of two; a wavefront has 64 / W
// rows.
template <class L, class S, class C, int FS, int EQ, bool SH, int W>
__global__ void __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(4)))
    k_bgk_tile(const StepArgs a, const Tile2D m, int FSX) {
  constexpr int Q = L::dimQ, ROWS = kTileRows<L, S, W>, STRIDE = kTileThreads / W;
  constexpr int B = int(sizeof(S));
  __shared__ S lds[Q * ROWS * W];

  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = b / m.tiles_y, by = b - bx * m.tiles_y;
  const int x0 = bx * m.tx, y0 = by * m.ty;
  const int hx = min(m.tx, a.nx - x0), hy = min(m.ty, a.ny - y0);
  // An axis that the tile covers whole wraps around in LDS; the other has a halo of
  // one cell for each step but the first, which pulls from memory.
  const bool whole_x = m.tx == a.nx, whole_y = m.ty == a.ny;
  const int halo_x = whole_x ? 0 : m.steps - 1, halo_y = whole_y ? 0 : m.steps - 1;
  const int rows = hx + 2 * halo_x, cols = hy + 2 * halo_y;

  // The thread's place in its rows (those beyond the tile idle at the last one) and
  // its first row, the same for a wavefront of one row.
  const int place = threadIdx.x % W, c = min(place, cols - 1);
  int row0 = threadIdx.x / W;
  if constexpr (W == 64) row0 = __builtin_amdgcn_readfirstlane(row0);
  const int y = wrap_index(y0 + c - halo_y, a.ny);
  const unsigned ys[3] = {(unsigned)(y == a.ny - 1 ? 0 : y + 1) * B, (unsigned)y * B,
                          (unsigned)(y == 0 ? a.ny - 1 : y - 1) * B};
  const int cm = c == 0 ? cols - 1 : c - 1, cp = c == cols - 1 ? 0 : c + 1;

  // Force components that do not vary along x, once for all steps.
  C held[2] = {C(0), C(0)};
  for (int d = 0; d < 2; ++d) {
    const C* t = static_cast<const C*>(a.ftab[d]);
    if (FS != SRC_ZERO && t && (a.fax[d] == 1 || a.fax[d] == 3)) held[d] = t[a.fax[d] == 1 ? y : 0];
  }

  const S* const src = static_cast<const S*>(a.src);
  S* const dst = static_cast<S*>(a.dst);
  // The others, of row r; read for the row after, ahead of its use.
  auto force_of = [&](int r, C* F) {
    int x = wrap_index(x0 + min(r, rows - 1) - halo_x, a.nx);
    if constexpr (W == 64) x = __builtin_amdgcn_readfirstlane(x);
    for (int d = 0; d < 2; ++d) {
      const C* t = static_cast<const C*>(a.ftab[d]);
      F[d] = held[d];
      if (FS != SRC_ZERO && t && a.fax[d] == 0) F[d] = t[x];
      if (FS != SRC_ZERO && t && a.fax[d] == 4) F[d] = t[x * a.ny + y];
    }
  };
  C ahead[2];
  force_of(row0, ahead);

  auto step = [&](int t, auto first_c, auto odd_c, auto last_c) {
    constexpr bool first = decltype(first_c)::value, odd = decltype(odd_c)::value,
                   last = decltype(last_c)::value;
    // cells that this step completes: the halo shrinks by one cell a step
    const int in_x = whole_x ? 0 : t - 1, in_y = whole_y ? 0 : t - 1;
    const bool active = place >= in_y && place < cols - in_y;
    // Slot of population i: even steps read the cell's own and leave the result
    // of i in the opposite one; odd steps find it there, at the neighbour it comes
    // from, and put theirs where they go -- into the slots that they have read.
    const int cc[3] = {odd ? cm : c, c, odd ? cp : c};
    for (int r = in_x + row0; r < rows - in_x; r += STRIDE) {
      C F[3] = {ahead[0], ahead[1], C(0)};
      force_of(r + STRIDE < rows - in_x ? r + STRIDE : in_x + (whole_x ? 0 : 1) + row0, ahead);
      if (!active) continue;
      int x = wrap_index(x0 + r - halo_x, a.nx);
      if constexpr (W == 64) x = __builtin_amdgcn_readfirstlane(x);
      const int rr[3] = {odd ? (r == 0 ? rows - 1 : r - 1) : r, r,
                         odd ? (r == rows - 1 ? 0 : r + 1) : r};
      int at[Q];
      static_for<Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value, o = opposite<L, i>();
        at[i] = ((odd ? o : i) * ROWS + rr[1 - cel<L, i, 0>()]) * W + cc[1 - cel<L, i, 1>()];
      });
      S p[Q];
      if constexpr (first) {
        const int xs[3] = {x == a.nx - 1 ? 0 : x + 1, x, x == 0 ? a.nx - 1 : x - 1};
        static_for<Q>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          const S* row = src + (size_t)i * (size_t)a.N;
          unsigned at = ys[cel<L, i, 1>() + 1];
          if constexpr (W == 64)
            row += (size_t)xs[cel<L, i, 0>() + 1] * a.ny;
          else
            at += (unsigned)xs[cel<L, i, 0>() + 1] * (unsigned)a.ny * B;
          p[i] = *reinterpret_cast<const S*>(reinterpret_cast<const char*>(row) + at);
        });
      } else {
        static_for<Q>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          p[i] = lds[at[i]];
        });
      }
      C rho, u[3];
      S v[Q];
      bgk_collide_stored<L, S, C, FS, EQ, SH>(a, p, F, rho, u, [&](auto ic, S s) {
        v[decltype(ic)::value] = s;
      });
      if constexpr (last) {
        static_for<Q>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          S* row = dst + (size_t)i * (size_t)a.N;
          unsigned at = ys[1];
          if constexpr (W == 64)
            row += (size_t)x * a.ny;
          else
            at += (unsigned)x * (unsigned)a.ny * B;
          *reinterpret_cast<S*>(reinterpret_cast<char*>(row) + at) = v[i];
        });
        if (a.store) {
          if constexpr (FS == SRC_ZERO) {  // the stored force is the configured one
            CellPos pos;
            pos.x = x;
            pos.y = y;
            pos.z = 0;
            force_of_cell<L, C>(a, pos, F);
          }
          store_fields<L, C>(a, x * a.ny + y, FSX, rho, u, F, 2.0);
        }
      } else {
        static_for<Q>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          lds[at[opposite<L, i>()]] = v[i];
        });
      }
    }
    __syncthreads();
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  step(1, yes, no, no);
  for (int t = 2; t < m.steps; ++t) {
    if (t & 1) step(t, no, no, no);
    else step(t, no, yes, no);
  }
  if (m.steps & 1) step(m.steps, no, no, yes);
  else step(m.steps, no, yes, yes);
}

}  // namespace lbm
