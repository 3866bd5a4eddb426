// fused_march.hpp -- two BGK steps of a 3D lattice in one pass over memory.
//
// The one-step kernels run at what the memory streams (D3Q19 256^3 FP32: 0.45 ms
// for the 2.55 GB that a step reads and writes), so the only way to a faster
// step is fewer bytes.  A workgroup owns a tile of y-z columns, extended by a
// rim of one column, and marches through the planes of an x range.  At plane x
// it pulls and collides the extended tile from the source lattice (step one),
// puts the populations that move within the plane into LDS, and gathers from
// there, column by column, the pulls of step two: those with c_x = -1 complete
// the cells of plane x - 1, those with c_x = 0 and +1 wait in registers for the
// cells of planes x and x + 1.  Completed cells collide and are stored, so that
// two steps read the lattice once (plus the rims) and write it once.
//
// The intermediate populations are rounded to the storage type and every cell
// collides as in the one-step kernels, so the result is that of two one-step
// launches to the bit.
//
// Tile: with the three populations that stay in their column held in
// registers, a column takes Q - 3 values of LDS, and the CU's 160 KB hold 2560
// columns of D3Q19 FP32.  Rows of the tile are whole rows of the domain where
// they fit (8 x 256 cells): the rim is then two rows, read a second time by the
// neighbours; a tile that splits the rows also fetches a whole cache line for
// each rim column (16 x 128 cells: 2.6 GB read for two steps against 1.5).  One
// workgroup of eight wavefronts has the whole CU, so that a lane has 256
// registers: each of its columns keeps Q populations waiting, and two columns
// have Q more in flight -- as soon as a column has collided, the pulls of the
// column after next are issued, across the end of the plane, and arrive while
// others collide.  (All four columns in flight: the compiler spills 20 registers
// of loads not yet there, whose waits cost a third of the time.)
//
// Measured, microseconds a step, one-step kernels -> this one: D3Q19 256^3 461 ->
// 257 (1.45 GB read and 1.28 GB written by a launch of 513 us, 5.3 TB/s; 64 % of
// the vector issue slots), D3Q27 193 x 161 x 130 Ma3 290 -> 129, product
// equilibrium 282 -> 152; FP64, one column a thread: D3Q19 192^3 422 -> 321, 171 x
// 150 x 133 257 -> 207 (60 % of the issue slots: before opposite populations shared
// their terms 246, with divisions by 6 and 24 304).  FP16 (D3Q27 384^3, waiting
// populations packed in pairs: 1162 against 1205, 72 % of the issue slots at half the
// bytes, but 192^3 1.01 to 1.21 and 64^3 2.2 times the one-step kernel's time) stays
// with the one-step kernels, and so does FP64 storage with FP32 arithmetic, whose
// kernels collide one population at a time: the pairwise form rounds its sums in
// another order, which FP64 populations show (1.7e-6 of them).
#pragma once

#include "fused_step.hpp"

namespace lbm {

// Threads, and the columns that the LDS holds: all of it, or (SIDE) beside force
// tables of kMarchSide rows and places for each component.
constexpr int kMarchThreads = 512, kMarchLds = 163840, kMarchSide = 264;
template <class L, class S, class C, bool SIDE>
constexpr int kMarchColumns = (kMarchLds - (SIDE ? 3 * kMarchSide * int(sizeof(C)) : 0)) /
                              ((L::dimQ - 3) * int(sizeof(S))) / 4 * 4;
// Interior columns per thread, and how many of them have pulls in flight.
template <class L, class S>
constexpr int kMarchUnits = sizeof(S) == 8 ? 1 : (L::dimQ > 19 ? 2 : 4);
template <class L, class S>
constexpr int kMarchAhead = kMarchUnits<L, S> == 1 ? 1 : 2;

// LDS slot of population i among those with (c_y, c_z) != 0, or -1.
template <class L, int i>
constexpr int march_slot() {
  if (L::C[i][1] == 0 && L::C[i][2] == 0) return -1;
  int k = 0;
  for (int j = 0; j < i; ++j)
    if (L::C[j][1] != 0 || L::C[j][2] != 0) ++k;
  return k;
}

// SIDE: forces that vary along y or z.
template <class L, class S, class C, int FS, int EQ, bool SH, bool SIDE>
__global__ void __launch_bounds__(kMarchThreads)
    __attribute__((amdgpu_waves_per_eu(2)))
    k_bgk_march(const StepArgs a, const MarchTiling m) {
  constexpr int Q = L::dimQ, U = kMarchUnits<L, S>, THREADS = kMarchThreads;
  constexpr int AHEAD = kMarchAhead<L, S>;
  static_assert(U % AHEAD == 0, "a plane's first columns find their registers free");
  constexpr int COLUMNS = kMarchColumns<L, S, C, SIDE>;
  __shared__ S lds[(Q - 3) * COLUMNS];
  __shared__ C side[SIDE ? 3 : 1][SIDE ? kMarchSide : 1];

  // tile and x range of the workgroup
  int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bz = b % m.tiles_z;
  b /= m.tiles_z;
  const int by = b % m.tiles_y, bx = b / m.tiles_y;
  const int y0 = by * m.ty, z0 = bz * m.tz;
  const int hy = min(m.ty, a.ny - y0), hz = min(m.tz, a.nz - z0);
  const int x0 = (int)((long long)bx * a.nx / m.ranges);
  const int x1 = (int)((long long)(bx + 1) * a.nx / m.ranges);
  // whole rows wrap around in the tile; parts of rows have a rim at both ends
  const bool whole = m.tiles_z == 1;
  const int rim_z = whole ? 0 : 1, pitch = m.tz + 2 * rim_z;

  // A column of the extended tile: row (0 and hy + 1 are rim) and place in the
  // row; -1 if the thread has none (it then reads row 1, place 1).
  auto column = [](int ey, int ez, bool active) { return active ? ey << 16 | ez : -1; };
  auto row_of = [](int c) { return c < 0 ? 1 : c >> 16; };
  auto place_of = [](int c) { return c < 0 ? 0 : c & 0xffff; };
  int own[U];
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const int t = threadIdx.x + k * THREADS;
    const int r = t / m.tz, z = t - r * m.tz;
    own[k] = column(r + 1, z + rim_z, r < hy && z < hz);
  }
  // rim column h: the rows above and below with their corners, then both ends
  const int rims = 2 * pitch + (whole ? 0 : 2 * hy);
  auto rim_column = [&](int h) {
    if (h < 2 * pitch) {
      const int r = h >= pitch ? 1 : 0, z = h - r * pitch;
      return column(r ? hy + 1 : 0, z, z < hz + 2 * rim_z);
    }
    const int k = h - 2 * pitch;
    return column(1 + (k >> 1), (k & 1) ? hz + 1 : 0, h < rims);
  };

  // Forces that vary along y or z, for the tile's rows and places; the others are
  // the same for a whole plane and are read as scalars.  (Read from memory at
  // each collision, they would wait behind the loads in flight.)
  if constexpr (SIDE) {
    for (int d = 0; d < 3; ++d) {
      const C* t = static_cast<const C*>(a.ftab[d]);
      if (!t || (a.fax[d] != 1 && a.fax[d] != 2)) continue;
      const bool along_y = a.fax[d] == 1;
      const int n = along_y ? hy + 2 : hz + 2 * rim_z;
      for (int e = threadIdx.x; e < n; e += THREADS)
        side[d][e] = t[along_y ? wrap_index(y0 + e - 1, a.ny)
                               : wrap_index(z0 + e - rim_z, a.nz)];
    }
    __syncthreads();
  }
  auto force_at = [&](int c, int x, C* F) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      typedef const __attribute__((address_space(4))) C* Scalar;
      const C* t = static_cast<const C*>(a.ftab[d]);
      F[d] = C(0);
      if (FS == SRC_ZERO || !t) continue;
      if (SIDE && a.fax[d] == 1)
        F[d] = side[SIDE ? d : 0][row_of(c)];
      else if (SIDE && a.fax[d] == 2)
        F[d] = side[SIDE ? d : 0][place_of(c)];
      else
        F[d] = ((Scalar)(unsigned long long)t)[a.fax[d] == 0 ? x : 0];
    }
  };

  const S* const src = static_cast<const S*>(a.src);
  S* const dst = static_cast<S*>(a.dst);
  const size_t plane = (size_t)a.ny * a.nz;

  // Step one's pulls of a column at plane x, as stored: scalar plane bases and
  // 32-bit byte offsets within the plane, formed anew for each plane (the empty
  // asm statement keeps the compiler from holding all of them for every column
  // across the loop).
  auto pull_column = [&](int c, int x_unwrapped, S (&f)[Q]) {
    const int x = wrap_index(x_unwrapped, a.nx);
    const int xm = x == 0 ? a.nx - 1 : x - 1, xp = x == a.nx - 1 ? 0 : x + 1;
    asm volatile("" : "+v"(c));
    const int y = wrap_index(y0 + row_of(c) - 1, a.ny);
    const int z = wrap_index(z0 + place_of(c) - rim_z, a.nz);
    const unsigned row = (unsigned)a.nz * (unsigned)sizeof(S);
    const unsigned ym = y == 0 ? a.ny - 1 : y - 1, yp = y == a.ny - 1 ? 0 : y + 1;
    const unsigned zm = z == 0 ? a.nz - 1 : z - 1, zp = z == a.nz - 1 ? 0 : z + 1;
    const unsigned rows[3] = {yp * row, (unsigned)y * row, ym * row};
    const unsigned cols[3] = {zp * (unsigned)sizeof(S), (unsigned)z * (unsigned)sizeof(S),
                              zm * (unsigned)sizeof(S)};
    static_for<Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr int cx = cel<L, i, 0>(), cy = cel<L, i, 1>(), cz = cel<L, i, 2>();
      const char* base = reinterpret_cast<const char*>(
          src + (size_t)i * (size_t)a.N + (size_t)(cx > 0 ? xm : (cx < 0 ? xp : x)) * plane);
      f[i] = *reinterpret_cast<const S*>(base + (rows[cy + 1] + cols[cz + 1]));
    });
  };

  // populations waiting for their cells: those with c_x = +1 for the next plane
  // to complete (wait) and the one after (ahead), those with c_x = 0 (wait)
  S wait[U][Q], ahead[U][Q];

  // The scheduling barriers keep each column's collision apart from the loads
  // around it.
  S f[AHEAD][Q];  // pulls in flight
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) pull_column(own[k], x0 - 1, f[k]);
  for (int x = x0 - 1; x <= x1; ++x) {
    const int xs = wrap_index(x, a.nx);
    S mine[U][3];  // the populations that stay in their column, by c_x + 1
    auto step_one = [&](int c, const S (&p)[Q], auto&& stays) {
      C F[3], rho, u[3];
      S* const to = lds + (row_of(c) * pitch + place_of(c));
      force_at(c, xs, F);
      bgk_collide_stored<L, S, C, FS, EQ, SH>(a, p, F, rho, u, [&](auto ic, S s) {
        constexpr int i = decltype(ic)::value, slot = march_slot<L, i>();
        if constexpr (slot >= 0) {
          if (c >= 0) to[slot * COLUMNS] = s;
        } else {
          stays(ic, s);
        }
      });
    };
    S fr[Q];
    int rim = rim_column(threadIdx.x);
    if (rim >= 0) pull_column(rim, x, fr);
#pragma unroll
    for (int k = 0; k < U; ++k) {
      __builtin_amdgcn_sched_barrier(0);
      step_one(own[k], f[k % AHEAD], [&](auto ic, S s) {
        mine[k][cel<L, decltype(ic)::value, 0>() + 1] = s;
      });
      __builtin_amdgcn_sched_barrier(0);
      if (k + AHEAD < U)
        pull_column(own[k + AHEAD], x, f[k % AHEAD]);
      else if (x < x1)
        pull_column(own[(k + AHEAD) % U], x + 1, f[k % AHEAD]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (rim >= 0) step_one(rim, fr, [](auto, S) {});
    for (int h = threadIdx.x + THREADS; h < rims; h += THREADS) {
      rim = rim_column(h);
      pull_column(rim, x, fr);
      step_one(rim, fr, [](auto, S) {});
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < U; ++k) {
      __builtin_amdgcn_sched_barrier(0);
      S g[Q];
      int c = own[k];
      asm volatile("" : "+v"(c));
      const int r = row_of(c) * pitch, z = place_of(c);
      const int zm = whole && z == 0 ? hz - 1 : max(z - 1, 0);
      const int zp = whole && z == hz - 1 ? 0 : min(z + 1, pitch - 1);
      const int rows[3] = {r + pitch, r, r - pitch}, places[3] = {zp, z, zm};
      static_for<Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value, slot = march_slot<L, i>();
        if constexpr (slot >= 0)
          g[i] = lds[slot * COLUMNS + rows[cel<L, i, 1>() + 1] + places[cel<L, i, 2>() + 1]];
        else
          g[i] = mine[k][cel<L, i, 0>() + 1];
      });
      if (x > x0 && c >= 0) {
        // plane x - 1 is complete
        const int xd = x - 1;
        S h[Q];
        C F[3], rho, u[3];
        static_for<Q>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          h[i] = cel<L, i, 0>() < 0 ? g[i] : wait[k][i];
        });
        force_at(c, xd, F);
        const unsigned cell = (unsigned)((y0 + row_of(c) - 1) * a.nz + (z0 + z - rim_z)) *
                              (unsigned)sizeof(S);
        bgk_collide_stored<L, S, C, FS, EQ, SH>(a, h, F, rho, u, [&](auto ic, S v) {
          constexpr int i = decltype(ic)::value;
          char* base = reinterpret_cast<char*>(dst + (size_t)i * (size_t)a.N + (size_t)xd * plane);
          __builtin_nontemporal_store(v, reinterpret_cast<S*>(base + cell));
        });
      }
      static_for<Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (cel<L, i, 0>() == 0) wait[k][i] = g[i];
        if constexpr (cel<L, i, 0>() > 0) {
          wait[k][i] = ahead[k][i];
          ahead[k][i] = g[i];
        }
      });
    }
    __syncthreads();
  }
}

}  // namespace lbm
