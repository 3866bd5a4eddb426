// fused_step.hpp -- BGK and entropic (ELBM) fused step kernels.
//
// Template parameters:
//   L   Lattice<...> descriptor              (Lattice.h)
//   S   storage type of populations          double | float | _Float16
//   C   compute type                         double | float
//   FS  collision source                     SRC_ZERO | SRC_GUO | SRC_EDM
//   EQ  equilibrium                          TruncationMa3 | Exact
//   SH  populations stored as f_i - w_i
// When C is double and SH is false every operator runs in the reference's
// operation order (parity build); otherwise the shifted/FMA form is used.
#pragma once

#include "entropy_series.hpp"
#include "mlp.hpp"
#include "step_kernels.hpp"

namespace lbm {

template <class L, class C>
__device__ __forceinline__ void store_fields(const StepArgs& a, int cell, int FS,
                                             C rho, const C* u, const C* F,
                                             double alpha) {
  a.rho_out[cell] = double(rho);
  if (FS == (int)ForcingSchemeType::None) {
    // ForcingScheme<None>::calculateHydrodynamicVelocity (ForcingScheme.h:50-57)
    for (int d = 0; d < L::dimD; ++d) a.uh_out[(size_t)d * a.N + cell] = double(u[d]);
  } else {
    // Generic: u + 0.5 / rho * F (ForcingScheme.h:26-33)
    const C h = C(0.5) / rho;
    for (int d = 0; d < L::dimD; ++d) {
      C v;
      if constexpr (std::is_same_v<C, float>) v = fmaf(F[d], h, u[d]);  // the same in each kernel
      else v = u[d] + F[d] * h;
      a.uh_out[(size_t)d * a.N + cell] = double(v);
    }
  }
  if (a.alpha_out) a.alpha_out[cell] = alpha;
  if (a.F_out)
    for (int d = 0; d < L::dimD; ++d) a.F_out[(size_t)d * a.N + cell] = double(F[d]);
}

// Index of the population with the opposite velocity.
template <class L, int i>
constexpr int opposite() {
  for (int j = 0; j < L::dimQ; ++j) {
    bool opp = true;
    for (int d = 0; d < L::dimD; ++d) opp = opp && L::C[j][d] == -L::C[i][d];
    if (opp) return j;
  }
  return -1;
}

// The single-precision BGK collision of one cell (Collision.h:134-151), two opposite
// populations at a time: they share every term of the Ma3 equilibrium and of the
// source up to the sign of the odd part (the two-step kernel on D3Q19 256^3 with the
// Guo source: 172 million vector instructions a launch instead of 248, addresses
// included).  Every kernel that one handle's steps may go through takes its arithmetic
// from here, so that a result does not depend on how steps are split over launches and
// calls.  For that each kernel has to round the same way, and the compiler, which in
// these files fuses any product that feeds a sum (pragmas or not), must have no choice:
// every fused operation is written out, and no rounded product is added or subtracted
// except as the addend of one.  SC: populations are in their FP16 storage scales
// (powers of two, so that the products with them, folded into the sums' and the results'
// factors, round nothing).
//
// The two rates add up to 1 exactly, the larger one in magnitude being the rounded one:
// rounded each by itself, omega_f + omega_eq lost mass and momentum at every collision,
// the same share in every cell, which was most of the result's error.  (EDM: omega_f (f -
// feq) + feq(v), for which any omega_f keeps them.)  The velocity is the rounded quotient
// (two operations a component: 0.2% of the 3D kernel's time, 1% of the 2D one's).  Error
// against 64 bits after 15 steps of noise on D3Q19 64^3 with tau 0.55 / 0.6624 / 0.8 / 1.3
// (relative 2-norm of f - w, Guo): 6.0e-7 / 2.7e-7 / 2.7e-7 / 1.5e-7; with each rate rounded
// and the product with 1 / rho 10e-7 / 6.8e-7 / 4.3e-7 / 4.4e-7; one population at a time,
// as it was before the pairs, 9.9e-7 / 5.2e-7 / 4.7e-7 / 5.1e-7; D2Q9 96^2, 2000 steps, tau
// 0.53: 2.8e-5, 8.3e-5 and 7.4e-5.

// Ma3: t(cu) = base + rho (P(cu) - 1), P the polynomial (Equilibrium.h:17-33), times
// `scale`, split into its even part e0 + cu^2 (e1 + e2 cu^2) and its odd part
// cu (o0 + o1 cu^2).
struct Ma3Split {
  float e0, e1, e2, o0, o1;
  __device__ __forceinline__ void set(float scale, float rho, float base, float u2) {
    const float sr = scale * rho;
    e0 = fmaf(sr, u2 * fmaf(1.125f, u2, -1.5f), scale * base);
    e1 = sr * fmaf(-6.75f, u2, 4.5f);
    e2 = sr * 3.375f;
    o0 = sr * fmaf(-4.5f, u2, 3.0f);
    o1 = sr * 4.5f;
  }
  __device__ __forceinline__ float even(float q, float more) const {
    return fmaf(q, fmaf(q, e2, e1), more);
  }
  __device__ __forceinline__ float odd(float q) const { return fmaf(q, o1, o0); }
};

// Product equilibrium: ExactShifted's factors e[d][c + 1] = phi_d^c - 1 with its fused
// operations written out, and s = sqrt(1 + 3 v^2) taken as 1 + sm1 throughout: half of the
// square roots just above 1 lie just below the middle of two floats and round down, which
// shows in the momentum (1e-8 of it a collision).
template <class L>
struct ExactTerms {
  float e[3][3];
  __device__ __forceinline__ void set(const float* u) {
    for (int d = 0; d < L::dimD; ++d) {
      const float v = u[d], t = 3.0f * v;
      const float sm1 = (t * v) / (1.0f + sqrtf(fmaf(t, v, 1.0f)));
      e[d][1] = -sm1;
      e[d][2] = fmaf(v, fmaf(-2.0f, sm1, 3.0f), fmaf(2.0f, sm1, -(t * v))) / (1.0f - v);
      e[d][0] = fmaf(v, sm1, fmaf(-3.0f, v, -2.0f * sm1)) / (fmaf(2.0f, v, 1.0f) + sm1);
    }
  }
  template <int i>
  __device__ __forceinline__ float p() const {
    const float e0 = e[0][cel<L, i, 0>() + 1], e1 = e[1][cel<L, i, 1>() + 1];
    float t = fmaf(e0, e1, e0 + e1);
    if constexpr (L::dimD == 3) {
      const float e2 = e[2][cel<L, i, 2>() + 1];
      t = fmaf(t, e2, t + e2);
    }
    return t;
  }
};

template <class L, int FS, int EQ, bool SH, bool SC>
struct PairCollision {
  static constexpr bool MA3 = EQ == (int)EquilibriumType::TruncationMa3;
  float rho, u[3];   // the moments
  float of, oe, sum; // sum: drho (SH) or rho
  float v[3];        // EDM: u + F / rho
  float G[3], uG;    // Guo: w (c.G - u.G + 3 (c.u) (c.G)), G = 3 (1 - 1 / (2 tau)) F
                     // (ForcingScheme.h:99-117)
  Ma3Split E, E2;
  ExactTerms<L> X, X2;

  template <int i>
  static constexpr float scale_of() {
    return SC ? float(kHalfScale<L, i>) : 1.0f;
  }

  __device__ __forceinline__ void set(const StepArgs& a, const float* f, const float* F) {
    constexpr int Q = L::dimQ, D = L::dimD;
    // 1 - oe is exact from 0.5 to 2, and then 1 - of from 0.5 to 1
    oe = float(a.omega_eq);
    of = oe < 0.5f ? float(a.omega_f) : 1.0f - oe;
    oe = oe < 0.5f ? 1.0f - of : oe;
    sum = f[0] * (1.0f / scale_of<0>());
    float j[3] = {0.0f, 0.0f, 0.0f};
    static_for<Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value, o = opposite<L, i>();
      if constexpr (i < o) {
        constexpr float inv = 1.0f / scale_of<i>();
        sum = SC ? fmaf(f[i] + f[o], inv, sum) : sum + (f[i] + f[o]);
        const float d = SC ? (f[i] - f[o]) * inv : f[i] - f[o];
        static_for<D>([&](auto dc) {
          constexpr int c = L::C[i][decltype(dc)::value];
          if constexpr (c > 0) j[decltype(dc)::value] += d;
          if constexpr (c < 0) j[decltype(dc)::value] -= d;
        });
      }
    });
    rho = SH ? 1.0f + sum : sum;
    const float r0 = __builtin_amdgcn_rcpf(rho);
    const float rr = fmaf(r0, fmaf(-rho, r0, 1.0f), r0);  // see moments_shifted_scaled
    u[2] = v[2] = 0.0f;
    for (int d = 0; d < D; ++d) {
      u[d] = j[d] * rr;
      // 1 / rho of a density below 1 rounds up more often than down: the quotient itself
      // (not for FP16 populations, whose own rounding is a thousand times that)
      if constexpr (!SC) u[d] = fmaf(fmaf(-rho, u[d], j[d]), rr, u[d]);
      asm("" : "+v"(u[d]));  // no longer a product: c.u adds them
    }
    if constexpr (FS == SRC_EDM)  // feq(rho, u + F / rho) - feq (ForcingScheme.h:184-197)
      for (int d = 0; d < D; ++d) v[d] = fmaf(F[d], rr, u[d]);
    uG = 0.0f;
    if constexpr (FS == SRC_GUO) {
      const float g = float(3.0 * a.guo_coef);
      // uG summed by itself: taken from E.e0 term by term, its roundings moved the mean
      // density by 1e-12 a step, always one way
      for (int d = 0; d < D; ++d) {
        G[d] = g * F[d];
        asm("" : "+v"(G[d]));  // likewise
        uG = fmaf(u[d], G[d], uG);
      }
    }
    if constexpr (MA3) {
      auto square = [](const float* w) {
        float s = w[0] * w[0];
        for (int d = 1; d < D; ++d) s = fmaf(w[d], w[d], s);
        return s;
      };
      E.set(FS == SRC_EDM ? -of : oe, rho, sum, square(u));
      if constexpr (FS == SRC_GUO) E.e0 -= uG;
      if constexpr (FS == SRC_EDM) {
        E2.set(1.0f, rho, sum, square(v));
        E.e0 += E2.e0;
      }
    } else {
      X.set(u);
      if constexpr (FS == SRC_EDM) X2.set(v);
    }
  }

  // Product equilibrium: omega_eq feq_i / w_i (less omega_eq if SH) and the source over
  // w_i, for EDM -omega_f feq_i(u) / w_i + feq_i(v) / w_i.
  template <int i>
  __device__ __forceinline__ float exact(float source) const {
    const float t = fmaf(rho, X.template p<i>(), sum);
    if constexpr (FS == SRC_EDM) return fmaf(-of, t, fmaf(rho, X2.template p<i>(), sum));
    else return fmaf(oe, t, source);
  }

  // Population 0 and the pair i, opposite<L, i>(): pulled to post-collision.
  __device__ __forceinline__ float rest(float f) const {
    constexpr float w = float(L::W[0]) * scale_of<0>();
    if constexpr (MA3) return fmaf(w, E.e0, of * f);
    else return fmaf(w, exact<0>(-uG), of * f);
  }
  template <int i>
  __device__ __forceinline__ void pair(float fi, float fo, float& to_i, float& to_o) const {
    constexpr int o = opposite<L, i>();
    constexpr float w = float(L::W[i]) * scale_of<i>();
    const float cu = cdot<L, i>(u);
    float cG = 0.0f;
    if constexpr (FS == SRC_GUO) cG = cdot<L, i>(G);
    float ti, to;
    if constexpr (MA3) {
      const float q = cu * cu;
      float even = E.even(q, E.e0);
      if constexpr (FS == SRC_ZERO) {
        const float odd = E.odd(q);
        ti = fmaf(cu, odd, even);
        to = fmaf(-cu, odd, even);
      } else {
        float odd;
        if constexpr (FS == SRC_GUO) {
          even = fmaf(3.0f * cu, cG, even);
          odd = fmaf(cu, E.odd(q), cG);
        } else {
          const float cv = cdot<L, i>(v), r = cv * cv;
          even = E2.even(r, even);
          odd = fmaf(cu, E.odd(q), cv * E2.odd(r));
        }
        ti = even + odd;
        to = even - odd;
      }
    } else if constexpr (FS == SRC_GUO) {
      const float even = fmaf(3.0f * cu, cG, -uG);
      ti = exact<i>(even + cG);
      to = exact<o>(even - cG);
    } else {
      ti = exact<i>(0.0f);
      to = exact<o>(0.0f);
    }
    to_i = fmaf(w, ti, of * fi);
    to_o = fmaf(w, to, of * fo);
  }
};

// BGK collision of one cell (Collision.h:134-151): f the pulled populations, F the
// force.  emit(i, v) takes the post-collision populations in order, v in the
// compute type (f_i - w_i when SH); rho and u are the moments.
template <class L, class C, int FS, int EQ, bool SH, class EMIT>
__device__ __forceinline__ void bgk_collide(const StepArgs& a, const C* f, const C* F, C& rho,
                                            C* u, EMIT&& emit) {
  constexpr int Q = L::dimQ;
  constexpr bool REF = std::is_same_v<C, double> && !SH;
  const C of = C(a.omega_f), oe = C(a.omega_eq), gc = C(a.guo_coef);
  u[0] = u[1] = u[2] = C(0);
  C u2;
  if constexpr (REF) {
    // calculateMoments (Collision.h:72-79)
    moments_ref<L>(f, rho, u, u2);
    const RefEquilibrium<L, EQ, C> E(rho, u, u2);
    C v[3] = {C(0), C(0), C(0)}, v2 = C(0);
    if constexpr (FS == SRC_EDM) {
      // ExactDifferenceMethod source: feq(rho, u + F / rho) - feq (ForcingScheme.h:184-197)
      const C k = C(1.0) / rho;
      for (int d = 0; d < L::dimD; ++d) v[d] = u[d] + F[d] * k;
      v2 = v[0] * v[0];
      for (int d = 1; d < L::dimD; ++d) v2 += v[d] * v[d];
    }
    const RefEquilibrium<L, EQ, C> E2(rho, v, v2);
    auto relax = [&](auto ic, C fe, C fe2) {
      constexpr int i = decltype(ic)::value;
      C s = C(0);
      if constexpr (FS == SRC_GUO) s = guo_ref<L, i>(gc, u, F);
      if constexpr (FS == SRC_EDM) s = fe2 - fe;
      emit(ic, of * f[i] + oe * fe + s);
    };
    static_for<Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value, o = opposite<L, i>();
      if constexpr (EQ != (int)EquilibriumType::TruncationMa3 || i == o) {
        relax(ic, E.template feq<i>(), FS == SRC_EDM ? E2.template feq<i>() : C(0));
      } else if constexpr (i < o) {
        C fe, fo, ge = C(0), go = C(0);
        feq_ma3_ref_pair<L, i>(rho, u, u2, fe, fo);
        if constexpr (FS == SRC_EDM) feq_ma3_ref_pair<L, i>(rho, v, v2, ge, go);
        relax(ic, fe, ge);
        relax(std::integral_constant<int, o>{}, fo, go);
      }
    });
  } else {
    C drho;
    if constexpr (SH) {
      moments_shifted<L>(f, drho, rho, u, u2);
    } else {
      moments_ref<L>(f, rho, u, u2);
      drho = rho - C(1);
    }
    const FastEquilibrium<L, EQ, C> E(u, u2);
    C v[3] = {C(0), C(0), C(0)}, v2 = C(0);
    if constexpr (FS == SRC_EDM) {
      const C k = C(1) / rho;
      for (int d = 0; d < L::dimD; ++d) v[d] = u[d] + F[d] * k;
      v2 = v[0] * v[0];
      for (int d = 1; d < L::dimD; ++d) v2 += v[d] * v[d];
    }
    const FastEquilibrium<L, EQ, C> E2(v, v2);
    C uF = u[0] * F[0];
    for (int d = 1; d < L::dimD; ++d) uF += u[d] * F[d];
    static_for<Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const C w = C(L::W[i]);
      const C p = E.template p<i>();
      // feq_i in the storage representation: w (drho + rho p) when shifted.
      const C eq = SH ? w * (drho + rho * p) : w * rho * (C(1) + p);
      C s = C(0);
      if constexpr (FS == SRC_GUO) {
        const C cF = cdot<L, i>(F);
        const C cu = cdot<L, i>(u);
        s = (C(3) * gc * w) * (cF - uF + C(3) * cu * cF);
      }
      if constexpr (FS == SRC_EDM) s = rho * w * (E2.template p<i>() - p);
      emit(ic, of * f[i] + oe * eq + s);
    });
  }
}

// Whether a number format has kernels of several steps (instantiate.hpp registers them
// by this), and whether its collisions therefore take the pairwise form in every kernel.
template <class L, class S, class C>
constexpr bool kSeveralSteps = L::dimD == 3 ? std::is_same_v<S, C> : sizeof(S) <= sizeof(C);
template <class L, class S, class C>
constexpr bool kPairs = std::is_same_v<C, float> && kSeveralSteps<L, S, C>;

// Stored populations to stored ones; emit(i, s) takes them, s in the storage type.  FP16
// populations of the pairwise form stay in their storage scales (D2Q9 2000^2, Guo: 23.8
// -> 21.3 us a step, 128^2 3% less, for two products a population less).  ORDERED: in the
// order of the populations, for kernels that wait for memory (D3Q27 193 x 161 x 130, one
// step, Guo with the product equilibrium: 269 us, 287 with each pair stored at once and
// 298 with all at the end; the compiler shares a pair's terms or forms them twice).
template <class L, class S, class C, int FS, int EQ, bool SH, bool ORDERED = false, class EMIT>
__device__ __forceinline__ void bgk_collide_stored(const StepArgs& a, const S* p, const C* F,
                                                   C& rho, C* u, EMIT&& emit) {
  constexpr bool SC = kPairs<L, S, C> && std::is_same_v<S, _Float16>;
  C f[L::dimQ];
  static_for<L::dimQ>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    f[i] = SC ? C(p[i]) : to_compute<L, i, S, C>(p[i]);
    // converted once, not again in each operation (mixed-precision ones are slower)
    if constexpr (SC) asm("" : "+v"(f[i]));
  });
  auto stored = [&](auto ic, C v) {
    constexpr int i = decltype(ic)::value;
    emit(ic, SC ? S(v) : to_storage<L, i, S, C>(v));
  };
  if constexpr (kPairs<L, S, C>) {
    PairCollision<L, FS, EQ, SH, SC> cell;
    cell.set(a, f, F);
    rho = cell.rho;
    for (int d = 0; d < 3; ++d) u[d] = cell.u[d];
    stored(std::integral_constant<int, 0>{}, cell.rest(f[0]));
    static_for<L::dimQ>([&](auto ic) {
      constexpr int i = decltype(ic)::value, o = opposite<L, i>();
      float vi, vo;
      if constexpr (ORDERED && i != o) {
        if constexpr (i < o) cell.template pair<i>(f[i], f[o], vi, vo);
        else cell.template pair<o>(f[o], f[i], vo, vi);
        stored(ic, vi);
      } else if constexpr (i < o) {
        cell.template pair<i>(f[i], f[o], vi, vo);
        stored(ic, vi);
        stored(std::integral_constant<int, o>{}, vo);
      }
    });
  } else {
    bgk_collide<L, C, FS, EQ, SH>(a, f, F, rho, u, stored);
  }
}

template <class L, class S, class C, int FS, int EQ, bool SH, int BLOCK, bool NT>
__global__ void __launch_bounds__(BLOCK) k_bgk(const StepArgs a, int FSX) {
  constexpr int Q = L::dimQ;
  const CellPos c = cell_of_thread<L, BLOCK>(a);
  if (!c.active) return;
  const int cell = self_index<L>(a, c);
  S* __restrict__ dst = static_cast<S*>(a.dst);

  S f[Q];
  pull_stored<L, S, NT>(a, c, f);
  C F[3];
  force_of_cell<L, C>(a, c, F);
  C rho, u[3];
  bgk_collide_stored<L, S, C, FS, EQ, SH, true>(a, f, F, rho, u, [&](auto ic, S v) {
    constexpr int i = decltype(ic)::value;
    __builtin_nontemporal_store(v, dst + (size_t)i * a.N + cell);
  });
  if (a.store) store_fields<L, C>(a, cell, FSX, rho, u, F, 2.0);
}

// ---- entropic collision ------------------------------------------------------

// FP64 view of one cell's pulled populations f and non-equilibrium parts n,
// held in the compute type C (f stored as f - w when SH).  Values are
// converted at each use, so the alpha solve keeps no FP64 copies of them
// (exact for C = double: the view then returns the stored values).
template <class L, class C, bool SH>
struct Fp64View {
  const C* fs;
  const C* ns;
  template <int i>
  __device__ __forceinline__ double f() const {
    return SH ? double(fs[i]) + L::W[i] : double(fs[i]);
  }
  template <int i>
  __device__ __forceinline__ double n() const {
    return double(ns[i]);
  }
  // The same values, converted afresh at each use: the empty asm statement
  // on the stored value keeps the compiler from hoisting the conversions out
  // of an iteration loop, which would hold 2Q doubles live across it.
  template <int i>
  __device__ __forceinline__ double f_fresh() const {
    C v = fs[i];
    asm volatile("" : "+v"(v));
    return SH ? double(v) + L::W[i] : double(v);
  }
  template <int i>
  __device__ __forceinline__ double n_fresh() const {
    C v = ns[i];
    asm volatile("" : "+v"(v));
    return double(v);
  }
  // f - w, and the non-equilibrium part in single precision.
  template <int i>
  __device__ __forceinline__ double shifted() const {
    return SH ? double(fs[i]) : double(fs[i]) - L::W[i];
  }
  template <int i>
  __device__ __forceinline__ float n32() const {
    return float(ns[i]);
  }
};

// The parity build's deviation test (Collision.h:284-303), with the
// reference's divisions.
template <class L, class V>
__device__ __forceinline__ bool small_deviation_ref(const V& p) {
  bool small = true;
  static_for<L::dimQ>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const double dev = fabs(p.template n<i>()) / p.template f<i>();
    if (dev > 1.0e-3) small = false;
  });
  return small;
}

// alphaMax (Collision.h:305-326).  True when it is below 2: the cell then
// takes alpha = 0.95 alphaMax (Collision.h:365-367) and needs no root.
// REFDIV keeps the reference's divisions; otherwise the smallest ratio is
// found by cross-multiplied comparisons (num / den < 2.5 tracked as a pair)
// and one division at the end instead of Q: the products round, so two ratios
// within an ulp may be ordered either way, which moves alphaMax by at most an
// ulp.
template <class L, bool REFDIV, class V>
__device__ __forceinline__ bool alpha_capped(const V& p, double& alpha, double& amax) {
  amax = 2.5;
  if constexpr (REFDIV) {
    static_for<L::dimQ>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const double fi = p.template f<i>(), ni = p.template n<i>();
      if (ni > 0) {
        const double t = fabs(fi) / ni;
        if (t < amax) amax = t;
      }
    });
  } else {
    double num = 2.5, den = 1.0;
    static_for<L::dimQ>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const double fi = fabs(p.template f_fresh<i>()), ni = p.template n_fresh<i>();
      if (ni > 0 && fi * den < num * ni) {
        num = fi;
        den = ni;
      }
    });
    if (den != 1.0 || num != 2.5) amax = num / den;
  }
  if (amax < 2.) {
    alpha = 0.95 * amax;
    return true;
  }
  return false;
}

// Newton on the entropy equation term by term, one library logarithm per
// population and iterate: the whole solve of the parity build, and of the
// cells beyond the power-sum series (entropy_series.hpp) in the others.
//  * tol == 0: the reference Newton-Raphson (EntropicStep.h:111-140 via
//    solveAlpha, Collision.h:328-349): warm start, |step| <= 1e-8, at most 50
//    iterations, the iterate before the last step is returned, alpha = 2 when
//    it fails or leaves (1, alphaMax).
//  * RESIDUAL: the same iteration stopped at |G| <= tol.  Like the reference's
//    loop it bounds alpha only at convergence: an iterate where a logarithm is
//    undefined (G is NaN there) or at or below 0 (from where the reference
//    converges to the trivial root) ends in the fallback alpha = 2.
// G and G' share one log per term: the library's of f / w in D2Q9 and the
// parity build, log_or_nan in 3D (27 library logarithms an iterate were most
// of its solve).  REFORDER keeps the reference's term order
// g += f A - fm lg (EntropicStep.h:31-62) with A_i = ln(f_i / w_i) held per
// term, for FP64 parity; otherwise the constant part is summed once, G =
// sum f A - sum fm lg, and the populations are converted afresh per iteration,
// so that neither Q FP64 values of A nor 2Q converted doubles are held (the
// solve's register footprint bounds its occupancy).
template <class L, bool REFORDER>
__device__ __forceinline__ double log_term(double v, double w) {
  if constexpr (REFORDER || L::dimQ <= 9)
    return log(v / w);
  else
    return log_or_nan(v * (1.0 / w));
}
template <class L, bool REFORDER, bool RESIDUAL, class V>
__device__ __forceinline__ double newton_termwise(const V& p, double guess, double amax,
                                                  double tol, int& branch, int& iterations) {
  constexpr int Q = L::dimQ;
  double A[REFORDER ? Q : 1];
  double SA = 0.0;
  static_for<Q>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const double fi = REFORDER ? p.template f<i>() : p.template f_fresh<i>();
    const double a = log_term<L, REFORDER>(fi, L::W[i]);
    if constexpr (REFORDER)
      A[i] = a;
    else
      SA += fi * a;
  });
  double x = guess, step = 0.0;
  bool ok = false;
  iterations = 0;
  for (int it = 1; it <= 50; ++it) {
    x = x - step;
    if (RESIDUAL && !(x > 0.0)) break;
    iterations = it;
    double g = REFORDER ? 0.0 : SA, dg = 0.0;
    static_for<Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      double fi, ni;
      if constexpr (REFORDER) {
        fi = p.template f<i>();
        ni = p.template n<i>();
      } else {
        fi = p.template f_fresh<i>();
        ni = p.template n_fresh<i>();
      }
      const double fm = fi - x * ni;
      const double lg = log_term<L, REFORDER>(fm, L::W[i]);
      if constexpr (REFORDER)
        g += fi * A[i] - fm * lg;
      else
        g -= fm * lg;
      dg += ni * (1 + lg);
    });
    // both sums end here: otherwise the compiler moves G' behind the test of G
    // and holds the Q logarithms until then (235 registers in D3Q27, not 140)
    if constexpr (RESIDUAL) asm volatile("" : "+v"(g), "+v"(dg));
    if (RESIDUAL && fabs(g) <= tol) {
      ok = (x > 1. && x < amax);
      break;
    }
    step = g / dg;
    if (!RESIDUAL && fabs(step) <= 1e-8) {
      ok = (x > 1. && x < amax);
      break;
    }
    // A NaN step (an iterate outside the logarithms' domain) makes every
    // later iterate NaN, so the reference's loop runs out its 50 iterations
    // and falls back: end now with the same outcome and iteration count.
    // (One such lane would otherwise hold its wavefront for all 50.)
    if (!RESIDUAL && step != step) {
      iterations = 50;
      break;
    }
  }
  if (!ok) {
    branch = 3;
    return 2.0;
  }
  branch = 2;
  return x;
}

// newton_termwise for one cell by a group of 32 lanes that all hold it: lane i
// takes the logarithm of population i, and every lane sums the terms in the
// same order as newton_termwise, so the results are the same to the bit.  For
// the short lists of the 3D lattices, whose launch lasts as long as its
// slowest cell: a solve of 27 logarithms an iterate, up to 50 iterates, took
// 127 us (D3Q27 256^3) with a lane to a cell and the library's logarithm.  lg: 64 doubles of LDS per
// wavefront.
constexpr int kGroupLanes = 32;

template <class L, bool RESIDUAL, class V>
__device__ __forceinline__ double newton_group(const V& p, double guess, double amax, double tol,
                                               double* lg, int& branch, int& iterations) {
  constexpr int Q = L::dimQ;
  static_assert(Q <= kGroupLanes, "one lane per population");
  const int lane = threadIdx.x & 63, mine = lane & (kGroupLanes - 1);
  const double* terms = lg + (lane & ~(kGroupLanes - 1));
  // lanes beyond Q repeat population 0
  double fl = p.template f<0>(), nl = p.template n<0>(), iwl = 1.0 / L::W[0];
  static_for<Q>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if (mine == i) {
      fl = p.template f<i>();
      nl = p.template n<i>();
      iwl = 1.0 / L::W[i];
    }
  });
  auto share = [&](double v) {
    wave_sync_lds();  // the previous terms have been read
    lg[lane] = v;
    wave_sync_lds();
  };
  share(log_or_nan(fl * iwl));
  double SA = 0.0;
  static_for<Q>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    SA += p.template f_fresh<i>() * terms[i];
  });
  double x = guess, step = 0.0;
  bool ok = false;
  iterations = 0;
  for (int it = 1; it <= 50; ++it) {
    x = x - step;
    if (RESIDUAL && !(x > 0.0)) break;
    iterations = it;
    share(log_or_nan((fl - x * nl) * iwl));
    double g = SA, dg = 0.0;
    static_for<Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const double fi = p.template f_fresh<i>(), ni = p.template n_fresh<i>();
      const double l = terms[i];
      g -= (fi - x * ni) * l;
      dg += ni * (1 + l);
    });
    if constexpr (RESIDUAL) asm volatile("" : "+v"(g), "+v"(dg));
    if (RESIDUAL && fabs(g) <= tol) {
      ok = (x > 1. && x < amax);
      break;
    }
    step = g / dg;
    if (!RESIDUAL && fabs(step) <= 1e-8) {
      ok = (x > 1. && x < amax);
      break;
    }
    // as in newton_termwise; the residual iteration is not a number from here
    // on either, and ends in the fallback
    if (step != step) {
      if (!RESIDUAL) iterations = 50;
      break;
    }
  }
  branch = ok ? 2 : 3;
  return ok ? x : 2.0;
}

__device__ __forceinline__ unsigned sample_hash(unsigned cell, unsigned salt) {
  unsigned h = cell * 0x9E3779B1u ^ salt;
  h ^= h >> 16;
  h *= 0x85EBCA6Bu;
  h ^= h >> 13;
  h *= 0xC2B2AE35u;
  return h ^ (h >> 16);
}

// Entropic step, one instantiation per alpha solver MODE so that no kernel
// carries the registers of another's solver:
//   6  reference Newton term by term (the parity build; small D2Q9 domains)
//   0  reference Newton from the power sums; the cells that need the terms are
//      listed for MODE 5, which solves those
//   4  plain Newton from the stored alpha to the residual tolerance: 3D from
//      the power sums, with a list for MODE 7; D2Q9 in the log1p form
//   1, 2  certified correction of the network's / the stored alpha, else plain
//      Newton: 3D from the same power sums, with a list for MODE 7; D2Q9 in the
//      log1p form, with a list for MODE 3.  MODE 1 makes one correction, MODE 2
//      up to two in 3D: from the stored alpha its iterates are the reference
//      Newton's own, so whatever it accepts is the root that Newton converges
//      to; from the network's a second step would also reach roots from which
//      the reference Newton, started at the stored alpha, diverges to its
//      alpha = 2 fallback, and the first stands only where that Newton provably
//      reaches it (reference_reaches)
// Plain Newton is the reference's iteration stopped at |G| <= residual_tol: it
// falls back to alpha = 2 exactly where the reference Newton does and otherwise
// reaches the same root.  A listed cell's populations, alpha and fields are
// left as they were for the second launch (whose order, set by atomics, enters
// no result): about 3% of the cells of MODE 0 in D2Q9 2048^2, which cost the
// whole wavefront the term-by-term solve when they took it in place (468 us a
// step), and 45 us in dense wavefronts of their own.
//
// Measured per step, term by term for every cell -> power sums and list:
// reference Newton D2Q9 2048^2 474 -> 190 us, D3Q27 256^3 5.75 -> 1.70 ms; plain
// Newton D3Q27 4.83 -> 1.65 ms, stored-alpha correction D3Q27 4.23 -> 1.70 ms.
// D2Q9's other modes take one or two evaluations in the log1p form already,
// most of what the power sums cost (plain Newton 173 us, the corrections 134 and 181 of
// which the network's inference is 47), and stay.
// Three phases so that the learned mode's wavefront-wide matrix-core
// inference runs with every lane present: (1) pull, moments, fneq and the
// deviation test per cell; (2) MODE 1 only: the network predicts alpha for
// every lane's cell at once on the matrix cores; (3) the alpha solve, the
// collision and the stores per cell.  The workgroup stages the network in
// LDS once, before phase 1, and one barrier before phase 2 publishes it (a
// copy per wavefront, as first built, needed four times the LDS and held a
// D3Q27 workgroup pair at the 160 KiB limit).
template <int MODE>
constexpr bool kListMode = MODE == 3 || MODE == 5 || MODE == 7;

// Minimum wavefronts per SIMD the register allocator must leave room for: the FP64 solve
// waits for its own results, so three gain over two where they spill little (FP32
// arithmetic up to 25 registers, D3Q19 in FP64 up to 60).  Two where three spilled more:
// D3Q27 in FP64 arithmetic (41 to 183; plain Newton 24^3 37 -> 22 us, 96 x 90 x 100 near
// equilibrium 228 -> 152, stored alpha 180 -> 147), and MODE 7 (FP32 64^3 with strong
// noise 83 -> 71, D3Q19 FP64 32^3 23 -> 17).
template <class L, class C, int MODE>
constexpr int elbm_min_waves() {
  if (L::Type == LatticeType::D2Q9) return kListMode<MODE> || MODE == 6 ? 2 : 4;
  if (std::is_same_v<C, double> && L::dimQ > 19) return 2;
  return MODE == 6 || MODE == 7 ? 2 : 3;
}

template <class L, class S, class C, int FS, int EQ, bool SH, int BLOCK, int MODE>
__global__ void __launch_bounds__(BLOCK)
    __attribute__((amdgpu_waves_per_eu(elbm_min_waves<L, C, MODE>())))
    k_elbm(const StepArgs a, int FSX) {
  constexpr int Q = L::dimQ;
  constexpr bool REF = std::is_same_v<C, double> && !SH;
  constexpr bool FLAT = L::dimQ <= 9;  // D2Q9
  // Solves from the power sums.
  constexpr bool SERIES = MODE == 0 || (!FLAT && (MODE == 1 || MODE == 2 || MODE == 4));
  // A short list of the 3D Newton modes gives each cell a group of lanes.
  constexpr bool GROUPS = !FLAT && (MODE == 5 || MODE == 7);
  __shared__ double s_group[GROUPS ? BLOCK : 1];
  using Shape = MlpShape<L>;
  __shared__ unsigned int s_cnt[6];
  extern __shared__ __align__(16) char s_lds[];
  if (a.stats && threadIdx.x < 6) s_cnt[threadIdx.x] = 0u;
  static_assert(MODE != 1 || Shape::NIN > 0, "no alpha network for this lattice");
  // MODE 1: the workgroup copies the packed network into its LDS now; the
  // copy completes while phase 1 runs, and one barrier before phase 2
  // publishes it.
  using Lay = MfmaLayout<Shape::NIN, Shape::H1, Shape::H2>;
  char* wave_tile = s_lds + Lay::NET + (threadIdx.x >> 6) * Lay::TILE;
  if constexpr (MODE == 1)
    copy_packed_network<Shape::NIN, Shape::H1, Shape::H2>(a.mlp_packed, s_lds);
  // List modes: a thread or a group of lanes per listed cell, the workgroups
  // striding over the list.  They tally their statistics per thread over the passes (branches
  // 0-3, Newton iterations, accepted corrections) and add them up once at the
  // end, so that the passes need no barrier.  Every other mode makes one pass.
  constexpr bool LIST = kListMode<MODE>;
  // The list is kept in shards (see DeferList); each has gridDim.x / shards
  // workgroups here.
  int n_listed = a.N, list_block = blockIdx.x, list_blocks = gridDim.x;
  const int* list = nullptr;
  if constexpr (LIST) {
    if (a.defer.cells) {
      const int shard = blockIdx.x % a.defer.shards;
      n_listed = (int)a.defer.count[shard * kDeferStride];
      list = a.defer.cells + (size_t)shard * a.defer.capacity;
      list_block = blockIdx.x / a.defer.shards;
      list_blocks = gridDim.x / a.defer.shards;
      if (list_block == 0 && threadIdx.x == 0) a.defer.next[shard * kDeferStride] = 0u;
    }
  }
  // at most one pass of groups: at 64 cells a shard and more, lanes are few
  // enough for one each
  const bool groups = GROUPS && n_listed <= list_blocks * (BLOCK / kGroupLanes);
  const int group_log2 = groups ? 5 : 0;
  static_assert(kGroupLanes == 32, "group_log2");
  unsigned tally[6] = {0u, 0u, 0u, 0u, 0u, 0u};
  for (long long list_base = (long long)list_block * (BLOCK >> group_log2);;
       list_base += (long long)list_blocks * (BLOCK >> group_log2)) {
  if constexpr (LIST) {
    if (list_base >= n_listed) break;  // uniform over the workgroup
  }
  CellPos c;
  if constexpr (LIST) {
    const long long t = list_base + (threadIdx.x >> group_log2);
    if (t < n_listed) {
      c = cell_from_index<L>(a, list ? list[t] : (int)t);
    } else {
      c = CellPos{};
      c.active = false;
    }
  } else {
    c = cell_of_thread<L, BLOCK>(a);
  }
  int branch = -1, its = 0;
  bool first = false, solve = false, deferred = false;
  int cell = 0;
  C f[Q], fneq[Q], eqv[Q], F[3];
  C rho = C(1), u[3] = {C(0), C(0), C(0)}, u2 = C(0), drho = C(0);
  double alpha = 2.0, amax = 2.5;
  CellRange range;
  // Every mode keeps the alpha state (Algorithm.h:103-106): it is the
  // reference Newton's warm start, also when that Newton is the fallback of
  // the residual modes.
  // ---- phase 1 ----
  if (c.active) {
    cell = self_index<L>(a, c);
    pull<L, S, C>(a, c, f);
    force_of_cell<L, C>(a, c, F);
    if constexpr (REF) {
      moments_ref<L>(f, rho, u, u2);
      const RefEquilibrium<L, EQ, C> E(rho, u, u2);
      // fneq parked per cell (Collision.h:232-236), here in registers.
      static_for<Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        fneq[i] = f[i] - E.template feq<i>();
      });
    } else {
      if constexpr (SH) {
        moments_shifted<L>(f, drho, rho, u, u2);
      } else {
        moments_ref<L>(f, rho, u, u2);
        drho = rho - C(1);
      }
      const FastEquilibrium<L, EQ, C> E(u, u2);
      static_for<Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const C w = C(L::W[i]);
        const C p = E.template p<i>();
        eqv[i] = SH ? w * (drho + rho * p) : w * rho * (C(1) + p);
        fneq[i] = f[i] - eqv[i];
      });
    }
    // The alpha solve runs in FP64 whatever the compute type.  Branch 0: the
    // deviation is small and alpha = 2 (Collision.h:356-359).
    const Fp64View<L, C, SH> p{f, fneq};
    if constexpr (REF && MODE == 6) {
      solve = !small_deviation_ref<L>(p);
    } else {
      range = cell_range<L>(p);
      solve = !small_deviation<L>(p, range);
    }
    if (!solve) branch = 0;
  }
  // ---- phase 2 ----
  double start = 2.0;
  if constexpr (MODE == 1) {
    float m[Shape::NIN];
    if (solve) {
      nonequilibrium_moments<L>(fneq, C(1) / rho, m);
    } else {
#pragma unroll
      for (int k = 0; k < Shape::NIN; ++k) m[k] = 0.0f;
    }
    __syncthreads();  // the staged network (every thread of the block reaches here)
    start = mlp_alpha_wave<Shape::NIN, Shape::H1, Shape::H2, typename Shape::Op>(s_lds,
                                                                                wave_tile, m);
  }
  // ---- phase 3 ----
  if (c.active) {
    S* __restrict__ dst = static_cast<S*>(a.dst);
    C* __restrict__ astate = static_cast<C*>(a.alpha_state);
    if (solve) {
      const Fp64View<L, C, SH> p{f, fneq};
      const double stored = double(astate[cell]);
      if constexpr (MODE == 5 || MODE == 6 || MODE == 7) {
        if (alpha_capped<L, REF && MODE == 6>(p, alpha, amax))
          branch = 1;
        else if (groups)
          alpha = newton_group<L, MODE == 7>(p, stored, amax, a.residual_tol,
                                             s_group + (GROUPS ? threadIdx.x & ~63 : 0), branch,
                                             its);
        else
          alpha = newton_termwise<L, REF && MODE == 6, MODE == 7>(p, stored, amax, a.residual_tol,
                                                                  branch, its);
      } else if constexpr (MODE == 3 || (FLAT && MODE == 4)) {
        // alphaMax is its cap 2.5 where every |n| / f is below 0.4
        if (!(range.x < 0.39f && ratios_hold<L>(range)) && alpha_capped<L, false>(p, alpha, amax))
          branch = 1;
        else
          alpha = newton_residual<L>(p, amax, stored, a.residual_tol, branch, its);
      } else if constexpr (SERIES) {
        // MODE 0: the reference Newton.  MODE 4: plain Newton from the stored
        // alpha to the residual tolerance.  MODES 1 and 2: the certified
        // correction of the network's or of the stored alpha, and plain Newton
        // where it does not settle the cell.
        int outcome = SOLVE_BEYOND;
        auto settled = [&](double x, double d) {
          if constexpr (std::is_same_v<C, double>) return true;
          return C(a.beta * (x - d)) == C(a.beta * (x + d)) && C(x - d) == C(x + d);
        };
        with_entropy_series<L>(p, range, stored, [&](const auto& s) {
          const double gnoise = log_form_noise<L>(rho);
          if constexpr (MODE == 0) {
            outcome = series_newton_reference(s, stored, gnoise, alpha, its, settled);
          } else {
            int before = 0;
            if constexpr (MODE != 4) {
              EvalCurv cv{};
              first = series_correction(s, MODE == 1 ? start : stored, a.residual_tol,
                                        MODE == 1 ? 1 : 2, alpha, before, cv);
              if constexpr (MODE == 1)
                first = first && reference_reaches(cv, alpha, stored, a.residual_tol);
            }
            if (first)
              outcome = SOLVE_DONE;
            else
              outcome = series_newton_residual(s, stored, a.residual_tol, gnoise, alpha, its,
                                               settled);
            its += before;
            if (MODE != 4 && outcome == SOLVE_BEYOND) its = before;
          }
        });
        if (outcome == SOLVE_BEYOND) {
          deferred = true;  // listed below, once the wavefront has reconverged
          if constexpr (MODE == 0 || MODE == 4) its = 0;
        } else {
          branch = outcome == SOLVE_DONE ? 2 : 3;
          if (outcome != SOLVE_DONE) alpha = 2.0;
        }
      } else if constexpr (MODE == 1 || MODE == 2) {
        // The same corrections in the log1p form (D2Q9); if the solve is not
        // accepted plain Newton decides -- in the MODE 3 launch that follows,
        // from the untouched stored alpha, with the reference's outcome.
        if constexpr (MODE == 2) start = stored;
        bool accepted = false;
        EvalCurv cv{};
        if (!(range.x < 0.39f && ratios_hold<L>(range)) && alpha_capped<L, false>(p, alpha, amax)) {
          branch = 1;
        } else {
          accepted = residual_correction<L>(p, amax, start, a.residual_tol, alpha, its, cv);
          if constexpr (MODE == 1)
            accepted = accepted && reference_reaches(cv, alpha, stored, a.residual_tol);
          if (accepted) {
            branch = 2;
            first = true;
          } else {
            deferred = true;
          }
        }
      }
      // The sample log records the Newton solves: every solve of the Newton
      // modes, of the correction modes those that the correction left to Newton,
      // here (3D) or in the list launch (the cells the network or the stored
      // alpha missed -- data to retrain on).
      if constexpr (Shape::NIN > 0 && (SERIES || (MODE != 1 && MODE != 2))) {
        if (a.log_cap > 0 && branch == 2 && !first &&
            (!groups || threadIdx.x % kGroupLanes == 0) &&
            sample_hash((unsigned)cell, a.log_salt) < a.log_threshold) {
          const unsigned long long k = atomicAdd(a.log_count, 1ull);
          if ((long long)k < a.log_cap) {
            // recomputed here rather than kept live from phase 2
            float m[Shape::NIN];
            nonequilibrium_moments<L>(fneq, C(1) / rho, m);
            for (int q = 0; q < Shape::NIN; ++q) a.log_x[k * Shape::NIN + q] = m[q];
            a.log_alpha[k] = alpha;
          }
        }
      }
    }
    // of a group the first lane speaks for the cell
    bool speaks = !deferred;
    if (groups && threadIdx.x % kGroupLanes != 0) {
      speaks = false;
      branch = -1;
      its = 0;
    }
    if (speaks) {
    astate[cell] = C(alpha);  // Algorithm.h:106
    const C gc = C(a.guo_coef);
    // tau = 1 / (alpha beta); collide with 1 / tau (Collision.h:240, 254).
    const double tau = 1.0 / (alpha * a.beta);
    const C rt = C(1.0 / tau);
    C v[3] = {C(0), C(0), C(0)}, v2 = C(0);
    if constexpr (FS == SRC_EDM) {
      const C k = C(1.0) / rho;
      for (int d = 0; d < L::dimD; ++d) v[d] = u[d] + F[d] * k;
      v2 = v[0] * v[0];
      for (int d = 1; d < L::dimD; ++d) v2 += v[d] * v[d];
    }
    C uF = u[0] * F[0];
    for (int d = 1; d < L::dimD; ++d) uF += u[d] * F[d];
    const RefEquilibrium<L, EQ, C> R2(rho, v, v2);
    const FastEquilibrium<L, EQ, C> E2(v, v2);
    // ELBM collideAndStream (Collision.h:243-258): feq := f - fneq.
    static_for<Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      C s = C(0);
      if constexpr (REF) {
        const C fe = f[i] - fneq[i];
        if constexpr (FS == SRC_GUO) s = guo_ref<L, i>(gc, u, F);
        if constexpr (FS == SRC_EDM) s = R2.template feq<i>() - fe;
      } else {
        const C w = C(L::W[i]);
        if constexpr (FS == SRC_GUO) {
          const C cF = cdot<L, i>(F);
          const C cu = cdot<L, i>(u);
          s = (C(3) * gc * w) * (cF - uF + C(3) * cu * cF);
        }
        if constexpr (FS == SRC_EDM) {
          const C e2 = SH ? w * (drho + rho * E2.template p<i>())
                          : w * rho * (C(1) + E2.template p<i>());
          s = e2 - eqv[i];
        }
      }
      const C out = f[i] - rt * fneq[i] + s;
      store_pop<L, i, S, C>(dst + (size_t)i * a.N + cell, out);
    });
    if (a.store) store_fields<L, C>(a, cell, FSX, rho, u, F, alpha);
    }
  }
  if constexpr (MODE == 1 || MODE == 2 || SERIES) {
    // One counter atomic per wavefront: the lanes' list slots follow from the
    // ballot.
    const unsigned long long mask = __ballot(deferred);
    if (mask) {
      const int lane = threadIdx.x & 63;
      const int leader = __ffsll((long long)mask) - 1;
      const int shard = blockIdx.x % a.defer.shards;
      unsigned base = 0u;
      if (lane == leader)
        base = atomicAdd(&a.defer.count[shard * kDeferStride], (unsigned)__popcll(mask));
      base = __shfl(base, leader);
      if (deferred)
        a.defer.cells[(size_t)shard * a.defer.capacity + base +
                      (unsigned)__popcll(mask & ((1ull << lane) - 1ull))] = cell;
    }
  }
  if (a.stats) {
    // a deferred cell counts its correction's evaluations here and its
    // branch and Newton iterations in the list launch
    if constexpr (LIST) {
      // static indices only: a runtime index would put the tally in scratch
      static_for<4>([&](auto bc) {
        constexpr int b = decltype(bc)::value;
        tally[b] += branch == b ? 1u : 0u;
      });
      tally[4] += (unsigned)its;
      tally[5] += first ? 1u : 0u;
    } else {
      __syncthreads();
      if (branch >= 0) atomicAdd(&s_cnt[branch], 1u);
      if (its) atomicAdd(&s_cnt[4], (unsigned)its);
      if (first) atomicAdd(&s_cnt[5], 1u);
    }
  }
  if constexpr (!LIST) break;
  }  // list passes
  if (a.stats) {
    if constexpr (LIST) {
      __syncthreads();
      static_for<6>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if (tally[k]) atomicAdd(&s_cnt[k], tally[k]);
      });
    }
    __syncthreads();
    if (threadIdx.x < 6 && s_cnt[threadIdx.x])
      atomicAdd(&a.stats[(blockIdx.x % kStatSlots) * kStatStride + threadIdx.x],
                (unsigned long long)s_cnt[threadIdx.x]);
  }
}

}  // namespace lbm
