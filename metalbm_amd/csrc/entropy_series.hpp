// entropy_series.hpp -- the entropic root solve from power sums.
//
// alpha is the nontrivial root of G(a) = H(f) - H(f - a n), H(v) = sum v ln(v/w)
// (EntropicStep.h:31-45).  Evaluated term by term every Newton iterate costs
// one FP64 logarithm per population, and those logarithms were the entropic
// step: D2Q9 2048^2 ran the reference Newton (2.85 iterates, 9 + 26 logarithms
// per cell) in 470 us and D3Q27 256^3 plain Newton (2.7 iterates, 27 + 73
// logarithms) in 4.76 ms, against 60 and 670 us for the bytes they move.
//
// Around a centre v = f - c n every f - a n = v (1 - b r) is close, r = n / v and
// b = a - c, and (1 + z) ln(1 + z) = z + sum_{k>=2} (-z)^k / (k (k - 1)), so
//   G(a)   = a S1 + E0 - sum_{k=2..K} P_k b^k / (k (k - 1))
//   G'(a)  =   S1      - sum_{k=2..K} P_k b^{k-1} / (k - 1)
//   -G''(a) =            sum_{k=2..K} P_k b^{k-2}
// with P_k = sum_i n_i r_i^{k-1}, S1 = sum_i n_i (1 + ln(v_i / w_i)) and
// E0 = sum_k P_k (-c)^k / (k (k - 1)).  One pass over the populations -- one
// logarithm and one quotient each -- gives the coefficients; every iterate
// after that is a polynomial in b.
//
// The centre:
//  * c = 1, the equilibrium, in 3D.  alpha is about 2, so both ends, a = 0 and
//    a = 2, are at |b| = 1, half the argument of c = 0.  D3Q27 turbulence has max
//    |r| 0.03 to 0.15 over a wavefront: orders 12 and 16.
//  * c = the stored alpha, from which Newton starts, where |r| is larger: b is
//    then small (alpha moves by about 1e-2 a step) and order 10 reaches any
//    |n| / f below 0.39, at the price of a second logarithm, G(c) itself, from
//    which E0 follows.
//  * c = 0 in D2Q9.  Its flows are near equilibrium (max |n| / f ~ 5e-3, order
//    10), and with v = f the one sum that carries rounding, sum n ln(f / w), is
//    the one its log1p-form solver takes.
//
// Truncation: the first term left out, relative to the curvature P_2 that
// turns an error of G into one of alpha, is at most 2 z^(K-1) / (K (K + 1)),
// z = max |r| max(c, |b|) (max |r| |b| where E0 is not a series).  The order is
// chosen per wavefront so that this stays below 1e-16 in D2Q9 and 1e-14 in 3D
// (kSeriesReach), under the rounding that the logarithms left in alpha (1e-10
// to 1e-13); a lane out of reach, or with a population at or below zero, takes
// the term-by-term solver.
#pragma once

#include "entropy_log.hpp"
#include "mlp.hpp"

namespace lbm {

enum : int { CENTRE_F = 0, CENTRE_E = 1, CENTRE_STORED = 2 };

// Largest z of a series of order K, and the orders built.
template <int CENTRE, int K>
constexpr double kSeriesReach = CENTRE == CENTRE_F   ? (K == 10 ? 0.0262 : 0.258)
                                : CENTRE == CENTRE_E ? (K == 12 ? 0.0797 : 0.162)
                                                     : 0.0433;

// Populations of the 3D pass in flight together.
constexpr int kSeriesGroup = 9;

// First look at one cell in FP32: the largest |n| / f, the smallest f and (D2Q9)
// the largest |f / w - 1|.  It settles the deviation test away from its threshold
// and chooses the orders; every decision it cannot settle is taken in FP64.
struct CellRange {
  float x = 0.0f, y = 0.0f, f = 3.0e38f;
};
// f is formed as (f - w) + w, with an error of up to 2^-23 (w + f): a cell's ratios are
// good to 3e-4 where every f is above 5e-4 of the largest weight (a population of
// the smallest weight then still reaches down to 3% of it).  Elsewhere, populations
// at or below zero among them, the cell is decided in FP64.
template <class L>
constexpr float largest_weight() {
  double w = 0.0;
  for (int i = 0; i < L::dimQ; ++i) w = L::W[i] > w ? L::W[i] : w;
  return float(w);
}
template <class L>
__device__ __forceinline__ bool ratios_hold(const CellRange& c) {
  return c.f > 5.0e-4f * largest_weight<L>();
}
template <class L, class V>
__device__ __forceinline__ CellRange cell_range(const V& p) {
  CellRange c;
  static_for<L::dimQ>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    constexpr float w = float(L::W[i]), inv_w = float(1.0 / L::W[i]);
    const float g = float(p.template shifted<i>()), n = float(p.template n32<i>());
    const float f = g + w;
    c.f = fminf(c.f, f);
    c.x = fmaxf(c.x, fabsf(n) * __builtin_amdgcn_rcpf(f));
    if constexpr (L::dimQ <= 9) c.y = fmaxf(c.y, fabsf(g) * inv_w);
  });
  return c;
}

// The deviation test max |n| / f <= 1e-3 (Collision.h:284-303).  Where the FP32
// ratios hold only a lane within 0.1% of the threshold is decided in FP64; so is one
// whose moments are not a number, which cell_range's maxima pass over (every n_i
// is then not a number, n_0 among them).
template <class L, class V>
__device__ __forceinline__ bool small_deviation(const V& p, const CellRange& c) {
  bool small = !(c.x > 1.0e-3f);
  const float n0 = p.template n32<0>();
  if (!ratios_hold<L>(c) || fabsf(c.x - 1.0e-3f) <= 1.0e-6f || n0 != n0) {
    small = true;
    static_for<L::dimQ>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const double fi = p.template f<i>(), ni = p.template n<i>();
      if (!(fabs(ni) <= 1.0e-3 * fi) && fi > 0.0) small = false;
    });
  }
  return small;
}

template <class L, int CENTRE, int K>
struct EntropySeries {
  double centre;              // c
  double s1, e0, rpos, rneg;  // rpos, rneg: largest r and -r, at least 0
  double c[K + 1];            // c[k] = P_k / (k (k - 1)), k = 2..K

  // One pass over the populations.  y bounds the cell's |f / w - 1|.
  template <class V>
  __device__ __forceinline__ void build(const V& p, float y, double stored) {
    centre = CENTRE == CENTRE_F ? 0.0 : (CENTRE == CENTRE_E ? 1.0 : stored);
    // sum n and sum n ln(v/w) apart: their sum is of the order of P_2, and
    // 1 + ln(v/w) rounded term by term would leave 1e-16 n in it.
    double sn = 0.0, sl = 0.0;
    e0 = 0.0;  // CENTRE_STORED: G(c) first
    rpos = rneg = 0.0;
    static_for<K - 1>([&](auto kc) { c[decltype(kc)::value + 2] = 0.0; });
    auto sums = [&](auto log1p_of) {
      static_for<L::dimQ>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        constexpr double inv_w = 1.0 / L::W[i];
        double ni, fi;
        if constexpr (CENTRE != CENTRE_F) {
          ni = p.template n_fresh<i>();
          fi = p.template f_fresh<i>();
        } else {
          ni = p.template n<i>();
          fi = p.template f<i>();
        }
        double vi, li;
        if constexpr (CENTRE == CENTRE_STORED) {
          vi = fi - centre * ni;
          li = log_or_nan(vi * inv_w);
          e0 += fi * log_or_nan(fi * inv_w) - vi * li;
        } else {
          vi = CENTRE == CENTRE_E ? fi - ni : fi;
          li = log1p_of(fma(vi, inv_w, -1.0));
        }
        sn += ni;
        sl = fma(ni, li, sl);
        const double r = quotient(ni, vi);
        rpos = fmax(rpos, r);
        rneg = fmax(rneg, -r);
        double t = ni;
        static_for<K - 1>([&](auto kc) {
          constexpr int k = decltype(kc)::value + 2;
          t *= r;
          c[k] += t;
        });
        // 3D: a few populations at a time.  The empty asm statements order each
        // group's sums before the next group's conversions; left alone, the
        // compiler computes every quotient first and the sums behind the first
        // iterate's tests, with 2Q doubles held between (256 registers and 224
        // spills at three wavefronts).
        if constexpr (CENTRE != CENTRE_F && i % kSeriesGroup == kSeriesGroup - 1) {
          static_for<K - 1>([&](auto kc) {
            asm volatile("" : "+v"(c[decltype(kc)::value + 2]));
          });
          asm volatile("" : "+v"(sl), "+v"(rpos), "+v"(rneg), "+v"(e0));
        }
      });
    };
    // ln(v/w) by a short series where every lane's |v/w - 1| allows it (D2Q9
    // near equilibrium; truncation below 1e-19 relative), else the logarithm.
    if (CENTRE == CENTRE_F && !__any(!(y <= 1.64e-2f)))
      sums([](double v) { return log1p_series<10>(v); });
    else
      sums([](double v) { return log1p_positive(v); });
    s1 = sn + sl;
    static_for<K - 1>([&](auto kc) {
      constexpr int k = K - decltype(kc)::value;  // smallest terms first
      c[k] *= 1.0 / (double(k) * (k - 1));
      if constexpr (CENTRE == CENTRE_E) e0 = k % 2 ? e0 - c[k] : e0 + c[k];
    });
    if constexpr (CENTRE == CENTRE_STORED) e0 = fma(-centre, s1, e0);
  }

  // Whether the series holds at alpha = a.
  __device__ __forceinline__ bool holds(double a) const {
    return fabs(a - centre) * fmax(rpos, rneg) <= kSeriesReach<CENTRE, K>;
  }
  // G and G': with H(b) = sum c_k b^(k-2) and its derivative in one Horner pass,
  // G = a S1 + E0 - b^2 H, G' = S1 - b (2 H + b H').
  __device__ __forceinline__ void eval(double a, double& g, double& dg) const {
    const double b = a - centre;
    double h = c[K], d = 0.0;
    static_for<K - 2>([&](auto kc) {
      constexpr int k = K - 1 - decltype(kc)::value;
      d = fma(d, b, h);
      h = fma(h, b, c[k]);
    });
    g = fma(a, s1, fma(-b * b, h, e0));
    dg = fma(-b, fma(b, d, h + h), s1);
  }
  // -G'' = sum n^2 / (f - a n) = sum k (k - 1) c_k b^(k-2) and max |n| / (f - a n),
  // at a > 1.
  __device__ __forceinline__ EvalCurv curvature(double a, double dg) const {
    const double b = a - centre;
    double h = 0.0;
    static_for<K - 1>([&](auto kc) {
      constexpr int k = K - decltype(kc)::value;
      h = fma(h, b, c[k] * (double(k) * (k - 1)));
    });
    const double r = fmax(rpos / (1.0 - b * rpos), rneg / (1.0 + b * rneg));
    return EvalCurv{a, dg, h, r * (1.0 + 1e-12)};
  }
};

// alphaMax = min(2.5, min_{n > 0} f / n) (Collision.h:305-326) is 2.5 wherever
// the series is used: |n| / f < 0.39.
constexpr double kSeriesAlphaMax = 2.5;

// Outcome of a solve from the series.
enum : int { SOLVE_DONE = 0, SOLVE_REJECTED = 1, SOLVE_BEYOND = 2 };

// Newton from the series, keeping the term-by-term solvers' results: to the bit in FP32
// arithmetic, their iterations and outcomes in FP64.
//
// Term by term, G carries rounding (gnoise, below), and so each step an error
// up to gnoise / |G'|; the series' own is a thousand times smaller.  At tau =
// 0.50003 a last-place change of one cell's relaxation rate grows to 1e-4 of its
// neighbourhood's populations within five steps, so where that error could
// change what the kernel applies or stores of alpha, or the number of
// iterations, the cell is left to the term-by-term solver, which decides as it
// always has (SOLVE_BEYOND; so are iterates that leave the series or are not a
// number).  settled(x, d): whether all of [x - d, x + d] rounds to one result.  In
// FP64 arithmetic no alpha is settled in that sense, and the series' is taken: it
// differs from the term-by-term one by that one's noise (4e-13 in D2Q9, 3e-14 in 3D
// on strong noise; 1e-10 where |G'| is smallest), so that a cell's alpha depends on
// whether its domain is large enough for the list.
//
// gnoise: the rounding of the 2Q quotients f / w under the logarithms, up to
// 2^-53 (sum f + sum (f - a n)) = 2^-52 rho: 1e-10 of alpha at D2Q9 2048^2, where
// alpha's step in FP32 is 2.4e-7 (3D, where f / w is the product with a rounded
// reciprocal, twice that).
template <class L>
__device__ __forceinline__ double log_form_noise(double rho) {
  return (L::dimQ <= 9 ? 0x1.1p-52 : 0x1.1p-51) * rho;
}

// The reference Newton (EntropicStep.h:111-140): warm start, |step| <= 1e-8, at
// most 50 iterations, the iterate before the last step, accepted inside
// (1, alphaMax).
template <class SERIES, class SETTLED>
__device__ __forceinline__ int series_newton_reference(const SERIES& s, double start,
                                                       double gnoise, double& alpha, int& evals,
                                                       SETTLED&& settled) {
  double x = start, before = 0.0;  // before: the error of x
  for (int it = 1; it <= 50; ++it) {
    if (!s.holds(x)) return SOLVE_BEYOND;
    double g, dg;
    s.eval(x, g, dg);
    evals = it;
    const double step = g / dg, noise = fabs(gnoise / dg);
    if (!(fabs(fabs(step) - 1e-8) > noise + before)) return SOLVE_BEYOND;
    if (fabs(step) <= 1e-8) {
      if (!settled(x, before)) return SOLVE_BEYOND;
      alpha = x;
      return x > 1.0 && x < kSeriesAlphaMax ? SOLVE_DONE : SOLVE_REJECTED;
    }
    x -= step;
    before = noise;
  }
  return SOLVE_REJECTED;
}

// Plain Newton: the same iteration stopped at |G| <= tol.
template <class SERIES, class SETTLED>
__device__ __forceinline__ int series_newton_residual(const SERIES& s, double start, double tol,
                                                      double gnoise, double& alpha, int& evals,
                                                      SETTLED&& settled) {
  double x = start, before = 0.0;
  for (int it = 1; it <= 50; ++it) {
    // an iterate at or below 0 ends as it does without the series
    if (!s.holds(x) || !(x > 0.0)) return SOLVE_BEYOND;
    double g, dg;
    s.eval(x, g, dg);
    evals = it;
    if (!(fabs(fabs(g) - tol) > gnoise + before * fabs(dg))) return SOLVE_BEYOND;
    if (fabs(g) <= tol) {
      if (!settled(x, before)) return SOLVE_BEYOND;
      alpha = x;
      return x > 1.0 && x < kSeriesAlphaMax ? SOLVE_DONE : SOLVE_REJECTED;
    }
    x -= g / dg;
    before = fabs(gnoise / dg);
  }
  return SOLVE_REJECTED;
}

// Certified correction: up to max_evals evaluations from `start` inside
// (1, alphaMax); accepts an iterate with |G| <= tol, or a Newton point a1 = a - s
// whose Taylor remainder bound is <= tol without evaluating G there: G(a1) =
// s^2/2 G''(xi) for some xi between a and a1, and f - xi n = (f - a n) +
// (a - xi) n >= (f - a n)(1 - |s| r), so |G''(xi)| <= h / (1 - |s| r); a relative
// allowance of 1e-6 covers the rounding of the bound.  Anything else defers
// the cell to plain Newton from the stored alpha.
template <class SERIES>
__device__ __forceinline__ bool series_correction(const SERIES& s, double start,
                                                  double tol, int max_evals, double& alpha,
                                                  int& evals, EvalCurv& cv) {
  double a = start;
  for (int it = 0; it < max_evals; ++it) {
    if (!(a > 1.0 && a < kSeriesAlphaMax) || !s.holds(a)) return false;
    double g, dg;
    s.eval(a, g, dg);
    cv = s.curvature(a, dg);
    evals = it + 1;
    if (fabs(g) <= tol) {
      alpha = a;
      return true;
    }
    const double step = g / dg;
    const double a1 = a - step;
    const double room = 1.0 - fabs(step) * cv.r;
    if (a1 > 1.0 && a1 < kSeriesAlphaMax && room > 0.0 &&
        0.5 * step * step * cv.h / room * (1.0 + 1e-6) <= tol) {
      alpha = a1;
      return true;
    }
    a = a1;
  }
  return false;
}

// Runs body(series) with the shortest series that holds for every active lane
// within reach (with some room above alpha = 2, of which alpha stays within a
// few percent), and returns true for those lanes; false for a lane out of
// reach.
template <class L, class V, class F>
__device__ __forceinline__ bool with_entropy_series(const V& p, const CellRange& c, double stored,
                                                    F&& body) {
  auto go = [&](auto centre, auto order) {
    EntropySeries<L, decltype(centre)::value, decltype(order)::value> s;
    s.build(p, c.y, stored);
    body(s);
  };
  if (!ratios_hold<L>(c) || !(c.x < 0.39f)) return false;
  if constexpr (L::dimQ <= 9) {
    using At = std::integral_constant<int, CENTRE_F>;
    const float r = 2.15f * c.x;
    if (!(r <= float(kSeriesReach<CENTRE_F, 24>))) return false;
    if (!__any(r > float(kSeriesReach<CENTRE_F, 10>)))
      go(At{}, std::integral_constant<int, 10>{});
    else
      go(At{}, std::integral_constant<int, 24>{});
  } else {
    using At = std::integral_constant<int, CENTRE_E>;
    const float r = c.x / (1.0f - c.x) * 1.08f;
    if (!__any(r > float(kSeriesReach<CENTRE_E, 12>)))
      go(At{}, std::integral_constant<int, 12>{});
    else if (!__any(r > float(kSeriesReach<CENTRE_E, 16>)))
      go(At{}, std::integral_constant<int, 16>{});
    else
      go(std::integral_constant<int, CENTRE_STORED>{}, std::integral_constant<int, 10>{});
  }
  return true;
}

}  // namespace lbm
