// Distance beyond which no bond is listed (host code, used when the pair tables are packed).
#pragma once
#include <cmath>
#include <limits>

namespace rxa {

// one kind of bond (sigma, pi, double pi) of a type pair: its part of BO' is factor exp(a (d / r)^b)
struct BondKind {
  bool on;
  double a, b, r, factor;
};

// A distance from which on the falling function f stays below limit, at most about 1e-6 beyond the first such one (a 2^-20th of the
// interval between two powers of two), or infinity past 1e6. Every pair_coeff calls it for every pair of types, so it stops there: 100
// halvings, for both orders of a pair, took 0.04 of 0.225 ms with 3 types and 0.4 of 2.9 ms with 9; now 0.188 and 2.53 ms.
template <class F>
double falls_below(F&& f, double limit) {
  double lo = 0.0, hi = 1.0;
  while (f(hi) >= limit) {
    lo = hi;
    hi *= 2.0;
    if (!(hi < 1e6)) return std::numeric_limits<double>::infinity();
  }
  for (int k = 0; k < 20; ++k) {
    const double m = 0.5 * (lo + hi);
    (f(m) >= limit ? lo : hi) = m;
  }
  return hi;
}

// Distance beyond which BO' stays below bo_cut: each kind of bond falls with the distance when its coefficient is negative and its power
// positive (then so does BO'); the bound is where BO' falls to bo_cut less 1e-3 of it, far beyond the rounding of the
// single-precision powers. Anything else: infinite, every candidate is evaluated.
inline double bond_reach(const BondKind (&kind)[3], double bo_cut) {
  const double inf = std::numeric_limits<double>::infinity();
  for (const BondKind& k : kind)
    if (k.on && !(k.a < 0.0 && k.b > 0.0 && k.r > 0.0)) return inf;
  const double limit = bo_cut * (1.0 - 1e-3);
  if (!(limit > 0.0)) return inf;
  return falls_below([&](double d) {
    double v = 0;
    for (const BondKind& k : kind)
      if (k.on) v += k.factor * std::exp(k.a * std::pow(d / k.r, k.b));
    return v;
  }, limit);
}

}  // namespace rxa
