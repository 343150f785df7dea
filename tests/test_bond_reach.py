"""The distance beyond which no bond is listed (csrc/bond_reach.hpp, host code), compiled here with the host compiler.

The bond build skips the bond-order evaluation of candidates beyond it, so for any parameters there must be no bond there: BO' in
double and in single precision (the orders of the FP64 / mixed and of the FP32 mode) is below the cutoff at every distance past the
bound. The bound is near enough to be of use (BO' just inside it reaches the cutoff less 1e-3 of it), it is infinite where BO' is not a falling
function, and finding it takes a few dozen evaluations, since every pair_coeff does it for every pair of types."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "metal-reax_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <random>
#include "bond_reach.hpp"
using namespace rxa;

template <class T> T order(const BondKind (&k)[3], double d) {
  T v = 0;
  for (const BondKind& b : k)
    if (b.on) v += (T)b.factor * std::exp((T)b.a * std::pow((T)d / (T)b.r, (T)b.b));
  return v;
}

int main() {
  std::mt19937_64 rng(7);
  auto uni = [&](double lo, double hi) { return lo + (hi - lo) * std::generate_canonical<double, 53>(rng); };
  int most = 0, bad = 0;
  for (int t = 0; t < 20000; ++t) {
    const double cut = std::pow(10.0, uni(-6.0, -0.5));
    const BondKind k[3] = {{true, -uni(0.01, 0.5), uni(1.0, 30.0), uni(0.5, 2.5), 1.0 + cut},
                           {t % 2 == 0, -uni(0.05, 0.6), uni(2.0, 40.0), uni(0.5, 2.0), 1.0},
                           {t % 3 == 0, -uni(0.05, 0.6), uni(2.0, 40.0), uni(0.5, 2.0), 1.0}};
    const double far = bond_reach(k, cut);
    int calls = 0;
    falls_below([&](double d) { ++calls; return order<double>(k, d); }, cut * (1.0 - 1e-3));
    if (calls > most) most = calls;
    if (!std::isfinite(far)) continue;   // out of range: everything is evaluated
    for (int s = 0; s < 20; ++s) {
      const double d = s == 0 ? std::nextafter(far, 1e9) : far * (1.0 + std::pow(10.0, uni(-9.0, 0.5)));
      if (order<double>(k, d) >= cut || order<float>(k, d) >= (float)cut) ++bad;
    }
    if (order<double>(k, far * (1.0 - 1e-5) - 1e-5) < cut * (1.0 - 1e-3)) ++bad;
  }
  auto inf = [&](BondKind s, BondKind p, double cut) { const BondKind k[3] = {s, p, {false, 0, 0, 0, 1.0}}; return std::isinf(bond_reach(k, cut)); };
  const BondKind good{true, -0.1, 6.0, 1.4, 1.001}, off{false, 0.3, -1.0, 0.0, 1.0};
  const double nan = std::nan("");
  const bool rule = !inf(good, off, 0.001) && inf(good, off, 0.0) && inf(good, off, -1.0) && inf(good, off, nan) &&
                    inf({true, 0.1, 6.0, 1.4, 1.0}, off, 0.001) && inf({true, 0.0, 6.0, 1.4, 1.0}, off, 0.001) &&
                    inf({true, -0.1, 0.0, 1.4, 1.0}, off, 0.001) && inf({true, -0.1, -6.0, 1.4, 1.0}, off, 0.001) &&
                    inf({true, -0.1, 6.0, 0.0, 1.0}, off, 0.001) && inf({true, nan, 6.0, 1.4, 1.0}, off, 0.001) &&
                    inf(good, {true, 0.2, 6.0, 1.2, 1.0}, 0.001) && inf({true, -1e-9, 1e-3, 1.4, 1.0}, off, 0.001);
  std::printf("%d %d %d\n", bad, most, (int)rule);
}
"""


@pytest.fixture(scope="module")
def result(tmp_path_factory):
    d = tmp_path_factory.mktemp("bond_reach")
    src = d / "reach.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(d / "reach")], check=True)
    return [int(v) for v in subprocess.run([str(d / "reach")], check=True, capture_output=True, text=True).stdout.split()]


def test_no_bond_beyond_the_bound(result):
    assert result[0] == 0


def test_few_evaluations(result):
    assert result[1] <= 48   # 20 halvings and the doublings before them


def test_infinite_where_the_order_does_not_fall(result):
    assert result[2] == 1
