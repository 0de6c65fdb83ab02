"""csrc/known_div.hpp on the host: infinities, NaN and zeros give what the
divisions give, and the quotients are the divisions' over the range of
magnitudes the header names."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include "known_div.hpp"
using namespace casl::dev;
static uint64_t bits(double x) { uint64_t b; std::memcpy(&b, &x, 8); return b; }
static bool same(double a, double b) { return bits(a) == bits(b) || (a != a && b != b); }
static long bad = 0;
static void one(double x, double d) {
  if (!same(div_known(x, d, 1.0 / d), x / d)) {
    std::printf("%a / %a: %a, not %a\n", x, d, div_known(x, d, 1.0 / d), x / d);
    ++bad;
  }
}
static void weighted(double x, double w) {
  volatile double p = x * w;
  if (!same(weighted_by(x, w, 1.0 / w), p / w)) {
    std::printf("(%a w) / w, w = %a: %a, not %a\n", x, w, weighted_by(x, w, 1.0 / w), p / w);
    ++bad;
  }
}
int main() {
  const double inf = HUGE_VAL, edges[] = {3.0, 2.5, 6.0, 0.3, 1.5e-3, 7e5, 2.9999999999999996};
  for (double e : edges)
    for (int l = 0; l < 16; ++l)
      for (double d : {std::ldexp(e, -l), std::ldexp(e * e, -l)})
        for (double x : {inf, -inf, inf - inf, 0.0, -0.0, 1.0, std::ldexp(1.0, -960), -std::ldexp(1.5, 900)}) {
          one(x, d);
          weighted(x, d);
        }
  std::mt19937_64 rng(5);
  std::uniform_real_distribution<double> u(1.0, 2.0);
  for (long k = 0; k < 4000000 && bad < 20; ++k) {
    const double x = std::ldexp(u(rng), int(rng() % 1921) - 960) * ((rng() & 1) ? 1 : -1);
    const double d = std::ldexp(u(rng), int(rng() % 121) - 60);
    one(x, d);
    if (std::fabs(x * d) >= std::ldexp(1.0, -960)) weighted(x, d);
  }
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_range(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "casl_p4est_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
