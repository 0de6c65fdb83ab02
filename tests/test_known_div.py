"""csrc/known_div.hpp on the host: division by a number with a known
reciprocal gives the correctly rounded quotient, and the weighted face value
is (x w) / w with both operations rounded, bit for bit -- on random operands
over many binades, on operands next to powers of two and halfway cases, and on
the edges and squared edges of the boxes that use them."""
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
int main() {
  std::mt19937_64 rng(11);
  long bad = 0;
  auto one = [&](double x, double d) {
    if (bits(div_known(x, d, 1.0 / d)) != bits(x / d)) ++bad;
    volatile double p = x * d;
    if (bits(weighted_by(x, d, 1.0 / d)) != bits(p / d)) ++bad;
  };
  auto mantissa = [&](int kind) {  // a double in [1, 2)
    uint64_t m = rng() >> 12;
    if (kind == 1) m &= 7;                        // just above a power of two
    if (kind == 2) m |= ~uint64_t(7) >> 12;       // just below one
    if (kind == 3) m &= uint64_t(0xfff) << 40;    // few significant bits
    uint64_t b = (uint64_t(1023) << 52) | m;
    double v;
    std::memcpy(&v, &b, 8);
    return v;
  };
  for (long k = 0; k < 4000000; ++k) {
    const double x = std::ldexp(mantissa(int(k & 3)), int(rng() % 121) - 60) * ((rng() & 1) ? 1 : -1);
    const double d = std::ldexp(mantissa(int((k >> 2) & 3)), int(rng() % 41) - 20);
    one(x, d);
  }
  const double edges[] = {3.0, 2.5, 0.3, 1.2, 6.283185307179586, 0.1, 7.0, 1.0, 0.5, 1.9999999999999998};
  for (double e : edges)
    for (int l = 0; l < 12; ++l) {
      const double q = std::ldexp(e, -l), q2 = q * q;
      for (long k = 0; k < 20000; ++k) {
        const double x = std::ldexp(mantissa(int(k & 3)), int(rng() % 41) - 40) * ((rng() & 1) ? 1 : -1);
        one(x, q);
        one(x, q2);
      }
      one(0.0, q);
      one(q, q);
      one(-q, q2);
    }
  std::printf("%ld\n", bad);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_known_division_is_correctly_rounded(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "casl_p4est_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    assert int(out) == 0
