// Division by a number whose reciprocal is known, correctly rounded (host and
// device; compile with -ffp-contract=off).
#pragma once

// functions shared by the host builder (g++) and the device kernels (hipcc)
#ifndef CASL_HD
#ifdef __HIPCC__
#define CASL_HD __host__ __device__
#else
#define CASL_HD
#endif
#endif

namespace casl {
namespace dev {

// The quotient v = x / d of a normal x and d, or what an infinite, NaN or zero x
// gives over d: on the device the instruction that ends the hardware's own
// division sequence.
CASL_HD inline double with_specials(double v, double x, double d) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_div_fixup(v, d, x);
#else
  return x - x != 0.0 || x == 0.0 ? x / d : v;
#endif
}
// x / d correctly rounded, for a d whose reciprocal rd = RN(1 / d) is known:
// two Newton corrections of q = x rd, each with the exact remainder an fma
// gives.  The first leaves q within one ulp; from there the second gives the
// correctly rounded quotient (Markstein, IBM J. Res. Dev. 34, 1990: q + r rd
// with r = x - q d rounds to x / d when rd is the correctly rounded
// reciprocal and q is within one ulp).  Five operations in place of the
// range-safe division sequence, a sixth for infinities, NaN and zeros (whose
// remainder is inf - inf, or loses a sign): 20 RK2 iterations on the 2.0M-node
// octree of 64 spheres in [0, 3]^3 2.99 ms without it, 3.06 with it, 3.30 with
// a test for a NaN behind every quotient, 3.74 with one for a range.  Numbers:
// |x| from 2^-960 to 2^1023 |d| and quotients from 2^-1020 (below, the
// remainder or the quotient is subnormal and the last place may differ; above,
// the division overflows and this gives a NaN).
CASL_HD inline double div_number(double x, double d, double rd) {
  double q = x * rd;
  q = __builtin_fma(__builtin_fma(-q, d, x), rd, q);
  return __builtin_fma(__builtin_fma(-q, d, x), rd, q);
}
CASL_HD inline double div_known(double x, double d, double rd) {
  return with_specials(div_number(x, d, rd), x, d);
}
// (x w) / w, both operations rounded: the reference's value of a face whose
// one nonzero-weight corner holds x.  The product p = x w is within half an
// ulp of exact, so x itself is within one ulp of p / w and the exact
// remainder p - x w corrects it in one step (the same theorem).  Numbers: |x|
// and |x w| from 2^-960.
CASL_HD inline double weighted_by(double x, double w, double rw) {
  const double p = x * w;
  return with_specials(__builtin_fma(__builtin_fma(-x, w, p), rw, x), p, w);
}

}  // namespace dev
}  // namespace casl
