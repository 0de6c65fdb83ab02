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

// x / d correctly rounded, for a d whose reciprocal rd = RN(1 / d) is known:
// two Newton corrections of q = x rd, each with the exact remainder an fma
// gives.  The first leaves q within one ulp; from there the second gives the
// correctly rounded quotient (Markstein, IBM J. Res. Dev. 34, 1990: q + r rd
// with r = x - q d rounds to x / d when rd is the correctly rounded
// reciprocal and q is within one ulp).  Five operations in place of the
// range-safe division sequence; x / d and the remainder must be normal
// numbers or x zero.
CASL_HD inline double div_known(double x, double d, double rd) {
  double q = x * rd;
  q = __builtin_fma(__builtin_fma(-q, d, x), rd, q);
  return __builtin_fma(__builtin_fma(-q, d, x), rd, q);
}
// (x w) / w, both operations rounded: the reference's value of a face whose
// one nonzero-weight corner holds x.  The product p = x w is within half an
// ulp of exact, so x itself is within one ulp of p / w and the exact
// remainder p - x w corrects it in one step (the same theorem).
CASL_HD inline double weighted_by(double x, double w, double rw) {
  const double p = x * w;
  return __builtin_fma(__builtin_fma(-x, w, p), rw, x);
}

}  // namespace dev
}  // namespace casl
