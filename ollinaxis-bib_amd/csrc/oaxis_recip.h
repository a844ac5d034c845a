// Quotients by one divisor through its reciprocal, for the horizon finder's
// sources.  Included by oaxis_ah.hip after oaxis_device.h (OA_HD), with
// floating-point contraction off.
#pragma once

// the estimate the refinement starts from, good to 2^-24
#ifndef OA_RCP
#define OA_RCP(d) __builtin_amdgcn_rcp(d)
#endif

namespace oax {

// Quotients by one divisor share its reciprocal: two Newton steps on the
// hardware's estimate, then per quotient a product and one residual correction
// (Markstein 1990); three instructions instead of eleven.  With the reciprocal
// rounded correctly the quotient is too, wherever numerator, divisor and
// quotient are normal numbers.  The second step leaves 2^-96 of the first
// one's error, so the reciprocal is rounded correctly unless it lies that close
// to the middle of two numbers (about one divisor in 2^40, such as 2 - 2^-52);
// by such a divisor a quotient can be the neighbour of the correctly rounded
// one (1 / (2 - 2^-52) is), never further off.  A division by zero or of an
// infinity gives NaN, which the sources refuse as they refuse an infinity.
struct AhRecip {
  double d, y;
  OA_HD explicit AhRecip(double div) : d(div) {
    y = OA_RCP(d);
    y = fma(y, fma(-d, y, 1.0), y);
    y = fma(y, fma(-d, y, 1.0), y);
  }
  OA_HD AhRecip(double div, double recip) : d(div), y(recip) {}
  OA_HD double of(double x) const {
    const double q = x * y;
    return fma(fma(-d, q, x), y, q);
  }
};

// x / n for the bicubic weights' n, 1 <= |n| <= 3
OA_HD double ah_over(double x, int n) {
  const int m = n < 0 ? -n : n;
  const double q = (m == 3) ? AhRecip(3.0, 1.0 / 3.0).of(x) : (m == 2) ? 0.5 * x : x;
  return n < 0 ? -q : q;
}

}  // namespace oax
