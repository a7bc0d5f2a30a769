// Arithmetic with one rounding.  No HIP here (constexpr functions are host and
// device functions to the compiler), so that it runs anywhere.
#pragma once

namespace ocsc {

// S / n - a b, rounded once: the rests of the quotient, of the product and of
// the difference are added back
template <class T>
constexpr T centred_difference(T S, T n, T a, T b) {
  const T q = S / n, rq = __builtin_fma(-q, n, S) / n;
  const T p = a * b, rp = __builtin_fma(a, b, -p);
  const T d = q - p, t = d - q, rd = (q - (d - t)) - (p + t);
  return d + (rd + (rq - rp));
}

}  // namespace ocsc
