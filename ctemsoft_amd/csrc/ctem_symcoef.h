// The polynomial of exp(B) - I for complex-symmetric B (ctem_sym.hip). With squares only, a product needs one
// operand on chip:
//   W = (B^2 + c B)^2 + d1 B^2,   p(B) = (r (W + d2 B))^2 + e1 W + g B^2 + B
// matches exp(B) - I through B^7 when c solves c^4 - 10 c^3 + 39 c^2 - 72 c + 60 = 0 (no real root; this one has
// the smallest coefficients), with r^2 = 1 / (20160 c), D = d1 + c^2 = 14 c - 2 c^2, d2 = 84 c - 2 c D,
// e1 = 1/24 - r^2 (D^2 + 4 c d2), g = 1/2 - r^2 d2^2 - e1 D; its B^8 coefficient is off by 0.73 of 1/8!.
//
// B itself enters once, exactly: B is nearly anti-Hermitian, and a complex coefficient on it would turn the rounding
// of its imaginary part into an error of the small real part of the result, which the intensities see in first order.
// tests/test_symcoef.py checks the coefficients.
#pragma once
#include <complex>

namespace ctem {

struct SymPoly { float c[2], d1[2], d2[2], r[2], e1[2], g[2]; };

inline SymPoly sym_poly() {
  typedef std::complex<double> C;
  C c(1.5347072799060086, 1.4831613630292302);
  for (int i = 0; i < 4; i++) {  // to the last bit by Newton's iteration
    const C p = (((c - 10.0) * c + 39.0) * c - 72.0) * c + 60.0, dp = ((4.0 * c - 30.0) * c + 78.0) * c - 72.0;
    c -= p / dp;
  }
  const C r2 = 1.0 / (20160.0 * c), D = 14.0 * c - 2.0 * c * c, d1 = D - c * c, d2 = 84.0 * c - 2.0 * c * D;
  const C e1 = 1.0 / 24.0 - r2 * (D * D + 4.0 * c * d2);
  // v rounded to FP32 into o; returns the rounded value
  auto put = [](C v, float* o) {
    o[0] = (float)v.real();
    o[1] = (float)v.imag();
    return C(o[0], o[1]);
  };
  SymPoly k;
  const C cf = put(c, k.c), d1f = put(d1, k.d1), d2f = put(d2, k.d2), rf = put(std::sqrt(r2), k.r), e1f = put(e1, k.e1);
  put(0.5 - (rf * d2f) * (rf * d2f) - e1f * (cf * cf + d1f), k.g);  // 1/2 for B^2 with the rounded others
  return k;
}

// ||B||_1 bound of that polynomial. Truncation alone, intensities in FP64 arithmetic (2-norm), bcc Fe of 8-25 and of
// 188-250 beams, fcc Ni of 29-39 and of 87-115: at most 2.4e-8 (at 0.9, half a squaring less: 2e-6, 7e-8, 2.6e-6, 2e-8;
// degree 8 at 5/4: 1e-7 to 5e-7).
constexpr double kThetaSym = 0.64;

}  // namespace ctem
