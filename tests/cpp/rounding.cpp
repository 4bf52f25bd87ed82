// TEST-ONLY: single formulas of the kernels' math (stage_math.hpp) over arrays, in
// double precision.  Built by tests/test_rounding.py.
#include <cstdint>

#include "../../zisafvm_amd/csrc/stage_math.hpp"

using namespace zfv;

extern "C" {

// y = x^(1/(gamma-1)) as the equilibria form it
void unit_eq_pow(double gamma, int n, const double *x, double *y) {
  Img m{};
  m.gamma = gamma;
  eq_pow_constants(gamma, m.eq_half, m.eq_db);
  for (int k = 0; k < n; ++k) y[k] = eq_pow(m, x[k], 1.0 / (gamma - 1.0));
}

// f (4 n) = the HLLC flux between uL and uR (4 n each) along the normals nn (2 n)
void unit_hllc(double gamma, int n, const double *uL, const double *uR, const double *nn, double *f) {
  for (int k = 0; k < n; ++k) hllc<2>(uL + 4 * k, uR + 4 * k, nn + 2 * k, gamma, f + 4 * k);
}

// the kernels' evaluation at the scaled point X of the polynomial of coefficients
// a over the basis X^alpha - c[alpha]: the moments in the nested form's constant
// coefficient, the mean beside it
double unit_poly(int dims, int degree, int dof, const double *a, const double *c, const double *X) {
  double b[16] = {0};
  for (int k = 1; k < dof; ++k) b[k] = a[k];
  for (int k = 1; k < dof; ++k) b[0] -= a[k] * c[k];
  double r = 0.0;
  if (dims == 2 && degree == 1) r = poly_nested<2, 1>(b, X);
  else if (dims == 2 && degree == 2) r = poly_nested<2, 2>(b, X);
  else if (dims == 2 && degree == 3) r = poly_nested<2, 3>(b, X);
  else if (dims == 3 && degree == 1) r = poly_nested<3, 1>(b, X);
  else r = poly_nested<3, 2>(b, X);
  return a[0] + r;
}

}  // extern "C"
