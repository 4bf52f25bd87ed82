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

}  // extern "C"
