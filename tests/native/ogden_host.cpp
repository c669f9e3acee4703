// Host build of the Ogden law's choice between its series and the principal
// directions (femtech_amd/csrc/ft_device.h) for CPU tests.  Test code only.
#include "../../femtech_amd/csrc/ft_device.h"

namespace {
// bit 0: the rule takes the series; bit 1: the series ends.  Z = diag(z); M6
// gets dev f(Z) / p by the series, V6 by the directions.
template <typename R>
int both(const double *z3, double alpha, double *M6, double *V6) {
  ft::Sym<R> Z = {{R(z3[0]), R(z3[1]), R(z3[2]), 0, 0, 0}}, Q = {{Z.v[0] * Z.v[0], Z.v[1] * Z.v[1], Z.v[2] * Z.v[2], 0, 0, 0}}, M, V;
  const R rho = ft::Num<R>::sqrt_(Q.v[0] + Q.v[1] + Q.v[2]), p = R(0.5) * R(alpha);
  const bool take = (float)rho <= ft::ogden_range<R>((float)p), ends = ft::ogden_series(Z, Q, rho, p, M);
  ft::ogden_principal(Z, p, V);
  for (int k = 0; k < 6; ++k) {
    M6[k] = ends ? (double)M.v[k] : 0.0;
    V6[k] = (double)V.v[k] / (0.5 * alpha);
  }
  return (take ? 1 : 0) | (ends ? 2 : 0);
}
}  // namespace

extern "C" int oh_both(int fp32, const double *z3, double alpha, double *M6, double *V6) {
  return fp32 ? both<float>(z3, alpha, M6, V6) : both<double>(z3, alpha, M6, V6);
}
