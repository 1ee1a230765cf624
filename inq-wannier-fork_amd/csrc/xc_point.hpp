// Point functions of the generalised gradient approximation.
#pragma once

#include <cmath>

namespace inqamd {

// PBE (Perdew, Burke, Ernzerhof 1996), one spin component: energy per
// particle e, vn = d(n e)/dn and vs = d(n e)/dsigma (sigma = |grad n|^2);
// the uniform-gas correlation is Perdew-Wang 1992 with libxc's LDA_C_PW_MOD
// parameters, as GGA_C_PBE uses it.
__device__ inline void pbe_exchange(double n, double sigma, double &e, double &vn, double &vs) {
  const double kappa = 0.8040, mu = 0.2195149727645171;
  const double ax = -0.75 * cbrt(3.0 / M_PI);
  const double n13 = cbrt(n);
  const double n83 = n13 * n13 * n * n;                                // n^(8/3)
  const double c = 4.0 * pow(3.0 * M_PI * M_PI, 2.0 / 3.0);
  const double x = sigma / (c * n83);                                  // s^2
  const double den = 1.0 + mu * x / kappa;
  const double F = 1.0 + kappa - kappa / den, dF = mu / (den * den);
  e = ax * n13 * F;
  vn = ax * n13 * ((4.0 / 3.0) * F - (8.0 / 3.0) * x * dF);
  vs = ax * n13 * n * dF / (c * n83);
}

__device__ inline void pbe_correlation(double n, double sigma, double &e, double &vn, double &vs) {
  const double beta = 0.06672455060314922, gamma = (1.0 - M_LN2) / (M_PI * M_PI);
  const double A0 = 0.0310907, a1 = 0.21370, b1 = 7.5957, b2 = 3.5876, b3 = 1.6382,
               b4 = 0.49294;
  const double rs = cbrt(3.0 / (4.0 * M_PI * n)), sq = sqrt(rs);
  const double q0 = -2.0 * A0 * (1.0 + a1 * rs);
  const double q1 = 2.0 * A0 * (b1 * sq + b2 * rs + b3 * rs * sq + b4 * rs * rs);
  const double q1p = A0 * (b1 / sq + 2.0 * b2 + 3.0 * b3 * sq + 4.0 * b4 * rs);
  const double lg = log(1.0 + 1.0 / q1);
  const double ec = q0 * lg;
  const double dec = (-2.0 * A0 * a1 * lg - q0 * q1p / (q1 * q1 + q1)) * (-rs / (3.0 * n));
  const double kf = cbrt(3.0 * M_PI * M_PI * n);
  const double ty = M_PI / (16.0 * kf * n * n);  // t^2 / sigma
  const double y = sigma * ty;
  const double ex = exp(-ec / gamma);
  const double A = (beta / gamma) / (ex - 1.0);
  const double dA = (beta / (gamma * gamma)) * ex / ((ex - 1.0) * (ex - 1.0));
  const double P = 1.0 + A * y, D = 1.0 + A * y + A * A * y * y;
  const double N = (beta / gamma) * y * P / D;
  const double H = gamma * log(1.0 + N);
  const double dNy = (beta / gamma) * ((P + A * y) * D - y * P * (A + 2.0 * A * A * y)) / (D * D);
  const double dNA = (beta / gamma) * y * (y * D - P * (y + 2.0 * A * y * y)) / (D * D);
  const double g = gamma / (1.0 + N);
  e = ec + H;
  vn = e + n * (dec + g * dNA * dA * dec - g * dNy * (7.0 / 3.0) * y / n);
  vs = n * g * dNy * ty;
}

// which: 1 = exchange, 2 = correlation, 3 = both; densities below 1e-15 give 0
__device__ inline void gga_point(double n, double sigma, int which, double &e, double &vn,
                                 double &vs) {
  e = vn = vs = 0.0;
  if (!(n >= 1e-15)) return;
  double e1, v1, s1;
  if (which & 1) {
    pbe_exchange(n, sigma, e1, v1, s1);
    e += e1, vn += v1, vs += s1;
  }
  if (which & 2) {
    pbe_correlation(n, sigma, e1, v1, s1);
    e += e1, vn += v1, vs += s1;
  }
}

}  // namespace inqamd
