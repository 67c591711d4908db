// qs_twiddles.hpp -- host tables of the transforms' twiddle factors W_n^m = exp(-2 pi i m/n),
// each rounded to two floats with its modulus kept.  (No device code: F2 is float2.)
//
// A modulus error is a gain that every transform applies again, and the sum over the slices
// of a run was the largest error of its detector sums: rounding both numbers to nearest, a
// 512-point transform loses 2.5e-8 of the amplitude.  Of the nine neighbouring pairs of
// floats the tables take the one whose squared error along the value, weighted against the
// error across it, is least; an error across it is noise.
#pragma once
#include <cmath>
#include <cstring>
#include <vector>

namespace qs {

// The k-th float after v (k = -1, 0, 1; v is not zero).
inline float float_step(float v, int k) {
  unsigned u;
  memcpy(&u, &v, sizeof u);
  u += k;
  memcpy(&v, &u, sizeof v);
  return v;
}

// Pair (p, q) next to (p0, q0) that represents exp(i a) = c + i s best; value(p, q, x, y) gives
// the complex number x + i y that the pair stands for.
template <class F2, class V>
F2 round_pair(float p0, float q0, double c, double s, double weight, V value) {
  F2 pair{p0, q0};
  double best = 1e300;
  for (int i = -1; i <= 1; i++)
    for (int k = -1; k <= 1; k++) {
      const float p = float_step(p0, i), q = float_step(q0, k);
      double x, y;
      value((double)p, (double)q, x, y);
      const double along = 0.5 * (x * x + y * y - 1.0), across = x * s - y * c;
      const double cost = weight * along * along + across * across;
      if (cost < best) {
        best = cost;
        pair = F2{p, q};
      }
    }
  return pair;
}

// (cos, sin) pairs, for the mixed-radix passes.
template <class F2>
std::vector<F2> twiddles(int n) {
  std::vector<F2> t(n);
  for (int m = 0; m < n; m++) {
    const double a = -2.0 * M_PI * m / n, c = cos(a), s = sin(a);
    if (4LL * m % n == 0) t[m] = F2{(float)rint(c), (float)rint(s)};  // quarter turns are exact
    else
      t[m] = round_pair<F2>((float)c, (float)s, c, s, 100.0, [](double p, double q, double& x, double& y) {
        x = p;
        y = q;
      });
  }
  return t;
}

// (cos, tan) pairs, for the fused butterflies of the power-of-two passes (bf_tw).  Where the
// cosine is zero it is 2^-28 and the tangent 2^28, off by 4e-9 of phase.
template <class F2>
std::vector<F2> butterfly_twiddles(int n) {
  std::vector<F2> t(n);
  for (int m = 0; m < n; m++) {
    const double a = -2.0 * M_PI * m / n, c = cos(a), s = sin(a);
    if (4LL * m % n == 0) {
      t[m] = fabs(c) > 0.5 ? F2{(float)rint(c), 0.f} : F2{0x1p-28f, (float)rint(s) * 0x1p28f};
      continue;
    }
    t[m] = round_pair<F2>((float)c, (float)(s / c), c, s, 3.0, [](double p, double q, double& x, double& y) {
      x = p;
      y = p * q;
    });
  }
  return t;
}

}  // namespace qs
