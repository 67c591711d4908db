// qs_twiddles.hpp -- host tables of the transforms' twiddle factors W_n^m = exp(-2 pi i m/n).
// (No device code: F2 is float2.)
#pragma once
#include <cmath>
#include <cstring>
#include <vector>

namespace qs {

// (cos, sin) pairs rounded to nearest, for the mixed-radix passes: of pairs chosen for their
// modulus as below, the passes' powers w^(k & ~3) w^(k & 3) gather the larger phase error
// (rms over the two-pass lengths: error 1.08e-7 here, 1.13e-7 so; gain 1.2e-8 and 1.1e-8).
template <class F2>
std::vector<F2> twiddles(int n) {
  std::vector<F2> t(n);
  for (int m = 0; m < n; m++) {
    const double a = -2.0 * M_PI * m / n;
    t[m] = F2{(float)cos(a), (float)sin(a)};
  }
  return t;
}

// (cos, tan) pairs, for the fused butterflies of the power-of-two passes (bf_tw).  Where the
// cosine is zero it is 2^-28 and the tangent 2^28, off by 4e-9 of phase.
//
// Rounded with the modulus kept: of the nine neighbouring pairs of floats, the one whose
// squared error along the value, weighted 10 to 1 against the error across it, is least.  A
// modulus error is a gain that every transform applies again, and the sum over the slices of
// a run was the largest error of its detector sums: with (cos, sin) rounded to nearest a
// 512-point transform loses 2.5e-8 of the amplitude, a 4096-point one 3.9e-8; so rounded
// 1.1e-8 and 3e-9.  (Weights 3, 10, 100: gain at 4096 6, 3, 6e-9; rms error at 512 0.98, 0.99,
// 1.00 of that of nearest pairs; dL/dV of probes of 256^2 5.0, 4.7, 4.9e-6.)
template <class F2>
std::vector<F2> butterfly_twiddles(int n) {
  // the k-th float after v (not zero)
  auto step = [](float v, int k) {
    unsigned u;
    memcpy(&u, &v, sizeof u);
    u += k;
    memcpy(&v, &u, sizeof v);
    return v;
  };
  std::vector<F2> t(n);
  for (int m = 0; m < n; m++) {
    const double a = -2.0 * M_PI * m / n, c = cos(a), s = sin(a);
    if (4LL * m % n == 0) {
      t[m] = fabs(c) > 0.5 ? F2{(float)rint(c), 0.f} : F2{0x1p-28f, (float)rint(s) * 0x1p28f};
      continue;
    }
    double best = 1e300;
    for (int i = -1; i <= 1; i++)
      for (int k = -1; k <= 1; k++) {
        const float p = step((float)c, i), q = step((float)(s / c), k);
        const double x = p, y = (double)p * q;
        const double along = 0.5 * (x * x + y * y - 1.0), across = x * s - y * c;
        const double cost = 10.0 * along * along + across * across;
        if (cost < best) {
          best = cost;
          t[m] = F2{p, q};
        }
      }
  }
  return t;
}

}  // namespace qs
