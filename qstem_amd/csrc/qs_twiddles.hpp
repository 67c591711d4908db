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
// squared error along the value, weighted 30 to 1 against the error across it, is least.  A
// modulus error is a gain that every transform applies again, and the sum over the slices of
// a run was the largest error of its detector sums: with (cos, sin) rounded to nearest a
// 512-point transform loses 2.5e-8 of the amplitude, a 4096-point one 3.9e-8; so rounded
// 1.3e-8 and 6e-9.  The weight is the one whose results were nearest to 64-bit ones: weights
// 10, 30 and 100 give rms errors of dL/dV of 24 images of various sizes of 4.0, 3.7 and
// 4.8e-6, and mean errors of dL/d(df0) of four sets of 1024 probes of 256^2 of 7.6, 2.0 and
// 1.6e-6.  The error of a 512-point transform of random data is 1.00 (weight 10) or 1.02 (30)
// of that with separate products by the nearest (cos, sin) at most.
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
        const double cost = 30.0 * along * along + across * across;
        if (cost < best) {
          best = cost;
          t[m] = F2{p, q};
        }
      }
  }
  return t;
}

}  // namespace qs
