// Reads "radix dir" and 2 R numbers per line, applies the twiddled radix-R butterfly of
// qs_fft.hpp with the constants of a transform's first thread (w = 1), and writes the 2 R
// results.  "table n" writes the n (cos, tan) pairs of butterfly_twiddles; "dft radix balanced
// dir" and 2 R numbers the results of qs_dft.hpp's DFT.
#include <cstdio>
#include <cstring>

#include "qs_dft.hpp"
#include "qs_fft.hpp"
#include "qs_twiddles.hpp"

using namespace qs;

template <int R, int DIR>
static void apply(float2* a) {
  constexpr int N = 4096;
  const auto table = butterfly_twiddles<float2>(N);
  float2 c[R / 2];
  tw_load<N, R>(c, table.data(), 0);
  dft_tw<R, DIR>(a, c);
}
template <int R>
static void apply(int dir, float2* a) {
  if (dir < 0) apply<R, -1>(a);
  else apply<R, +1>(a);
}

template <int R>
static bool plain(int r, int balanced, int dir, float2* a) {
  if (r != R) return false;
  if (balanced && dir < 0) dft_any<R, -1, true>(a);
  else if (balanced) dft_any<R, +1, true>(a);
  else if (dir < 0) dft_any<R, -1, false>(a);
  else dft_any<R, +1, false>(a);
  return true;
}
template <int... R>
static void plain_of(int r, int balanced, int dir, float2* a) {
  (plain<R>(r, balanced, dir, a) || ...);
}

int main() {
  char word[16];
  while (scanf("%15s", word) == 1) {
    int r, dir;
    if (!strcmp(word, "table")) {
      if (scanf("%d", &r) != 1) return 1;
      for (const float2& w : butterfly_twiddles<float2>(r)) printf("%.9g %.9g\n", w.x, w.y);
      continue;
    }
    if (!strcmp(word, "dft")) {
      int balanced;
      float2 a[32];
      if (scanf("%d %d %d", &r, &balanced, &dir) != 3 || r > 32) return 1;
      for (int k = 0; k < r; k++)
        if (scanf("%f %f", &a[k].x, &a[k].y) != 2) return 1;
      plain_of<3, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16, 18, 20, 21, 24, 25, 28, 30>(r, balanced, dir, a);
      for (int k = 0; k < r; k++) printf("%.9g %.9g\n", a[k].x, a[k].y);
      continue;
    }
    if (sscanf(word, "%d", &r) != 1 || scanf("%d", &dir) != 1 || r > 16) return 1;
    float2 a[16];
    for (int k = 0; k < r; k++)
      if (scanf("%f %f", &a[k].x, &a[k].y) != 2) return 1;
    if (r == 2) apply<2>(dir, a);
    else if (r == 4) apply<4>(dir, a);
    else if (r == 8) apply<8>(dir, a);
    else apply<16>(dir, a);
    for (int k = 0; k < r; k++) printf("%.9g %.9g\n", a[k].x, a[k].y);
  }
  return 0;
}
