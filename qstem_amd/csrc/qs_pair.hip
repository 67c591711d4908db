// qs_pair.hip -- per-length instantiation of the two-pass sweeps (qs_pair.hpp).
// Compiled once per length of QS_PAIR_SIZES with -DQS_PAIR_N=<n> so the lengths build in
// parallel.
#include "qs_pair.hpp"

#ifndef QS_PAIR_N
#error "compile with -DQS_PAIR_N=<a length of QS_PAIR_SIZES>"
#endif
#define QS_CAT2(a, b) a##b
#define QS_CAT(a, b) QS_CAT2(a, b)

namespace qs {
static_assert(pair_r1(QS_PAIR_N) > 0, "no pair of radices for this length");
void QS_CAT(pair_rows_, QS_PAIR_N)(const GenRowArgs& a, hipStream_t st) { launch_pair_rows_t<QS_PAIR_N>(a, st); }
void QS_CAT(pair_cols_, QS_PAIR_N)(const GenColArgs& a, int nblocks, hipStream_t st) {
  launch_pair_cols_t<QS_PAIR_N>(a, nblocks, st);
}
int QS_CAT(pair_cpb_, QS_PAIR_N)() { return Pair<QS_PAIR_N>::CPB; }
}  // namespace qs
