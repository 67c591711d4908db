// qs_pair.hip -- per-length instantiation of the two-pass sweeps (qs_pair.hpp).
// Compiled once per length of QS_PAIR_SIZES that runs, with -DQS_PAIR_N=<n>, so the lengths
// build in parallel.
#include "qs_pair.hpp"

#ifndef QS_PAIR_N
#error "compile with -DQS_PAIR_N=<a length of QS_PAIR_SIZES>"
#endif
namespace qs {
static_assert(pair_r1(QS_PAIR_N) > 0, "no pair of radices for this length");
template <int N> int pair_cpb() { return Pair<N>::CPB; }
template void launch_pair_rows_t<QS_PAIR_N>(const GenRowArgs&, hipStream_t);
template void launch_pair_cols_t<QS_PAIR_N>(const GenColArgs&, int, hipStream_t);
template int pair_cpb<QS_PAIR_N>();
}  // namespace qs
