// qs_mix.hip -- per-length instantiation of the compiled-plan sweeps (qs_mix.hpp).
// Compiled once per length of QS_MIX_RUN with -DQS_MIX_N=<n> so the lengths build in
// parallel.
#include "qs_mix.hpp"

#ifndef QS_MIX_N
#error "compile with -DQS_MIX_N=<a length of QS_MIX_SIZES>"
#endif
namespace qs {
static_assert(MixPlan<QS_MIX_N>::E > 0, "no compiled plan for this length");
template <int N> int mix_cols_block() { return mix_cpb<N>(); }
template void launch_mix_rows_t<QS_MIX_N>(const GenRowArgs&, hipStream_t);
template void launch_mix_cols_t<QS_MIX_N>(const GenColArgs&, int, hipStream_t);
template int mix_cols_block<QS_MIX_N>();
}  // namespace qs
