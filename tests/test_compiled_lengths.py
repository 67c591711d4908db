"""The build compiles one plan per length: no length's kernels are built that the dispatch
(compiled_plan of qs_generic.hip, over the same lists of qs_internal.hpp) does not reach."""
from qstem_amd import build


def test_one_compiled_plan_per_length():
    mix, pair = build.mix_sizes(), build.pair_sizes()
    assert len(set(mix)) == len(mix) and len(set(pair)) == len(pair)
    assert not set(mix) & set(pair)
    assert set(mix) <= set(build._listed("QS_MIX_SIZES"))
    assert set(mix) | set(pair) == set(build._listed("QS_MIX_RUN")) | set(build._listed("QS_PAIR_SIZES"))
