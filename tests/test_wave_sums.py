"""Sums over a wavefront's lanes (wave_sum, detector_sums, __shfl_xor) stand only where all of
its lanes arrive: HIP leaves open what a shuffle reads from a lane that is switched off.  The
kernels' sources are searched for such a call inside a branch on anything but values that
are the same for the whole wavefront."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qstem_amd", "csrc")
CALL = re.compile(r"\b(wave_sum\(|detector_sums<|__shfl_xor\()")
# conditions on kernel arguments alone, or on a probe per wavefront (k_reduce_partials: p)
UNIFORM = {"rec", "a.rec", "p >= nprobe"}


def _enclosing(text, at):
    """Heads of the blocks that hold position `at`, innermost first, up to the function."""
    depth, heads, i = 0, [], at
    while i > 0:
        i -= 1
        if text[i] == "}":
            depth += 1
        elif text[i] == "{":
            if depth:
                depth -= 1
                continue
            start = max(text.rfind(c, 0, i) for c in ";{}")
            heads.append(" ".join(text[start + 1:i].split()))
            if text[start + 1:i].lstrip().startswith(("template", "__global__", "__device__")):
                break
    return heads


def _statement(text, at):
    start = max(text.rfind(c, 0, at) for c in ";{}")
    return " ".join(text[start + 1:at].split())


@pytest.mark.parametrize("name", sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".hpp"))))
def test_lane_sums_are_not_inside_lane_branches(name):
    text = re.sub(r"//[^\n]*|^[ \t]*#[^\n]*", "", open(os.path.join(CSRC, name)).read(), flags=re.M)
    for m in CALL.finditer(text):
        for head in [_statement(text, m.start())] + _enclosing(text, m.start()):
            for cond in re.findall(r"\bif \((.*?)\)(?= |$)", re.sub(r"\bif constexpr \([^)]*\)", "", head)):
                assert cond in UNIFORM, "%s: %s inside if (%s)" % (name, m.group(1), cond)
            assert not re.search(r"\belse$", head), "%s: %s inside an else branch" % (name, m.group(1))
