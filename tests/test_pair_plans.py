"""The two-pass plans (qstem_amd/csrc/qs_pair.hpp) on the CPU: QS_PAIR_SIZES is every
product of two of its radices from 64 to 1024, each length's transforms fit a wavefront and
its slot, and the kernels' index scheme (element j + k RB of lane j in, exchange at
k (RB | 1) + j, twiddles W_N^(k j), element j + k RA out) run with numpy DFTs gives numpy's
FFT in both directions, first radix R0 then R1 and R1 then R0."""
import os
import re

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qstem_amd", "csrc")


def _sizes():
    text = open(os.path.join(CSRC, "qs_internal.hpp")).read()
    m = re.search(r"#define QS_PAIR_SIZES\(X\)((?:[ \t]*\\\n|[ \t]*X\(\d+\))+)", text)
    return [int(n) for n in re.findall(r"X\((\d+)\)", m.group(1))]


def _radices():
    text = open(os.path.join(CSRC, "qs_pair.hpp")).read()
    return [int(r) for r in re.search(r"constexpr int set\[\] = \{([^}]*)\}", text).group(1).split(",")]


def _pair(n):
    return next(((n // r, r) for r in range(8, 33) if n % r == 0 and r in _radices() and n // r in _radices() and n // r <= r), None)


def _slot(n, r0, r1):
    ld = max(n, r0 * (r1 | 1), r1 * (r0 | 1))
    want = 1 if 64 // r1 >= 4 else 4
    while ld % 32 != want:
        ld += 1
    return ld


def _dft(x, sign):
    k = np.arange(len(x))
    return np.exp(sign * 2j * np.pi * np.outer(k, k) / len(x)) @ x


def _transform(x, ra, rb, ld, sign):
    n = ra * rb
    slot = np.full(ld, np.nan + 0j)
    for t in range(rb):
        y = _dft(np.array([x[t + k * rb] for k in range(ra)]), sign)
        for k in range(ra):
            assert np.isnan(slot[k * (rb | 1) + t])
            slot[k * (rb | 1) + t] = y[k]
    out = np.empty(n, complex)
    for t in range(ra):
        v = np.array([slot[t * (rb | 1) + k] * np.exp(sign * 2j * np.pi * k * t / n) for k in range(rb)])
        out[[t + k * ra for k in range(rb)]] = _dft(v, sign)
    return out


def test_sizes_are_the_products_of_the_radices():
    s = _radices()
    assert sorted(_sizes()) == sorted({a * b for a in s for b in s if 64 <= a * b <= 1024})


@pytest.mark.parametrize("n", _sizes())
def test_pair_transforms(n):
    r0, r1 = _pair(n)
    ld = _slot(n, r0, r1)
    assert r0 * r1 == n and r0 <= r1 <= 32
    assert 4 * (64 // r1) * ld * 8 <= 160 * 1024  # a block's slots
    x = np.random.default_rng(n).standard_normal((n, 2)) @ [1, 1j]
    for sign, ref in ((-1, np.fft.fft(x)), (+1, np.fft.ifft(x) * n)):
        assert np.allclose(_transform(x, r0, r1, ld, sign), ref, atol=1e-9 * n)
        assert np.allclose(_transform(x, r1, r0, ld, sign), ref, atol=1e-9 * n)
