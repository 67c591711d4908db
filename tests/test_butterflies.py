"""The twiddled butterflies of qstem_amd/csrc/qs_fft.hpp compiled for the CPU: each output is as
exact as its own size allows, also where the inputs share a much larger mean, and the
(cos, tan) table of their constants; the DFTs of qs_dft.hpp for the mixed-radix passes."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "qstem_amd", "csrc")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("butterfly") / "harness")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-I" + os.path.join(HERE, "hip_host"), "-I" + CSRC,
                    os.path.join(HERE, "butterfly_harness.cpp"), "-o", exe], check=True)

    def call(text):
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
        return np.array(out.split(), dtype=np.float64).reshape(-1, 2) @ [1, 1j]
    return call


@pytest.mark.parametrize("radix", [2, 4, 8, 16])
@pytest.mark.parametrize("sign", [-1, 1])
def test_differences_keep_their_own_precision(harness, radix, sign):
    rng = np.random.default_rng(radix + 100 * sign + 200)
    noise = 2.0 ** -14
    reps = 200
    # multiples of 2^-23 around 1: first differences are exact (Sterbenz), and the odd outputs
    # are built from them alone
    x = 1.0 + np.round(rng.uniform(-noise, noise, (reps, radix)) * 2 ** 23) / 2 ** 23
    y = np.round(rng.uniform(-noise, noise, (reps, radix)) * 2 ** 23) / 2 ** 23
    a = x + 1j * y
    text = "".join("%d %d %s\n" % (radix, sign, " ".join("%.9g %.9g" % (v.real, v.imag) for v in row)) for row in a)
    got = harness(text).reshape(reps, radix)
    k = np.arange(radix)
    want = a @ np.exp(sign * 2j * np.pi * np.outer(k, k) / radix)
    # each of the later stages (three at most) rounds four times at most, and its constant
    # thrice, values below R sqrt(2) 2 noise
    stages = int(np.log2(radix)) - 1
    odd = slice(1, None, 2)
    bound = max(stages, 1) * 7 * 2.0 ** -24 * radix * np.sqrt(2) * 2 * noise
    assert np.abs(got - want)[:, odd].max() <= bound
    # the others: the same number of roundings at the size of the sums
    assert np.abs(got - want).max() <= (stages + 1) * 7 * 2.0 ** -24 * radix * 1.01


@pytest.mark.parametrize("n", [64, 128, 256, 512, 1024, 2048, 4096])
def test_table_of_cosines_and_tangents(harness, n):
    pairs = harness("table %d\n" % n)
    w = pairs.real * (1 + 1j * pairs.imag)
    exact = np.exp(-2j * np.pi * np.arange(n) / n)
    assert np.all(np.isfinite(w))
    # cosine and tangent within one step (2^-23) of themselves
    assert np.abs(w - exact).max() <= 2 * 2.0 ** -23
    # chosen for the modulus: no worse than the two numbers rounded to nearest
    near = exact.real.astype(np.float32).astype(np.float64)
    with np.errstate(divide="ignore", invalid="ignore"):
        near = near * (1 + 1j * (exact.imag / exact.real).astype(np.float32).astype(np.float64))
    ok = np.abs(exact.real) > 1e-9
    assert np.sum((np.abs(w) - 1)[ok] ** 2) <= np.sum((np.abs(near) - 1)[ok] ** 2)


RADICES = [3, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16, 18, 20, 21, 24, 25, 28, 30]


def _dft(harness, radix, balanced, sign, a):
    a = a.astype(np.complex64)
    return harness("".join("dft %d %d %d %s\n" % (radix, balanced, sign, " ".join("%.9g %.9g" % (v.real, v.imag) for v in row))
                           for row in a)).reshape(a.shape)


@pytest.mark.parametrize("radix", RADICES)
@pytest.mark.parametrize("balanced", [0, 1])
@pytest.mark.parametrize("sign", [-1, 1])
def test_dft_is_linear_in_complex_factors(harness, radix, balanced, sign):
    rng = np.random.default_rng(radix)
    a = (rng.standard_normal((50, radix)) + 1j * rng.standard_normal((50, radix))).astype(np.complex64)
    got = _dft(harness, radix, balanced, sign, a)
    k = np.arange(radix)
    want = a.astype(np.complex128) @ np.exp(sign * 2j * np.pi * np.outer(k, k) / radix)
    # at most five binary or three larger stages, each with a rounded constant: 2^-24 times
    # about twenty roundings of the values' size
    assert np.linalg.norm(got - want) <= 20 * 2.0 ** -24 * np.linalg.norm(want)
    # the real and the imaginary part go through the same constants, so that i times the input
    # (exact) gives i times the output, bit for bit
    assert np.array_equal(_dft(harness, radix, balanced, sign, 1j * a), 1j * got)


def test_constants_rounded_to_nearest_where_not_balanced(harness):
    # the runtime-planned kernels' 7-point DFT: sin(2 pi 3/7) to nearest, the balanced one a step above
    a = np.zeros((1, 7))
    a[0, 1] = 1.0
    near, up = (_dft(harness, 7, b, -1, a)[0] for b in (0, 1))
    s3 = np.float32(np.sin(6 * np.pi / 7))
    assert np.float32(-near[3].imag) == s3 and np.float32(-up[3].imag) == np.nextafter(s3, np.float32(2))
    # 16 points: cos(pi/8) likewise in the turns by 3 and 9 sixteenths alone
    b = np.zeros((1, 16))
    b[0, 1] = 1.0
    near = _dft(harness, 16, 0, -1, b)[0]
    assert np.max(np.abs(near - np.exp(-2j * np.pi * np.arange(16) / 16))) <= 2.0 ** -25
