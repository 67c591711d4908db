"""Gradients of several probes in one call equal the sum of single-probe calls: the reverse
row sweep that sums dL/dt of a transmission row in LDS (groups of rows per wavefront, partial
groups and chunks, windows wider than the LDS area, repeated and distinct x offsets)."""
import numpy as np
import pytest

from cases import smooth_potential

pytestmark = pytest.mark.gpu

# n, potNx, potNy, probes: rows per wavefront 4 (64, 128), 2 (256), 1 (512, 1024), block-wide 2048;
# potNx not a multiple of the group; 1824 and 2560 columns exceed the summed span at 256 and 512
CASES = [(64, 67, 80, 2), (64, 131, 64, 37), (128, 129, 150, 70), (256, 301, 259, 21), (256, 258, 2080, 5),
         (512, 515, 521, 9), (512, 512, 2560, 3), (1024, 1026, 1024, 3), (2048, 2048, 2048, 2)]


@pytest.mark.parametrize("n,potx,poty,probes", CASES)
def test_many_probes_equal_the_sum_of_single_ones(n, potx, poty, probes):
    from qstem_amd import Multislice, StemConfig
    cfg = StemConfig(nx=n, ny=n, resolutionX=0.05, resolutionY=0.05, v0=200.0, slices=2, sliceThickness=1.9525,
                     potNx=potx, potNy=poty, bandlimittrans=0, Cs=1.0e4, df0=-50.0, alpha=20.0, electronScale=1.0)
    rng = np.random.default_rng(n + probes)
    # a few distinct x offsets, the corners among them, so that neighbours share one
    xs = np.unique(np.concatenate([[0, potx - n], rng.integers(0, potx - n + 1, 4)]))
    ipos = np.stack([rng.choice(xs, probes), rng.integers(0, poty - n + 1, probes)], 1).astype(np.int32)
    ipos[0], ipos[-1] = (0, 0), (potx - n, poty - n)
    target = rng.uniform(0.0, 2.0 / (n * n), (probes, n, n)).astype(np.float32)
    with Multislice(cfg) as ms:
        ms.set_potential(smooth_potential(2, potx, poty, seed=n))
        ms.make_probe()
        many = ms.adjoint(ipos, target)
        one = [ms.adjoint(ipos[i:i + 1], target[i:i + 1]) for i in range(probes)]
    # sums of `probes` single-precision terms in another order differ by at most
    # 2 (probes + 1) 2^-24 of the sum of their magnitudes; the three transforms between the
    # states and a term are the same instructions on both sides
    size = sum(np.abs(o["grad_V"].astype(np.float64)) for o in one)
    total = sum(o["grad_V"].astype(np.float64) for o in one)
    # dL/dV takes two components of the summed dL/dt, each of which may be larger than their
    # difference: 4 for the pair, and the largest pixel's size as the scale of a component
    bound = 4 * 2 * (probes + 1) * 2.0 ** -24 * np.maximum(size, size.max())
    assert np.all(np.abs(many["grad_V"] - total) <= bound)
    for key in ("grad_df0", "grad_Cs"):
        want = sum(o[key] for o in one)
        assert abs(many[key] - want) <= 1e-5 * sum(abs(o[key]) for o in one) + 1e-30
