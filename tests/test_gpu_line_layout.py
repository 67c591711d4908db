"""Windows whose two axes use different kernels of the sweeps: the state's lines of four rows
at nx = 4096 under every row transform, and every column kernel under rows of 4096, against
the FP64 oracle; gradients of several probes there against the sum of single-probe calls."""
import numpy as np
import pytest

from cases import probe_positions, rel_l2, small_config, smooth_potential

pytestmark = pytest.mark.gpu

# a transform's rms error stays below 2e-7; four transforms per slice
TOL = 4 * 2e-7
SHAPES = [(4096, 64), (4096, 128), (4096, 256), (4096, 512), (4096, 1024), (4096, 2048), (64, 4096), (128, 4096),
          (256, 4096), (512, 4096), (2048, 4096)]


def _config(nx, ny, pad, slices):
    cfg = small_config(nx=nx, ny=ny, pad=pad, slices=slices, dx=0.04, bandlimit=0)
    cfg.potNx, cfg.potNy = nx + (pad if nx < 2048 else 0), ny + (pad if ny < 2048 else 0)
    return cfg


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_mixed_axes_match_oracle(oracle, nx, ny):
    from qstem_amd import Multislice
    cfg = _config(nx, ny, 7, 2)
    V = smooth_potential(cfg.slices, cfg.potNx, cfg.potNy, seed=nx + ny)
    ipos = probe_positions(cfg, 2, seed=4)
    bins, nbins = oracle.record_bins(cfg.slices, outputInterval=1)
    with Multislice(cfg) as ms:
        ms.set_potential(V)
        psi0 = ms.make_probe()
        t = ms.get_trans()
        out = ms.run_stem(ipos, bins=bins, nbins=nbins, want_exit=True, want_diff=True)
    ex, det, diff = oracle.multislice(cfg, t.astype(np.complex128), ipos, psi0.astype(np.complex128), bins=bins,
                                      nbins=nbins, want_diff=True)
    tol = cfg.slices * TOL
    assert rel_l2(out["exit"], ex) < tol
    assert rel_l2(out["diff"], diff) < 2 * tol
    assert rel_l2(out["det"], det) < 4 * tol


@pytest.mark.parametrize("nx,ny", [(4096, 64), (4096, 512), (64, 4096), (256, 128), (128, 512)])
def test_gradients_of_mixed_axes(nx, ny):
    from qstem_amd import Multislice
    cfg = _config(nx, ny, 9, 2)
    probes = 3
    ipos = probe_positions(cfg, probes, seed=2)
    rng = np.random.default_rng(nx)
    target = rng.uniform(0.0, 2.0 / (nx * ny), (probes, nx, ny)).astype(np.float32)
    with Multislice(cfg) as ms:
        ms.set_potential(smooth_potential(cfg.slices, cfg.potNx, cfg.potNy, seed=ny))
        ms.make_probe()
        many = ms.adjoint(ipos, target)
        one = [ms.adjoint(ipos[i:i + 1], target[i:i + 1]) for i in range(probes)]
    # sums of three single-precision terms in another order: 2 (probes + 1) 2^-24 of the sum
    # of their magnitudes for each of the two components of a pixel of dL/dt (4 for the pair)
    size = sum(np.abs(o["grad_V"].astype(np.float64)) for o in one)
    total = sum(o["grad_V"].astype(np.float64) for o in one)
    bound = 4 * 2 * (probes + 1) * 2.0 ** -24 * np.maximum(size, size.max())
    assert np.all(np.abs(many["grad_V"] - total) <= bound)
    # one context's loss: the intensity of the oracle-checked forward run
    want = sum(o["loss"] for o in one)
    assert abs(many["loss"] - want) <= 1e-5 * abs(want)
