"""The two-pass sweeps (qs_pair.hpp) against the FP64 oracle and against the runtime-planned
kernels: one to eight transforms per wavefront, unequal and equal radices, radix 27 and 32,
partial column blocks and row steps, powers of two beside other lengths."""
import numpy as np
import pytest

from cases import probe_positions, rel_l2, small_config, smooth_potential

pytestmark = pytest.mark.gpu

SHAPES = [(64, 72), (80, 64), (96, 126), (135, 100), (225, 240), (243, 81), (336, 480), (400, 400), (512, 210),
          (288, 1024), (630, 560), (900, 128), (729, 135), (960, 70)]


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_pair_sweeps_match_oracle_and_runtime_plans(oracle, monkeypatch, nx, ny):
    from qstem_amd import Multislice
    cfg = small_config(nx=nx, ny=ny, pad=7, slices=3, dx=0.04)
    V = smooth_potential(cfg.slices, cfg.potNx, cfg.potNy, seed=nx)
    ipos = probe_positions(cfg, 5, seed=ny)
    bins, nbins = oracle.record_bins(cfg.slices, outputInterval=2)
    outs = []
    for plans in ("1", "0"):
        monkeypatch.setenv("QSTEM_COMPILED_PLANS", plans)
        with Multislice(cfg) as ms:
            ms.set_potential(V)
            psi0 = ms.make_probe()
            trans = ms.get_trans()
            ms.set_batch(3)
            outs.append(ms.run_stem(ipos, bins=bins, nbins=nbins, want_exit=True, want_diff=True, want_intensity=True))
            if plans == "1":  # other rows per slot: the same sums in the same order
                ms.set_tuning(1, 0)
                again = ms.run_stem(ipos, bins=bins, nbins=nbins, want_exit=True)
                assert np.array_equal(again["exit"], outs[0]["exit"])
    ex, det, diff = oracle.multislice(cfg, trans.astype(np.complex128), ipos, psi0.astype(np.complex128), bins=bins,
                                      nbins=nbins, want_diff=True)
    # a transform's rms error stays below 4e-7 (two passes of at most five binary stages, and
    # twiddles that are products of two rounded ones); four transforms in each of three slices
    tol = 12 * 4e-7
    for out in outs:
        assert rel_l2(out["exit"], ex) < tol
        assert rel_l2(out["diff"], diff) < 2 * tol
        for b in range(nbins):
            for d in range(det.shape[1]):
                if np.any(det[b, d]):
                    assert rel_l2(out["det"][b, d], det[b, d]) < 2 * tol
        assert np.allclose(out["intensity"], np.sum(np.abs(ex) ** 2, axis=(1, 2)) / (nx * ny), rtol=2 * tol)
    assert rel_l2(outs[0]["exit"], outs[1]["exit"]) < 2 * tol
