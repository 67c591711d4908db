"""Runs of small windows in one launch (qs_slab.hip) against the two sweeps (which per-launch
profiling keeps) and the FP64 oracle: every window shape, one and many probes, phonon
configurations, detectors with shifts, outputs at several slices, a continued run, and more
slices than one launch takes."""
import numpy as np
import pytest

from cases import probe_positions, rel_l2, small_config, smooth_potential

pytestmark = pytest.mark.gpu

# a transform's rms error stays below 2e-7 on either side; four transforms per slice
TOL = 4 * 2e-7


@pytest.mark.parametrize("nx,ny,probes", [(64, 64, 1), (64, 128, 5), (128, 64, 3), (128, 128, 24), (128, 128, 300)])
def test_slab_matches_sweeps_and_oracle(oracle, nx, ny, probes):
    from qstem_amd import Multislice
    cfg = small_config(nx=nx, ny=ny, pad=9, slices=6, dx=0.04)
    V = [smooth_potential(cfg.slices, cfg.potNx, cfg.potNy, seed=k) for k in (3, 4)]
    ipos = probe_positions(cfg, probes, seed=5)
    config = (np.arange(probes) % 2).astype(np.int32)
    bins, nbins = oracle.record_bins(cfg.slices, outputInterval=2)
    kw = dict(bins=bins, nbins=nbins, config=config, want_exit=True, want_diff=True, want_intensity=True)
    with Multislice(cfg) as ms:
        ms.set_configs(2)
        for k in range(2):
            ms.select_config(k)
            ms.set_potential(V[k])
        psi0 = ms.make_probe()
        one = ms.run_stem(ipos, **kw)
        first = ms.run_stem(ipos, nslice=4, bins=bins[:4], nbins=nbins, config=config)
        rest = ms.run_stem(ipos, nslice=2, first_slice=4, start=1, bins=bins[4:], nbins=nbins, det=first["det"],
                           config=config, want_exit=True)
        ms.set_graph(True)
        graph = [ms.run_stem(ipos, **kw) for _ in range(3)]
        ms.set_graph(False)
        ms.set_profiling(True)
        two = ms.run_stem(ipos, **kw)
        ms.set_profiling(False)
        ms.select_config(1)
        t1 = ms.get_trans()
    assert np.array_equal(rest["exit"], one["exit"]) and np.array_equal(rest["det"], one["det"])
    for g in graph:
        assert all(np.array_equal(g[k], one[k]) for k in ("exit", "det", "diff", "intensity"))
    tol = cfg.slices * TOL
    assert rel_l2(one["exit"], two["exit"]) < 2 * tol
    assert rel_l2(one["diff"], two["diff"]) < 4 * tol
    assert rel_l2(one["det"], two["det"]) < 4 * tol
    assert np.allclose(one["intensity"], two["intensity"], rtol=4 * tol)
    sel = np.nonzero(config == 1)[0][:2]
    if len(sel):
        ex, det, diff = oracle.multislice(cfg, t1.astype(np.complex128), ipos[sel], psi0.astype(np.complex128),
                                          bins=bins, nbins=nbins, want_diff=True)
        assert rel_l2(one["exit"][sel], ex) < tol
        assert rel_l2(one["diff"][sel], diff) < 2 * tol
        for b in range(nbins):
            for d in range(det.shape[1]):
                if np.any(det[b, d]):
                    assert rel_l2(one["det"][b, d, sel], det[b, d]) < 2 * tol


def test_slab_more_slices_than_one_launch():
    from qstem_amd import Multislice, record_bins
    cfg = small_config(nx=64, ny=64, pad=2, slices=1030)
    V = smooth_potential(cfg.slices, cfg.potNx, cfg.potNy, seed=9, vmax=2.0)
    ipos = probe_positions(cfg, 2, seed=1)
    bins, nbins = record_bins(cfg.slices, outputInterval=500)
    with Multislice(cfg) as ms:
        ms.set_potential(V)
        ms.make_probe()
        one = ms.run_stem(ipos, bins=bins, nbins=nbins, want_exit=True)
        ms.set_profiling(True)
        two = ms.run_stem(ipos, bins=bins, nbins=nbins, want_exit=True)
    assert rel_l2(one["exit"], two["exit"]) < 2 * cfg.slices * TOL
    assert rel_l2(one["det"], two["det"]) < 4 * cfg.slices * TOL
