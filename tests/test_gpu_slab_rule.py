"""Which kernels a small window's run takes: the one-launch kernel, or the two sweeps (which
per-launch profiling keeps too) for the per-probe launch sequence of a group size of 1; and
the autotuner, which leaves the group size of such windows to the library."""
import numpy as np
import pytest

from cases import probe_positions, small_config, smooth_potential

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,probes", [(64, 64, 1), (64, 128, 3), (128, 128, 30), (128, 128, 5)])
def test_set_group_size_and_autotuner(nx, ny, probes):
    from qstem_amd import Multislice
    cfg = small_config(nx=nx, ny=ny, pad=9, slices=9, dx=0.04)
    ipos = probe_positions(cfg, probes, seed=7)
    with Multislice(cfg) as ms:
        ms.set_potential(smooth_potential(cfg.slices, cfg.potNx, cfg.potNy, seed=nx))
        ms.make_probe()
        whole = ms.run_stem(ipos, want_exit=True)["exit"]
        ms.set_profiling(True)
        sweeps = ms.run_stem(ipos, want_exit=True)["exit"]
        ms.set_profiling(False)
        one_launch = nx * ny < 128 * 128 or probes >= 24
        assert np.array_equal(whole, sweeps) == (not one_launch)
        for batch, want in ((1, sweeps), (4, whole)):
            ms.set_batch(batch)
            assert np.array_equal(ms.run_stem(ipos, want_exit=True)["exit"], want)
        ms.set_batch(0)
        best = ms.autotune(ipos)
        assert best["batch"] == 0 and ms.get_tuning()[2] == 0 and best["rate"] > 0
        assert np.array_equal(ms.run_stem(ipos, want_exit=True)["exit"], whole)
        ms.autotune(ipos)  # from the cache
        assert np.array_equal(ms.run_stem(ipos, want_exit=True)["exit"], whole)
