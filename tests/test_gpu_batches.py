"""Batched queries of every size on a simulator that has fewer envs than the batch has items: the
number of wavefronts that serve a batch follows the batch, not the envs.  Compared with the oracle
bit for bit."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 513, 2304, 2305, 9001])
def test_batch_sizes(oracle, n):
    """Up to 2304 path queries get a block of two wavefronts each (nine blocks on each of 256 CUs),
    more share them; up to 8192 snaps get a wavefront each."""
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: batches of {n}", flush=True)
    blob = scenes.config_scene(2, 3)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    pts = scenes.sample_points(blob, 17, 2 * n) + np.random.default_rng(n).normal(0, 0.2, (2 * n, 3)).astype(np.float32)
    xo, ro = cpu.snap(pts)
    xg, rg = gpu.snap_points(0, pts)
    assert np.array_equal(ro, rg) and np.array_equal(common.bits(xo), common.bits(xg))
    d = gpu.geodesic(0, xo[:n], ro[:n], xo[n:], ro[n:])
    assert np.array_equal(common.bits(cpu.geodesic(xo[:n], ro[:n], xo[n:], ro[n:])), common.bits(d))
    cpu.close()
    gpu.close()
