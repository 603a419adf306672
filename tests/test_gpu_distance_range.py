"""Path searches over distances whose squares are infinite, the largest floats, no normal ones, or zero, against the oracle bit for bit."""
import numpy as np
import pytest

from tests import common

pytestmark = pytest.mark.gpu


# calls that a search per block serves, with the whole pool in LDS and without, and calls beyond
@pytest.mark.parametrize("n", [600, 1500, 4000])
@pytest.mark.parametrize("unit", [1e18, 1e17, 1e16, 1e-3, 1e-18, 1e-21, 1e-22, 1e-23, 1e-24, 1e-25, 3e-26])
def test_distances_of_all_sizes_match_oracle(oracle, unit, n):
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: portals {unit} apart, {n} searches", flush=True)
    for seed in range(4):
        blob, near = common.crossing_portals(seed, 100, unit)
        cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
        refs = cpu.poly_info()[0]
        (a, ar), (b, br) = near(refs, 600), near(refs, 600)
        a[::3] *= np.float32(1e-3)   # (points with infinite squares on both sides count as one place)
        b[::5] *= np.float32(1e-4)
        want = cpu.geodesic(a, ar, b, br)
        at = np.arange(n) % 600
        got = gpu.geodesic(0, a[at], ar[at], b[at], br[at])
        pops = gpu.counters()["astar_pops"]
        cpu.close()
        gpu.close()
        assert np.isfinite(want).mean() > 0.5 and pops > n
        differ = np.nonzero(common.bits(want)[at] != common.bits(got))[0]
        assert len(differ) == 0, (seed, len(differ), differ[:8], want[at][differ[:5]], got[differ[:5]])
