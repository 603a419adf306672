"""The path search's open list between its two places, against the oracle bit for bit: halls without obstacles, whose lists
come to 38 up to 224 entries (54 are sorted at most), so that entries are moved out of the registers and come back, those of
nodes that have been updated meanwhile among them, and the longest lists go on as the reference's heap."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


# calls that a search per block serves, with the whole pool in LDS and without, and calls beyond
@pytest.mark.parametrize("n", [300, 1500, 4000])
@pytest.mark.parametrize("edge,outgrown", [(4.0, False), (7.0, False), (11.0, False), (11.0, True)])
def test_lists_of_all_lengths_match_oracle(oracle, edge, outgrown, n):
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: a hall of {edge} m, {n} searches", flush=True)
    blob = scenes.gen_scene(scenes.BOX_ROOM, 3, cell=5, size_x=edge, size_z=edge, num_boxes=0)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    x, r = cpu.snap(scenes.sample_points(blob, 21, 600))
    a, ar, b, br = x[:300], r[:300], x[300:].copy(), r[300:]
    # one in three leaves the mesh: its totals differ by their last bits only, or, further out, are the same for hundreds of nodes
    b[::3, 0] += np.float32(1e7 if outgrown else 2e3)
    want = cpu.geodesic(a, ar, b, br)
    at = np.arange(n) % 300
    got = gpu.geodesic(0, a[at], ar[at], b[at], br[at])
    c = gpu.counters()
    cpu.close()
    gpu.close()
    assert np.array_equal(common.bits(want)[at], common.bits(got))
    assert (c["geo_exact_runs"] > 0) == outgrown, c
