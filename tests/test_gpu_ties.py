"""Path searches in which many open nodes share the smallest total, against the oracle bit for bit.  The
end point lies in a polygon of the mesh by its reference and far away by its coordinates, as far as the
interface allows: a step's length is lost in the rounding of the totals, which then collapse to a few
values or to one.  The order in which the reference's heap has equal totals decides the corridor."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


# calls small enough for a wavefront with the whole pool in LDS each, for a block each, and beyond both
@pytest.mark.parametrize("n,whole_block", [(400, True), (1600, True), (4000, False)])
def test_equal_totals_match_oracle(oracle, n, whole_block):
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: {n} searches of equal totals", flush=True)
    # 1936 polygons: a search of the whole room stays within the reference's pool of 2048 nodes
    blob = scenes.gen_scene(scenes.BOX_ROOM, 7, cell=5, size_x=11.0, size_z=11.0, num_boxes=0)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    pts = scenes.sample_points(blob, 9, 800)
    x, r = cpu.snap(pts)
    assert (r != 0).all()
    a, ar, b, br = x[:400], r[:400], x[400:].copy(), r[400:]
    # one distance in four as it is; up to 84 equal totals; over 700; all of them infinite
    for k, far in enumerate((0.0, 1e6, 1e10, 1e25)):
        b[k::4, 0] += np.float32(far)
    want = cpu.geodesic(a, ar, b, br)
    assert np.isfinite(want).all()
    at = np.arange(n) % 400
    got = gpu.geodesic(0, a[at], ar[at], b[at], br[at])
    c = gpu.counters()   # of a new simulator: this call's
    differ = np.nonzero(common.bits(want)[at] != common.bits(got))[0]
    assert len(differ) == 0, (len(differ), differ[:8] % 4, want[at][differ[:5]], got[differ[:5]])
    assert c["geo_tie_replays"] > n and c["geo_exact_runs"] >= n // 2
    assert c["geo_heap_spills"] > n // 20      # heaps that outgrow LDS, of 379, 511 and 383 entries
    assert (c["geo_long_path"] == n) == whole_block
    cpu.close()
    gpu.close()


# rooms whose open lists come to up to 67, 140, 218 and 354 entries: the reference's heap grows and shrinks through
# the sizes up to which a pop is one round of accesses to 64, 128 and 256 entries, and beyond
@pytest.mark.parametrize("edge,far", [(6.0, 3e5), (8.0, 1e7), (11.0, 1e7), (8.0, 1e10)])
def test_replayed_heaps_of_all_sizes_match_oracle(oracle, edge, far):
    n = 64
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: a room of {edge} m, end points {far} m away", flush=True)
    blob = scenes.gen_scene(scenes.BOX_ROOM, 5, cell=5, size_x=edge, size_z=edge, num_boxes=0)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    pts = scenes.sample_points(blob, 3, 2 * n)
    x, r = cpu.snap(pts)
    a, ar, b, br = x[:n], r[:n], x[n:].copy(), r[n:]
    b[::2, 0] += np.float32(far)
    want = cpu.geodesic(a, ar, b, br)
    got = gpu.geodesic(0, a, ar, b, br)
    c = gpu.counters()
    assert c["geo_tie_replays"] + c["geo_exact_runs"] > n // 2
    assert np.array_equal(common.bits(want), common.bits(got))
    cpu.close()
    gpu.close()


# more searches than blocks that have a second wavefront for the reference's heap (eight on a CU): some blocks have
# several searches one after the other, and that wavefront begins anew for each
@pytest.mark.parametrize("over", [1, 512])
def test_equal_totals_one_search_after_the_other(oracle, over):
    import torch
    test_equal_totals_match_oracle(oracle, 8 * torch.cuda.get_device_properties(0).multi_processor_count + over, True)
