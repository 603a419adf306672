"""String pulling sixteen portals at a time, against the oracle bit for bit: strips of quadrilaterals whose edges run straight
for some portals and bend, so that points lie on one line with the apex and rounding alone decides which of them is the
narrower (comparisons of rounded areas are not transitive there), with corridors of every length from two polygons to the
reference's limit."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


def strip(rng, n, run, origin):
    """Navmesh of n quadrilaterals one after the other along x, its middle line straight for `run` of them at a time."""
    bends = np.repeat(rng.integers(-4, 5, n // run + 1), run)[:n]
    z = np.concatenate([[0], np.cumsum(bends)])
    z -= z.min()
    step, width = int(rng.integers(4, 9)), int(rng.integers(6, 20))
    verts = [(step * k, 0, int(z[k]) + w) for k in range(n + 1) for w in (0, width)]
    polys = [(2 * k, 2 * k + 1, 2 * k + 3, 2 * k + 2) for k in range(n)]
    neis = [(k - 1, -1, k + 1 if k + 1 < n else -1, -1) for k in range(n)]
    return scenes.navmesh_from_polys(np.array(verts, np.int64), polys, neis, bmin=(origin, 0.0, origin))


@pytest.mark.parametrize("n,run", [(4, 2), (16, 5), (17, 7), (33, 7), (60, 9), (120, 20), (256, 7), (260, 30)])
def test_strips_match_oracle(oracle, n, run):
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: strips of {n} polygons", flush=True)
    rng = np.random.default_rng(n)
    blobs = [strip(rng, n, run, origin) for origin in (0.0, 0.0, 0.0, 0.0, 3.3, 3.3, -1000.0, 40.0)]
    gpu = nav_only(blobs)
    for s, blob in enumerate(blobs):
        cpu = bpo.Nav(oracle, blob)
        x, r = cpu.snap(scenes.sample_points(blob, 7 + s, 600))
        a, ar, b, br = x[:300], r[:300], x[300:], r[300:]
        want = cpu.geodesic(a, ar, b, br)
        got = gpu.geodesic(s, a, ar, b, br)
        cpu.close()
        assert np.isfinite(want).mean() > 0.9
        assert np.array_equal(common.bits(want), common.bits(got)), s
    gpu.close()
