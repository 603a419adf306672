"""Points between many floors, snapped by calls of more of them than wavefronts: each is over twelve polygons and beside a hundred of the first box,
so that a wavefront's candidates are more than its lists hold of either kind, and up to three floors are equally near (all within the climb).
Bit for bit the oracle's."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


def floors(levels, cells):
    """squares of 0.3 m, 0.15 m between the floors, each joined to none"""
    verts, polys = [], []
    for y in range(levels):
        for x in range(cells):
            for z in range(cells):
                at = len(verts)
                verts += [(6 * x, 3 * y, 6 * z), (6 * x, 3 * y, 6 * z + 6), (6 * x + 6, 3 * y, 6 * z + 6), (6 * x + 6, 3 * y, 6 * z)]
                polys.append([at, at + 1, at + 2, at + 3])
    return scenes.navmesh_from_polys(verts, polys, [[-1] * 4] * len(polys))


@pytest.mark.parametrize("per", [1, 2, 5, 16])
def test_points_between_floors(oracle, per):
    import torch
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    blob = floors(12, 8)
    waves = 16 * torch.cuda.get_device_properties(0).multi_processor_count
    n = (per - 1) * waves + 77 if per > 1 else waves
    rng = np.random.default_rng(per)
    q = rng.uniform(-0.5, 2.9, (n, 3)).astype(np.float32)
    grid = rng.integers(0, 3, n) == 0   # on vertices and edges, floors and the middles between them
    q[grid] = (np.round(q[grid] / 0.15) * 0.15).astype(np.float32)
    print(f"case: {n} points between floors", flush=True)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    (xo, ro), (xg, rg) = cpu.snap(q), gpu.snap_points(0, q)
    bad = np.nonzero((ro != rg) | (common.bits(xo) != common.bits(xg)).any(axis=1))[0]
    assert len(bad) == 0, (len(bad), q[bad[:5]], xo[bad[:5]], xg[bad[:5]])
    assert (rg != 0).all() and len(np.unique(rg)) > 12 * 8 * 8 // 2
    cpu.close()
    gpu.close()
