"""tryStep by a row of eight lanes, against the oracle bit for bit: moves from a millimetre to several
metres from points on the mesh, from polygon vertices and edges, into walls, off the mesh, and long ones
through many small polygons, which meet the reference's limits (a pool of 64 nodes, 48 in the queue)."""
import os

import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common
from tests.test_gpu_snap import bv_nodes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["1", "2", "3", "4", "recast_room", "recast_two_floors"])
def test_moves_match_oracle(oracle, name):
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: moves on {name}", flush=True)
    if name.isdigit():
        blob = scenes.config_scene(int(name), 1)
    else:
        with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", name + ".navmesh"), "rb") as f:
            blob = f.read()
    rng = np.random.default_rng(11)
    _, _, xyz = bv_nodes(blob)
    n = 1503
    pts = np.concatenate([scenes.sample_points(blob, 3, n), xyz[rng.integers(0, len(xyz), n)],
                          xyz[rng.integers(0, len(xyz) - 1, n)[:, None] + np.arange(2)].mean(axis=1).astype(np.float32)])
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    x, r = cpu.snap(pts)
    ok = r != 0
    x, r = x[ok], r[ok]
    for reach in (1e-3, 0.25, 1.0, 6.0):
        ang, d = rng.uniform(0, 2 * np.pi, len(x)), rng.uniform(0, reach, len(x))
        end = (x + np.stack([d * np.cos(ang), 0.1 * d, d * np.sin(ang)], axis=1)).astype(np.float32)
        end[::50] = x[::50]
        end[1::97, 0] = np.nan
        end[2::97, 2] = np.inf
        ref = r.copy()
        ref[3::89] = 0
        so, sro = cpu.try_step(x, ref, end)
        sg, srg = gpu.try_steps(0, x, ref, end)
        bad = np.nonzero((sro != srg) | (common.bits(so) != common.bits(sg)).any(axis=1))[0]
        assert len(bad) == 0, (reach, len(bad), x[bad[:3]], end[bad[:3]], so[bad[:3]], sg[bad[:3]])
    cpu.close()
    gpu.close()


@pytest.mark.parametrize("config", [1, 3, 4])
def test_samples_match_oracle(oracle, config):
    """The polygon by eight pivots at once, at the ends of the range too."""
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: samples on configuration {config}", flush=True)
    blob = scenes.config_scene(config, 2)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    u = np.random.default_rng(5).random((4001, 3), dtype=np.float32)
    u[:4, 0] = [0.0, 1e-30, np.nextafter(np.float32(1), np.float32(0)), 0.5]
    assert np.array_equal(common.bits(cpu.sample(u)), common.bits(gpu.random_points(0, u)[0]))
    cpu.close()
    gpu.close()
