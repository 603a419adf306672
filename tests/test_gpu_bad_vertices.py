"""Path searches over navmeshes with vertices that are not finite numbers, which the loader accepts as the
reference's does: there the costs of a path through such a vertex are NaN.  Where the reference's search
ends the distances are the oracle's bit for bit; where it does not (A* around a cycle, the funnel at an
infinite vertex or at a second one that is no number) the call still returns."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common
from tests.golden import meshes
from tests.test_gpu_snap import bv_nodes

pytestmark = pytest.mark.gpu

NANS = np.array([0x7fc00000, 0xffc00000, 0x7fffffff, 0x7f800000], np.uint32).view(np.float32)   # either sign, largest payload, infinity


def with_x(blob, which, value):
    """The navmesh with another x coordinate of the vertices `which(xyz)` names."""
    _, _, xyz = bv_nodes(blob)
    b = bytearray(blob)
    v = np.frombuffer(b, np.float32, xyz.size, 148).reshape(-1, 3)
    at = np.nonzero(which(xyz))[0]
    assert len(at)
    v[at, 0] = value
    return bytes(b)


def corridor(rng, m):
    """Twelve squares of 2 m in a row, without a cycle, and m pairs of points well inside of them."""
    blob = meshes._rects_to_mesh([(2 * i, 0, 2 * i + 2, 2) for i in range(12)])
    cell = rng.integers(0, 12, (2, m))
    pts = np.stack([2 * cell + rng.uniform(0.2, 1.8, (2, m)), np.zeros((2, m)), rng.uniform(0.2, 1.8, (2, m))], axis=-1).astype(np.float32)
    return blob, cell, pts


# the three forms of the kernel
@pytest.mark.parametrize("m", [300, 1600, 3000])
@pytest.mark.parametrize("value", NANS[:3])
def test_one_vertex_that_is_no_number_matches_oracle(oracle, m, value):
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: corridor with {value}, {m} searches", flush=True)
    blob, cell, (a, b) = corridor(np.random.default_rng(m), m)
    blob = with_x(blob, lambda v: (v[:, 0] == 12) & (v[:, 2] == 2), value)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    refs = cpu.poly_info()[0]
    want = cpu.geodesic(a, refs[cell[0]], b, refs[cell[1]])
    assert np.array_equal(common.bits(want), common.bits(gpu.geodesic(0, a, refs[cell[0]], b, refs[cell[1]])))
    cpu.close()
    gpu.close()


@pytest.mark.parametrize("m", [300, 1600, 3000])
def test_searches_end_where_the_reference_does_not(oracle, m):
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    for value in NANS:
        print(f"case: two vertices of {value}, {m} searches", flush=True)
        blob, cell, (a, b) = corridor(np.random.default_rng(m), m)
        blob = with_x(blob, lambda v: np.isin(v[:, 0], (12, 14)) & (v[:, 2] == 2), value)
        cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
        refs = cpu.poly_info()[0]
        got = gpu.geodesic(0, a, refs[cell[0]], b, refs[cell[1]])
        off = (cell < 5).all(axis=0)   # these paths meet neither
        want = cpu.geodesic(a[off], refs[cell[0]][off], b[off], refs[cell[1]][off])
        assert np.array_equal(common.bits(want), common.bits(got[off]))
        gpu.close()
        cpu.close()
        # a room of many cycles with one such vertex
        print(f"case: room with {value}, {m} searches", flush=True)
        blob = scenes.config_scene(1, 0)
        _, _, xyz = bv_nodes(blob)
        x, r = (v.reshape(2, m, -1) for v in nav_points(oracle, blob, 2 * m))
        inner = int(np.argmin(np.abs(xyz - xyz.mean(axis=0)).sum(axis=1)))
        gpu = nav_only([with_x(blob, lambda v: np.arange(len(v)) == inner, value)])
        assert len(gpu.geodesic(0, x[0], r[0].ravel(), x[1], r[1].ravel())) == m
        gpu.close()


def nav_points(oracle, blob, n):
    from oracle import bpo
    cpu = bpo.Nav(oracle, blob)
    x, r = cpu.snap(scenes.sample_points(blob, 4, n))
    cpu.close()
    return x, r
