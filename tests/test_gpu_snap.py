"""snapPoint by a wavefront, for one point and for several at once: the box that grows with the best distance against the oracle's walk of the
whole 4 x 8 x 4 m box, bit for bit, on points where the two could part: on vertices, edges and
midpoints shared by polygons, above and below the mesh, between rooms, at the mesh's corners (where the
tree's spare zero leaf counts) and outside; and on navmeshes whose BV tree does not allow the growing
box or does not bound its leaves."""
import os
import struct

import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


def bv_nodes(blob):
    """(offset, count) of the BV nodes in the bytes of a one-tile navmesh, and its polygons' vertices."""
    head = struct.unpack_from("<15i", blob, 48)
    polys, verts, links, details, dverts, dtris, nodes = head[6], head[7], head[8], head[9], head[10], head[11], head[12]
    off = 48 + 100
    xyz = np.frombuffer(blob, np.float32, verts * 3, off).reshape(-1, 3)
    for size in (12 * verts, 32 * polys, 12 * links, 12 * details, 12 * dverts, 4 * dtris):
        off += (size + 3) & ~3
    return off, nodes, xyz


def changed(blob, how):
    """The navmesh with other bounds in its tree: every 7th leaf, or the first inner node below the root,
    shrunk to one corner."""
    off, count, _ = bv_nodes(blob)
    b = bytearray(blob)
    nodes = np.frombuffer(b, np.dtype([("min", "<u2", 3), ("max", "<u2", 3), ("i", "<i4")]), count, off)
    which = np.nonzero(nodes["i"] >= 0)[0][3::7] if how == "leaves" else np.nonzero(nodes["i"] < 0)[0][1:2]
    assert len(which)
    for k in which:
        nodes["max"][k] = nodes["min"][k]
    return bytes(b)


def points(blob, seed, n):
    rng = np.random.default_rng(seed)
    _, _, xyz = bv_nodes(blob)
    on = scenes.sample_points(blob, seed, n)
    v = xyz[rng.integers(0, len(xyz), n)]
    w = xyz[rng.integers(0, len(xyz) - 1, n)[:, None] + np.arange(2)].mean(axis=1).astype(np.float32)
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    anywhere = rng.uniform(lo - 2.5, hi + 2.5, (n, 3)).astype(np.float32)
    corners = np.array([[x, y, z] for x in (lo[0], hi[0]) for y in (lo[1], hi[1]) for z in (lo[2], hi[2])], np.float32)
    corners = np.repeat(corners, 40, axis=0) + rng.normal(0, 1.0, (320, 3)).astype(np.float32)
    tall = on + np.array([0, 1, 0], np.float32) * rng.uniform(-6, 6, (n, 1)).astype(np.float32)
    near = on + rng.normal(0, 0.6, on.shape).astype(np.float32)
    odd = np.array([[np.nan, 0, 0], [np.inf, 0, 0], [1e30, 0, 0], [5, 1e30, 5], [-3000, 0, 5]], np.float32)
    return np.concatenate([on, v, w, anywhere, corners, tall, near, odd]).astype(np.float32)


@pytest.mark.parametrize("name", ["1", "2", "3", "4", "recast_room", "recast_two_floors", "2 leaves", "3 leaves", "2 inner", "recast_room leaves"])
def test_snap_matches_the_walk_of_the_whole_box(oracle, name):
    import torch
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: snaps on {name}", flush=True)
    base, *how = name.split()
    if base.isdigit():
        blob = scenes.config_scene(int(base), 1)
    else:
        with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", base + ".navmesh"), "rb") as f:
            blob = f.read()
    if how:
        blob = changed(blob, how[0])
    q = points(blob, 5, 1500)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    xo, ro = cpu.snap(q)
    # a wavefront for each point, as the resets snap them, and several points to a wavefront
    waves = 16 * torch.cuda.get_device_properties(0).multi_processor_count
    assert len(q) > waves
    for per_call in (waves, len(q)):
        parts = [gpu.snap_points(0, q[i:i + per_call]) for i in range(0, len(q), per_call)]
        xg, rg = (np.concatenate(v) for v in zip(*parts))
        bad = np.nonzero((ro != rg) | (common.bits(xo) != common.bits(xg)).any(axis=1))[0]
        assert len(bad) == 0, (per_call, len(bad), q[bad[:5]], xo[bad[:5]], xg[bad[:5]])
    cpu.close()
    gpu.close()


@pytest.mark.parametrize("name", ["1", "4", "2 leaves"])
def test_many_points_snap_like_few(name):
    """A call of more points than wavefronts gives each several points and evaluates their candidates
    together; every point's result is that of a call of few, bit for bit, whatever its neighbours are
    and however the last wavefront is filled."""
    import torch
    from bps_nav_amd.bps_sim import nav_only
    base, *how = name.split()
    blob = scenes.config_scene(int(base), 1)
    if how:
        blob = changed(blob, how[0])
    waves = 16 * torch.cuda.get_device_properties(0).multi_processor_count
    q = points(blob, 6, 2000)
    q = q[np.random.default_rng(7).permutation(len(q))]
    gpu = nav_only([blob])
    parts = [gpu.snap_points(0, q[i:i + 1000]) for i in range(0, len(q), 1000)]
    x, r = (np.concatenate(v) for v in zip(*parts))
    for n in (waves, waves + 1, 2 * waves + 5, 15 * waves + 1, 17 * waves + 3):
        print(f"case: {n} snaps on {name}", flush=True)
        at = np.arange(n) % len(q)
        xn, rn = gpu.snap_points(0, q[at])
        assert np.array_equal(rn, r[at])
        assert np.array_equal(common.bits(xn), common.bits(x[at]))
    gpu.close()
