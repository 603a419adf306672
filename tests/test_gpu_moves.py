"""tryStep by a row of eight lanes, against the oracle bit for bit: moves from a millimetre to several
metres from points on the mesh, from polygon vertices and edges, into walls, off the mesh, and long ones
through many small polygons, which may meet the limit of the reference's pool of 64 nodes and are then done
again by one lane.  (The limit of its queue, 48 nodes, lies behind that one: a polygon has at most six
neighbours, among them the one it was entered from.)"""
import os
import struct

import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common
from tests.test_gpu_snap import bv_nodes

pytestmark = pytest.mark.gpu


POLY = np.dtype([("link", "<u4"), ("verts", "<u2", 6), ("neis", "<u2", 6), ("flags", "<u2"), ("nv", "u1"), ("area", "u1")])


def neighbours_met(blob, first, a, b):
    """How many neighbours a move from a to b meets if it starts in polygon `first` and no limit stops it:
    of the polygons entered one after the other, until one holds b; those whose edge is near enough are."""
    _, _, xyz = bv_nodes(blob)
    head = struct.unpack_from("<15i", blob, 48)
    polys = np.frombuffer(blob, POLY, head[6], 148 + 12 * head[7])
    middle, near = ((a + b) / 2)[[0, 2]], (np.linalg.norm(b - a) / 2 + 1e-3) ** 2
    entered, met, k = [first], 1, 0
    while k < len(entered) and met <= 128:
        p = polys[entered[k]]
        v = xyz[p["verts"][:p["nv"]]][:, [0, 2]]
        e = np.roll(v, -1, axis=0) - v
        side = e[:, 0] * (b[2] - v[:, 1]) - e[:, 1] * (b[0] - v[:, 0])
        if (side > 0).all() or (side < 0).all():
            break
        for j in range(p["nv"]):
            n = int(p["neis"][j])
            if n == 0 or n & 0x8000:
                continue
            met += 1
            d = v[j] + np.clip((middle - v[j]) @ e[j] / (e[j] @ e[j]), 0, 1) * e[j] - middle
            if d @ d <= near and n - 1 not in entered:
                entered.append(n - 1)
        k += 1
    return met


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
    refs = cpu.poly_info()[0]
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
        if name.isdigit() and reach in (0.25, 6.0):
            # on either side of the limit of 64, and well clear of it
            met = np.array([neighbours_met(blob, int(np.nonzero(refs == r[k])[0][0]), x[k], end[k])
                            for k in range(4, 200) if np.isfinite(end[k]).all()])
            assert (met > 80).sum() > 20 if reach > 1 else (met < 50).all()
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
