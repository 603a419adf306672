"""Shared builders for the tests: scenes of the benchmark configurations at reduced agent
counts, with episode tables measured by the CPU oracle."""
import numpy as np

from bps_nav_amd import episodes, scenes
from oracle import bpo

# config -> (geodesic range of the episodes, forward probability of the action stream)
CONFIGS = {1: (1.0, 10.0, None), 2: (1.0, 30.0, 0.6), 3: (1.0, 30.0, 0.7), 4: (15.0, 40.0, 0.8)}


def oracle_geodesic_fn(nav):
    def f(s, g):
        sx, sr = nav.snap(s)
        gx, gr = nav.snap(g)
        return nav.geodesic(sx, sr, gx, gr)
    return f


def build_scenes(oracle, config, num_scenes, episodes_per_scene=64):
    """[(navmesh bytes, episodes f32[E,10])] for scenes 0..num_scenes-1 of a configuration."""
    dmin, dmax, _ = CONFIGS[config]
    out = []
    for i in range(num_scenes):
        blob = scenes.config_scene(config, i)
        nav = bpo.Nav(oracle, blob)
        eps = episodes.make_episodes(blob, 2000 + i, episodes_per_scene, dmin, dmax, oracle_geodesic_fn(nav))
        nav.close()
        out.append((blob, eps))
    return out


def action_stream(config, steps, n):
    rng = np.random.default_rng(3000 + config)
    return [episodes.random_actions(rng, n, CONFIGS[config][2]) for _ in range(steps)]


def bits(a):
    a = np.ascontiguousarray(a)
    return a.view(np.uint32) if a.dtype == np.float32 else a


def crossing_portals(seed, n, unit):
    """Navmesh of n polygons, each joined to three others at random, whose portals' middles all have x = z = 0 and heights of up
    to 1000 units: the distances of a search within it are of any size that floats have.  And the middle's neighbourhood
    in it: f(count) -> points and polygons."""
    rng = np.random.default_rng(seed)
    while True:
        ends = rng.permutation(np.repeat(np.arange(n), 3)).reshape(-1, 2)
        if (ends[:, 0] != ends[:, 1]).all() and len(np.unique(np.sort(ends, 1), axis=0)) == len(ends):
            break
    verts, joined = [], [[] for _ in range(n)]
    for k, (p, q) in enumerate(ends.tolist()):
        x, z = (int(v) for v in rng.integers(1, 60, 2) * rng.choice([-1, 1], 2))
        verts += [(64 + x, int(rng.integers(0, 1000)), 64 + z), (64 - x, int(rng.integers(0, 1000)), 64 - z)]
        joined[p].append((q, 2 * k, 2 * k + 1))
        joined[q].append((p, 2 * k + 1, 2 * k))
    polys = [[v for _, a, b in j for v in (a, b)] for j in joined]
    neis = [[v for q, _, _ in j for v in (q, -1)] for j in joined]
    blob = scenes.navmesh_from_polys(verts, polys, neis, bmin=(-4.0, 0.0, -4.0), cs=0.0625, ch=unit)

    def near(refs, count):
        at = rng.integers(-1000, 1001, (count, 3))
        at[:, 1] = np.abs(at[:, 1])
        return (at * np.float64(unit)).astype(np.float32), refs[rng.integers(0, n, count)]
    return blob, near
