"""Batched queries of every size on a simulator that has fewer envs than the batch has items: the
number of wavefronts that serve a batch follows the batch, not the envs.  Compared with the oracle
bit for bit."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


def compute_units():
    import torch
    return torch.cuda.get_device_properties(0).multi_processor_count


def limit(name):
    """The largest batch that is served one way; one more item goes the next way.  Path queries: a block with
    the whole node pool in LDS each (three on a CU), blocks of a search each with a window (eight on a CU, which
    serve up to ten), blocks of two searches.  Snaps: a wavefront each (sixteen on a CU), several to a
    wavefront.  Allocation-free path queries: a block with the whole pool in LDS for each of 768, more in blocks
    of two searches."""
    return {"pool": 3, "block": 10, "snap": 16, "static": 3}[name] * (256 if name == "static" else compute_units())


def points(oracle, n):
    from oracle import bpo
    blob = scenes.config_scene(2, 3)
    pts = scenes.sample_points(blob, 17, 2 * n) + np.random.default_rng(n).normal(0, 0.2, (2 * n, 3)).astype(np.float32)
    return blob, bpo.Nav(oracle, blob), pts


SIZES = [1, 2, 3, 513, 2304, 2305, 9001] + [(name, k) for name in ("pool", "block", "snap") for k in (-1, 0, 1)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: str(s) if isinstance(s, int) else f"{s[0]}{s[1]:+d}")
def test_batch_sizes(oracle, size):
    """Small and odd sizes, and each side of the limits above."""
    from bps_nav_amd.bps_sim import nav_only
    n = size if isinstance(size, int) else limit(size[0]) + size[1]
    print(f"case: batches of {n}", flush=True)
    blob, cpu, pts = points(oracle, n)
    gpu = nav_only([blob])
    xo, ro = cpu.snap(pts[:n])
    xg, rg = gpu.snap_points(0, pts[:n])
    assert np.array_equal(ro, rg) and np.array_equal(common.bits(xo), common.bits(xg))
    x2, r2 = cpu.snap(pts[n:])
    d = gpu.geodesic(0, xo, ro, x2, r2)
    assert np.array_equal(common.bits(cpu.geodesic(xo, ro, x2, r2)), common.bits(d))
    assert gpu.search_kernel() == ("k_geodesic_few" if n <= limit("pool") else "k_geodesic_mid" if n <= limit("block") else "k_geodesic")
    # every search with larger LDS structures up to the second limit, none beyond
    c = gpu.counters()
    assert c["geo_long_path"] == (c["geodesic_queries"] if n <= limit("block") else 0)
    cpu.close()
    gpu.close()


@pytest.mark.parametrize("size", [1, 383, 385, ("static", -1), ("static", 0), ("static", 1), 4096],
                         ids=lambda s: str(s) if isinstance(s, int) else f"{s[0]}{s[1]:+d}")
def test_allocation_free_sizes(oracle, size):
    """The allocation-free entry point, which shares 384 blocks among more queries than it has pools for."""
    import torch
    from bps_nav_amd.bps_sim import nav_only
    n = size if isinstance(size, int) else limit(size[0]) + size[1]
    print(f"case: {n} allocation-free path queries", flush=True)
    blob, cpu, pts = points(oracle, n)
    gpu = nav_only([blob])
    x, r = cpu.snap(pts)
    dev = [torch.from_numpy(v).cuda() for v in (x[:n], r[:n].view(np.int32), x[n:], r[n:].view(np.int32))]
    got = gpu.geodesic_static(0, *dev).cpu().numpy()
    assert np.array_equal(common.bits(cpu.geodesic(x[:n], r[:n], x[n:], r[n:])), common.bits(got))
    c = gpu.counters()
    assert gpu.search_kernel() == ("k_geodesic_few" if n <= limit("static") else "k_geodesic")
    assert c["geodesic_queries"] == n and c["geo_long_path"] == (n if n <= limit("static") else 0)
    cpu.close()
    gpu.close()


def test_batch_without_room_for_pools_of_its_own(oracle):
    """With too little device memory left for node pools of its own a batch is served with the simulator's
    (some room for everything else stays: of 650 MB for this batch 400 are there)."""
    import torch
    from bps_nav_amd.bps_sim import nav_only
    print("case: a batch of path queries on a full device", flush=True)
    n = 5000
    blob, cpu, pts = points(oracle, n)
    gpu = nav_only([blob])
    x, r = cpu.snap(pts)
    gpu.geodesic(0, x[:64], r[:64], x[n:n + 64], r[n:n + 64])   # pools of its own, which the next call has to give up
    room = 400 << 20
    taken = [torch.empty(torch.cuda.mem_get_info()[0] - room, dtype=torch.uint8, device="cuda")]
    # (the runtime reports less than there is before the first large allocation)
    if torch.cuda.mem_get_info()[0] > room:
        taken.append(torch.empty(torch.cuda.mem_get_info()[0] - room, dtype=torch.uint8, device="cuda"))
    assert torch.cuda.mem_get_info()[0] < room + (64 << 20)
    got = gpu.geodesic(0, x[:n], r[:n], x[n:], r[n:])
    few = gpu.geodesic(0, x[:64], r[:64], x[n:n + 64], r[n:n + 64])
    del taken
    torch.cuda.empty_cache()
    assert np.array_equal(common.bits(cpu.geodesic(x[:n], r[:n], x[n:], r[n:])), common.bits(got))
    assert np.array_equal(common.bits(got[:64]), common.bits(few))
    again = gpu.geodesic(0, x[:n], r[:n], x[n:], r[n:])         # with room again
    assert np.array_equal(common.bits(got), common.bits(again))
    cpu.close()
    gpu.close()


# calls whose arrays pass through pinned memory of at most 16 MiB, and calls beyond, which copy, as do calls of more than 256
# KiB until eight times as much has been copied as the largest needs: 28 bytes a snap or sample, 44 a move, 36 a distance
@pytest.mark.parametrize("call,each", [("snap", 28), ("sample", 28), ("move", 44), ("distance", 36)])
def test_calls_beyond_the_pinned_memory(oracle, call, each):
    from bps_nav_amd.bps_sim import nav_only
    few = 1000
    blob, cpu, pts = points(oracle, few)
    cpu.close()
    pts = pts[:few]
    u = np.random.default_rng(5).random((few, 3), dtype=np.float32)
    gpu = nav_only([blob])
    x, r = gpu.snap_points(0, pts)
    to = x + np.float32(0.2)
    gx, gr = gpu.snap_points(0, x + np.float32(0.4))
    rep = lambda v, at: np.ascontiguousarray(v[at])  # noqa: E731
    ask = {"snap": lambda at: gpu.snap_points(0, rep(pts, at)), "sample": lambda at: gpu.random_points(0, rep(u, at)),
           "move": lambda at: gpu.try_steps(0, rep(x, at), rep(r, at), rep(to, at)),
           "distance": lambda at: (gpu.geodesic(0, rep(x, at), rep(r, at), rep(gx, at), rep(gr, at)),)}[call]
    want = ask(np.arange(few))
    most, at_once, middle = (size // each for size in (16 * 2 ** 20, 256 * 2 ** 10, 2 ** 21))
    assert gpu.batch_route() == "pinned"   # of the 1000
    routes = [(at_once - 60, "pinned"), (at_once, "copied")]   # the arrays take up to 1536 bytes more than their own
    for n in (at_once + 1000, middle, most - 100):
        routes += [(n, "copied")] * 8 + [(n, "pinned")] * 2
    for n, route in routes + [(most + 1, "copied"), (7, "pinned")]:
        print(f"case: {call} of {n}", flush=True)
        at = np.arange(n) % few
        for w, g in zip(want, ask(at)):
            assert np.array_equal(common.bits(w)[at], common.bits(g))
        assert gpu.batch_route() == route
    gpu.close()


def test_a_call_after_one_that_failed(oracle):
    """A call that finds an error of an earlier one behind its launches fails, but not before these are done: the next one's
    arrays take the place of its own in the pinned memory."""
    from bps_nav_amd import _lib
    from bps_nav_amd.bps_sim import nav_only
    n = 5000
    blob, cpu, pts = points(oracle, n)
    pts = np.resize(pts, (n, 3))
    few = pts[:50]
    want = cpu.snap(few)
    cpu.close()
    gpu = nav_only([blob])
    print("case: a call after one that failed", flush=True)
    for _ in range(5):
        assert _lib.lib().hipSetDevice(1 << 20) != 0   # (of the runtime that the library is bound to)
        with pytest.raises(RuntimeError):
            gpu.snap_points(0, pts)
        x, r = gpu.snap_points(0, few)
        assert np.array_equal(common.bits(x), common.bits(want[0])) and np.array_equal(r, want[1])
    gpu.close()
