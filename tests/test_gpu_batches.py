"""Batched queries of every size on a simulator that has fewer envs than the batch has items: the
number of wavefronts that serve a batch follows the batch, not the envs.  Compared with the oracle
bit for bit."""
import numpy as np
import pytest

from bps_nav_amd import scenes
from tests import common

pytestmark = pytest.mark.gpu


def points(oracle, n):
    from oracle import bpo
    blob = scenes.config_scene(2, 3)
    pts = scenes.sample_points(blob, 17, 2 * n) + np.random.default_rng(n).normal(0, 0.2, (2 * n, 3)).astype(np.float32)
    return blob, bpo.Nav(oracle, blob), pts


@pytest.mark.parametrize("n", [1, 2, 3, 513, 2304, 2305, 9001])
def test_batch_sizes(oracle, n):
    """Up to 2304 path queries get a block of two wavefronts each (nine blocks on each of 256 CUs),
    more share them; up to 8192 snaps get a wavefront each."""
    from bps_nav_amd.bps_sim import nav_only
    from oracle import bpo
    print(f"case: batches of {n}", flush=True)
    blob = scenes.config_scene(2, 3)
    cpu, gpu = bpo.Nav(oracle, blob), nav_only([blob])
    pts = scenes.sample_points(blob, 17, 2 * n) + np.random.default_rng(n).normal(0, 0.2, (2 * n, 3)).astype(np.float32)
    xo, ro = cpu.snap(pts)
    xg, rg = gpu.snap_points(0, pts)
    assert np.array_equal(ro, rg) and np.array_equal(common.bits(xo), common.bits(xg))
    d = gpu.geodesic(0, xo[:n], ro[:n], xo[n:], ro[n:])
    assert np.array_equal(common.bits(cpu.geodesic(xo[:n], ro[:n], xo[n:], ro[n:])), common.bits(d))
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
