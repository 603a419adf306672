"""Resets of whole groups against the oracle.  Up to 1024 blocks of four starts and goals, one launch draws the episodes and snaps
both; two launches do beyond.  Sizes on both sides, and blocks that are not full."""
import numpy as np
import pytest

from tests import common
from tests.test_gpu_parity import assert_step_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("task", ["PointNav", "Flee", "Exploration"])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 2047, 2049, 4097])
def test_resets_match_oracle(oracle, task, mode, n):
    import torch
    from bps_nav_amd import bps_sim
    from oracle import bpo
    sc = common.build_scenes(oracle, 1, 1)
    number = ["PointNav", "Flee", "Exploration"].index(task)
    cpu = bpo.Sim(oracle, sc, n, reset_mode=mode, seed=n, threads=4, task=number)
    gen = getattr(bps_sim, task + "RolloutGenerator")("", "", n, 1, scenes=sc, reset_mode=mode, seed=n)
    state, infos = gen.get_state(0), gen.get_infos(0)
    rng = np.random.default_rng(n)
    for t in range(3):
        print(f"case: {task}, mode {mode}, {n} agents, reset {t}", flush=True)
        cpu.reset()
        gen.reset(0)
        cs = cpu.state()
        for k in ("poly_ref", "goal_ref", "step", "episode", "num_resets", "position", "rotation"):
            assert np.array_equal(cs[k].view(np.uint32), state[k].cpu().numpy().view(np.uint32)), f"{k} differs"
        np.testing.assert_allclose(gen.get_polars(0).cpu().numpy()[:, 0], cpu.outputs()["polars"][:, 0], rtol=1e-6, atol=1e-6)
        for _ in range(t):
            a = rng.integers(0, 4, n)
            cpu.step(a)
            gen.step(0, torch.from_numpy(a).cuda())
            assert_step_equal(cpu, gen, 0, state, infos, f"after reset {t}")
    assert gen.counters()["resets"] == int(cpu.state()["num_resets"].sum())
    gen.check_errors()
    gen.close()
