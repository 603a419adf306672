"""Steps of exploring agents, one launch each, against the oracle: from no episode to all of them ending in one step, whose starts the
launch's blocks of 32 agents snap four at a time next to the moves and eight at a time behind them."""
import numpy as np
import pytest

from tests import common
from tests.test_gpu_parity import assert_step_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n", [1, 32, 33, 100])
def test_ends_of_any_number_match_oracle(oracle, n, mode):
    import torch
    from bps_nav_amd import bps_sim
    from oracle import bpo
    sc = common.build_scenes(oracle, 1, 1)
    cpu = bpo.Sim(oracle, sc, n, reset_mode=mode, seed=5, threads=4, task=2, max_steps=9)
    gen = bps_sim.ExplorationRolloutGenerator("", "", n, 1, scenes=sc, reset_mode=mode, seed=5, max_steps=9)
    cpu.reset()
    gen.reset(0)
    state, infos = gen.get_state(0), gen.get_infos(0)
    rng = np.random.default_rng(n)
    for t, ending in enumerate([0, 1, 2, 3, 4, 5, 0, 8, 12, 13, 31, 32, 0, 0, 0, 0, 0, 0, 0, 0, 32, 4, 1]):
        # the steps at which all agents of an episode of nine steps stand at its end are among them
        print(f"case: {n} agents, mode {mode}, step {t}: {ending} of 32 stop", flush=True)
        a = rng.integers(1, 4, n)
        for b in range(0, n, 32):
            k = min(32, n - b)
            a[b + rng.permutation(k)[:ending]] = 0
        if t % 5 == 4:
            gen.set_profiling(t % 2 == 0)   # (a timed step is followed by ones that are not)
        cpu.step(a)
        gen.step(0, torch.from_numpy(a).cuda())
        _, cs = assert_step_equal(cpu, gen, 0, state, infos, f"at step {t}")
    c = gen.counters()
    assert c["agent_steps"] == 23 * n and c["resets"] == int(cs["num_resets"].sum())
    gen.check_errors()
    gen.close()


# on both sides of the sizes (of 256 compute units 2048, 4096 and 16384) at which a block has 8, 16 or 32 agents, with and without wavefronts that begin episodes
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("per_cu,more", [(8, 0), (8, 1), (16, 0), (16, 1), (64, 0), (64, 1)])
def test_ends_in_blocks_of_every_size_match_oracle(oracle, per_cu, more, mode):
    import torch
    from bps_nav_amd import bps_sim
    from oracle import bpo
    n = per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more
    sc = common.build_scenes(oracle, 2, 1)
    cpu = bpo.Sim(oracle, sc, n, reset_mode=mode, seed=7, threads=8, task=2, max_steps=5)
    gen = bps_sim.ExplorationRolloutGenerator("", "", n, 1, scenes=sc, reset_mode=mode, seed=7, max_steps=5)
    cpu.reset()
    gen.reset(0)
    state, infos = gen.get_state(0), gen.get_infos(0)
    rng = np.random.default_rng(n)
    # of each 32 agents, and at the fourth and fifth steps those of them as well that have taken five
    for t, share in enumerate([0.0, 0.05, 0.3, 0.7, 0.2, 1.0, 0.1]):
        print(f"case: {n} agents, mode {mode}, step {t}: {share:.2f} of them stop", flush=True)
        a = np.where(rng.random(n) < share, 0, rng.integers(1, 4, n))
        cpu.step(a)
        gen.step(0, torch.from_numpy(a).cuda())
        _, cs = assert_step_equal(cpu, gen, 0, state, infos, f"at step {t}")
    c = gen.counters()
    assert c["agent_steps"] == 7 * n and c["resets"] == int(cs["num_resets"].sum())
    gen.check_errors()
    gen.close()
