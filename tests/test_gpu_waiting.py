"""What a host-synchronous step or reset has written can be read as soon as the call has returned, on any stream and without a
further wait: the step's last launch itself tells the host of its end, from a block or two up to the most agents that do so and
one pair beyond (an event is waited for there), between timed and stream-ordered steps, steps that are given to streams in turn
and steps behind which the stream has been given longer work."""
import numpy as np
import pytest

from tests import common
from tests.test_gpu_parity import assert_step_equal, make_gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("task", [0, 2])
@pytest.mark.parametrize("n", [2, 514, 16384, 16386])
def test_outputs_are_there_when_the_call_returns(oracle, n, task):
    import torch
    from bps_nav_amd import bps_sim
    from oracle import bpo
    sc = common.build_scenes(oracle, 2, 2)
    cpu = bpo.Sim(oracle, sc, n, double_buffered=True, seed=3, threads=4, max_steps=11, task=task)
    if task == 0:
        gen = make_gen(sc, n, double_buffered=True, seed=3, max_steps=11)
    else:
        gen = bps_sim.ExplorationRolloutGenerator("", "", n, len(sc), scenes=sc, double_buffered=True, seed=3, max_steps=11)
    streams = [torch.cuda.Stream() for _ in range(3)]   # two that the steps are given, one that reads
    state = [gen.get_state(g) for g in (0, 1)]
    infos = [gen.get_infos(g) for g in (0, 1)]
    rng = np.random.default_rng(n + task)
    for t in range(24):
        g = t % 2
        a = rng.integers(0, 4, n // 2)
        print(f"case: {n} agents, task {task}, step {t}", flush=True)
        if t % 10 == 6:
            gen.set_profiling(True)
        if t % 10 == 8:
            gen.set_profiling(False)
        ordered = t in (12, 13)
        gen.set_stream_ordered(ordered)
        if t < 2 or t in (16, 17):
            cpu.reset(g)
            with torch.cuda.stream(streams[t % 3 % 2]):
                gen.reset(g)
            with torch.cuda.stream(streams[2]):
                for k in ("poly_ref", "goal_ref", "step", "num_resets", "position"):
                    assert np.array_equal(cpu.state(g)[k].view(np.uint32), state[g][k].cpu().numpy().view(np.uint32)), f"{k} after reset {t}"
        with torch.cuda.stream(streams[t % 3 % 2]):
            cpu.step(a, g)
            gen.step_start(g, torch.from_numpy(a).cuda() if t % 4 < 2 else a)
            if t == 20:
                torch.cuda._sleep(20_000_000)   # some ten milliseconds
                behind = streams[t % 3 % 2].record_event()
            gen.step_end(g)
            if t == 20:
                assert not behind.query(), "step_end has waited for what the stream does behind the step"
        if ordered:
            streams[t % 3 % 2].synchronize()
        with torch.cuda.stream(streams[2]):
            assert_step_equal(cpu, gen, g, state[g], infos[g], f"after step {t}")
    gen.check_errors()
    gen.close()
