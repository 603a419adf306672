"""Entry points that are called between step_start and step_end: each that says it waits for the step in flight does, also where the
step's last launch tells the host of its end and no event is recorded behind it.  Longer work in front of the step, on a stream of its
own, keeps it from running until after the call has been made."""
import numpy as np
import pytest

from tests import common
from tests.test_gpu_parity import assert_step_equal

pytestmark = pytest.mark.gpu

CALLS = ["synchronize", "check_errors", "counters", "reset"]


@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("n", [64, 16386])   # two groups of agents, whose steps tell, and of one more than tell
@pytest.mark.parametrize("task", ["PointNav", "Exploration"])
def test_calls_wait_for_the_step_in_flight(oracle, task, n, ordered):
    import torch
    from bps_nav_amd import bps_sim
    from oracle import bpo
    sc = common.build_scenes(oracle, 2, 2)
    number = ["PointNav", "Flee", "Exploration"].index(task)
    cpu = bpo.Sim(oracle, sc, n, double_buffered=True, seed=3, threads=4, task=number)
    gen = getattr(bps_sim, task + "RolloutGenerator")("", "", n, len(sc), scenes=sc, double_buffered=True, seed=3)
    gen.set_stream_ordered(ordered)
    slow, other = torch.cuda.Stream(), torch.cuda.Stream()
    state, infos = [gen.get_state(g) for g in (0, 1)], [gen.get_infos(g) for g in (0, 1)]
    for g in (0, 1):
        cpu.reset(g)
        gen.reset(g)
    rng = np.random.default_rng(n)
    steps = 0
    for t in range(8):
        g, call = t // 4, CALLS[t % 4]
        print(f"case: {task}, {n} agents, stream-ordered {ordered}, {call} while a step of group {g} is in flight", flush=True)
        a = rng.integers(0, 4, n // 2)
        b = torch.from_numpy(a).cuda()
        torch.cuda.synchronize()
        with torch.cuda.stream(slow):
            torch.cuda._sleep(20_000_000)   # some ten milliseconds
            began = slow.record_event()
            gen.step_start(g, b)
        assert not began.query()
        steps += n // 2
        with torch.cuda.stream(other):
            if call == "reset":
                gen.reset(1 - g)
            elif call == "counters":
                assert gen.counters()["agent_steps"] == steps
            else:
                getattr(gen, call)()
            assert began.query(), f"{call} did not wait"   # (the step itself is over some microseconds before its stream says so)
            cpu.step(a, g)
            assert_step_equal(cpu, gen, g, state[g], infos[g], f"after {call}")
            if call == "reset":
                cpu.reset(1 - g)
                cs = cpu.state(1 - g)
                for k in ("poly_ref", "goal_ref", "step", "episode", "num_resets", "position"):
                    assert np.array_equal(cs[k].view(np.uint32), state[1 - g][k].cpu().numpy().view(np.uint32)), f"{k} of the group that was reset"
        gen.step_end(g)
        # and steps go on from there, of both groups, the one behind the other
        for h in (1 - g, g):
            a = rng.integers(0, 4, n // 2)
            cpu.step(a, h)
            gen.step(h, torch.from_numpy(a).cuda())
            steps += n // 2
            gen.synchronize()
            assert_step_equal(cpu, gen, h, state[h], infos[h], f"in the step of group {h} after {call}")
    # an action that is none, in a step that has not run yet
    a = np.full(n // 2, 3)
    a[-1] = 4
    b = torch.from_numpy(a).cuda()
    torch.cuda.synchronize()
    with torch.cuda.stream(slow):
        torch.cuda._sleep(20_000_000)
        gen.step_start(0, b)
    with torch.cuda.stream(other), pytest.raises(RuntimeError, match="action id"):
        gen.check_errors()
    gen.step_end(0)
    gen.close()
