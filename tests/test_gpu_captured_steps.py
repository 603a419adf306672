"""Host-synchronous steps that a HIP graph captures, as steps that run: step_end after the capture has nothing to wait for, and what the
replays write does not reach the host's waits for other steps."""
import numpy as np
import pytest

from tests import common
from tests.test_gpu_parity import assert_step_equal

pytestmark = pytest.mark.gpu


def test_replays_do_not_meet_the_waits_of_other_steps(oracle):
    import torch
    from bps_nav_amd import bps_sim
    from oracle import bpo
    n = 100
    sc = common.build_scenes(oracle, 2, 2)
    # (exploring agents: a step of theirs keeps no queue that is another's in the next step, so that one graph can be replayed)
    cpu = bpo.Sim(oracle, sc, n, seed=3, threads=4, task=2, max_steps=9)
    gen = bps_sim.ExplorationRolloutGenerator("", "", n, len(sc), scenes=sc, seed=3, max_steps=9)
    state, infos = gen.get_state(0), gen.get_infos(0)
    rng = np.random.default_rng(4)
    a = [rng.integers(0, 4, n) for _ in range(40)]
    d = torch.from_numpy(np.stack(a)).cuda()
    actions = d[0].clone()
    cpu.reset()
    gen.reset(0)
    cpu.step(a[0])
    gen.step(0, actions)
    busy = torch.cuda.Stream()

    def while_another_stream_is_busy(f, what):
        torch.cuda.synchronize()
        with torch.cuda.stream(busy):
            torch.cuda._sleep(20_000_000)   # some ten milliseconds
        f()
        assert not busy.query(), f"{what} waited for all of the device"
        torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    print("case: capture", flush=True)
    with torch.cuda.graph(graph):
        gen.step_start(0, actions)
    while_another_stream_is_busy(lambda: gen.step_end(0), "step_end of a captured step")
    for t in range(1, 20, 2):
        print(f"case: a step, and a replay behind it, {t}", flush=True)

        def step():
            gen.step_start(0, d[t])
            actions.copy_(d[t + 1])
            graph.replay()
            gen.step_end(0)
        while_another_stream_is_busy(step, "step_end in front of a replay")
        cpu.step(a[t])
        cpu.step(a[t + 1])
        assert_step_equal(cpu, gen, 0, state, infos, f"after step {t} and a replay")
        if t % 4 == 1:
            while_another_stream_is_busy(lambda: gen.reset(0), "a reset behind a replay")
            cpu.reset()
    gen.check_errors()
    gen.close()
