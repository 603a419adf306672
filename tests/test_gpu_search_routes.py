"""Steps on both sides of the sizes at which another kernel serves their searches and another launch takes the snaps
of their new episodes, against the oracle after every step."""
import pytest

from tests import common
from tests.test_gpu_parity import assert_step_equal

pytestmark = pytest.mark.gpu


# A step expects three queries for four agents: up to 3 for each CU they have a block with the whole node pool in LDS,
# up to 18 a block of their own with a window, in both of which the snaps run next to the searches, and beyond
# that two share a block.  The last ones are between the lines, where the snaps are another task's.
KERNELS = {(3, 0): "k_geodesic_few", (3, 1): "k_geodesic_mid", (18, 0): "k_geodesic_mid", (18, 1): "k_geodesic"}


@pytest.mark.parametrize("task, per_cu, over, mode", [(0, p, o, m) for p in (3, 18) for o in (0, 1) for m in (0, 1)] +
                         [(1, 3, 0, 1), (1, 3, 1, 0), (1, 6, 0, 0), (1, 6, 1, 1)])
def test_steps_at_the_lines_between_kernels(oracle, task, per_cu, over, mode):
    import torch
    from bps_nav_amd.bps_sim import FleeRolloutGenerator, PointNavRolloutGenerator
    from oracle import bpo
    n = per_cu * torch.cuda.get_device_properties(0).multi_processor_count * 4 // 3 + over
    print(f"case: steps of {n} agents, task {task}, mode {mode}", flush=True)
    sc = common.build_scenes(oracle, 2, 1, episodes_per_scene=32)
    cpu = bpo.Sim(oracle, sc, n, reset_mode=mode, seed=41, threads=8, task=task)
    gen = (PointNavRolloutGenerator, FleeRolloutGenerator)[task]("", "", n, len(sc), scenes=sc, reset_mode=mode, seed=41)
    cpu.reset()
    gen.reset(0)
    state, infos = gen.get_state(0), gen.get_infos(0)
    before = gen.counters()
    begun = 0
    for t, a in enumerate(common.action_stream(2, 16, n)):
        cpu.step(a)
        gen.step(0, a)
        co, _ = assert_step_equal(cpu, gen, 0, state, infos, f"at step {t}")
        begun += int((co["masks"] == 0).sum())
        assert gen.search_kernel() == KERNELS.get((per_cu, over), "k_geodesic_mid")
    assert begun > n // 8
    after = gen.counters()
    queries, alone = (after[k] - before[k] for k in ("geodesic_queries", "geo_long_path"))
    assert queries > n and (alone == queries) == (gen.search_kernel() != "k_geodesic")
    gen.check_errors()
    gen.close()
    cpu.close()
