"""gxt_run limited to a number of iterations: the tracks go through that many at
most, and a run continued to the end gives the same events.

An iteration is at most four transports of a track, each a step (up to 8 of a
photon) that makes three tracks of it at most, so one primary takes no more than
8 (1 + 3 + ... + 3^(4 k - 1)) steps in k iterations."""
import numpy as np
import pytest

from geantexascalepilot_amd import abi
import oracle_harness as O
from test_gpu_step_loop import COUNTS, ENERGIES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("species", [abi.GAMMA, abi.ELECTRON])
@pytest.mark.parametrize("pool", [4096, 2_000_000])
def test_one_iteration_is_a_few_steps(gpu_lib, species, pool):
    print("iterations: species %d, pool %d" % (species, pool), flush=True)
    cfg = abi.config_lead_block(max_events=1, pool_capacity=pool)
    with gpu_lib.Transport(cfg) as t:
        t.submit(gpu_lib.make_primaries(12345, species, 2000.0, 2000.0, 0.0, 1), 1)
        steps = [0]
        t.run(max_iterations=1)
        steps.append(int(t.stats().track_steps))
        assert 1 <= steps[1] <= 8 * (3 ** 4 - 1) // 2
        while not t.poll():
            t.run(max_iterations=1)
            steps.append(int(t.stats().track_steps))
            assert steps[-1] > steps[-2]
        # (the shower's longest chain has some 70 transports)
        assert len(steps) > 10
        gpu = t.event_tallies(1, 1)
    ref = O.Oracle(cfg)
    ref.run(O.make_primaries(12345, species, 2000.0, 2000.0, 0.0, 1), 1)
    cpu = ref.event_tallies(1)
    for k in COUNTS:
        assert np.array_equal(gpu[k], cpu[k]), k
    assert steps[-1] == cpu["n_steps"].sum()


# 3: launches of one transport; 10**6: launches of their whole time, and a limit that is never reached
@pytest.mark.parametrize("first", [3, 20_000, 10 ** 6, 2 ** 62])
def test_limited_run_then_the_rest(gpu_lib, first):
    print("iterations: %d, then the rest" % first, flush=True)
    n = 300
    cfg = abi.config_lead_block(max_events=n, pool_capacity=100_000)
    with gpu_lib.Transport(cfg) as t:
        t.submit(gpu_lib.make_primaries(12345, abi.ELECTRON, 500.0, 500.0, 0.0, n), 1)
        t.run(max_iterations=first)
        assert bool(t.poll()) == (first > 3)
        t.run()
        gpu = t.event_tallies(1, n)
    ref = O.Oracle(cfg)
    ref.run(O.make_primaries(12345, abi.ELECTRON, 500.0, 500.0, 0.0, n), 8)
    cpu = ref.event_tallies(n)
    for k in COUNTS:
        assert np.array_equal(gpu[k], cpu[k]), k
    for k in ENERGIES:
        np.testing.assert_allclose(gpu[k], cpu[k], rtol=1e-9, atol=1e-9, err_msg=k)
