"""What admission learns from events that come and go between two snapshots of
the counters: their peaks come from the device, and events that tell nothing of
the tracks per GeV leave the estimate alone."""
import numpy as np
import pytest

from geantexascalepilot_amd import abi
import oracle_harness as O
from test_gpu_many_jobs import run_jobs
from test_gpu_step_loop import COUNTS, ENERGIES

pytestmark = pytest.mark.gpu


def test_low_energy_events_do_not_open_the_pool(gpu_lib):
    """64 photons of 5 MeV, whose tracks are within every event's reserve, then on the
    same context 400 e- of 1 GeV, of which a pool of 8192 holds some 80 at a time."""
    n = 400
    print("admission: 64 photons of 5 MeV, then %d e- of 1 GeV" % n, flush=True)
    cfg = abi.config_lead_block(max_events=n, pool_capacity=8192)
    with gpu_lib.Transport(cfg) as t:
        t.submit(gpu_lib.make_primaries(12345, abi.GAMMA, 5.0, 5.0, 0.0, 64), 1)
        t.run()
        t.submit(gpu_lib.make_primaries(12345, abi.ELECTRON, 1000.0, 1000.0, 0.0, n), 2)
        t.run()
        gpu = t.event_tallies(2, n)
    ref = O.Oracle(cfg)
    ref.run(O.make_primaries(12345, abi.ELECTRON, 1000.0, 1000.0, 0.0, n), 8)
    cpu = ref.event_tallies(n)
    for k in COUNTS:
        assert np.array_equal(gpu[k], cpu[k]), k
    for k in ENERGIES:
        np.testing.assert_allclose(gpu[k], cpu[k], rtol=1e-9, atol=1e-9, err_msg=k)


@pytest.mark.parametrize("n,pool", [(300, 2048), (120, 1024)])
def test_short_showers_fill_a_small_pool(gpu_lib, n, pool):
    """Showers of 300 MeV end within a launch or two; more of them than the pool holds."""
    run_jobs(gpu_lib, 1, n, pool, 300.0, True)


@pytest.mark.parametrize("n", [1, 100])
def test_peak_of_a_run_within_one_launch(gpu_lib, n):
    """max_live of n photons of 10 MeV is at least n, where no launch ends with one
    of them alive."""
    cfg = abi.config_lead_block(max_events=n)
    with gpu_lib.Transport(cfg) as t:
        t.submit(gpu_lib.make_primaries(12345, abi.GAMMA, 10.0, 10.0, 0.0, n), 1)
        t.run()
        st, ev = t.stats(), t.event_tallies(1, n)
    assert n <= st.max_live <= n + ev["n_secondaries"].sum()
