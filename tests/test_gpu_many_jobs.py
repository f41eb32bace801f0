"""Many jobs in flight at once: the tracks that they inject share pages, so that
pools which hold the tracks hold the jobs.

Jobs only decide when an event's tracks are stepped, so the bounds are those of
the event parity tests: counts equal to the oracle's, energies within 1e-9
relative (FP64 sums in another order)."""
import numpy as np
import pytest

from geantexascalepilot_amd import abi
import oracle_harness as O
from test_gpu_step_loop import COUNTS, ENERGIES

pytestmark = pytest.mark.gpu


def _primaries(make, n, ekin, mixed, first=0):
    """Events [first, first + n): photons, or photons, e- and e+ in turn."""
    if not mixed:
        return make(12345, abi.GAMMA, ekin, ekin, 0.0, n, first, 1 << 40)
    parts = [make(12345, s, ekin, ekin, 0.0, n, first, 1 << 40) for s in (abi.GAMMA, abi.ELECTRON, abi.POSITRON)]
    p = abi.primaries_array(n)
    for i in range(n):
        p[i] = parts[(first + i) % 3][i]
    return p


def run_jobs(gpu_lib, jobs, per, pool, ekin, mixed):
    """`jobs` jobs of `per` events each, all submitted before the run, against the oracle."""
    print("jobs: %d of %d events, %g MeV, pool %d%s" % (jobs, per, ekin, pool, ", mixed" if mixed else ""), flush=True)
    n = jobs * per
    cfg = abi.config_lead_block(max_events=n, max_jobs=jobs, pool_capacity=pool)
    with gpu_lib.Transport(cfg) as t:
        for j in range(jobs):
            t.submit(_primaries(gpu_lib.make_primaries, per, ekin, mixed, j * per), j)
        t.run()
        ev = [t.event_tallies(j, per) for j in range(jobs)]
    ref = O.Oracle(cfg)
    ref.run(_primaries(O.make_primaries, n, ekin, mixed), 8)
    cpu = ref.event_tallies(n)
    for k in COUNTS + ENERGIES:
        gpu = np.concatenate([e[k] for e in ev])
        if k in COUNTS:
            assert np.array_equal(gpu, cpu[k]), k
        else:
            np.testing.assert_allclose(gpu, cpu[k], rtol=1e-9, atol=1e-9, err_msg=k)


# one primary for each workgroup and job (97 and 256 of them) and one more, jobs of one event,
# more jobs than one injection takes, both species classes
@pytest.mark.parametrize("jobs,per,pool,ekin,mixed", [
    (300, 1, 8192, 1.0, False), (65, 3, 65536, 5.0, True), (200, 97, 400_000, 1.0, False), (120, 98, 400_000, 1.0, False),
    (400, 256, 2_000_000, 1.0, False)])
def test_jobs_share_pages(gpu_lib, jobs, per, pool, ekin, mixed):
    run_jobs(gpu_lib, jobs, per, pool, ekin, mixed)


def test_one_event_of_both_species_classes_fills_the_pool(gpu_lib):
    """1.9 M photons and e- of 30 keV in turn in one event, in a pool of 2 M; one
    in a thousand outside the block, whose energy leaks."""
    n, e = 1_900_000, 0.03
    print("jobs: one event of %d primaries" % n, flush=True)
    cfg = abi.config_lead_block(max_events=1, pool_capacity=2_000_000)
    p = gpu_lib.make_primaries(12345, abi.GAMMA, e, e, 0.0, n)
    a = np.frombuffer(p, dtype=np.dtype(abi.Primary))
    a["event"] = 0
    a["species"][1::2] = abi.ELECTRON
    a["pos"][::1000, 2] = -1000.0
    with gpu_lib.Transport(cfg) as t:
        t.submit(p, 1)
        t.run()
        gpu = t.event_tallies(1, 1)
    assert gpu["leak"][0] >= e * (n // 1000) * (1 - 1e-9)
    assert abs((gpu["edep"][0] + gpu["leak"][0]) / (e * n) - 1.0) < 1e-9
    assert gpu["n_steps"][0] >= n - n // 1000


# the smallest pools, of one workgroup: jobs of one event, up to the default
# max_jobs and more, and jobs whose showers use most of what the pool holds
@pytest.mark.parametrize("jobs,per,pool,ekin,mixed", [
    (17, 1, 1024, 10.0, False), (64, 1, 1024, 10.0, False), (62, 1, 4096, 10.0, False), (200, 1, 4096, 10.0, False),
    (1, 16, 1024, 300.0, True), (1, 31, 1024, 1000.0, True), (10, 30, 1024, 20.0, True), (2, 10, 1500, 2000.0, True)])
def test_smallest_pools(gpu_lib, jobs, per, pool, ekin, mixed):
    run_jobs(gpu_lib, jobs, per, pool, ekin, mixed)
