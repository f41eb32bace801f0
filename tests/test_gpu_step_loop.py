"""The step loop's pages at the sizes where they can go wrong: one primary and
one more or fewer than a page, jobs of both species classes, pools of one and
two workgroups and capacities that are not whole pages, more pages than the
workgroups of one launch take, and events continued over many launches.

The pages only decide which wave steps a track when, so the bounds are those
of the event parity tests: counts equal to the oracle's, energies within
1e-9 relative (FP64 sums in another order)."""
import numpy as np
import pytest

from geantexascalepilot_amd import abi
import oracle_harness as O

pytestmark = pytest.mark.gpu

COUNTS = ("n_steps", "n_pairs", "n_annihil", "n_secondaries")
ENERGIES = ("edep", "visible", "leak", "charged_length")


def _mixed(make, n, ekin):
    """n primaries of the three species in turn, n events, distinct substreams."""
    parts = [make(12345, s, ekin, ekin, 0.0, n, 1000 * s, 1 << 40) for s in range(3)]
    p = abi.primaries_array(n)
    for i in range(n):
        p[i] = parts[i % 3][i]
    return p


@pytest.mark.parametrize("n,pool", [(1, 4096), (63, 4096), (64, 8192), (65, 8191), (257, 65537), (1025, 2_000_000)])
def test_pages_give_the_oracle_events(gpu_lib, n, pool):
    print("pages: %d events, pool %d" % (n, pool), flush=True)
    cfg = abi.config_lead_block(max_events=n, pool_capacity=pool)
    ekin = 50.0
    with gpu_lib.Transport(cfg) as t:
        t.submit(_mixed(gpu_lib.make_primaries, n, ekin), 1)
        t.run()
        gpu = t.event_tallies(1, n)
        st = t.stats()
    ref = O.Oracle(cfg)
    ref.run(_mixed(O.make_primaries, n, ekin), 8)
    cpu = ref.event_tallies(n)
    for k in COUNTS:
        assert np.array_equal(gpu[k], cpu[k]), k
    for k in ENERGIES:
        np.testing.assert_allclose(gpu[k], cpu[k], rtol=1e-9, atol=1e-9, err_msg=k)
    assert st.track_steps == gpu["n_steps"].sum()


def test_more_pages_than_one_launch_takes(gpu_lib):
    """5.2 M photons of 30 keV in one event: 81,000 pages, of which the
    workgroups of a launch take at most 256 each; the rest wait in the list."""
    n = 5_200_000
    print("pages: %d primaries in one event" % n, flush=True)
    cfg = abi.config_lead_block(max_events=1, pool_capacity=8_000_000)
    pg = gpu_lib.make_primaries(12345, abi.GAMMA, 0.03, 0.03, 0.0, n)
    dt = np.dtype(abi.Primary)
    np.frombuffer(pg, dtype=dt)["event"] = 0
    with gpu_lib.Transport(cfg) as t:
        t.submit(pg, 1)
        t.run()
        gpu = t.event_tallies(1, 1)
    # the oracle's events of a sample of the primaries, and the energy balance of all
    total = gpu["edep"][0] + gpu["leak"][0]
    assert abs(total / (0.03 * n) - 1.0) < 1e-9
    m = 200_000
    ref = O.Oracle(cfg)
    pc = O.make_primaries(12345, abi.GAMMA, 0.03, 0.03, 0.0, m)
    np.frombuffer(pc, dtype=dt)["event"] = 0
    ref.run(pc, 1)
    cpu = ref.event_tallies(1)
    # 10^5 independent photons: means within 5 standard errors (a photon's steps
    # and secondaries have a spread of about their mean)
    for k in ("n_steps", "n_secondaries"):
        a, b = np.sum(gpu[k]) / n, np.sum(cpu[k]) / m
        assert abs(a / b - 1.0) < 5.0 / np.sqrt(m), k


def test_interrupted_run_continues(gpu_lib):
    """gxt_run stopped after each launch leaves the tracks in their pages; the
    following calls finish the same events."""
    n = 200
    cfg = abi.config_pbwo4_block(max_events=n)
    p = gpu_lib.make_primaries(cfg.seed, abi.ELECTRON, 2000.0, 2000.0, 0.0, n)
    with gpu_lib.Transport(cfg) as t:
        t.submit(p, 1)
        t.run()
        whole = t.event_tallies(1, n)
        t.submit(p, 2)
        for _ in range(10000):
            t.run(max_iterations=1)
            if any(r.job_id == 2 for r in t.poll()):
                break
        parts = t.event_tallies(2, n)
    for k in COUNTS:
        assert np.array_equal(whole[k], parts[k]), k
    for k in ENERGIES:
        np.testing.assert_allclose(parts[k], whole[k], rtol=1e-9, atol=1e-9, err_msg=k)


def test_every_page_comes_back(gpu_lib):
    """A pool of one workgroup has 64 pages: 300 short jobs, one after the
    other, each with launches that find no track left, need every page back."""
    cfg = abi.config_lead_block(max_events=1, pool_capacity=4096)
    p = gpu_lib.make_primaries(cfg.seed, abi.GAMMA, 5.0, 5.0, 0.0, 1)
    with gpu_lib.Transport(cfg) as t:
        steps = set()
        for job in range(300):
            t.submit(p, job)
            t.run()
            steps.add(int(t.event_tallies(job, 1)["n_steps"][0]))
    assert len(steps) == 1
