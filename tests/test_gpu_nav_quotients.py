"""Distances of the volume-tree navigator where a direction component is at the
edge of the range of its shared reciprocal: bit-exact against the CPU oracle,
which divides."""
import numpy as np
import pytest

import oracle_harness as O
from geantexascalepilot_amd import abi
from test_gpu_nav import _same
from test_gpu_parity import _flush
from test_nav import _unit, many_daughters_tree, random_tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tree", ["calo", "random", "many"])
@pytest.mark.parametrize("small", [0.0, 1e-300, 0.999e-150, 1e-150, 1.001e-150, 1e-12])
def test_small_direction_components_bit_exact(gpu_lib, tree, small):
    _flush("nav quotients: %s, component %g" % (tree, small))
    rs = np.random.default_rng(31)
    vols, pls, world = (abi.reference_calorimeter_tree() if tree == "calo" else
                        (random_tree if tree == "random" else many_daughters_tree)(rs) + (0,))
    g, c = gpu_lib.Navigator(vols, pls, world), O.Navigator(vols, pls, world)
    try:
        n = 3001
        pos = rs.uniform(-1.0, 1.0, (3, n)) * np.array(vols[world][0])[:, None]
        pos[0, ::5] = 0.0
        d = _unit(rs, n)
        ax = np.arange(n) % 3
        d[ax, np.arange(n)] = small * np.where(rs.random(n) < 0.5, -1.0, 1.0)
        d /= np.linalg.norm(d, axis=0)
        t = g.locate(pos, d)
        np.testing.assert_array_equal(t, c.locate(pos, d))
        ins = t >= 0
        assert ins.any()
        _same(g.step(t[ins], pos[:, ins], d[:, ins]), c.step(t[ins], pos[:, ins], d[:, ins]))
    finally:
        g.close()
