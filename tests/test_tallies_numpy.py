"""abi.tallies_to_numpy takes an EventTally array or any sequence of event tallies."""
import numpy as np
import pytest

from geantexascalepilot_amd import abi


def _tallies(n):
    t = (abi.EventTally * n)()
    for i in range(n):
        for k, f in enumerate(("edep", "visible", "leak", "charged_length")):
            setattr(t[i], f, 1.5 * i + k)
        t[i].n_secondaries[:] = [3 * i, 3 * i + 1, 3 * i + 2]
        t[i].n_steps, t[i].n_pairs, t[i].n_annihil = 2 ** 40 + i, 10 + i, 20 + i
    return t


@pytest.mark.parametrize("n", [0, 1, 5])
@pytest.mark.parametrize("as_given", [lambda t: t, list, tuple, lambda t: t[:]])
def test_every_field_of_a_sequence(n, as_given):
    out = abi.tallies_to_numpy(as_given(_tallies(n)))
    i = np.arange(n)
    for k, f in enumerate(("edep", "visible", "leak", "charged_length")):
        assert out[f].dtype == np.float64
        np.testing.assert_array_equal(out[f], 1.5 * i + k)
    for f in ("n_secondaries", "n_steps", "n_pairs", "n_annihil"):
        assert out[f].dtype == np.int64
    np.testing.assert_array_equal(out["n_secondaries"], np.arange(3 * n).reshape(n, 3))
    np.testing.assert_array_equal(out["n_steps"], 2 ** 40 + i)
    np.testing.assert_array_equal(out["n_pairs"], 10 + i)
    np.testing.assert_array_equal(out["n_annihil"], 20 + i)


def test_slice_of_an_array():
    t = _tallies(6)
    np.testing.assert_array_equal(abi.tallies_to_numpy(t[2:5])["n_pairs"], [12, 13, 14])
