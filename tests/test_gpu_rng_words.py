"""Draws from states with words of the moduli and above, up to 2^32 - 1, which no
jump or draw gives but gxt_rng_draw takes: the recurrence's exact residues, and
the words that no draw has replaced as they were.  Whole numbers: bit-exact
against the CPU oracle."""
import numpy as np
import pytest

import oracle_harness as O

pytestmark = pytest.mark.gpu

M = (4294967087, 4294944443)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 33])
def test_draws_from_words_beyond_the_moduli(gpu_lib, k):
    print("rng words, %d draws" % k, flush=True)
    rs = np.random.default_rng(17)
    n = 4096
    st = rs.integers(0, 2**32, (n, 6), dtype=np.uint64).astype(np.uint32)
    for j in range(6):
        edge = rs.integers(M[j // 3] - 2, 2**32, n, dtype=np.uint64).astype(np.uint32)
        st[:, j] = np.where(rs.random(n) < 0.5, edge, st[:, j])
    st[0] = 0xffffffff
    st[1, :3], st[1, 3:] = M[0], M[1]
    g, gs = gpu_lib.rng_draw(st, k)
    c, cs = O.rng_draw(st, k)
    np.testing.assert_array_equal(g, c)
    np.testing.assert_array_equal(gs, cs)
