"""The pair search's rounds (16 lanes per row, one cell each, a cell's first 64
decisions kept as bits; src/pairlist/pair_r.cc:95-170, pair_s.cc:98-186) and
the sort below it, where they take another branch: cells with more than 64
members, fewer search cells than a round, a last round that is partial, row
counts around a workgroup's 16 rows, and more than 2 M cells (the scan's
three-launch form). The sets are whole numbers: equal to the oracle's.
"""
import numpy as np
import pytest

from conftest import uniform_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box,cutoff,spread", [
    (300, 40.0, 8.0, 1.2),      # clustered: cells with more than 64 members
    (900, 9.0, 4.4, 0.0),       # 4 cells a side, 14 members each
    (16, 12.0, 3.0, 0.0), (17, 12.0, 3.0, 0.0), (1, 12.0, 3.0, 0.0),
    (2000, 200.0, 3.0, 0.0),    # 133^3 cells
])
@pytest.mark.parametrize("mode", ["R", "S"])
@pytest.mark.parametrize("poly", [False, True])
def test_pairs_equal_oracle(sdt, orc, n, box, cutoff, spread, mode, poly):
    pos, rdi = uniform_system(n, box, 900 + n)
    rng = np.random.default_rng(n)
    if spread > 0:
        pos = (0.45 * box + spread * rng.standard_normal((n, 3))).reshape(-1)
    if poly:
        rdi = rng.uniform(0.5, 1.5, n)
    ia, ja = sdt.pairlist(pos, rdi, box, cutoff, mode)
    oia, oja = orc.pairlist(pos, rdi, box, cutoff, mode)
    assert np.array_equal(ia, oia) and np.array_equal(ja, oja)


def test_update_with_crowded_cells_matches_oracle(sdt, orc):
    # every particle in one tile or two, and clustered: long ranges in the
    # sort's ranks and in the spread's candidate lists
    n, box, K = 600, 20.0, 32
    rng = np.random.default_rng(12)
    pos = (10.0 + 0.8 * rng.standard_normal((n, 3))).reshape(-1)
    rdi = np.ones(n)
    f = rng.standard_normal((3 * n, 6))
    o = orc.MobSpme(n, rdi, box, 0.9, 5.0, K, 6)
    assert o.init()
    o.update(pos, rdi)
    ref = o.mul_vector(f)
    for prec, tol in ((sdt.FP64, 1e-11), (sdt.FP32, 1e-5)):
        g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, 6, prec)
        assert g.init()
        g.update(pos)
        assert orc.frob_rel_err(ref, g.mul_vector(f)) < tol, prec
