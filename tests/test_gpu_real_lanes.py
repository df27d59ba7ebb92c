"""The real-space product (src/mob/mob_spme.cc:135-202) either side of the lines
between 16, 8 and 4 lanes per row (128 and 256 workgroups at 4 lanes: 64 rows a
workgroup, 8 FP64 or 16 FP32 columns), with row counts that do not fill a wave, and
rows with more and fewer pairs than lanes: against the oracle, FP64 1e-12 (sums
of a few hundred products), FP32 2e-6.
"""
import numpy as np
import pytest

from conftest import uniform_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box,b", [
    (17, 20.0, 8), (301, 40.0, 9), (1500, 24.0, 20), (5461, 40.0, 24), (5462, 40.0, 24),
    (8193, 40.0, 16),
    (2688, 30.0, 24), (2689, 30.0, 24), (5440, 40.0, 24), (5441, 40.0, 24),   # FP64: 126, 129, 255, 258
    (4032, 36.0, 24), (4097, 36.0, 24), (8128, 48.0, 24),                     # FP32: 126, 130, 254
])
@pytest.mark.parametrize("poly", [False, True])
def test_real_product_matches_oracle(sdt, orc, n, box, b, poly):
    pos, rdi = uniform_system(n, box, 1500 + n)
    if poly:
        rdi = np.random.default_rng(n).uniform(0.5, 1.5, n)
    f = np.random.default_rng(1600 + n).standard_normal((3 * n, b))
    o = orc.MobSpme(n, rdi, box, 0.9, 5.0, 32, 6)
    assert o.init()
    o.update(pos, rdi)
    ref = o.mul_vector(f, mode="real")
    for prec, tol in ((sdt.FP64, 1e-12), (sdt.FP32, 2e-6)):
        g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, 32, 6, prec)
        assert g.init()
        g.update(pos)
        g.set_launch_width(32)
        assert orc.frob_rel_err(ref, g.real_mul_vector(f)) < tol, prec
