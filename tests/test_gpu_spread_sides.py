"""The point-owner spread (src/mob/spme.cc:313-363) at the launches where its
kernel takes another branch: mesh sides that are not multiples of 4 (partial
blocks of 2 points, rows on 8-byte boundaries), sides below 32 + p - 1 (a
stencil reaches both ends of a block), FP32 column counts below a full column
block, unequal radii as two columns per right-hand side, one and several column
blocks per workgroup, and a stage that overflows.

Reciprocal products against the oracle: FP64 to 1e-12 (sums of p^3 products and
a K^3 transform in 64 bits, measured 2e-15), FP32 to 2e-6 (measured 2e-7 to
5e-7). The forms' sums keep candidate order, so they agree to the bit.
"""
import numpy as np
import pytest

from conftest import uniform_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,p", [(24, 4), (30, 6), (32, 8), (36, 6), (50, 5), (54, 6), (90, 6)])
@pytest.mark.parametrize("poly", [False, True])
def test_recip_columns_match_oracle(sdt, orc, K, p, poly):
    n, box = 700, 18.0
    pos, rdi = uniform_system(n, box, 500 + K)
    if poly:
        rdi = np.random.default_rng(K).uniform(0.5, 1.5, n)
    o = orc.MobSpme(n, rdi, box, 0.9, 5.0, K, p)
    assert o.init()
    o.update(pos, rdi)
    f = np.random.default_rng(600 + K).standard_normal((3 * n, 35))
    ref = o.mul_vector(f, mode="recip")
    full = o.mul_vector(f[:, :9])
    for prec, tol in ((sdt.FP64, 1e-12), (sdt.FP32, 2e-6)):
        g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, p, prec)
        assert g.init(), g.init_error
        g.update(pos)
        g.set_launch_width(64)
        for b in (1, 2, 4, 5, 8, 15, 17, 35):
            got = g.recip_mul_vector(f[:, :b])
            assert orc.frob_rel_err(ref[:, :b], got) < tol, (prec, b)
        assert orc.frob_rel_err(full, g.mul_vector(f[:, :9])) < tol


# 50 (FP64) and 90: a workgroup takes several column blocks in turn in form 0
@pytest.mark.parametrize("K", [30, 50, 90])
@pytest.mark.parametrize("prec", [0, 1])
def test_forms_identical_on_partial_blocks(sdt, K, prec):
    n, box = 700, 18.0
    pos, rdi = uniform_system(n, box, 700 + K)
    g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, 6, prec)
    assert g.init()
    g.update(pos)
    g.set_launch_width(64)
    f = np.random.default_rng(K).standard_normal((3 * n, 35))
    out = {}
    for form in (0, 1, 3):
        g.set_forms(0, 0, form)
        out[form] = g.recip_mul_vector(f)
        assert np.array_equal(out[0], out[form]), form


@pytest.mark.parametrize("K,p", [(16, 4), (18, 4), (20, 5), (24, 6)])
@pytest.mark.parametrize("prec", [0, 1])
def test_forms_identical_on_short_sides(sdt, K, p, prec):
    # one x block of 16 to 24 points: waves of the comparison form lie past it
    n, box = 700, 18.0
    pos, rdi = uniform_system(n, box, 800 + K)
    g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, p, prec)
    assert g.init(), g.init_error
    g.update(pos)
    f = np.random.default_rng(K).standard_normal((3 * n, 9))
    ref = g.recip_mul_vector(f)
    g.set_forms(0, 0, 1)
    assert np.array_equal(ref, g.recip_mul_vector(f))


@pytest.mark.parametrize("prec", [0, 1])
def test_dense_blocks_overflow_the_stage(sdt, orc, prec):
    # 1500 particles in a box of 9 on 24^3: a block's candidates exceed every
    # stage, which is then filled and summed in parts for each column block
    n, box, K = 1500, 9.0, 24
    pos, rdi = uniform_system(n, box, 77)
    o = orc.MobSpme(n, rdi, box, 0.9, 4.0, K, 6)
    assert o.init()
    o.update(pos, rdi)
    g = sdt.MobSpme(n, rdi, box, 0.9, 4.0, K, 6, prec)
    assert g.init()
    g.update(pos)
    g.set_launch_width(64)
    f = np.random.default_rng(78).standard_normal((3 * n, 40))
    ref = o.mul_vector(f, mode="recip")
    for b in (1, 3, 12, 40):
        assert orc.frob_rel_err(ref[:, :b], g.recip_mul_vector(f[:, :b])) < (1e-12, 2e-6)[prec], b
