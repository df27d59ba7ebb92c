"""The SPME transforms (src/mob/spme.cc:549-618) at the mesh sides where their
kernels differ: the smallest two-stage sides, odd radices, the largest fused
planes, the separate x and y passes on both sides of that line (FP32 192 / 200,
FP64 128 / 144), the components' three-step z pass (unequal radii in FP64 from a
second radix of 8 up: 64, 72, 80, 90, ...; 54 and 60 below; 256 in FP64), and the general radix chain (250, 360).

FP64 against the oracle's reciprocal product: the sums of a product of
K^3 log K^3 operations in 64 bits, 1e-12 of the result (measured 2e-15); FP32
the single-precision gate 2e-6 (measured 2e-7 to 5e-7).
"""
import numpy as np
import pytest

from conftest import uniform_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,p,poly", [
    (16, 4, False), (20, 4, True), (24, 6, False), (30, 6, True), (50, 6, False), (54, 6, True),
    (60, 6, True), (64, 6, True), (80, 6, True), (96, 6, True), (90, 6, True), (100, 6, False), (128, 6, True), (144, 6, False), (162, 6, True),
    (180, 6, False), (192, 8, False), (200, 8, False), (240, 6, True), (250, 6, False), (256, 8, False),
    (324, 6, False), (360, 6, False),
])
def test_recip_matches_oracle_at_every_kind_of_side(sdt, orc, K, p, poly):
    n, box, nrhs = 150, 14.0, 1 if K > 150 else 3
    pos, rdi = uniform_system(n, box, 300 + K)
    if poly:
        rdi = np.random.default_rng(K).uniform(0.5, 1.5, n)
    f = np.random.default_rng(400 + K).standard_normal((3 * n, nrhs))
    o = orc.MobSpme(n, rdi, box, 0.9, 5.0, K, p)
    assert o.init()
    o.update(pos, rdi)
    ref = o.mul_vector(f, mode="recip")
    for prec, tol in ((sdt.FP64, 1e-12), (sdt.FP32, 2e-6)):
        g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, p, prec)
        assert g.init(), g.init_error
        g.update(pos)
        got = g.recip_mul_vector(f)
        assert orc.frob_rel_err(ref, got) < tol, prec
        # nothing of one call is left for the next
        assert np.array_equal(got, g.recip_mul_vector(f))


@pytest.mark.parametrize("poly", [False, True])
def test_side_18_matches_plain_path(sdt, orc, poly):
    # the smallest radix-3 side, which the oracle's spread blocking excludes:
    # against the plain form's stored tables and library transforms
    n, box, K = 150, 14.0, 18
    pos, rdi = uniform_system(n, box, 318)
    if poly:
        rdi = np.random.default_rng(K).uniform(0.5, 1.5, n)
    f = np.random.default_rng(418).standard_normal((3 * n, 3))
    plain = sdt.PlainMobSpme(n, rdi, box, 0.9, 5.0, K, 4)
    plain.update(pos)
    ref = plain.mul_vector(f, mode=2)
    for prec, tol in ((sdt.FP64, 1e-12), (sdt.FP32, 2e-6)):
        g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, 4, prec)
        assert g.init(), g.init_error
        g.update(pos)
        assert orc.frob_rel_err(ref, g.recip_mul_vector(f)) < tol, prec


@pytest.mark.parametrize("prec", [0, 1])
def test_separate_passes_equal_fused_planes(sdt, prec):
    # the same stages and operations: the same bits, at a side with odd radices
    n, box, K = 150, 14.0, 150 if prec == 1 else 128
    pos, rdi = uniform_system(n, box, 7)
    g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, 6, prec)
    assert g.init()
    g.update(pos)
    f = np.random.default_rng(8).standard_normal((3 * n, 5))
    fused = g.recip_mul_vector(f)
    g.set_forms(0, 0, 0, 1)
    assert np.array_equal(fused, g.recip_mul_vector(f))
