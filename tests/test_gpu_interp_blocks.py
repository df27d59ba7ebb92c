"""The interpolation (src/mob/spme.cc:163-198) at the launches where its kernel
takes another branch: tiles of 4, 5, 6 and 8 points, blocks that are partial in
each dimension, regions longer than the mesh, blocks with more particles than a
chunk and with none, few and many columns, unequal radii, and the strips that
large sparse meshes keep.

Reciprocal products against the oracle: FP64 1e-12 (measured 2e-15), FP32 2e-6
(measured 2e-7 to 5e-7).
"""
import numpy as np
import pytest

from conftest import uniform_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box,K,p", [
    (300, 12.0, 16, 4),      # 4-point tiles, a region as long as the mesh
    (900, 18.0, 50, 6),      # 5-point tiles, 10 of them: partial blocks
    (900, 18.0, 54, 6),      # 6-point tiles, 9 of them
    (4000, 18.0, 40, 6),     # 8-point tiles, 5 of them; dense
    (3000, 12.0, 24, 6),     # 890 particles in a block of 16^3: chunks
    (60, 30.0, 64, 8),       # mostly empty blocks
    (700, 18.0, 64, 7),
    (300, 40.0, 200, 6),     # sparse
])
@pytest.mark.parametrize("poly", [False, True])
def test_recip_matches_oracle(sdt, orc, n, box, K, p, poly):
    pos, rdi = uniform_system(n, box, 1200 + n)
    if poly:
        rdi = np.random.default_rng(n).uniform(0.5, 1.5, n)
    o = orc.MobSpme(n, rdi, box, 0.9, 5.0, K, p)
    assert o.init()
    o.update(pos, rdi)
    cols = (1, 3) if K == 200 else (1, 3, 9, 21)
    f = np.random.default_rng(1300 + K).standard_normal((3 * n, cols[-1]))
    ref = o.mul_vector(f, mode="recip")
    for prec, tol in ((sdt.FP64, 1e-12), (sdt.FP32, 2e-6)):
        g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, p, prec)
        assert g.init(), g.init_error
        g.update(pos)
        g.set_launch_width(64)
        for b in cols:
            got = g.recip_mul_vector(f[:, :b])
            assert orc.frob_rel_err(ref[:, :b], got) < tol, (prec, b)
            acc = g.recip_mul_vector(f[:, :b], 1.5, -0.5, f[:, :b])
            assert orc.frob_rel_err(1.5 * ref[:, :b] - 0.5 * f[:, :b], acc) < tol, (prec, b)
        g.set_interp_form(1)     # strips
        assert orc.frob_rel_err(ref, g.recip_mul_vector(f)) < tol, prec


def test_sparse_large_mesh_takes_strips(sdt, orc):
    # 8-point tiles, few particles per block, a grid above the line
    n, box, K = 400, 40.0, 192
    pos, rdi = uniform_system(n, box, 1400)
    g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, 6, sdt.FP32)
    assert g.init()
    assert g.interp_plan(3) == ("strips",)
    g.update(pos)
    o = orc.MobSpme(n, rdi, box, 0.9, 5.0, K, 6)
    assert o.init()
    o.update(pos, rdi)
    f = np.random.default_rng(1).standard_normal((3 * n, 3))
    assert orc.frob_rel_err(o.mul_vector(f, mode="recip"), g.recip_mul_vector(f)) < 2e-6


@pytest.mark.parametrize("n,K,p,prec,b,plan", [
    # FP32 blocks of 3 x 2 x 1 tiles: 768 on 128^3, 2304 on 192^3 (grid line 2048)
    (400, 128, 6, 1, 8, ("blocks", (3, 2, 1), 4)),
    (400, 128, 6, 1, 9, ("strips",)),
    # 48 particles in a block of 3072 points of 192^3
    (110591, 192, 6, 1, 1, ("strips",)),
    (110593, 192, 6, 1, 1, ("blocks", (3, 2, 1), 1)),
    # FP64 cubes of 2 tiles: 1728 on 192^3
    (400, 192, 6, 0, 4, ("blocks", (2, 2, 2), 4)),
    (400, 192, 6, 0, 5, ("strips",)),
    # 6-point tiles stay with blocks
    (400, 180, 6, 1, 16, ("blocks", (3, 2, 2), 4)),
])
def test_rule_between_strips_and_blocks(sdt, n, K, p, prec, b, plan):
    g = sdt.MobSpme(n, np.ones(n), 0.5 * K, 0.9, 5.0, K, p, prec)
    assert g.init(), g.init_error
    assert g.interp_plan(b) == plan
    g.set_interp_form(1)
    assert g.interp_plan(b) == ("strips",)
