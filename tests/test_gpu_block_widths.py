"""Block-Lanczos kernels at the edges of their launch choices: Gram chunks of
128 to 2048 rows, the 8- and 32-row product tiles (either side of 32 768 rows),
Cholesky widths padded to 4, 8 and 16 (src/brwn/brwn_lanczos.cc:36-221).

Gram tiles against numpy: sums of n products in 64 bits, 1e-12 of the norms.
Lanczos at 1e-9 of the oracle for a tolerance of 1e-4, where the iterate does
not depend on rounding (it moves by 1e-14 under a perturbation of 1e-15 up to 8
iterations, by 1e-10 up to about 20).
"""
import numpy as np
import pytest

from conftest import uniform_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 127, 128, 129, 6144, 6145, 98303, 98305, 120001])
@pytest.mark.parametrize("btot,bs", [(3, 3), (20, 8), (25, 11), (16, 16), (13, 4)])
def test_gram_groups_match_numpy(sdt, n, btot, bs):
    rng = np.random.default_rng(n + btot)
    A, B = rng.standard_normal((n, btot)), rng.standard_normal((n, btot))
    G = sdt.debug_gram_groups(A, B, bs)
    for g in range((btot + bs - 1) // bs):
        a, b = A[:, g * bs:(g + 1) * bs], B[:, g * bs:(g + 1) * bs]
        ref = a.T @ b
        tol = 1e-12 * np.linalg.norm(a) * np.linalg.norm(b)
        assert np.abs(G[g][:ref.shape[0], :ref.shape[1]] - ref).max() <= tol, g


@pytest.mark.parametrize("bs", [1, 3, 4, 5, 8, 9, 16])
def test_lanczos_block_widths_match_oracle(sdt, orc, bs):
    n, box = 300, 20.0
    pos, rdi = uniform_system(n, box, 61)
    z = np.random.default_rng(62).standard_normal((3 * n, 2 * bs + 1 if bs > 1 else 3))
    g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, 32, 6, sdt.FP64)
    assert g.init()
    g.update(pos)
    o = orc.MobSpme(n, rdi, box, 0.9, 5.0, 32, 6)
    assert o.init()
    o.update(pos, rdi)
    bl = sdt.BrwnLanczos(3 * n, 100, bs, 1e-4)
    assert bl.init()
    y, ok = bl.compute(g, z)
    oy, _ = orc.lanczos(o, z, 100, bs, 1e-4)
    assert ok and orc.frob_rel_err(oy, y) < 1e-9


@pytest.mark.parametrize("n,dim", [(10922, 64), (10923, 64)])
def test_lanczos_around_the_tile_line(sdt, n, dim):
    # 32 766 and 32 769 rows: |y|^2 = z^T M z per column at convergence
    box = (4.0 * np.pi * n / (3.0 * 0.2)) ** (1.0 / 3.0)
    pos = sdt.rsa_positions(n, box, 1.0, 63)
    g = sdt.MobSpme(n, np.ones(n), box, 0.8, 5.0, dim, 6, sdt.FP64)
    assert g.init()
    g.update(pos)
    z = np.random.default_rng(64).standard_normal((3 * n, 5))
    bl = sdt.BrwnLanczos(3 * n, 100, 4, 1e-6)
    assert bl.init()
    y, ok = bl.compute(g, z)
    zmz = (z * g.mul_vector(z)).sum(0)
    # the criterion bounds the error of y at 1e-6 |z|; its square enters here
    # through the component along y
    assert ok and np.abs((y * y).sum(0) - zmz).max() < 1e-5 * zmz.max()
