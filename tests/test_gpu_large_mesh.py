"""The reciprocal product (src/mob/spme.cc:714-839) on a mesh of more than 2^32
bytes (FP64 from K = 813 up): particles everywhere, both interpolation kernels.

FP32 meshes stay below 2^32 bytes, so the single-precision product of the same
system is the reference, at the single-precision gate 2e-6 (measured 2e-7 to
5e-7). A shift by whole mesh points along z leaves the product as it is up to
the rounding of the coordinates (1e-16 of L, which enters the weights through
the offset times K / L) and of the sums: 1e-10 of the result.
"""
import numpy as np
import pytest

from conftest import uniform_system

pytestmark = pytest.mark.gpu


def test_fp64_mesh_above_4_gib(sdt, orc):
    n, K, h = 200, 900, 0.5
    box = K * h
    pos, rdi = uniform_system(n, box, 900)
    f = np.random.default_rng(901).standard_normal((3 * n, 1))
    g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, 6, sdt.FP32)
    assert g.init(), g.init_error
    g.update(pos)
    ref = g.recip_mul_vector(f)
    del g
    g = sdt.MobSpme(n, rdi, box, 0.9, 5.0, K, 6, sdt.FP64)
    assert g.init(), g.init_error
    out = {}
    for shift in (0, 300, 600):
        g.update((pos.reshape(n, 3) + [0.0, 0.0, shift * h]).reshape(-1))
        for form in (0, 1):      # blocks of tiles (6-point tiles), strips
            g.set_interp_form(form)
            out[shift, form] = g.recip_mul_vector(f)
            assert orc.frob_rel_err(ref, out[shift, form]) < 2e-6, (shift, form)
    for k in out:
        assert orc.frob_rel_err(out[0, 0], out[k]) < 1e-10, k
