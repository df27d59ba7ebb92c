"""A system whose spread candidates pass 2^31 (a stencil of order 6 reaches 18
mesh blocks, so from 119.3 M particles up) is accepted as smaller ones are: the
candidate offsets have 64 bits. Init only; no list of that size is built."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_init_accepts_120_million_particles(sdt):
    n = 120_000_000
    g = sdt.MobSpme(n, np.ones(n), 1000.0, 0.9, 20.0, 64, 6, sdt.FP32)
    assert g.init(), g.init_error
