"""The serving loop admits a job by its predicted device footprint, so no job may
use more than it reserved: the device memory that one whole mobility interval of
the same system takes (the step of src/simbox/simbox_bd.cc:296-366), against the
reservation of the submitted job. Few iterations and columns, where the particle
arrays weigh most; many; unequal radii; both precisions.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = [
    # n, K, order, precision, columns of an interval, iterations, unequal radii
    (1000000, 64, 6, 1, 1, 5, False),
    (1000000, 64, 8, 0, 1, 5, False),
    (1000000, 64, 6, 0, 8, 5, False),
    (200000, 64, 6, 1, 12, 20, True),
    (200000, 64, 6, 1, 40, 20, False),
    (200000, 96, 6, 0, 20, 20, True),
    (20000, 96, 6, 1, 100, 100, False),
    (500, 24, 6, 1, 1, 5, False),
]


def _system(n, poly):
    a = 1.5 if poly else 1.0
    box = a * (4.0 * np.pi * n / (3.0 * 0.1)) ** (1.0 / 3.0)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    grid = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    rng = np.random.default_rng(n)
    pos = (grid * (box / m) + rng.uniform(0.0, 0.1, (n, 3))).reshape(-1)
    return pos, rng.uniform(0.5, 1.5, n) if poly else np.ones(n), box


def _bd(sdt, pos, rdi, box, K, p, prec, mi, iters):
    bd = sdt.BDSim(pos, rdi, box, 0.896, 4.0, K, p, prec, iters, 8, 1e-1, 2.0, 125.0, 1e-3, mi, 3)
    bd.init()
    bd.advance(1)
    return bd


@pytest.mark.parametrize("n,K,p,prec,mi,iters,poly", ROWS)
def test_job_stays_within_its_reservation(sdt, n, K, p, prec, mi, iters, poly):
    pos, rdi, box = _system(500, poly)       # the library's and runtime's own memory first
    _bd(sdt, pos, rdi, box, 24, 6, prec, 40, 5)
    pos, rdi, box = _system(n, poly)
    sv = sdt.Server(sdt.SERVE_FP32 if prec == 1 else sdt.SERVE_FP64, 1e12, 1, porder=p,
                    max_iters=iters, mob_interval=mi)
    sv.submit(pos, rdi, box, 0.896, 4.0, K, 1, 3, 0.0)
    free = sdt.device_memory()[0]
    bd = _bd(sdt, pos, rdi, box, K, p, prec, mi, iters)
    used = free - sdt.device_memory()[0]
    reserved = sv.job(0)["bytes"]
    print("used %.1f MB of %.1f" % (used / 1e6, reserved / 1e6))
    assert used <= reserved
    del bd
