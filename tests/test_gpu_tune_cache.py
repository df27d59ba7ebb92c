"""A tuning cache holds choices timed on the kernels of its entries' version:
entries without one (the first form of the key) and of another one are not read.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("version", ["", "kernels=1 "])
def test_entries_of_other_kernels_are_not_read(sdt, tmp_path, version):
    n, box = 300, 20.0
    pos = sdt.rsa_positions(n, box, 1.0, 5)

    def tuned(cache):
        bd = sdt.BDSim(pos, np.ones(n), box, 0.896, 5.0, 24, 6, sdt.FP32, 100, 4, 1e-6, 2.0,
                       125.0, 1e-3, 16, 6)
        bd.init()
        return bd.autotune(cache)[:2]

    cache = tmp_path / "tune.txt"
    tuned(cache)
    lines = cache.read_text().splitlines()
    assert len(lines) == 2
    # the same systems with choices that no tuning makes (a chunk of 33)
    keys = [ln.split(" b=")[0] + " b=" + ln.split(" b=")[1].split()[0] for ln in lines]
    current = tmp_path / "current.txt"
    current.write_text("".join(k + " 0 4 33 17\n" for k in keys))
    assert [tuple(c) for c in tuned(current)] == [(0, 4, 33, 17)] * 2
    other = tmp_path / "other.txt"
    other.write_text("".join(k.replace("kernels=2 ", version) + " 0 4 33 17\n" for k in keys))
    assert all(tuple(c) != (0, 4, 33, 17) for c in tuned(other))
    assert len(other.read_text().splitlines()) == 4
