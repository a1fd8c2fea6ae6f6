"""GPU: LINE systems some of whose lines cannot run on their factored rows (a
pivot out of the corrected quotient's range)."""
import numpy as np
import pytest

from tests.cases import make_system

pytestmark = pytest.mark.gpu


def _small_pivot(p, c):
    """Row c with next to no diagonal, uncoupled from its J neighbours: its pivot is 1e-19."""
    p[3, c] = -1e-19
    p[1, c] = p[1, c + 1] = 0.0


def test_working_launches_are_counted(gpu):
    """Every colour phase that ran counts as a working launch, also where the
    lines of a system that streams are solved by DGTSV itself."""
    dims = (195, 255, 195)
    gpu.grid_init(*dims)
    a, b = make_system(1, *dims, seed=5)
    _small_pivot(a.reshape(7, b.size), 2 * 257 * 197 + 3 * 257 + 100)
    D = gpu.DeviceArray.from_host
    dx, da, db = D(np.zeros(b.size)), D(a), D(b)
    gpu.prof_enable(1, True)
    try:
        r = gpu.bicgs_dev(dx, da, db, pc="LINE", tol=1e-30, itmax=2)
        p = gpu.prof_read(1)
    finally:
        gpu.prof_enable(1, False)
    assert r.stats["iterations"] == 2
    assert p["launches"] == 2 * 2 * 4     # two applications an iteration, four phases each
