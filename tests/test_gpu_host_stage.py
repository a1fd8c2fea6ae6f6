"""GPU: the host-array entry moves its arrays in chunks through pinned memory
by one or several threads.  Grids of less than a chunk, of a chunk and a
remainder, and of more chunks than slots give what the same solve on device
arrays gives, bit for bit: solution, scaled matrix and right-hand side."""
import os

import numpy as np
import pytest

from tests.cases import make_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,cpus", [((3, 2, 1), 0), ((31, 62, 62), 0), ((49, 53, 47), 0), ((80, 70, 60), 0),
                                       ((80, 70, 60), 1), ((80, 70, 60), 2)])
def test_same_as_on_the_device(gpu, dims, cpus):
    gpu.grid_init(*dims)
    a, b = make_system(1, *dims, seed=3)
    da, db, dx = gpu.DeviceArray.from_host(a), gpu.DeviceArray.from_host(b), gpu.DeviceArray.from_host(np.zeros(b.size))
    gpu.bicgs_dev(dx, da, db, pc="LINE", tol=1e-8, itmax=20)
    x, aa, bb = np.zeros(b.size), a.copy(), b.copy()
    before = os.sched_getaffinity(0)  # (one thread a processor that the process may use, up to four)
    if cpus:
        os.sched_setaffinity(0, set(sorted(before)[:cpus]))
    try:
        gpu.leq_bicgs("u", 1, x, aa, bb, "RSRS", 1e-8, "LINE", 20)
    finally:
        os.sched_setaffinity(0, before)
    np.testing.assert_array_equal(x, dx.download())
    np.testing.assert_array_equal(aa, da.download())
    np.testing.assert_array_equal(bb, db.download())
