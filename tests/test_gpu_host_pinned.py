"""GPU: the host-array entry on arrays in pinned memory, which the runtime moves
from where they are, on pageable ones and on some of each: the same bits."""
import ctypes as C

import numpy as np
import pytest

from tests.cases import make_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pinned(gpu):
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip, held = C.CDLL(path), []

    def make(a):
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(a.nbytes), C.c_uint(0)) == 0
        held.append(p)
        v = np.frombuffer((C.c_char * a.nbytes).from_address(p.value), dtype=np.float64)
        v[:] = a
        return v
    yield make
    for p in held:
        assert hip.hipHostFree(p) == 0


@pytest.mark.parametrize("dims", [(3, 2, 1), (49, 53, 47), (80, 70, 60)])
def test_same_bits(gpu, pinned, dims):
    gpu.grid_init(*dims)
    a, b = make_system(1, *dims, seed=3)
    x = np.linspace(-1.0, 1.0, b.size)
    want = None
    for px, pa, pb in ((0, 0, 0), (1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1)):
        vx, va, vb = (pinned(v) if p else v.copy() for p, v in ((px, x), (pa, a), (pb, b)))
        gpu.leq_bicgs("u", 1, vx, va, vb, "RSRS", 1e-8, "LINE", 20)
        got = vx.copy(), va.copy(), vb.copy()
        want = want or got
        for v, w in zip(got, want):
            np.testing.assert_array_equal(v, w)
