"""GPU: what mfix_leq_autotune reports can be pinned by mfix_leq_set_shape and
mfix_leq_set_line_block, and solves are the same bits either way."""
import ctypes as C

import numpy as np
import pytest

from mfix_amd import _lib
from tests.cases import make_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
def test_the_choice_can_be_pinned(gpu, mixed):
    L, n = _lib.load(), 24
    gpu.grid_init(n, n, n)
    a, b = make_system(1, n, n, n, seed=3)
    D = gpu.DeviceArray.from_host

    def solve():
        dx, da, db = D(np.zeros(b.size)), D(a), D(b)
        r = gpu.bicgs_dev(dx, da, db, pc="LINE", tol=1e-10, itmax=100, mixed=mixed)
        return r.ier, r.stats["iterations"], dx.download()
    shape, lines = C.c_int(), C.c_int()
    try:
        _lib.check(L.mfix_leq_autotune(n, n, n, int(mixed), C.byref(shape), C.byref(lines)), "autotune")
        tuned = solve()
        _lib.check(L.mfix_leq_set_shape(n, n, n, int(mixed), shape.value // 100, shape.value % 100), "set_shape")
        gpu.set_line_block(n, n, n, lines.value, mixed=mixed)
        pinned = solve()
    finally:
        _lib.check(L.mfix_leq_set_shape(n, n, n, int(mixed), 256, 1), "set_shape")
        gpu.set_line_block(n, n, n, 0, mixed=mixed)
    assert tuned[:2] == pinned[:2]
    np.testing.assert_array_equal(tuned[2], pinned[2])
