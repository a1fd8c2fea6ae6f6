"""GPU: blocks of up to eight lines with row interchanges, solved by eight lanes
a line (whole_forward_swap8, whole_back_swap8), against the oracle's LEQ_MSOLVE,
bit for bit: line lengths around the groups of eight rows, interchanges next to
a group's ends and in neighbouring rows, and a block whose last lines are
missing; and blocks of more lines, which one lane a line solves, give the same."""
import numpy as np
import pytest

from tests.cases import make_system, rng_vec
from tests.test_gpu_line_whole import _msolve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jmax", [1, 2, 4, 5, 6, 7, 8, 13, 14, 15, 22, 30, 62, 255])
def test_row_counts(gpu, oracle_mod, jmax):
    _msolve(gpu, oracle_mod, (5, jmax, 4), False, 0)


@pytest.mark.parametrize("rows", [(1,), (7,), (8,), (9,), (7, 8), (15, 16, 17), (28, 29, 30), tuple(range(1, 31))])
def test_interchanges_at_group_ends(gpu, oracle_mod, rows):
    def change(p):
        nj = 31
        for q in rows:                  # the coupling below row q - 1 outweighs its pivot
            p[1, q::nj] = np.where(p[1, q::nj] != 0.0, 1.7, 0.0)
    _msolve(gpu, oracle_mod, (14, 29, 11), False, 1, change)


def test_more_lines_a_block(gpu):
    im, jm, km = 40, 37, 30
    gpu.grid_init(im, jm, km)
    a, b = make_system(0, im, jm, km, seed=5)
    r = rng_vec(b.size, 3)
    da, dr, dz = gpu.DeviceArray.from_host(a), gpu.DeviceArray.from_host(r), gpu.DeviceArray(r.size)
    out = []
    for lines in (0, 16, 32):
        gpu.set_line_block(im, jm, km, lines)
        gpu.msolve_dev("LINE", "RSRS", da, dr, dz)
        out.append(dz.download())
    gpu.set_line_block(im, jm, km, 0)
    np.testing.assert_array_equal(out[0], out[1])
    np.testing.assert_array_equal(out[0], out[2])
