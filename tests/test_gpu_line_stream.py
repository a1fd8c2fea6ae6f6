"""GPU: the red-black line phases of systems of more than one round of blocks
(k_line_stream) against k_line_whole, which a pinned number of lines per block
selects and tests/test_gpu_line_whole.py holds against the oracle: the same
operations, so the same bits.

Line lengths at which a block holds its most lines, a remainder of them and one,
2-D and 3-D, with and without row interchanges; and the inputs that leave the
factored lines for DGTSV itself.
"""
import numpy as np
import pytest

from tests.cases import make_system, rng_vec

pytestmark = pytest.mark.gpu


def _both(gpu, dims, no_k, kind, change=None, rhs=None):
    im, jm, km = dims
    gpu.grid_init(im, jm, km, no_k=no_k)
    a, b = make_system(kind, im, jm, km, no_k, seed=5)
    p = a.reshape(7, b.size)
    d = p[3].copy()
    d[d == 0.0] = 1.0
    p /= -d        # rows scaled to A0 = -1, as the solver's set-up leaves them
    if change is not None:
        change(p)
    r = rng_vec(b.size, 3) if rhs is None else rhs(b.size)
    da, dr, dz = gpu.DeviceArray.from_host(a), gpu.DeviceArray.from_host(r), gpu.DeviceArray(r.size)
    out = []
    for lines in (0, 16):
        gpu.set_line_block(im, jm, km, lines)
        gpu.msolve_dev("LINE", "RSRS", da, dr, dz)
        out.append(dz.download())
    gpu.set_line_block(im, jm, km, 0)
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("dims,no_k,kind", [((511, 34, 511), False, 1), ((195, 255, 195), False, 0),
                                            ((194, 254, 196), False, 1), ((200, 246, 198), False, 0), ((80, 1534, 78), False, 0),
                                            ((6500, 1534, 1), True, 1)])
def test_sizes(gpu, dims, no_k, kind):
    _both(gpu, dims, no_k, kind)


def test_interchanges_in_some_blocks_and_a_value_out_of_range(gpu):
    def change(p):
        p[1, p.shape[1] // 2 + 3] = 7.0

    def rhs(n):
        r = rng_vec(n, 9)
        r[n // 3:n // 3 + 1000] *= 1e-303
        r[n // 4] = np.inf
        return r
    _both(gpu, (195, 255, 195), False, 1, change, rhs)


def test_zero_pivot(gpu):
    nj, ni = 257, 197

    def change(p):
        c = 2 * nj * ni + 3 * nj
        p[3, c] = 0.0
        p[1, c + 1] = 0.0
    _both(gpu, (ni - 2, nj - 2, 195), False, 1, change)
