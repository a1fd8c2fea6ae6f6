"""GPU: LINE systems some of whose lines cannot run on their factored rows (a
pivot, or values of the solution, out of the corrected quotient's range)."""
import numpy as np
import pytest

from tests.cases import make_system, rng_vec
from tests.test_gpu_line_stream import _both
from tests.test_gpu_line_whole import _msolve

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


@pytest.mark.parametrize("dims,no_k", [((195, 255, 195), False), ((6500, 1534, 1), True)])
def test_clamped_lines_read_their_own_start_values(gpu, dims, no_k):
    """The lines on an end of I or K have themselves as outward neighbour: with
    an outward coupling their right-hand side holds the values they start from,
    also when part of a block's solution is out of range and it is solved
    again.  Streamed lines against k_line_whole, the same bits."""
    im, jm, km = dims
    nk, ni, nj = 1 if no_k else km + 2, im + 2, jm + 2

    def change(p):
        q = p.reshape(7, nk, ni, nj)
        q[2, :, 0] = 0.21
        q[4, :, -1] = 0.17
        if not no_k:
            q[0, 0] = 0.13
            q[6, -1] = 0.11

    def rhs(n):
        r = np.random.default_rng(9).uniform(-1.0, 1.0, (nk, ni, nj))
        r[:, 0, ::3] *= 1e-303            # out of range beside values in range
        r[:, -1, nj // 2] = np.inf
        r[nk // 2, ni // 2:ni // 2 + 20, :9] *= 1e-300
        if not no_k:
            r[0, ::7] *= 1e-305
            r[-1, ni // 3, 5] = -np.inf
        return r.reshape(-1)
    _both(gpu, dims, no_k, 1, change, rhs)


@pytest.mark.parametrize("kind", [0, 1])
def test_small_pivots_beside_interchanges(gpu, oracle_mod, kind):
    """Blocks with a pivot out of range, with interchanged rows (kind 0 has
    them) and with neither, in one system: the oracle's bits."""
    def change(p):
        nj = 31
        for line in (0, 17, 40, 41, 42, 150, 215):
            _small_pivot(p, line * nj + 3 + line % 20)
        _small_pivot(p, 100 * nj)            # a first row
        p[3, 120 * nj + 30] = 1e19           # a last row's pivot, above the range
    _msolve(gpu, oracle_mod, (14, 29, 12), False, kind, change)


@pytest.mark.parametrize("kind", [0, 1])
def test_small_pivots_in_streamed_lines(gpu, kind):
    def change(p):
        for line in range(1, 197 * 197, 2411):
            _small_pivot(p, line * 257 + 1 + line % 255)
    _both(gpu, (195, 255, 195), False, kind, change)


def _decaying(n, rows):
    """A few sources in J lines whose solution falls below the range within the line."""
    r = np.zeros(n)
    r[5::7 * rows] = 1.0
    r[rows * 11 + rows - 2::13 * rows] = -3.0
    return r


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("what", ["decay", "small", "large", "mixed"])
@pytest.mark.parametrize("dims", [(14, 29, 12), (5, 61, 4), (2, 1, 2), (9, 383, 3)])
def test_values_out_of_range(gpu, oracle_mod, dims, what, kind):
    """Right-hand sides out of range and solutions that leave it: the oracle's bits."""
    def change(p):
        if what == "decay":      # 2^-30 a row
            for q in (1, 5):
                p[q] *= 1e-9

    def rhs(n):
        r = rng_vec(n, 8)
        if what == "decay":
            return _decaying(n, dims[1] + 2)
        if what == "mixed":
            r[n // 3:n // 2] *= 1e-300
            r[n // 4] = np.nan
            r[n - 5] = -np.inf
            return r
        return r * {"small": 1e-290, "large": 1e290}[what]
    _msolve(gpu, oracle_mod, dims, False, kind, change, rhs=rhs)


@pytest.mark.parametrize("kind", [0, 1])
def test_decaying_solutions_in_streamed_lines(gpu, kind):
    def change(p):
        for q in (1, 5):
            p[q, ::2] *= 1e-9
    _both(gpu, (195, 255, 195), False, kind, change, lambda n: _decaying(n, 257))
