"""GPU: the whole-line red-black kernel of the LINE preconditioner
(k_line_factor + k_line_whole) against the oracle's LEQ_MSOLVE
(model/leqsol_mod.f:286-598, DGTSV per line), bit for bit.

Line lengths around the kernel's row groups (four rows a step, eight a
register set, 768 rows a loading step) up to its longest line and the first
one past it, one to many lines per block, and the inputs that leave the
factored path for DGTSV itself: a row interchange or a zero pivot anywhere in
the system, and solutions outside the range of the corrected quotient.
"""
import numpy as np
import pytest

from tests.cases import make_system, rng_vec

pytestmark = pytest.mark.gpu


def _msolve(gpu, oracle_mod, dims, no_k, kind, change=None, rhs=None, seed=5):
    im, jm, km = dims
    gpu.grid_init(im, jm, km, no_k=no_k)
    og = oracle_mod.grid(im, jm, km, no_k=no_k)
    a, b = make_system(kind, im, jm, km, no_k, seed=seed)
    a, b, _ = oracle_mod.unit_scale(og, a, b)
    if change is not None:
        change(a.reshape(7, b.size))
    r = rng_vec(b.size, 3) if rhs is None else rhs(b.size)
    z_ref, info = oracle_mod.msolve(og, "LINE", a, r, "RSRS")
    da, dr, dz = gpu.DeviceArray.from_host(a), gpu.DeviceArray.from_host(r), gpu.DeviceArray(r.size)
    gpu.msolve_dev("LINE", "RSRS", da, dr, dz)
    np.testing.assert_array_equal(dz.download(), z_ref)


@pytest.mark.parametrize("jmax", [1, 2, 3, 4, 5, 6, 7, 13, 14, 15, 16, 29, 62, 130, 254, 255, 383, 766, 767, 1534, 1535])
def test_row_counts(gpu, oracle_mod, jmax):
    _msolve(gpu, oracle_mod, (4, jmax, 3), False, 1)


@pytest.mark.parametrize("dims,no_k", [((1, 1, 1), False), ((1, 9, 1), True), ((40, 90, 1), True), ((70, 5, 66), False),
                                       ((48, 37, 45), False)])
def test_grids(gpu, oracle_mod, dims, no_k):
    _msolve(gpu, oracle_mod, dims, no_k, 0)


def test_one_interchange_in_the_system(gpu, oracle_mod):
    def change(p):
        c = p.shape[1] // 2 + 3
        p[1, c] = 7.0
    _msolve(gpu, oracle_mod, (12, 30, 9), False, 1, change)


def test_zero_pivot_line_keeps_its_values(gpu, oracle_mod):
    nj, ni = 21, 9   # the line of cell (i, k) = (4, 3): its first row has no pivot and no coupling below

    def change(p):
        c = 2 * nj * ni + 3 * nj
        p[3, c] = 0.0
        p[1, c + 1] = 0.0
    _msolve(gpu, oracle_mod, (ni - 2, nj - 2, 8), False, 1, change)


@pytest.mark.parametrize("scale", [1e-305, 1e-290, 1e290])
def test_solutions_outside_the_quotient_range(gpu, oracle_mod, scale):
    _msolve(gpu, oracle_mod, (12, 30, 9), False, 1, rhs=lambda n: scale * rng_vec(n, 8))


def test_some_blocks_outside_the_range(gpu, oracle_mod):
    def rhs(n):
        r = rng_vec(n, 9)
        r[n // 3:n // 2] *= 1e-300
        r[:n // 8] = 0.0
        r[n // 4] = np.inf
        return r
    _msolve(gpu, oracle_mod, (30, 30, 30), False, 1, rhs=rhs)


def test_fp32_lines_past_the_several_lane_kernels(gpu, oracle_mod):
    """FP32 lines of more than 512 rows take DGTSV in LDS; the bar is the FP32
    line tests' 2e-5 of max |z|."""
    im, jm, km = 4, 600, 3
    gpu.grid_init(im, jm, km)
    og = oracle_mod.grid(im, jm, km)
    a, b = make_system(1, im, jm, km, False, seed=5)
    a, b, _ = oracle_mod.unit_scale(og, a, b)
    a32 = np.zeros((8, b.size), np.float32)
    a32[:7] = a.reshape(7, b.size)
    a32[7] = a32[3]
    r = rng_vec(b.size, 4).astype(np.float32)
    z_ref, info = oracle_mod.msolve(og, "LINE", a32[:7].astype(np.float64).reshape(-1), r.astype(np.float64), "RSRS")
    assert info == 0
    da, dr = gpu.DeviceArray.from_host(a32.reshape(-1)), gpu.DeviceArray.from_host(r)
    dz = gpu.DeviceArray(b.size, np.float32)
    gpu.msolve32_dev("RSRS", da, dr, dz)
    assert np.max(np.abs(dz.download() - z_ref)) <= 2e-5 * np.max(np.abs(z_ref))
