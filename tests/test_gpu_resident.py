"""GPU: FP64 DIAG and NONE solves that run as one resident launch (k_resident)
against the same solves as launched iterations (set_graphs(False)), bit for
bit: VAR, the scaled A_M and B_M, IER, iterations, residual norms and the exit
taken.

The grids end on and beside 256-cell blocks, from one block to the 512 the
device holds and one more (launched in both cases), in 2-D and with cyclic
axes; the options are those of the scalar logic (the interior dot product,
MINIMIZE_DOTPRODUCTS with ICHECK_BICGS) and the ways a solve ends.
"""
import numpy as np
import pytest

from mfix_amd.leq import DeviceArray
from tests.cases import make_system

pytestmark = pytest.mark.gpu

GRIDS = [
    ((1, 1, 1), False, (0, 0, 0)), ((5, 4, 3), False, (0, 0, 0)), ((6, 6, 2), False, (1, 0, 1)),     # 1 block (256: full)
    ((6, 6, 3), False, (0, 1, 0)), ((30, 62, 1), True, (0, 0, 0)), ((17, 29, 1), True, (1, 0, 0)),
    ((20, 20, 20), False, (0, 0, 0)), ((32, 32, 32), False, (0, 0, 0)),
    ((62, 62, 30), False, (0, 0, 0)), ((62, 62, 31), False, (0, 0, 0)),                              # 512 blocks, one plane more
]


def _solve(gpu, a, b, graphs, **kw):
    gpu.set_graphs(graphs)
    try:
        da, db = DeviceArray.from_host(a), DeviceArray.from_host(b)
        dx = DeviceArray.from_host(np.linspace(-1.0, 1.0, b.size))
        r = gpu.bicgs_dev(dx, da, db, seed=3, **kw)
    finally:
        gpu.set_graphs(True)
    st = {k: r.stats[k] for k in ("iterations", "iter_tot_increment", "exit_reason", "rnorm0", "rnorm")}
    return (r.ier, st), dx.download(), da.download(), db.download()


def _both(gpu, a, b, **kw):
    want, got = _solve(gpu, a, b, False, **kw), _solve(gpu, a, b, True, **kw)
    assert repr(got[0]) == repr(want[0])
    for x, y in zip(got[1:], want[1:]):
        np.testing.assert_array_equal(x, y)
    return got


@pytest.mark.parametrize("pc", ["DIAG", "NONE"])
@pytest.mark.parametrize("dims,no_k,cyc", GRIDS)
def test_grids(gpu, dims, no_k, cyc, pc):
    gpu.grid_init(*dims, no_k=no_k, cyclic=tuple(bool(c) for c in cyc))
    a, b = make_system(0, *dims, no_k, seed=2)
    for itmax in (1, 2, 40):
        _both(gpu, a, b, pc=pc, tol=1e-10, itmax=itmax)


@pytest.mark.parametrize("opts", [dict(is_serial=False), dict(minimize_dotproducts=True, icheck_bicgs=1),
                                  dict(minimize_dotproducts=True, icheck_bicgs=7, is_serial=False)])
def test_scalar_logic(gpu, opts):
    gpu.grid_init(14, 15, 13, **opts)
    a, b = make_system(1, 14, 15, 13, False, seed=4)
    for tol, itmax in ((1e-10, 500), (1e-3, 500), (1e-30, 33)):
        _both(gpu, a, b, pc="DIAG", tol=tol, itmax=itmax)


def test_ways_to_end(gpu):
    dims = (9, 10, 8)
    gpu.grid_init(*dims)
    a, b = make_system(0, *dims, False, seed=5)
    n3 = b.size
    ident = np.zeros(7 * n3)
    ident[3 * n3:4 * n3] = -1.0
    _both(gpu, ident, b, pc="DIAG", tol=1e-14, itmax=50)                      # S-norm exit
    zero = a.copy()
    zero.reshape(7, n3)[:, n3 // 2] = 0.0
    assert _both(gpu, zero, b, pc="DIAG", tol=1e-10, itmax=50)[0][0] == -2    # a row of zeros
    _both(gpu, a, b, pc="DIAG", tol=1e-10, itmax=0)
    bad = b.copy()
    bad[n3 // 3] = np.nan
    _both(gpu, a, bad, pc="DIAG", tol=1e-10, itmax=6)                         # NaN runs to ITMAX
