"""GPU: CALC_RESID of domains of which FLAG leaves out parts, none or nearly all,
on grids around the residual pass's blocks of 2,048 cells and the XCDs' turns of
them, against the oracle: counts and location exact, sums (another order) to
relative 1e-13 as in the residual tests."""
import numpy as np
import pytest

import oracle
from tests.cases import make_system, rng_vec
from tests.test_gpu_resid import _check, _grid_init

pytestmark = pytest.mark.gpu


def _flags(what, nk, ni, nj):
    """Fluid cells: all, none, one, a cylinder along J, the lower rows, every other cell of a sixth."""
    f = np.full((nk, ni, nj), 1, np.int32)
    k, i, j = np.meshgrid(np.arange(nk), np.arange(ni), np.arange(nj), indexing="ij")
    out = {"all": k < 0, "none": k >= 0, "one": (k != nk // 2) | (i != ni // 2) | (j != nj - 2),
           "cylinder": ((k - nk / 2) / max(nk, 1)) ** 2 + ((i - ni / 2) / ni) ** 2 > 0.06, "low": j > nj // 3,
           "sparse": (i > ni // 6) | ((i + j + k) % 2 == 0)}[what]
    f[out] = 100
    ghost = np.ones(f.shape, bool)
    (ghost[0] if nk == 1 else ghost[1:-1])[..., 1:-1, 1:-1] = False
    f[ghost] = 100
    return f.reshape(-1)


@pytest.mark.parametrize("what", ["all", "none", "one", "cylinder", "low", "sparse"])
@pytest.mark.parametrize("dims,no_k", [((2, 3, 2), False), ((14, 14, 6), False), ((30, 62, 1), True), ((70, 83, 61), False),
                                       ((301, 199, 1), True), ((130, 6, 140), False)])
def test_parts_left_out(gpu, dims, no_k, what):
    im, jm, km = dims
    a, b = make_system(0, im, jm, km, no_k, seed=31)
    g = oracle.grid(im, jm, km, no_k=no_k)
    _grid_init(gpu, g)
    x, ep_s = rng_vec(b.size, 3), np.random.default_rng(4).uniform(0, 2e-4, b.size)
    flag = _flags(what, 1 if no_k else km + 2, im + 2, jm + 2)
    D = gpu.DeviceArray.from_host
    dx, da, db, df, de = D(x), D(a), D(b), D(flag), D(ep_s)
    for kind in ("C", "S", "PP"):
        opt = dict(tol=0.2, norm=0.5)
        got = gpu.calc_resid_dev(kind, b=db, flag=df, var=dx, a=da, ep_s=de if kind == "S" else None, **opt)
        _check(got, oracle.calc_resid(g, kind, x, a, b, flag, ep_s=ep_s if kind == "S" else None, **opt))
