"""GPU: a resident solve whose waits run out (here: after none or a few tries)
gives up without a trace, and the launched iterations solve the system: the same
VAR, A_M, B_M, IER and iterations, bit for bit."""
import os

import pytest

from tests.cases import make_system
from tests.test_gpu_resident import _both

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[0, 1, 3, 40])
def tries(request, gpu):
    gpu.finalize()
    os.environ["MFIX_LEQ_RESIDENT_SPINS"] = str(request.param)
    try:
        gpu.init(0)
        yield request.param
    finally:
        del os.environ["MFIX_LEQ_RESIDENT_SPINS"]
        gpu.finalize()
        gpu.init(0)


@pytest.mark.parametrize("pc", ["DIAG", "NONE"])
@pytest.mark.parametrize("dims,no_k", [((1, 1, 1), False), ((2, 4, 1), True), ((6, 6, 2), False), ((17, 29, 1), True),
                                       ((20, 20, 20), False), ((62, 62, 30), False)])
def test_launched_instead(gpu, tries, dims, no_k, pc):
    gpu.grid_init(*dims, no_k=no_k)
    a, b = make_system(0, *dims, no_k, seed=2)
    for itmax in (1, 40):
        _both(gpu, a, b, pc=pc, tol=1e-10, itmax=itmax)
