"""GPU: k_conv_dif_phi's axis tables by scalar loads against the oracle, bit for
bit, at J rows around the wave's 64 lanes (a wave within one row, across two,
across more) and short ones, in 2-D, 3-D and with cyclic axes."""
import numpy as np
import pytest

import oracle
from tests.phi_cases import phi_fields, phi_flags, reference_chain
from tests.test_gpu_phi import _device_run, _grid_init, _oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cyc", [(0, 0, 0), (1, 0, 1), (0, 1, 0)])
@pytest.mark.parametrize("dims", [(9, 61, 5), (9, 62, 5), (9, 63, 5), (3, 126, 4), (40, 3, 6), (21, 30, 3), (7, 62, 1),
                                  (30, 20, 1)])
def test_rows(gpu, dims, cyc):
    im, jm, km = dims
    no_k = km == 1
    if no_k:
        cyc = (cyc[0], cyc[1], 0)
    g = oracle.grid(im, jm, km, no_k=no_k, cyclic=cyc)
    n3 = oracle.n3_of(g)
    fields, b_in = phi_fields(n3, im + 2, jm + 2, 1 if no_k else km + 2, no_k, 7)
    case = dict(grid=g, flag=phi_flags(im, jm, km, no_k, cyc, 6), fields=fields, b_in=b_in, ur=0.7)
    _grid_init(gpu, g)
    got, want = (reference_chain(case, run(case)) for run in (lambda c: _device_run(gpu, c), _oracle_run))
    for (a, b), (ao, bo) in zip(got, want):
        np.testing.assert_array_equal(a, ao)
        np.testing.assert_array_equal(b, bo)
