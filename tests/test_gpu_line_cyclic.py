"""GPU: LINE on a cyclic axis with an odd number of cells, where the first and
the last line along it have the same colour and are neighbours.  The lines of a
colour take the values that it started from: against that rule in numpy with
the oracle's DGTSV, bit for bit, for colours of up to 64 lines."""
import numpy as np
import pytest

from tests.cases import rng_vec

pytestmark = pytest.mark.gpu


def _phases(oracle_mod, p, r, nk, ni, nj, cyc, no_k):
    """LEQ_MSOLVE's R passes (model/leqsol_mod.f:497-522, IKSWEEP :851-921)."""
    def shift(t, n, d, c):
        inner, s = 0 < t < n - 1, t + d
        if c and inner:
            return n - 2 if s == 0 else 1 if s == n - 1 else s
        return min(max(s, 0), n - 1)
    p, r = p.reshape(7, nk, ni, nj), r.reshape(nk, ni, nj)
    z = r.copy()
    for _ in range(2):
        for param in (1, 0):
            new = z.copy()
            for v in range(nk):
                for u in range(ni):
                    if ((u + 1 if no_k else u + v) & 1) != param:
                        continue
                    b = r[v, u] - p[2, v, u] * z[v, shift(u, ni, -1, cyc[0])] - p[4, v, u] * z[v, shift(u, ni, 1, cyc[0])]
                    if not no_k:
                        b = b - p[0, v, u] * z[shift(v, nk, -1, cyc[2]), u] - p[6, v, u] * z[shift(v, nk, 1, cyc[2]), u]
                    new[v, u] = oracle_mod.dgtsv(p[1, v, u, 1:], p[3, v, u], p[5, v, u, :-1], b)[0]
            z = new
    return z.reshape(-1)


@pytest.mark.parametrize("dims,no_k,cyc", [((21, 30, 1), True, (1, 0, 0)), ((63, 9, 1), True, (1, 0, 0)),
                                           ((9, 20, 7), False, (1, 0, 1)), ((8, 45, 9), False, (0, 0, 1)),
                                           ((7, 6, 8), False, (1, 1, 0))])
def test_same_colour_neighbours(gpu, oracle_mod, dims, no_k, cyc):
    im, jm, km = dims
    nk, ni, nj = 1 if no_k else km + 2, im + 2, jm + 2
    gpu.grid_init(im, jm, km, no_k=no_k, cyclic=tuple(bool(c) for c in cyc))
    g = np.random.default_rng(6)
    p = g.uniform(0.02, 0.2, (7, nk, ni, nj))
    p[3] = -1.0
    if no_k:
        p[0] = p[6] = 0.0
    r = rng_vec(nk * ni * nj, 7)
    want = _phases(oracle_mod, p, r, nk, ni, nj, cyc, no_k)
    da, dr, dz = gpu.DeviceArray.from_host(p.reshape(-1)), gpu.DeviceArray.from_host(r), gpu.DeviceArray(r.size)
    for _ in range(3):
        gpu.msolve_dev("LINE", "RSRS", da, dr, dz)
        np.testing.assert_array_equal(dz.download(), want)
