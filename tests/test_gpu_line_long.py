"""GPU: long J lines, of which whole lines in LDS are one or two a block, on both
sides of where they go to k_line_color_sys instead: the oracle's line solve
(DGTSV's bits), FP64."""
import numpy as np
import pytest

from tests.cases import rng_vec

pytestmark = pytest.mark.gpu


# (rows 748: two lines an entry; 1,148: one)  entries of a block: 7, 8; 6, 7
@pytest.mark.parametrize("dims", [(14334, 746, 1), (14340, 746, 1), (6140, 1146, 1), (6146, 1146, 1)])
def test_both_sides(gpu, oracle_mod, dims):
    im, jm, _ = dims
    ni, nj = im + 2, jm + 2
    gpu.grid_init(im, jm, 1, no_k=True)
    g = np.random.default_rng(4)
    p = g.uniform(0.02, 0.2, (7, ni * nj))
    p[3] = -1.0
    p[0] = p[6] = 0.0
    p[1, ::977] = 1.3                       # some rows interchange
    r = rng_vec(ni * nj, 5)
    z, info = oracle_mod.msolve(oracle_mod.grid(im, jm, 1, no_k=True), "LINE", p.reshape(-1), r, "RSRS")
    assert info == 0
    da, dr, dz = gpu.DeviceArray.from_host(p.reshape(-1)), gpu.DeviceArray.from_host(r), gpu.DeviceArray(r.size)
    gpu.msolve_dev("LINE", "RSRS", da, dr, dz)
    np.testing.assert_array_equal(dz.download(), z)


@pytest.mark.parametrize("dims,no_k", [((509, 600, 1), True), ((510, 600, 1), True), ((511, 600, 1), True),
                                       ((20, 1100, 22), False)])
def test_fp32_lines_past_the_several_lane_kernels(gpu, oracle_mod, dims, no_k):
    """FP32 lines of more than 512 rows, on both sides of 256 lines a colour; the
    bar is the FP32 line tests' 2e-5 of max |z|."""
    im, jm, km = dims
    gpu.grid_init(im, jm, km, no_k=no_k)
    n3 = (im + 2) * (jm + 2) * (1 if no_k else km + 2)
    g = np.random.default_rng(4)
    a32 = np.zeros((8, n3), np.float32)
    a32[:7] = g.uniform(0.02, 0.15, (7, n3))
    if no_k:
        a32[0] = a32[6] = 0.0
    a32[3] = a32[7] = -1.0
    r = rng_vec(n3, 4).astype(np.float32)
    z, info = oracle_mod.msolve(oracle_mod.grid(im, jm, km, no_k=no_k), "LINE",
                                a32[:7].astype(np.float64).reshape(-1), r.astype(np.float64), "RSRS")
    assert info == 0
    da, dr, dz = gpu.DeviceArray.from_host(a32.reshape(-1)), gpu.DeviceArray.from_host(r), gpu.DeviceArray(n3, np.float32)
    gpu.msolve32_dev("RSRS", da, dr, dz)
    assert np.max(np.abs(dz.download() - z)) <= 2e-5 * np.max(np.abs(z))
