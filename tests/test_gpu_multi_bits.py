"""hbem_sigma_sweep_multi gives the bits of hbem_sigma_sweep of each instance alone
where the two could take different ways:

* orders next to 1024 and 2048, where the LU changes its step width, padded across
  them, alone and beside instances of the other side;
* fewer than 32 wavenumbers, on the bands, on the node loops (7 panels; kappa times
  the panel diameter beyond the last tier) and on both in one call.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def instance(H, N, ks, seed, order=3, nvert=5, c_i=6.0):
    sp = H.ContinuousSpace1()
    bd = H.BuilderData(H.random_polygon_mesh(seed, nvert, N), sp, sp, order)
    return bd, np.asarray(ks, dtype=float), 1.0, c_i, H.gaussian_test_matrix(2 * N, 2, seed)


def check(H, items, bucket, proj):
    got = H.sigma_sweep_batched(items, 2, proj=proj, bucket=bucket)
    for (bd, ks, c_o, c_i, R), s in zip(items, got):
        alone = H.sigma_sweep(bd, ks, c_o, c_i, R, 2, proj=proj)
        assert np.all(np.isfinite(s)) and np.all(s > 0)
        assert np.array_equal(s, alone), (bd.getNumPanels(), bucket, np.abs(s - alone).max())


@pytest.mark.parametrize("sizes,bucket", [((500,), 768), ((500,), 2048), ((512,), 1536), ((513, 511), 1536),
                                          ((500, 700, 512), 2048), ((1000,), 768), ((1020, 1030, 1024), 2304)])
def test_orders_padded_across_the_step_widths(H, sizes, bucket):
    check(H, [instance(H, N, [3.0, 9.5], 50 + i) for i, N in enumerate(sizes)], bucket, proj=False)


@pytest.mark.parametrize("nk", [1, 3, 31, 33])
@pytest.mark.parametrize("where", ["bands", "loops", "beyond", "both"])
def test_any_number_of_wavenumbers(H, nk, where):
    rng = np.random.default_rng(nk)
    sizes = (7, 6) if where == "loops" else (40, 61, 37)
    lo, hi = {"bands": (2.0, 8.0), "loops": (2.0, 8.0), "beyond": (400.0, 900.0), "both": (5.0, 300.0)}[where]
    items = [instance(H, N, np.sort(rng.uniform(lo, hi, nk)), 70 + i, order=8) for i, N in enumerate(sizes)]
    for bucket in (32, 256):
        check(H, items, bucket, proj=True)
