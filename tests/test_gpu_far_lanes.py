"""Coefficients of the far bands (hbem_radial.hip, k_radial_far), with 64 lanes to a
pair of hats where there are few pairs and with 16 where there are many: panel counts
on both sides of that line (512 tiles of 16 pairs, near 125 panels) and the fewest,
orders whose nodes leave some of the lanes idle or fill them several times.  Against
the oracle, at the plain path's matrix bar of 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kd", [0.4, 4.0])
@pytest.mark.parametrize("n,order", [(9, 3), (9, 12), (40, 17), (118, 3), (118, 8), (126, 8), (134, 3), (134, 8)])
def test_far_bands(n, order, kd, H, O):
    m = H.polygon_mesh([(0, 0), (1, 0), (1.2, 0.7), (0.1, 1)], n)
    d = max(float(np.hypot(*(np.array(p[1.0]) - np.array(p[0.0])))) for p in m.getPanels())
    sp = H.ContinuousSpace1()
    gb = H.GalerkinBuilder(H.BuilderData(m, sp, sp, order))
    gb.assembleDense(kd / d, 1.0, H.LayerType.ALL, 0)
    for ref, out in zip(O.assemble(m, order, kd / d, 1.0, d=0), (gb.getDoubleLayer(0), gb.getHypersingular(0), gb.getSingleLayer(0))):
        assert np.linalg.norm(out - ref[0]) <= 1e-12 * np.linalg.norm(ref[0])
