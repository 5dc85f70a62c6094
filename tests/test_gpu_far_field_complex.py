"""HBEM_FLAG_FAR_FIELD applies to real positive wavenumbers only: at complex and
negative ones a context with the flag gives the plain context's bits, in every tier
of kappa times the panel diameter and for every layer and k-derivative, also after
real wavenumbers of the same tier; at real positive ones it differs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def layers(H, bd, k, d):
    gb = H.GalerkinBuilder(bd)
    gb.assembleDense(k, 4.0, H.LayerType.ALL, d)
    return [f(t) for f in (gb.getDoubleLayer, gb.getHypersingular, gb.getSingleLayer) for t in range(d + 1)]


@pytest.mark.parametrize("kd", [0.4, 1.0, 2.0, 4.0])
def test_complex_wavenumbers_keep_the_full_rule(kd, H):
    sp = H.ContinuousSpace1()
    mesh = H.random_polygon_mesh(4, 7, 150)
    d = max(float(np.hypot(*(np.array(p[1.0]) - np.array(p[0.0])))) for p in mesh.getPanels())
    plain = H.BuilderData(mesh, sp, sp, 8)
    far = H.BuilderData(mesh, sp, sp, 8, flags=H.FLAG_FAR_FIELD)
    k = kd / (2.0 * d)
    assert not all(np.array_equal(a, b) for a, b in zip(layers(H, plain, k, 2), layers(H, far, k, 2)))
    for z in (k + 0.02j / d, k + 0.5j / d, complex(-k, 0.0)):
        for a, b in zip(layers(H, plain, z, 2), layers(H, far, z, 2)):
            assert np.array_equal(a, b), (kd, z, np.abs(a - b).max())


def test_batch_with_a_negative_wavenumber(H):
    """(which is evaluated as a complex one throughout)"""
    sp = H.ContinuousSpace1()
    mesh = H.random_polygon_mesh(4, 7, 90)
    ks = np.array([1.5, -2.0, 3.0])
    R = H.gaussian_test_matrix(180, 2, 0)
    a, b = (H.sigma_sweep(H.BuilderData(mesh, sp, sp, 8, flags=f), ks, 1.0, 4.0, R, 2) for f in (0, H.FLAG_FAR_FIELD))
    assert np.array_equal(a, b)
