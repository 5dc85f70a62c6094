"""Meshes whose consecutive panels do not all meet: several closed curves in one
panel list, an open arc, curves far apart.  The hat over such a seam reaches from
one curve's end to the other's start, so its pairs' distances spread wider than the
bands of hbem_radial.hip, and the context has to sum panel pair by panel pair.

Every layer and k-derivative against the oracle within 1e-12 relative Frobenius (the
matrix bar of the plain path); the sweep's sigma is the oracle's within its bar of
1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def circles(H, *rest):
    """circles of (panels, radius, centre)"""
    return H.ParametrizedMesh([p for n, r, c in rest for p in H.circle_mesh(n, r, c).getPanels()])


MESHES = {
    "two_circles": lambda H: circles(H, (40, 0.4, (0.0, 0.0)), (40, 0.3, (2.0, 0.5))),
    "two_circles_near": lambda H: circles(H, (20, 0.4, (0.0, 0.0)), (24, 0.3, (0.75, 0.0))),
    "far_apart": lambda H: circles(H, (12, 0.4, (0.0, 0.0)), (13, 0.4, (50.0, 0.0))),
    "three": lambda H: circles(H, (9, 0.2, (0.0, 0.0)), (8, 0.2, (1.0, 1.0)), (10, 0.2, (-1.5, 0.3))),
    "open_arc": lambda H: H.ParametrizedMesh(H.ParametrizedLine((0, 0), (1, 0)).split(20)
                                             + H.ParametrizedLine((1, 0), (1.5, 1)).split(20)),
    "gap": lambda H: H.ParametrizedMesh(H.ParametrizedLine((0, 0), (1, 0)).split(15)
                                        + H.ParametrizedLine((1.2, 0), (1.2, 1)).split(15)
                                        + H.ParametrizedLine((1.2, 1), (0, 0)).split(20)),
}


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("k", [3.0, 3.0 + 0.05j])
def test_layers(name, k, H, O):
    m = MESHES[name](H)
    sp = H.ContinuousSpace1()
    gb = H.GalerkinBuilder(H.BuilderData(m, sp, sp, 8))
    gb.assembleDense(k, 4.0, H.LayerType.ALL, 2)
    K, W, V = O.assemble(m, 8, k, 4.0, d=2)
    # k-derivatives of W: the rounding of its curl part over (kappa h)^2 (tests/test_gpu_radial.py)
    h = min(float(np.hypot(*(np.array(p[1.0]) - np.array(p[0.0])))) for p in m.getPanels())
    curl = 8 * 2.0 ** -52 / (abs(k) * 2.0 * h) ** 2
    for t in range(3):
        for get, ref, lab in ((gb.getDoubleLayer, K, "K"), (gb.getHypersingular, W, "W"), (gb.getSingleLayer, V, "V")):
            tol = max(TOL, curl) if lab == "W" and t else TOL
            if name == "far_apart":
                tol = max(tol, 1e-11)   # points at 50 are rounded to 1e-14, nodes lie 2e-2 apart and v.n is r^2
            assert rel(get(t), ref[t]) <= tol, (name, k, lab, t, rel(get(t), ref[t]))


@pytest.mark.parametrize("name", ["two_circles", "three"])
def test_sweep(name, H, O):
    m = MESHES[name](H)
    sp = H.ContinuousSpace1()
    bd = H.BuilderData(m, sp, sp, 8)
    n = 2 * m.getNumPanels()
    R = H.gaussian_test_matrix(n, 2, 3)
    ks = np.linspace(1.0, 5.0, 33)
    s = H.sigma_sweep(bd, ks, 1.0, 4.0, R, 2, proj=False)
    ref = O.SolOp(m, 8, proj=False).sigma_sweep(ks[[0, 17, 32]], 1.0, 4.0, R, 2)
    assert np.all(np.abs(s[[0, 17, 32]] - ref) <= 1e-10 * ref), (s[[0, 17, 32]], ref)
