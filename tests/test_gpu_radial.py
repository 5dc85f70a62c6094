"""The banded assembly (hbem_radial.hip) at the edges of its ranges, against the
oracle: every layer and k-derivative within 1e-12 relative Frobenius (the
matrix bar of the plain path; 8 units of rounding over (kappa h)^2, h the
shortest panel, for the k-derivatives of W where that is more: the curl part's
large constant cancels between neighbouring panels, in the oracle's own
rounding too) for

* each tier of kappa times the largest panel diameter, from far below the
  first edge to beyond the last one, where the node loops take over;
* curves whose pairs of hats fall into the bands in unusual ways: the fewest
  panels (8; 7 takes the node loops), a needle-sharp corner, two arms closer
  than a panel, panels of very different length, arcs, a trigonometric curve,
  a spline;
* quadrature orders 3, 8 and 16;
* complex wavenumbers on both sides of the near band's limit, and negative ones;
* odd numbers of columns, unsorted wavenumbers of several tiers in one call.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def dmax(mesh):
    """Largest panel chord."""
    return max(float(np.hypot(*(np.array(p[1.0]) - np.array(p[0.0])))) for p in mesh.getPanels())


def shortest(mesh):
    return min(float(np.hypot(*(np.array(p[1.0]) - np.array(p[0.0])))) for p in mesh.getPanels())


def graded(H):
    """A square whose lower side has panels 40 times shorter than the others'."""
    v = [(0, 0), (1, 0), (1, 1), (0, 1)]
    panels = H.ParametrizedLine(v[0], v[1]).split(40)
    for a, b in ((1, 2), (2, 3), (3, 0)):
        panels += H.ParametrizedLine(v[a], v[b]).split(1)
    return H.ParametrizedMesh(panels)


def spline(H):
    from helmholtzbem_amd import scatterer
    import os
    path = os.path.join(os.path.dirname(__file__), "golden", "scatterers", "scatterer_circle.dat")
    return H.ParametrizedMesh(scatterer.SmoothScatterer(path).panelize(30))


MESHES = {
    "fewest": lambda H: H.polygon_mesh([(0, 0), (1, 0), (1, 0.7), (0, 1)], 8),
    "loops7": lambda H: H.polygon_mesh([(0, 0), (1, 0), (0.3, 0.8)], 7),
    "needle": lambda H: H.polygon_mesh([(0, 0), (2, 0.02), (2, 0.3)], 61),
    "slit": lambda H: H.polygon_mesh([(0, 0), (1, 0), (1, 0.5), (0.45, 0.5), (0.45, 0.02), (0.44, 0.02), (0.44, 0.5), (0, 0.5)], 67),
    "graded": graded,
    "arcs": lambda H: H.circle_mesh(33, 0.4, (0.1, 0.2)),
    "star": lambda H: H.star_mesh(45),
}


@pytest.fixture(scope="module", params=sorted(MESHES))
def mesh(request, H):
    return request.param, MESHES[request.param](H)


def compare(H, O, name, mesh, order, k, c, d, flags=0):
    sp = H.ContinuousSpace1()
    gb = H.GalerkinBuilder(H.BuilderData(mesh, sp, sp, order, flags=flags))
    gb.assembleDense(k, c, H.LayerType.ALL, d)
    K, W, V = O.assemble(mesh, order, k, c, d=d)
    curl = 8 * 2.0 ** -52 / (abs(k) * np.sqrt(c) * shortest(mesh)) ** 2
    for t in range(d + 1):
        for get, ref, lab in ((gb.getDoubleLayer, K, "K"), (gb.getHypersingular, W, "W"), (gb.getSingleLayer, V, "V")):
            assert rel(get(t), ref[t]) <= (max(TOL, curl) if lab == "W" and t else TOL), (name, order, k, lab, t, rel(get(t), ref[t]))
        assert np.array_equal(gb.getSingleLayer(t), gb.getSingleLayer(t).T)
        assert np.array_equal(gb.getHypersingular(t), gb.getHypersingular(t).T)


@pytest.mark.parametrize("kd", [1e-3, 0.6249, 0.626, 1.3, 2.51, 5.1, 10.5, 21.0])
def test_tiers(mesh, kd, H, O):
    name, m = mesh
    c = 4.0
    compare(H, O, name, m, 8, kd / (dmax(m) * np.sqrt(c)), c, 2)


@pytest.mark.parametrize("order", [3, 16])
def test_orders(mesh, order, H, O):
    name, m = mesh
    compare(H, O, name, m, order, 0.5 / dmax(m), 1.0, 1)


@pytest.mark.parametrize("im", [0.02, 0.049, 0.2, -0.0])
def test_complex_wavenumbers(mesh, im, H, O):
    """kappa d = 0.4 + i im: the near band serves Im kappa up to 0.05 / dmax;
    im = -0.0: the negative real wavenumber of that size."""
    name, m = mesh
    d = dmax(m)
    k = complex(0.4 / d, im / d) if im else complex(-0.4 / d, 0.0)
    compare(H, O, name, m, 8, k, 1.0, 2)


def test_spline_panels(H, O):
    m = spline(H)
    compare(H, O, "spline", m, 8, 0.7 / dmax(m), 2.0, 2)


@pytest.mark.parametrize("nk", [1, 5, 17, 33])
def test_unsorted_wavenumbers_of_several_tiers(nk, H):
    """Each column of a batched call, and each sigma of a sweep, is the one of a
    call of its own: the same bits whatever the other wavenumbers, their order
    and number."""
    m = H.polygon_mesh([(0, 0), (1, 0), (1.2, 0.7), (0.1, 1)], 40)
    sp = H.ContinuousSpace1()
    bd = H.BuilderData(m, sp, sp, 8)
    rng = np.random.default_rng(nk)
    ks = rng.uniform(0.1, 6.0, nk) / dmax(m)
    out = H.assemble_dense_batch(bd, ks, 3.0, H.LayerType.ALL, 1)
    gb = H.GalerkinBuilder(bd)
    for i in sorted({0, nk // 2, nk - 1}):
        gb.assembleDense(ks[i], 3.0, H.LayerType.ALL, 1)
        for t in range(2):
            assert np.array_equal(out[H.LayerType.DOUBLE][i, t], gb.getDoubleLayer(t))
            assert np.array_equal(out[H.LayerType.HYPERSINGULAR][i, t], gb.getHypersingular(t))
            assert np.array_equal(out[H.LayerType.SINGLE][i, t], gb.getSingleLayer(t))
    R = H.gaussian_test_matrix(80, 2, 1)
    sig = H.sigma_sweep(bd, ks, 1.0, 3.0, R, 2)
    rev = H.sigma_sweep(bd, ks[::-1], 1.0, 3.0, R, 2)
    assert np.array_equal(sig, rev[::-1])
