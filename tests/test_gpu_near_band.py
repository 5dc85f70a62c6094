"""Accuracy of the near band (hbem_radial.hip) against extended precision: the
entries of the double and single layer between hats at most three panels apart, where
the kernel falls by orders of magnitude over the band, evaluated in 80-bit arithmetic
with the reference's quadrature rules (the oracle's doubles) and the Bessel functions
by Miller's recurrence and Neumann's series.

Bar: 8 units of rounding (the last roundings of coefficients, basis and sums), plus the
phase that rounded node positions put on H(kappa r): coordinates up to 1.3 are 18 panel
diameters here, so a difference of two is off by up to 36 units of d, and the 64 nodes
of a panel pair average it to an eighth; 8 kappa d units are allowed.  Beyond kappa d =
5 the real ones of these calls take the node loops, whose tables of the Bessel functions are good to
1e-14: 1e-14 more there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD, CL = np.longdouble, np.clongdouble
PI = 4 * np.arctan(LD(1))
EULER = LD("0.57721566490153286060651209008240243")
U = 2.0 ** -53
ORDER, N, APART = 8, 64, 3
VERTICES = [(0.0, 0.0), (1.0, 0.1), (1.3, 0.9), (0.5, 0.6), (-0.2, 1.1)]


def hankel(z):
    """H0, H1 (first kind) of real or complex z in extended precision."""
    a = float(np.abs(z).max())
    n = 2 * (int(a + 60 + 12 * a ** (1 / 3)) // 2)
    hi, lo = np.zeros_like(z), np.full_like(z, LD("1e-2000"))
    s = np.zeros_like(z)
    y0, y1 = np.zeros_like(z), np.zeros_like(z)
    for k in range(n, 0, -1):
        m = k // 2
        if k % 2 == 0:
            s = s + 2 * lo
            y0 = y0 + (-1) ** (m + 1) * 2 * lo / m
        elif m:
            y1 = y1 + (-1) ** (m + 1) * (2 * m + 1) * lo / LD(m * (m + 1))
        hi, lo = lo, 2 * k / z * lo - hi
    s = s + lo
    j0, j1, y0, y1 = lo / s, hi / s, y0 / s, y1 / s
    g = np.log(z / 2) + EULER
    return j0 + CL(1j) * (2 / PI) * (g * j0 + y0), j1 + CL(1j) * (2 / PI) * ((g - 1) * j1 + y1 - j0 / z)


def layers(O, mesh, kap):
    """K and V of the pairs of hats at most APART apart (galerkin_builder.cpp:17-346)."""
    pan = mesh.packed
    a0, tau = pan[:, 1:3].astype(LD), (pan[:, 3:5] - pan[:, 1:3]).astype(LD)
    a1, nrm = pan[:, 3:5].astype(LD), np.sqrt((tau ** 2).sum(1))
    xg, wg = (v.astype(LD) for v in O.gauss_rule(ORDER))
    xc, wc = (v.astype(LD) for v in O.composite_rule(ORDER))
    K, V = np.zeros((N, N), CL), np.zeros((N, N), CL)
    reach = APART + 1
    for i in range(N):
        for off in range(reach + 1):
            j = (i + off) % N                 # panel j follows i
            if off == 0:
                t, x = np.broadcast_arrays(xc[None, :], 1 - xc[:, None])
                rules = [(t * x, t, t * wc[:, None] * wc[None, :])]
            elif off == 1:                    # end of i = start of j: the nodes run from there
                t, x = np.broadcast_arrays(xc[:, None], xc[None, :])
                w = t * wc[:, None] * wc[None, :]
                rules = [(1 - t * x, t, w), (1 - t, t * x, w)]
            else:
                s, t = np.broadcast_arrays(xg[:, None], xg[None, :])
                rules = [(s, t, wg[:, None] * wg[None, :])]
            for s, t, w in rules:
                # positions are doubles in the library
                zi = [(a1[i][q] - tau[i][q] * (1 - s) if off == 1 else a0[i][q] + tau[i][q] * s).astype(float).astype(LD) for q in (0, 1)]
                zj = [(a0[j][q] + tau[j][q] * t).astype(float).astype(LD) for q in (0, 1)]
                vx, vy = zi[0] - zj[0], zi[1] - zj[1]
                r = np.sqrt(vx * vx + vy * vy)
                h0, h1 = hankel((kap * r).astype(CL if np.iscomplexobj(kap) else LD))
                hi, hj = (s, 1 - s), (t, 1 - t)
                k1 = kap * h1 / r * w
                kij = (vx * tau[j][1] - vy * tau[j][0]) * nrm[i] * k1
                kji = (vy * tau[i][0] - vx * tau[i][1]) * nrm[j] * k1
                v = nrm[i] * nrm[j] * h0 * w
                flat = max(np.abs((vx * tau[j][1] - vy * tau[j][0]) * nrm[i]).max(),
                           np.abs((vy * tau[i][0] - vx * tau[i][1]) * nrm[j]).max()) < 2.0 ** -52
                for a in (0, 1):
                    for b in (0, 1):
                        m, n = (i + 1 - a) % N, (j + 1 - b) % N
                        pairs = [(m, n, hi[a] * hj[b])] if off else [(m, n, hi[a] * hj[b] + hj[a] * hi[b])]
                        for p, q, f in pairs:
                            V[p, q] += (v * f).sum()
                            if off:
                                V[q, p] += (v * f).sum()
                            if off and not flat:
                                K[p, q] += (kij * f).sum()
                                K[q, p] += (kji * f).sum()
    return CL(1j) / 4 * K, CL(1j) / 4 * V


@pytest.mark.parametrize("kd", [0.3, 0.62, 2.4, 4.9, 9.9, 19.9, 0.4 + 0.03j, 4.5 + 0.045j, 9.0 + 0.045j, -4.5, -9.0])
def test_entries_next_to_the_diagonal(kd, H, O):
    if np.finfo(LD).eps > 1e-18:
        pytest.skip("long double is no wider than double here")
    mesh = H.polygon_mesh(VERTICES, N)
    d = max(float(np.hypot(*(np.array(p[1.0]) - np.array(p[0.0])))) for p in mesh.getPanels())
    k = complex(kd) / d
    sp = H.ContinuousSpace1()
    gb = H.GalerkinBuilder(H.BuilderData(mesh, sp, sp, ORDER))
    gb.assembleDense(k, 1.0)
    kap = CL(complex(0)) + LD(k.real) + CL(1j) * LD(k.imag) if k.imag or k.real < 0 else LD(k.real)
    m, n = np.indices((N, N))
    near = np.minimum((m - n) % N, (n - m) % N) <= APART
    bar = (8 + 8 * abs(kd)) * U + (1e-14 if np.isreal(kd) and kd > 5 else 0.0)
    for name, got, ref in zip("KV", (gb.getDoubleLayer(), gb.getSingleLayer()), layers(O, mesh, kap)):
        e = np.linalg.norm((got[near].astype(CL) - ref[near]).astype(complex)) / np.linalg.norm(ref[near].astype(complex))
        print("%s kd %s: %.1e of %.1e" % (name, kd, e, bar))
        assert e <= bar, (name, kd, e, bar)
