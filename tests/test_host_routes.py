"""Which way a call's wavenumbers take -- the bands or the node loops -- read off the
kernels it launches, on the CPU with the HIP runtime double of test_host_memory.py.

kappa d is kappa times the largest panel diameter: builder calls (single matrices,
batches of them, solutions operators, transmission solves) take the bands up to 5 at
real wavenumbers and up to 20 at complex ones, sweeps up to 20, all only where
consecutive panels meet and there are 8 of them."""
import pytest

from test_host_memory import run, stub  # noqa: F401

BODY = """
from helmholtzbem_amd.solvers import tp
N = %(panels)d
mesh = H.polygon_mesh([(0, 0), (1, 0), (1.2, 0.7), (0.1, 1)], N)
bd = H.BuilderData(mesh, SP, SP, 8, flags=%(flags)d)
d = max(float(np.hypot(*(np.array(p[1.0]) - np.array(p[0.0])))) for p in mesh.getPanels())
k = %(kd)s / (2.0 * d)
R = H.gaussian_test_matrix(2 * N, 2, 1)
u, g = (lambda x, y: complex(x, y)), (lambda x, y: (1j, 1.0))
calls = {
    "layers": lambda: H.GalerkinBuilder(bd).assembleDense(k, 4.0),
    "batch": lambda: H.assemble_dense_batch(bd, np.full(%(nk)d, k), 4.0, H.LayerType.ALL, 0),
    "operator": lambda: H.SolutionsOperator(bd).gen_sol_op(k, 1.0, 4.0),
    "transmission": lambda: tp.direct_second_kind.solve(mesh, u, g, 8, k, 1.0, 4.0),
    "sweep": lambda: H.sigma_sweep(bd, np.full(%(nk)d, k), 1.0, 4.0, R, 2),
    "multi": lambda: H.sigma_sweep_batched([(bd, np.full(%(nk)d, k), 1.0, 4.0, R)], 2),
}
launches()
calls[%(call)r]()
log = launches()
bands, loops = (any(s in x for x in log) for s in ("k_band_eval", "k_records_from_locals"))
print(bands, loops)
assert (bands, loops) == %(want)r, sorted({x.split()[0] for x in log})
"""
BANDS, LOOPS = (True, False), (False, True)
BUILDER, SWEEP = ("layers", "batch", "operator", "transmission"), ("sweep", "multi")


@pytest.mark.parametrize("call", BUILDER + SWEEP)
@pytest.mark.parametrize("nk", [1, 33])
@pytest.mark.parametrize("kd", ["0.5", "4.9", "5.1", "19.0", "21.0"])
def test_real_wavenumbers(stub, call, nk, kd):  # noqa: F811
    want = BANDS if float(kd) <= (5.0 if call in BUILDER else 20.0) else LOOPS
    run(stub, BODY % dict(panels=40, flags=0, kd=kd, nk=nk, call=call, want=want))


@pytest.mark.parametrize("kd,want", [("(0.5 + 0.03j)", BANDS), ("(0.5 + 0.2j)", LOOPS), ("(9 + 0.03j)", BANDS), ("-0.5", BANDS), ("-9.0", BANDS), ("(21 + 0.03j)", LOOPS)])
def test_complex_wavenumbers(stub, kd, want):  # noqa: F811
    run(stub, BODY % dict(panels=40, flags=0, kd=kd, nk=1, call="layers", want=want))


@pytest.mark.parametrize("call", ["layers", "sweep"])
def test_few_panels(stub, call):  # noqa: F811
    run(stub, BODY % dict(panels=7, flags=0, kd="0.5", nk=1, call=call, want=LOOPS))
