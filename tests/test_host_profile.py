"""The profile's phases (hbem_profile_query) hold every assembly launch: on the bands
the far products (0) and the near band's (1), on the node loops the three classes of
panel pairs (0-2).  On the CPU, with the HIP runtime double of test_host_memory.py."""
import pytest

from test_host_memory import run, stub  # noqa: F401

BODY = """
mesh = H.polygon_mesh([(0, 0), (1, 0), (1.2, 0.7), (0.1, 1)], %(panels)d)
bd = H.BuilderData(mesh, SP, SP, 8)
ks = np.linspace(1.0, 3.0, 5)
R = H.gaussian_test_matrix(2 * %(panels)d, 2, 1)
H.sigma_sweep(bd, ks, 1.0, 4.0, R, 2, der=%(der)d)
H.profile_enable(bd)
launches()
H.sigma_sweep(bd, ks, 1.0, 4.0, R, 2, der=%(der)d)
eval_ = [x for x in launches() if "k_band_eval" in x]
q = [H.profile_query(bd, w) for w in range(7)]
print(q, eval_)
assert [x[1] for x in q[:3]] == %(want)r, q
assert all((x[1] > 0) == (x[2] > 0) for x in q[:3]), q
assert len(eval_) == %(evals)d, eval_
assert all(x[1] == 1 for x in q[3:6]), q
"""


@pytest.mark.parametrize("der", [0, 1, 2])
@pytest.mark.parametrize("panels,want,evals", [(120, [1, 1, 0], 2), (7, [1, 1, 1], 0)])
def test_every_assembly_launch_has_a_phase(stub, panels, want, evals, der):  # noqa: F811
    run(stub, BODY % dict(panels=panels, want=want, evals=evals, der=der))
