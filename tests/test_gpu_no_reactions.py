"""The implicit integrators walk their reactions from 0 to nreactions, so a negative count is a
mechanism without reactions (streams_compute_chemistry refuses it, these two do not): the same
bits as with none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("version", [1, 2])
def test_negative_count_is_no_reaction(pkg, h2_tables, version):
    from test_gpu_cells import _state
    shape, ng = (5, 4, 3), 3
    w, tg = _state(pkg, h2_tables, shape, ng, 6)
    w[0, ng] *= -1.0                      # clipped by ROS4 even where nothing reacts
    be = pkg.solver.HipBackend()
    out = []
    for nr in (0, -1):
        num = pkg.solver.Numerics(enable_chemistry=2, rosenbrock_version=version, ros_maxsteps=5)
        s = pkg.solver.Solver(be, h2_tables, *shape, ng, [1e-4] * 3, numerics=num)
        s.set_state(w, tg)
        be.fill_(s.w_aux[s.ns + 11], 0.5)
        s.nr = nr
        (s.rosenbrock if version == 1 else s.rosenbrock_krylov)(1.0e-9)
        be.sync()
        out.append((be.to_numpy(s.w), be.to_numpy(s.w_aux)))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
