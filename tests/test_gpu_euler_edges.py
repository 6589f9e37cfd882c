"""Fields with order-reduced and zeroed faces above and below the size up to which the cells and
the edges of a direction share a launch (768 workgroups of 256 cells): the edges are then listed,
along x from 1024 cells at a time, whose last group is only partly filled; lines whose ends are most
of them.  Against the oracle within 1e-12 of each variable's largest right-hand side, as the
other sizes."""
import pytest

from test_gpu_routine_cells import TOL, _fl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [0, 1, 2])
@pytest.mark.parametrize("shape,ng,order,force", [((67, 61, 53), 4, 8, [1, 0, 0, 1, 1, 1]),
                                                  ((8, 160, 154), 3, 6, [0, 1, 1, 0, 0, 0]),
                                                  ((8, 160, 153), 3, 6, None)])
def test_reduced_ends_of_large_fields(pkg, oracle, h2_tables, d, shape, ng, order, force):
    num = pkg.solver.Numerics(ep_order=order, visc_order=order, sensor_threshold=2.0, correct_bound_ord=1)
    print(f"[euler edges] {shape} order {order} direction {d}", flush=True)
    err = _fl(pkg, oracle, h2_tables, shape, ng, num, lambda s: s.euler(d), (2,) * 6, force)
    assert err.max() < TOL, err
