"""Rows of lanes that take more than one cell each: fields larger than the 8192 cells that the
Rosenbrock rows have in flight, against one lane per cell, bit for bit; some cells are not finite, so
that the turn after such a cell starts clean, and among the others are a few whose energy column of
the Jacobian is not finite while the species' columns are."""
import numpy as np
import pytest

from test_gpu_cells import _tables
from test_gpu_rosenbrock_rows import _run
from test_gpu_routine_cells import _general_nasa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mech,shape,pasr,limits", [
    ("h2", (25, 20, 18), False, {"ros_maxsteps": 4}),
    ("h2", (40, 32, 32), True, {"ros_maxsteps": 2}),
    ("h2", (41, 32, 32), False, {"ros_maxsteps": 1}),
    ("keromnes", (32, 32, 26), False, {"ros_maxsteps": 2}),
    ("davis", (33, 32, 26), False, {"ros_maxsteps": 1}),
])
def test_rosenbrock_rows_take_several_cells(pkg, mech, shape, pasr, limits):
    tb = _tables(pkg, mech)
    be = pkg.solver.HipBackend()
    print(f"[rosenbrock turns] {mech} {shape} {pasr} {limits}", flush=True)
    rows = _run(pkg, be, tb, shape, 2.0e-9, pasr, True, **limits)
    lanes = _run(pkg, be, _general_nasa(tb), shape, 2.0e-9, pasr, True, **limits)
    for a, b in zip(rows, lanes):
        np.testing.assert_array_equal(a, b)
    good = np.isfinite(rows[0]).all(axis=0)
    assert good.any() and not good.all()
