"""Half waves that take more than one cell each: fields larger than the 4096 cells that the Krylov rows
have in flight, up to the largest that they take and just above.  The step control amplifies
rounding in the stiffer of these random states: the difference from one lane per cell is held, at its
median, its 90 and 99 per cent points and its largest value over the cells, to ten times the one-lane
kernel's own response to a change of its input by 1e-15, or 1e-9 where that is smaller; a cell
that took another's state or a stale one would be off by its whole change."""
import numpy as np
import pytest

from parity_util import interior
from test_gpu_cells import _state, _tables
from test_gpu_rosenbrock_rows import NG
from test_gpu_routine_cells import _general_nasa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mech,shape,forced", [("h2", (17, 16, 16), False), ("h2", (24, 16, 16), True),
                                               ("h2", (25, 16, 16), False), ("keromnes", (32, 16, 16), False)])
def test_krylov_rows_take_several_cells(pkg, mech, shape, forced):
    tb = _tables(pkg, mech)
    ns = tb.n_species
    be = pkg.solver.HipBackend()
    num = pkg.solver.Numerics(enable_chemistry=2, rosenbrock_version=2)
    w, tg = _state(pkg, tb, shape, NG, 8)
    rng = np.random.default_rng(4)
    z = np.where(rng.uniform(size=tg.shape) < 0.2, 1.0, 0.5)
    f = None
    if forced:
        f = be.asarray(rng.standard_normal((ns + 4,) + shape[::-1]) * 1e-3 * np.abs(interior(w, NG)) / 1e-8)

    def run(tables, scale=1.0):
        s = pkg.solver.Solver(be, tables, *shape, NG, [2.0e-5 * n for n in shape], numerics=num, rho0=0.3, u0=150.0)
        s.set_state(w * scale, tg)
        aux = be.to_numpy(s.w_aux).copy()
        aux[ns + 10], aux[ns + 11] = w[:ns].sum(axis=0), z       # J_R, J_Z
        be.copy_(s.w_aux, be.asarray(aux))
        s.rosenbrock_krylov(1.0e-8, f)
        be.sync()
        return interior(be.to_numpy(s.w), NG)

    print(f"[krylov turns] {mech} {shape} {forced}", flush=True)
    rows, lanes = run(tb), run(_general_nasa(tb))
    def apart(a):
        d = (np.abs(a - lanes) / np.abs(lanes).max(axis=(1, 2, 3), keepdims=True)).max(axis=0)
        return np.quantile(d, (0.5, 0.9, 0.99, 1.0))

    difference, response = apart(rows), apart(run(_general_nasa(tb), 1.0 + 1e-15))
    print("[krylov turns] difference", difference, "response", response, "change", apart(interior(w, NG)), flush=True)
    assert (difference < np.maximum(1e-9, 10.0 * response)).all()
    still = interior(z, NG) > 0.9
    np.testing.assert_array_equal(rows[:, still], interior(w, NG)[:, still])
    assert (rows[:, ~still] != interior(w, NG)[:, ~still]).any(axis=0).all()
