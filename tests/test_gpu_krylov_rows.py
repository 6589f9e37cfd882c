"""Rosenbrock-Krylov chemistry with half a wave per cell against one lane per cell (taken by the
same mechanism with an additional zero T^5 term in its NASA polynomials): boxes that leave half
a wave or a workgroup empty, 9, 13 and 14 species, the PaSR closure, the transport forcing, a
mixture fraction outside the window in some cells, which stay untouched.  The operations are the same
but for the compiler's contraction, so the bound is that of the oracle comparison, 1e-9; with
the forcing the step control amplifies rounding and the bound is ten times the one-lane kernel's own
response to a change of its input by 1e-15, as there."""
import dataclasses

import numpy as np
import pytest

from parity_util import interior, rel_maxnorm
from test_gpu_cells import _state, _tables
from test_gpu_routine_cells import _general_nasa

pytestmark = pytest.mark.gpu
NG = 3


@pytest.mark.parametrize("mech,shape,pasr,forced", [
    ("h2", (1, 1, 1), False, False), ("h2", (3, 1, 1), True, False), ("davis", (5, 3, 2), True, False),
    ("keromnes", (7, 5, 1), False, False), ("h2", (7, 5, 1), False, True)])
def test_rows_match_one_lane_per_cell(pkg, mech, shape, pasr, forced):
    tb = _tables(pkg, mech)
    ns = tb.n_species
    be = pkg.solver.HipBackend()
    num = pkg.solver.Numerics(enable_chemistry=2, rosenbrock_version=2)
    if pasr:
        num = dataclasses.replace(num, enable_les=1, les_model=2, les_pr=0.7, les_sc=0.7, les_c_wale=0.3,
                                  les_c_yoshi=0.1, les_c_eps=1.0, les_c_mix=0.1)
    w, tg = _state(pkg, tb, shape, NG, 8)
    rng = np.random.default_rng(4)
    z = np.where(rng.uniform(size=tg.shape) < 0.2, 1.0, 0.5)
    z[NG, NG, NG] = 0.5
    f = None
    if forced:
        f = be.asarray(rng.standard_normal((ns + 4,) + shape[::-1]) * 1e-3 * np.abs(interior(w, NG)) / 1e-8)

    def run(tables, scale=1.0):
        s = pkg.solver.Solver(be, tables, *shape, NG, [2.0e-5 * n for n in shape], numerics=num, rho0=0.3, u0=150.0)
        s.set_state(w * scale, tg)
        aux = be.to_numpy(s.w_aux).copy()
        aux[ns + 10], aux[ns + 11], aux[ns + 7] = w[:ns].sum(axis=0), z, 5.0e-5      # J_R, J_Z, J_MU
        if pasr:
            aux[2 * ns + 13] = 1.0e-4
        be.copy_(s.w_aux, be.asarray(aux))
        s.rosenbrock_krylov(1.0e-8, f)
        be.sync()
        return interior(be.to_numpy(s.w), NG)

    print(f"[krylov rows] {mech} {shape} {pasr} {forced}", flush=True)
    rows, lanes = run(tb), run(_general_nasa(tb))
    bound = 1e-9
    if forced:
        bound = max(bound, 10.0 * rel_maxnorm(run(_general_nasa(tb), 1.0 + 1e-15), lanes).max())
    assert rel_maxnorm(rows, lanes).max() < bound
    assert not np.array_equal(rows, interior(w, NG))
    still = interior(z, NG) > 0.9
    np.testing.assert_array_equal(rows[:, still], interior(w, NG)[:, still])
