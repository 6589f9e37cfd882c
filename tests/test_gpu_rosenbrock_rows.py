"""Implicit chemistry of a field with a row of 16 lanes per cell against one lane per cell, bit
for bit: the same mechanism with an additional zero T^5 term in its NASA polynomials takes the
one-lane kernel, whose sums that term leaves as they are.  Boxes that leave rows of a wave empty (1,
3, 30, 105 cells), temperatures about the polynomials' 1000 K limit (a range changes within
the temperature iteration), a negative first species, the PaSR closure, species counts that fill
9, 13 and 14 lanes, steps cut off by maxsteps and maxtry, a state that is not finite; and a
mechanism with five species on a side, which stays with the one-lane kernel."""
import dataclasses

import numpy as np
import pytest

from parity_util import interior
from test_gpu_cells import _state, _tables
from test_gpu_routine_cells import _general_nasa

pytestmark = pytest.mark.gpu
NG = 3


def _run(pkg, be, tb, shape, dt, pasr=False, spoil=False, **limits):
    num = pkg.solver.Numerics(enable_chemistry=2, operator_splitting=1, **limits)
    if pasr:
        num = dataclasses.replace(num, enable_les=1, les_model=2, les_pr=0.7, les_sc=0.7, les_c_wale=0.3,
                                  les_c_yoshi=0.1, les_c_eps=1.0, les_c_mix=0.1)
    w, tg = _state(pkg, tb, shape, NG, 8)
    ns = tb.n_species
    rng = np.random.default_rng(2)
    T = rng.uniform(950.0, 1050.0, tg.shape)
    rho = w[:ns].sum(axis=0)
    Y = np.moveaxis(w[:ns] / rho, 0, -1)
    e = tb.e_from_T_many(T.ravel(), Y.reshape(-1, ns)).reshape(T.shape)
    w[ns + 3] = rho * e + 0.5 * (w[ns:ns + 3] ** 2).sum(0) / rho
    w[0].ravel()[::3] *= -1.0e-6
    if spoil:
        w[1].ravel()[::5] = np.inf
    s = pkg.solver.Solver(be, tb, *shape, NG, [2.0e-5 * n for n in shape], numerics=num, rho0=0.3, u0=150.0)
    s.set_state(w, T + rng.uniform(-80.0, 80.0, T.shape))
    aux = be.to_numpy(s.w_aux).copy()
    aux[ns + 10] = rho                    # J_R
    aux[ns + 7] = 5.0e-5                  # J_MU
    if pasr:
        aux[2 * ns + 13] = rng.uniform(1.0e-5, 1.0e-3, T.shape)
    be.copy_(s.w_aux, be.asarray(aux))
    s.rosenbrock(dt)
    be.sync()
    return interior(be.to_numpy(s.w), NG), interior(be.to_numpy(s.w_aux), NG)


@pytest.mark.parametrize("mech,shape,pasr,spoil,limits", [
    ("h2", (1, 1, 1), False, False, {}),
    ("h2", (3, 1, 1), True, False, {}),
    ("davis", (5, 3, 2), False, False, {}),
    ("keromnes", (7, 5, 3), True, False, {}),
    ("h2", (7, 5, 3), False, False, {"ros_maxsteps": 2}),
    ("h2", (7, 5, 3), False, False, {"ros_maxtry": 2}),
    ("h2", (5, 3, 2), False, True, {"ros_maxsteps": 3}),
])
def test_rows_match_one_lane_per_cell(pkg, mech, shape, pasr, spoil, limits):
    tb = _tables(pkg, mech)
    be = pkg.solver.HipBackend()
    print(f"[rosenbrock rows] {mech} {shape} {pasr} {spoil} {limits}", flush=True)
    rows = _run(pkg, be, tb, shape, 2.0e-9, pasr, spoil, **limits)
    lanes = _run(pkg, be, _general_nasa(tb), shape, 2.0e-9, pasr, spoil, **limits)
    for a, b in zip(rows, lanes):
        np.testing.assert_array_equal(a, b)
    if spoil:                            # the unspoiled states of davis hold a few such cells as well
        assert not np.isfinite(rows[0]).all()
    assert np.isfinite(rows[0]).all(axis=0).any()


def test_wide_sides_take_one_lane_per_cell(pkg, h2_tables):
    """Both calls take the one-lane kernel; a row kernel would drop the fifth species."""
    r = np.array(h2_tables.r_coeffs)
    r[0] = 0.0
    r[0, :5] = (1.0, 0.5, 1.0, 1.0, 0.5)
    tb = dataclasses.replace(h2_tables, r_coeffs=r)
    be = pkg.solver.HipBackend()
    a = _run(pkg, be, tb, (5, 3, 2), 2.0e-9)
    b = _run(pkg, be, _general_nasa(tb), (5, 3, 2), 2.0e-9)
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])
    assert not np.array_equal(a[0], _run(pkg, be, h2_tables, (5, 3, 2), 2.0e-9)[0])
