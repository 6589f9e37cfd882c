"""The one-thread-per-cell forms of the convective, viscous and chemistry routines where they can
go wrong: ragged boxes, every KEEP order and energy split, faces of reduced order and faces whose
flux is zeroed on short axes, NASA tables in the general form, mechanisms that do not fit the
packed records (a side of five species) or the local memory (a reaction set repeated until it
exceeds it), against the oracle within 1e-12 of each variable's largest right-hand side, the
tolerance of the routines' other parity tests."""
import dataclasses

import numpy as np
import pytest

from parity_util import rel_maxnorm

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _fl(pkg, oracle, tb, shape, ng, num, stage, bctags=(0,) * 6, force=None, seed=5, stretched=False):
    import oracle_backend
    from test_gpu_cells import _state
    w, tg = _state(pkg, tb, shape, ng, seed)
    maps = [lambda x, h=2.0e-5: x + 0.2 * h * np.sin(x / h)] * 3 if stretched else None
    out = []
    for be in (oracle_backend.OracleBackend(oracle), pkg.solver.HipBackend()):
        s = pkg.solver.Solver(be, tb, *shape, ng, [2.0e-5 * n for n in shape], bctags=bctags, numerics=num, rho0=0.3,
                              u0=150.0, mappings=maps)
        s.set_state(w, tg)
        if force is not None:
            s.force_zero_flux = force
        if not out:
            s.bcswap()
            s.compute_aux()
            ref = s
        else:                            # the oracle's auxiliaries, so one routine is compared
            be.copy_(s.w_aux, be.asarray(ref.w_aux))
            be.copy_(s.w, be.asarray(ref.w))
        stage(s)
        be.sync()
        out.append(be.to_numpy(s.fl).copy())
    return rel_maxnorm(out[1], out[0])


@pytest.mark.parametrize("d", [0, 1, 2])
@pytest.mark.parametrize("shape,ng,order,nkeep,bc,force", [
    ((37, 5, 3), 4, 8, 0, (0,) * 6, None),
    ((5, 37, 9), 3, 4, -1, (0,) * 6, None),
    ((9, 6, 41), 3, 2, 0, (0,) * 6, None),
    ((11, 13, 12), 4, 8, 0, (2, 2, 2, 2, 2, 2), [1, 0, 0, 1, 1, 1]),
    ((7, 8, 9), 3, 6, -1, (2, 2, 2, 2, 2, 2), [0, 1, 1, 1, 0, 1]),
])
def test_euler_without_sensor(pkg, oracle, h2_tables, d, shape, ng, order, nkeep, bc, force):
    num = pkg.solver.Numerics(ep_order=order, visc_order=order, nkeep=nkeep, sensor_threshold=2.0,
                              weno_scheme=min(ng, 3), correct_bound_ord=int(bc[0] != 0))
    err = _fl(pkg, oracle, h2_tables, shape, ng, num, lambda s: s.euler(d), bc, force)
    assert err.max() < TOL, err


def _general_nasa(tb):
    """The same polynomials with a zero T^5 term: a form that has no staged variant."""
    n = tb.indx_cp_r - tb.indx_cp_l + 1
    grow = lambda a: np.insert(a, n, 0.0, axis=0)  # noqa: E731
    return dataclasses.replace(tb, indx_cp_r=tb.indx_cp_r + 1, cp_coeff=grow(tb.cp_coeff), cv_coeff=grow(tb.cv_coeff))


@pytest.mark.parametrize("shape,mech,general", [((37, 5, 3), "h2", False), ((6, 21, 19), "keromnes", False),
                                                ((5, 7, 33), "davis", True)])
def test_viscous_faces(pkg, oracle, shape, mech, general):
    from test_gpu_cells import _tables
    tb = _tables(pkg, mech)
    if general:
        tb = _general_nasa(tb)
    err = _fl(pkg, oracle, tb, shape, 3, pkg.solver.Numerics(), lambda s: s.visflx(1), stretched=True)
    assert err.max() < TOL, err


@pytest.mark.parametrize("shape,mech,change", [((37, 5, 3), "h2", "none"), ((64, 2, 2), "keromnes", "none"),
                                               ((5, 7, 33), "h2", "general"), ((9, 8, 7), "h2", "five"),
                                               ((9, 8, 7), "h2", "many"), ((9, 8, 7), "h2", "three"),
                                               ((150, 60, 40), "h2", "none")])
def test_chemistry_tables(pkg, oracle, shape, mech, change):
    """(150, 60, 40): more cells than the grid's threads, so a workgroup takes several rounds."""
    from test_gpu_cells import _tables
    tb = _tables(pkg, mech)
    if change == "general":
        tb = _general_nasa(tb)
    elif change == "five":
        r = np.array(tb.r_coeffs)
        r[0] = 0.0
        r[0, :5] = (1.0, 0.5, 2.0, 1.0, 0.25)
        tb = dataclasses.replace(tb, r_coeffs=r)
    elif change in ("many", "three"):            # beyond the local memory, and most of it
        rep = 6 if change == "many" else 3
        cat = lambda a, ax=0: np.concatenate([np.asarray(a)] * rep, axis=ax)  # noqa: E731
        kc = np.asarray(tb.kc_tab)
        rows = {f: cat(getattr(tb, f)) for f in ("reac_ty", "isRev", "arr_a", "arr_b", "arr_ea", "falloff_coeffs",
                                                 "tb_eff", "r_coeffs", "p_coeffs")}
        tb = dataclasses.replace(tb, nreactions=rep * tb.nreactions, kc_tab=cat(kc, kc.ndim - 1), **rows)
    err = _fl(pkg, oracle, tb, shape, 3, pkg.solver.Numerics(), lambda s: s.compute_chemistry())
    assert err.max() < TOL, err
