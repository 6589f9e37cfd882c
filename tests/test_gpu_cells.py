"""streams_rhs_cells, the one-pass right-hand side of 3-D boxes on which every face takes the
KEEP flux of one order: the fused step on boxes that leave its 32 x 4 x 2 tiles and 8-tile
bands partly filled (down to two cells along an axis), with 9, 13 and 14 species, sixth and
eighth order, stretched grids, walls, chemistry on and off, against the oracle run routine by
routine, within 1e-12 of each variable's largest right-hand side and 1e-11 of its largest value
after a Runge-Kutta step, the tolerances of the sweeps it replaces; and against the sweeps
themselves on the GPU."""
import numpy as np
import pytest

from parity_util import box_state, interior, rel_maxnorm

pytestmark = pytest.mark.gpu

CASES = [
    # shape, mechanism, ng, order, boundaries, chemistry, stretched
    ((33, 5, 3), "h2", 3, 6, (0,) * 6, 1, False),
    ((32, 36, 2), "h2", 3, 6, (0,) * 6, 1, False),
    ((64, 4, 4), "h2", 4, 8, (0,) * 6, 1, False),
    ((2, 9, 5), "h2", 4, 8, (0, 0, 0, 0, 0, 0), 0, False),
    ((19, 14, 11), "davis", 3, 6, (0,) * 6, 1, False),
    ((21, 35, 3), "keromnes", 3, 6, (0, 0, 8, 2, 0, 0), 1, True),
    ((40, 3, 9), "h2", 4, 6, (2, 2, 0, 0, 8, 8), 0, True),
]


def _tables(pkg, mech):
    if mech == "h2":
        return pkg.cases.h2_air_mechanism().tables()
    name = {"davis": "davis2005_13sp.yaml", "keromnes": "keromnes2013_14sp.yaml"}[mech]
    return pkg.mechanism.Mechanism(str(pkg.cases.mechanism_path(name))).tables()


def _state(pkg, tb, shape, ng, seed):
    """A seeded smooth periodic state of any mechanism (padded) and the temperature guess."""
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    ns = tb.n_species
    T = 1250.0 + 150.0 * rng.uniform(-1, 1, (nz, ny, nx))
    Y = rng.dirichlet(np.full(ns, 2.0), (nz, ny, nx))
    rho = 101325.0 / ((Y @ tb.rgas) * T)
    vel = 120.0 * rng.uniform(-1, 1, (3, nz, ny, nx))
    e = tb.e_from_T_many(T.ravel(), Y.reshape(-1, ns)).reshape(T.shape)
    w = np.empty((ns + 4, nz, ny, nx))
    w[:ns] = np.moveaxis(rho[..., None] * Y, -1, 0)
    w[ns:ns + 3] = rho * vel
    w[ns + 3] = rho * (e + 0.5 * (vel ** 2).sum(0))
    pad = lambda a: np.pad(a, [(0, 0)] * (a.ndim - 3) + [(ng, ng)] * 3, mode="wrap")  # noqa: E731
    return pad(w), pad(T)


@pytest.mark.parametrize("shape,mech,ng,order,bc,chem,stretched", CASES)
def test_cells_match_oracle_and_sweeps(pkg, oracle, shape, mech, ng, order, bc, chem, stretched):
    import oracle_backend
    tb = _tables(pkg, mech)
    w, tg = _state(pkg, tb, shape, ng, 11)
    num = pkg.solver.Numerics(ep_order=order, visc_order=order, enable_chemistry=chem, weno_scheme=min(ng, 3))
    length = [2.0e-5 * n for n in shape]
    maps = None
    if stretched:
        maps = [lambda x: x, lambda x, h=2.0e-5: x + 0.2 * h * np.sin(x / h), None]
    out = []
    for be, cells in ((pkg.solver.HipBackend(), True), (pkg.solver.HipBackend(), False),
                      (oracle_backend.OracleBackend(oracle), None)):
        s = pkg.solver.Solver(be, tb, *shape, ng, length, bctags=bc, numerics=num, rho0=0.3, u0=150.0, mappings=maps)
        s.set_state(w, tg)
        s.compute_aux()
        s.dt = 2.0e-9
        if cells:
            assert s.cells_supported()
        elif cells is False:
            s.cells_supported = lambda: False
        print(f"[cells] {shape} {mech} order {order} cells={cells}", flush=True)
        s.rk_sync(fused=cells is not None)
        be.sync()
        out.append((be.to_numpy(s.fl).copy(), interior(be.to_numpy(s.w), ng).copy(), be.to_numpy(s.fln).copy()))
    for other in out[1:]:
        assert rel_maxnorm(out[0][0], other[0]).max() < 1e-12
        assert rel_maxnorm(out[0][1], other[1]).max() < 1e-11
        assert rel_maxnorm(out[0][2], other[2]).max() < 1e-12


def test_cells_refuse_what_they_do_not_cover(pkg, h2_tables):
    """A sensor, an order reduction, another energy split, a forced-zero face or a flat axis
    keep the sweeps."""
    be = pkg.solver.HipBackend()
    N = pkg.solver.Numerics

    def solver(num=None, shape=(8, 6, 4), bc=(0,) * 6, ng=4):
        return pkg.solver.Solver(be, h2_tables, *shape, ng, [1e-3] * 3, bctags=bc, numerics=num or N())

    assert solver().cells_supported()
    assert not solver(N(sensor_threshold=0.5)).cells_supported()
    assert not solver(N(nkeep=2)).cells_supported()
    assert not solver(N(nkeep=-1)).cells_supported()
    assert not solver(N(ep_order=4, visc_order=4)).cells_supported()
    assert not solver(N(visc_order=4)).cells_supported()
    assert not solver(N(correct_bound_ord=1), bc=(8, 2, 0, 0, 0, 0)).cells_supported()
    assert not solver(shape=(8, 1, 4)).cells_supported()
    s = solver()
    s.force_zero_flux[2] = 1
    assert not s.cells_supported()
