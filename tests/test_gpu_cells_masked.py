"""Arguments of streams_rhs_cells that the fused step's other tests leave out: a mask of solid cells,
with and without the next substep's init folded in, against the sweeps and the tail that take the
same mask (masked cells keep their bits, the rest agrees within the 1e-11 of its largest value
that holds without a mask); and the eighth-order instance with 13 and 14 species, against the oracle and
the sweeps with the bounds of the other orders."""
import numpy as np
import pytest

import test_gpu_cells as cells
from parity_util import interior, rel_maxnorm

pytestmark = pytest.mark.gpu


class _Masked:
    """A backend that passes its mask where the solver passes none."""

    def __init__(self, be, mask):
        self._be, self._mask = be, mask

    def __getattr__(self, name):
        return getattr(self._be, name)

    def call(self, name, *args):
        if name in ("rhs_cells", "rhs_finish", "rhs_finish_next"):
            assert args[-2] is None
            args = args[:-2] + (self._mask, args[-1])
        return self._be.call(name, *args)


@pytest.mark.parametrize("fold", [False, True])
@pytest.mark.parametrize("shape,mech,ng,order", [((33, 9, 5), "h2", 3, 6), ((19, 14, 11), "davis", 4, 8)])
def test_masked_cells_stay(pkg, shape, mech, ng, order, fold):
    tb = cells._tables(pkg, mech)
    w, tg = cells._state(pkg, tb, shape, ng, 12)
    be = pkg.solver.HipBackend()
    solid = (np.random.default_rng(1).uniform(size=w.shape[1:]) < 0.2).astype(np.int32)
    num = pkg.solver.Numerics(ep_order=order, visc_order=order)
    out = []
    for use in (True, False):
        s = pkg.solver.Solver(_Masked(be, be.asarray(solid, "i4")), tb, *shape, ng, [2.0e-5 * n for n in shape],
                              numerics=num, rho0=0.3, u0=150.0)
        assert s.cells_supported()
        s.cells_supported = lambda use=use: use
        s.fold_substeps = fold
        s.set_state(w, tg)
        s.compute_aux()
        s.dt = 2.0e-9
        print(f"[cells masked] {shape} {mech} order {order} fold {fold} cells {use}", flush=True)
        s.rk_sync(fused=True)
        be.sync()
        out.append((interior(be.to_numpy(s.w), ng), be.to_numpy(s.fl), be.to_numpy(s.fln)))
    still = interior(solid, ng) == 1
    w0 = interior(w, ng)
    for a in out:
        np.testing.assert_array_equal(a[0][:, still], w0[:, still])
        assert (a[0][:, ~still] != w0[:, ~still]).any(axis=0).all()
    for a, b, tol in zip(out[0], out[1], (1e-11, 1e-12, 1e-12)):
        assert rel_maxnorm(a, b).max() < tol


@pytest.mark.parametrize("shape,mech,bc", [((37, 9, 5), "keromnes", (0,) * 6), ((9, 35, 10), "davis", (0, 0, 2, 2, 0, 0))])
def test_eighth_order_with_many_species(pkg, oracle, shape, mech, bc):
    cells.test_cells_match_oracle_and_sweeps(pkg, oracle, shape, mech, 4, 8, bc, 1, False)
