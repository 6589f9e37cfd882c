"""Which solvers may take the one-pass right-hand side: it has no WENO stencil, but a solver whose
WENO stencil does not exist or does not fit the ghost layers is refused by the sweeps, as it is
by the routines, and must reach them."""
import pytest

import oracle_backend


class _Cells(oracle_backend.OracleBackend):
    """The oracle's backend with the fused entry points listed."""

    def has(self, name):
        return True


@pytest.mark.parametrize("scheme,ng,taken", [(1, 3, True), (3, 3, True), (4, 4, True), (4, 3, False), (5, 5, False),
                                             (0, 3, False)])
def test_weno_stencil_must_fit(pkg, oracle, h2_tables, scheme, ng, taken):
    num = pkg.solver.Numerics(weno_scheme=scheme)
    s = pkg.solver.Solver(_Cells(oracle), h2_tables, 6, 5, 4, ng, [1e-3] * 3, numerics=num)
    assert s.cells_supported() == taken
