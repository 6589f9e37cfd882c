"""All periodic axes of a halo exchange in one launch: every combination of axes shorter than the
ghost layer (lines kept in registers, and deeper layers than those hold), longer and equal to it,
against the oracle, bit for bit; and the six faces of bcextr_var in one launch on flat boxes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,ng,nv", [((70, 5, 3), 4, 3), ((1, 1, 1), 3, 2), ((2, 300, 1), 4, 1), ((3, 2, 90), 3, 13),
                                         ((4, 7, 300), 4, 17), ((20, 3, 1), 10, 2), ((2, 13, 9), 9, 1)])
@pytest.mark.parametrize("periodic", [(1, 1, 1), (0, 1, 1), (1, 0, 0), (0, 0, 0)])
def test_exchange_and_extrapolation(pkg, oracle, shape, ng, nv, periodic):
    import oracle_backend
    nx, ny, nz = shape
    a = np.random.default_rng(9).standard_normal((nv, nz + 2 * ng, ny + 2 * ng, nx + 2 * ng))
    per = np.array(periodic, dtype=np.int32)
    hip, cpu = pkg.solver.HipBackend(), oracle_backend.OracleBackend(oracle)
    for name, args in (("bcswap", (nx, ny, nz, ng, nv)), ("bcextr_var", (nx, ny, nz, ng))):
        g, c = hip.asarray(a), a.copy()
        tail = (per,) if name == "bcswap" else ()
        hip.call(name, *args, g, *tail, hip.stream)
        cpu.call(name, *args, c, *tail, None)
        np.testing.assert_array_equal(hip.to_numpy(g), c)
