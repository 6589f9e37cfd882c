"""The rate forms of compute_chemistry on each of its table walks (records in local memory;
dense tables because the reactions exceed it, or because a side has five species): one
irreversible reaction with k = A T^10 among others of rate zero, against 80-bit arithmetic at
the temperatures and concentrations that the kernel itself works with.  pow is good to 1 ulp and
the products of the rate and its source take at most eleven roundings, 12 * 1.1e-16 in all: below
1.4e-15.  A rate folded into exp(b ln T) has an exponent of about 70, whose rounding alone is
up to 7e-15."""
import dataclasses

import numpy as np
import pytest

from parity_util import interior

pytestmark = pytest.mark.gpu
NG = 3


def _one_reaction(tb, count, wide):
    """`count` reactions of which only the first has a rate."""
    ns = tb.n_species
    a, b, z = np.zeros((count, 2)), np.zeros((count, 2)), np.zeros((count, 2))
    a[:, 1] = 1.0
    a[0, 0], b[0, 0] = 1.0e-24, 10.0
    r, p = np.zeros((count, ns)), np.zeros((count, ns))
    r[:, 0] = p[:, 1] = 1.0
    r[0, :5 if wide else 2] = 1.0
    p[0] = 0.0
    p[0, 6] = 1.0
    kc = np.ones((tb.num_t_tab + 1, count))
    return dataclasses.replace(tb, nreactions=count, reac_ty=np.zeros(count, dtype=np.int32),
                               isRev=np.zeros(count, dtype=np.int32), arr_a=a, arr_b=b, arr_ea=z, r_coeffs=r,
                               p_coeffs=p, kc_tab=kc, falloff_coeffs=np.zeros((count, 5)), tb_eff=np.ones((count, ns)))


@pytest.mark.parametrize("count,wide", [(5, False), (77, False), (5, True)])
def test_rates_keep_their_forms(pkg, h2_tables, count, wide):
    from test_gpu_cells import _state
    tb = _one_reaction(h2_tables, count, wide)
    shape = (9, 8, 7)
    w, tg = _state(pkg, h2_tables, shape, NG, 5)
    be = pkg.solver.HipBackend()
    s = pkg.solver.Solver(be, tb, *shape, NG, [2.0e-5 * n for n in shape], rho0=0.3, u0=150.0)
    s.set_state(w, tg)
    s.compute_chemistry()
    be.sync()
    ns = tb.n_species
    T = interior(be.to_numpy(s.w_aux), NG)[ns + 4].astype(np.longdouble)
    v = interior(w, NG)[:ns]
    rho = v[0]
    for q in range(1, ns):
        rho = rho + v[q]
    conc = (rho * (v * (1.0 / rho))) / np.asarray(tb.mw)[:, None, None, None]
    q = np.longdouble(tb.arr_a[0, 0]) * T ** 10
    for k in range(5 if wide else 2):
        q = q * conc[k].astype(np.longdouble)
    want = np.zeros((ns,) + T.shape, dtype=np.longdouble)
    for k in range(ns):
        want[k] = -np.longdouble(tb.p_coeffs[0, k] - tb.r_coeffs[0, k]) * q * np.longdouble(tb.mw[k])
    got = be.to_numpy(s.fl)[:ns]
    used = np.flatnonzero(tb.p_coeffs[0] != tb.r_coeffs[0])
    err = np.abs((got[used] - want[used]) / want[used]).max()
    print(f"[chemistry forms] {count} reactions, wide {wide}: {float(err):.2e}", flush=True)
    assert err < 1.4e-15
    assert not got[np.setdiff1d(np.arange(ns), used)].any()
