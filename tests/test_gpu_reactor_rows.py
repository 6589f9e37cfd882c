"""The species-block reactor kernel gives a reactor 16 lanes: batches that leave rows of a
wave, waves or workgroups partly empty (1, 3, 4, 15, 17, 65 reactors) give every reactor the
bits it has in a batch of 130, at constant volume and at constant pressure, in whole calls
and resumed under a step budget, for species counts that fill 10, 14 and 15 of the lanes; and
the FP64 block's states agree with the plain FP64 form (the same method with a
central-difference Jacobian) within 1e-6 of the state's scale, the bound the other reactor
tests hold the forms to."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tables(pkg, mech):
    if mech == "h2":
        return pkg.cases.h2_air_mechanism().tables()
    name = {"davis": "davis2005_13sp.yaml", "keromnes": "keromnes2013_14sp.yaml"}[mech]
    return pkg.mechanism.Mechanism(str(pkg.cases.mechanism_path(name))).tables()


def _inputs(pkg, tb, n, pressure):
    rng = np.random.default_rng(3)
    ns = tb.n_species
    T = rng.uniform(1100.0, 1900.0, n)
    Y = pkg.serving.premixed(tb, np.exp(rng.uniform(-1.0, 1.0, n)), {"H2": 1.0} if ns == 9 else {"H2": 0.5, "CO": 0.5})
    w = np.zeros((ns + 4, n))
    if pressure:
        w[:ns] = Y.T
        w[ns + 3] = pkg.serving.enthalpy_many(tb, T, Y)
    else:
        rho = 101325.0 / ((Y @ tb.rgas) * T)
        w[:ns] = (rho[:, None] * Y).T
        w[ns + 3] = rho * tb.e_from_T_many(T, Y)
    return w, T


@pytest.mark.parametrize("mech", ["h2", "davis", "keromnes"])
@pytest.mark.parametrize("pressure", [False, True])
@pytest.mark.parametrize("form", [1, 2])
def test_ragged_batches_give_the_same_bits(pkg, mech, pressure, form):
    tb = _tables(pkg, mech)
    be = pkg.solver.HipBackend()
    R = pkg.reactors.ReactorBatchGPU(be, tb)
    w0, t0 = _inputs(pkg, tb, 130, pressure)
    horizon = 2e-6

    def run(n, mixed, budget=0):
        w, tg = be.asarray(np.ascontiguousarray(w0[:, :n])), be.asarray(t0[:n])
        first, end = be.asarray(np.full(n, 1e-9)), be.asarray(np.full(n, horizon))
        pres = be.asarray(np.full(n, 101325.0)) if pressure else None
        nacc, nrej = be.zeros((n,), "i4"), be.zeros((n,), "i4")
        if budget:
            td, dn = be.zeros((n,)), be.zeros((n,))
            for _ in range(60):
                R.integrate(w, tg, first, end, mixed=mixed, pressure=pres, t_done=td, dt_next=dn, maxsteps=budget)
            assert np.all(be.to_numpy(td) == horizon)
            return be.to_numpy(w)
        R.integrate(w, tg, first, end, nacc, nrej, mixed=mixed, pressure=pres)
        return be.to_numpy(w), be.to_numpy(tg), be.to_numpy(nacc), be.to_numpy(nrej)

    print(f"[rows] {mech} pressure {pressure} form {form}", flush=True)
    whole = run(130, form)
    assert np.all(np.isfinite(whole[0])) and whole[2].min() > 3
    for n in (1, 3, 4, 15, 17, 65):
        for a, b in zip(run(n, form), whole):
            np.testing.assert_array_equal(a, b[..., :n])
    np.testing.assert_array_equal(run(17, form, budget=7)[:, :17], run(17, form, budget=50))
    if form == 2:
        ref = run(130, 0)[0]
        scale = np.abs(ref[:tb.n_species]).sum(axis=0)
        assert np.max(np.abs(whole[0] - ref)[:tb.n_species] / scale) < 1e-6


@pytest.mark.parametrize("mech", ["h2", "keromnes"])
@pytest.mark.parametrize("first", [1e-9, 1e-7])
@pytest.mark.parametrize("budget", [0, 1])
def test_large_fp64_block_batches_give_the_same_bits(pkg, mech, first, budget):
    """From 65536 constant-volume reactors on, form 2 takes one lane per reactor where the first step
    spans the interval (first = the horizon), rows elsewhere: the same bits as in small batches,
    also resumed, with some reactors finished before."""
    tb = _tables(pkg, mech)
    be = pkg.solver.HipBackend()
    R = pkg.reactors.ReactorBatchGPU(be, tb)
    n, few, horizon = 65536 + 77, 300, 1e-7
    w0, t0 = _inputs(pkg, tb, 512, False)
    pick = np.arange(n) % 512

    def run(count):
        w, tg = be.asarray(np.ascontiguousarray(w0[:, pick[:count]])), be.asarray(t0[pick[:count]])
        dt, end = be.asarray(np.full(count, first)), be.asarray(np.full(count, horizon))
        nacc, nrej = be.zeros((count,), "i4"), be.zeros((count,), "i4")
        td = dn = None
        if budget:
            td, dn = be.asarray(np.where(np.arange(count) % 5 == 0, horizon, 0.0)), be.zeros((count,))
        R.integrate(w, tg, dt, end, nacc, nrej, mixed=2, t_done=td, dt_next=dn, maxsteps=budget or None)
        return [be.to_numpy(a) for a in (w, tg, nacc, nrej) + ((td, dn) if budget else ())]

    print(f"[lanes] {mech} first {first} budget {budget}", flush=True)
    for a, b in zip(run(few), run(n)):
        np.testing.assert_array_equal(a, b[..., :few])
