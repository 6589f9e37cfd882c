"""The species-block forms of large batches: one lane per reactor for the first steps, rows of 16
lanes for what is left.  Batches of the sizes at which that changes end bit for bit where their
reactors end in a batch of 300, which rows integrate from the first step, with the same step
counts, times and next steps: whole calls in which reactors take some ten to a hundred steps
(beyond the lanes' 24), calls of one step, resumed calls whose budget ends before, in and after
the lanes' part, some reactors finished before, a state that is not finite, few and many
species, NASA9 tables, both forms, constant volume and pressure, and the call recorded in a graph,
where no workspace is taken."""
import dataclasses

import numpy as np
import pytest

from test_gpu_reactor_rows import _inputs, _tables

pytestmark = pytest.mark.gpu
FEW = 300


def _runner(pkg, mech, pressure, form, horizon, first, budget, nasa9=False):
    tb, state = _tables(pkg, "h2" if mech == "premix" else mech), None
    if mech == "premix":                    # the nine species' states among eleven
        state = _inputs(pkg, tb, 512, pressure), [n.upper() for n in tb.names]
        tb = pkg.mechanism.Mechanism(str(pkg.cases.mechanism_path("h2_premix_11sp.yaml"))).tables()
    be = pkg.solver.HipBackend()
    if state is None:
        w0, t0 = _inputs(pkg, tb, 512, pressure)
    else:
        (w9, t0), names = state
        w0 = np.zeros((tb.n_species + 4, 512))
        w0[[[n.upper() for n in tb.names].index(n) for n in names]] = w9[:len(names)]
        w0[tb.n_species:] = w9[len(names):]
    w0[1, 7] = np.inf
    if nasa9:                               # the same polynomials with T^-2 and T^-1 terms of zero
        grow = lambda a: np.concatenate([np.zeros((2,) + a.shape[1:]), a])  # noqa: E731
        tb = dataclasses.replace(tb, indx_cp_l=-2, cp_coeff=grow(tb.cp_coeff), cv_coeff=grow(tb.cv_coeff))
    R = pkg.reactors.ReactorBatchGPU(be, tb)

    def inputs(count):
        pick = np.arange(count) % 512                     # every reactor recurs 512 places on
        w, tg = be.asarray(np.ascontiguousarray(w0[:, pick])), be.asarray(t0[pick])
        dt, end = be.asarray(np.full(count, first)), be.asarray(np.full(count, horizon))
        kw = dict(nacc=be.zeros((count,), "i4"), nrej=be.zeros((count,), "i4"), mixed=form,
                  pressure=be.asarray(np.full(count, 101325.0)) if pressure else None)
        if budget:
            kw.update(t_done=be.asarray(np.where(pick % 5 == 0, horizon, 0.0)), dt_next=be.zeros((count,)),
                      maxsteps=budget)
        return (w, tg, dt, end), kw

    def run(count):
        args, kw = inputs(count)
        R.integrate(*args, **kw)
        out = [args[0], args[1], kw["nacc"], kw["nrej"]] + ([kw["t_done"], kw["dt_next"]] if budget else [])
        return [be.to_numpy(a) for a in out]

    return be, R, inputs, run


@pytest.mark.parametrize("mech,n", [("h2", 12288), ("h2", 65536), ("h2", 65537), ("keromnes", 40961),
                                    ("keromnes", 131072 + 77), ("h2", 131072)])
@pytest.mark.parametrize("pressure", [False, True])
@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("horizon,first,budget", [(3e-6, 1e-9, 0), (1e-8, 1e-8, 0), (3e-6, 1e-9, 7), (3e-6, 1e-9, 24),
                                                  (3e-6, 1e-9, 40), (3e-6, 1e-9, 300)])
def test_large_batches_give_the_same_bits(pkg, mech, n, pressure, form, horizon, first, budget):
    _compare(pkg, mech, n, pressure, form, horizon, first, budget)


@pytest.mark.parametrize("mech,n,nasa9", [("h2", 65537, True), ("premix", 131072 + 5, False), ("premix", 40961, True)])
@pytest.mark.parametrize("pressure", [False, True])
@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("horizon,first,budget", [(3e-6, 1e-9, 0), (1e-8, 1e-8, 0), (3e-6, 1e-9, 7)])
def test_other_tables_give_the_same_bits(pkg, mech, n, nasa9, pressure, form, horizon, first, budget):
    """NASA9 tables, and a species count between those above."""
    _compare(pkg, mech, n, pressure, form, horizon, first, budget, nasa9)


def _compare(pkg, mech, n, pressure, form, horizon, first, budget, nasa9=False):
    print(f"[lanes] {mech} {n} nasa9 {nasa9} pressure {pressure} form {form} horizon {horizon} budget {budget}", flush=True)
    run = _runner(pkg, mech, pressure, form, horizon, first, budget, nasa9)[-1]
    few, many = run(FEW), run(n)
    last = n // 512 * 512 - 512
    for a, b in zip(few, many):
        np.testing.assert_array_equal(a, b[..., :FEW])
        np.testing.assert_array_equal(a, b[..., last:last + FEW])
    if horizon > 1e-6 and budget in (0, 300):
        assert few[2].max() > 24


def test_recorded_call_gives_the_same_bits(pkg):
    """Recorded in a graph and replayed, with the inputs put back between the replays."""
    be, R, inputs, run = _runner(pkg, "h2", False, 2, 3e-6, 1e-9, 0)
    n = 65537
    want = run(n)
    args, kw = inputs(n)
    kept = [a.clone() for a in args[:2]]
    torch = be.torch
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        R.integrate(*args, **kw)
    for _ in range(3):
        for a, b in zip(args, kept):
            a.copy_(b)
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip((args[0], args[1], kw["nacc"], kw["nrej"]), want):
            np.testing.assert_array_equal(be.to_numpy(a), b)
