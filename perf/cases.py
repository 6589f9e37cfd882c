"""The work this framework is measured on, through its public entry points.

Three families, as its users run it:

* a field advanced in time (``solver.Solver``): boxes of decaying turbulence with explicit
  chemistry, from a few thousand cells to the 256^3 box of the benchmark, by the fused
  substeps and routine by routine (the order a Fortran host calls the entry points in); an
  LES with the PaSR closure; the syngas mixing layer with WENO on about a tenth of its faces,
  with explicit and with Strang-split batched chemistry; the 1-D reactive shock tube;
* batches of independent 0-D reactors (``reactors.ReactorBatchGPU``): the constant-volume
  batch of the benchmark, one tick of the reactor server, the FP64 form it falls back to;
* the reactor server itself (``serving.ReactorServer``).
"""
from __future__ import annotations

import functools
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parents[1]
NG = 3
DEV = "cuda:0"
MECHS = ("h2air9", "davis13", "keromnes14")
LES = dict(enable_les=1, les_model=2, les_pr=0.9, les_sc=0.7, les_c_wale=0.5, les_c_yoshi=0.0886, les_c_eps=1.048,
           les_c_mix=0.1)


def package():
    if "prop_streams2_amd" in sys.modules:
        return sys.modules["prop_streams2_amd"]
    d = ROOT / "prop-streams2_amd"
    spec = importlib.util.spec_from_file_location("prop_streams2_amd", d / "__init__.py",
                                                  submodule_search_locations=[str(d)])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["prop_streams2_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


@functools.lru_cache(maxsize=None)
def tables(mech: str):
    pkg = package()
    if mech == "h2air9":
        return pkg.cases.h2_air_mechanism().tables()
    if mech == "keromnes14":
        return pkg.cases.keromnes_mechanism().tables()
    if mech == "davis13":
        return pkg.mechanism.Mechanism(str(pkg.cases.mechanism_path("davis2005_13sp.yaml"))).tables()
    return pkg.cases.shock_tube_mechanism().tables(p0=7173.0)


# ------------------------------------------------------------------------------ the cases
def listed():
    return [
        # the benchmark's box: 256^3 cells, 9 species, 21 reactions, one RK3 step
        dict(name="box_256", kind="box", mech="h2air9", nx=256, ny=256, nz=256, fused=True),
        # an ordinary subdomain of odd sizes with a 13-species syngas mechanism
        dict(name="box_117x90x77_13sp", kind="box", mech="davis13", nx=117, ny=90, nz=77, fused=True),
        # a box as small as a test's: launches and latency
        dict(name="box_19x14x11", kind="box", mech="h2air9", nx=19, ny=14, nz=11, fused=True),
        # the same step through the routine-by-routine entry points, as a Fortran host calls them
        dict(name="routines_96x72x60", kind="box", mech="h2air9", nx=96, ny=72, nz=60, fused=False),
        # LES (WALE, PaSR closure) with the cell-by-cell Rosenbrock chemistry, Strang splitting
        dict(name="les_40x30x24", kind="les", mech="h2air9", nx=40, ny=30, nz=24),
        # the plain-method configuration: 800-cell reactive shock tube, WENO5 on every face,
        # Rosenbrock-Krylov chemistry, dt recomputed every step
        dict(name="tube_800", kind="tube", mech="tube9", nx=800),
        # the syngas mixing layer, WENO5 on about a tenth of the faces, explicit chemistry
        dict(name="layer_160x96x64", kind="layer", mech="keromnes14", nx=160, ny=96, nz=64, form=-1),
        # the same flow with Strang splitting, its cells one mixed-precision reactor batch
        dict(name="layer_strang_64x48x32", kind="layer", mech="keromnes14", nx=64, ny=48, nz=32, form=1),
        # the batched-chemistry workload: constant volume, random radical pools, 1 us, mixed
        dict(name="reactors_131072", kind="reactors", mech="h2air9", n=131072, form=1, budget=0),
        # one tick of the reactor server: constant-pressure premixed syngas, a step budget
        dict(name="tick_1500", kind="tick", mech="keromnes14", n=1500, form=1, budget=60),
        # the FP64 form that the server falls back to, on a handful of reactors
        dict(name="fallback_60", kind="tick", mech="h2air9", n=60, form=0, budget=12),
        # the reactor server on a burst of requests of two mechanisms
        dict(name="serve", kind="serve", mech="both", requests=8, most=400, budget=100),
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(("box", "box", "box", "routines", "les", "tube", "layer", "strang", "reactors", "tick", "tick",
                       "serve"))
    if kind in ("box", "routines"):
        most = 200 if kind == "box" else 110
        return dict(kind="box", mech=rng.choice(MECHS), nx=log(12, most), ny=log(9, most), nz=log(9, most),
                    fused=kind == "box")
    if kind == "les":
        return dict(kind="les", mech="h2air9", nx=log(10, 48), ny=log(9, 40), nz=log(9, 32))
    if kind == "tube":
        return dict(kind="tube", mech="tube9", nx=log(200, 2400))
    if kind == "layer":
        return dict(kind="layer", mech="keromnes14", nx=log(32, 180), ny=log(32, 120), nz=log(16, 80), form=-1)
    if kind == "strang":
        return dict(kind="layer", mech="keromnes14", nx=log(16, 80), ny=log(24, 64), nz=log(12, 40),
                    form=rng.choice((1, 2)))
    if kind == "reactors":
        return dict(kind="reactors", mech="h2air9", n=log(70000, 131072), form=rng.choice((1, 2)), budget=0)
    if kind == "tick":
        form = rng.choice((1, 1, 2, 0))
        return dict(kind="tick", mech=rng.choice(("h2air9", "keromnes14")), n=log(1, 4096) if form else log(1, 200),
                    form=form, budget=rng.randint(20, 80) if form else rng.randint(5, 12))
    return dict(kind="serve", mech="both", requests=rng.randint(3, 10), most=log(60, 400),
                budget=rng.choice((0, 60, 100)))


# ------------------------------------------------------------------------- inputs
def _dev(a):
    return torch.as_tensor(np.array(a, dtype=np.float64), device=DEV)


def _range_of(tb, T):
    """0-based temperature range of every species (N_S, ...)."""
    tr = _dev(tb.trange)
    m = torch.zeros((tb.n_species,) + tuple(T.shape), dtype=torch.int64, device=T.device)
    for q in range(1, tb.nsetcv):
        m += (T[None] >= tr[:, q].reshape((-1,) + (1,) * T.dim())).long()
    return m


def _poly(tb, coeff, T, s, m, integral):
    """cp or cv of species s (or, integral, h or e) from the NASA rows at T in range m."""
    c = _dev(coeff[:, s, :])
    lo, hi = tb.indx_cp_l, tb.indx_cp_r
    out = c[hi + 1 - lo][m] if integral else torch.zeros_like(T)
    for l in range(lo, hi + 1):
        a = c[l - lo][m]
        if not integral:
            out = out + a * T ** l
        elif l == -1:
            out = out + a * torch.log(T)
        else:
            out = out + a / (l + 1.0) * T ** (l + 1)
    return out


def _energy(tb, T, Y):
    """Mixture internal energy; Y (N_S, ...)."""
    m = _range_of(tb, T)
    e = torch.zeros_like(T)
    for s in range(tb.n_species):
        e = e + Y[s] * _poly(tb, tb.cv_coeff, T, s, m[s], True)
    return e


def _weights(tb, x):
    y = np.array([x.get(n.upper(), 0.0) for n in tb.names]) * tb.mw
    return _dev(y / y.sum())


def _fuel(mech):
    return {"H2": 1.0} if mech == "h2air9" else {"H2": 0.5, "CO": 0.5}


def _smooth(shape, gen, count, k0):
    """`count` smooth random periodic fields (count, nz, ny, nx) of unit rms and, for three
    of them read as a vector, the wave numbers to make it solenoidal with."""
    nz, ny, nx = shape
    h = torch.fft.rfftn(torch.randn((count,) + shape, dtype=torch.float64, device=DEV, generator=gen), dim=(1, 2, 3))
    k = torch.meshgrid(torch.fft.fftfreq(nz, 1.0 / nz, dtype=torch.float64, device=DEV),
                       torch.fft.fftfreq(ny, 1.0 / ny, dtype=torch.float64, device=DEV),
                       torch.fft.rfftfreq(nx, 1.0 / nx, dtype=torch.float64, device=DEV), indexing="ij")
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    k2[0, 0, 0] = 1.0
    amp = k2 / k0 ** 2 * torch.exp(-k2 / k0 ** 2)          # Passot-Pouquet: E(k) ~ k^4 exp(-2 k^2/k0^2)
    amp = amp / k2.sqrt()
    amp[0, 0, 0] = 0.0
    return h * amp, k, k2


def _turbulence(tb, mech, shape, seed):
    """Interior conserved variables (nv, nz, ny, nx) and T of a box of reacting decaying
    turbulence: solenoidal velocity at M_t about 0.3, mixture fraction and temperature
    (900-1500 K) varying smoothly, traces of burnt gas and radicals, 1 atm."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) % (1 << 62))
    k0 = 4.0 if min(shape) >= 64 else 1.5
    h, (kz, ky, kx), k2 = _smooth(shape, gen, 6, k0)
    dot = (kx * h[0] + ky * h[1] + kz * h[2]) / k2
    h[0] -= kx * dot
    h[1] -= ky * dot
    h[2] -= kz * dot
    f = torch.fft.irfftn(h, s=shape, dim=(1, 2, 3))
    del h, dot, kz, ky, kx, k2
    vel = f[:3] / f[:3].square().sum(0).mean().sqrt() * 230.0
    g = (f[3:] / f[3:].square().mean(dim=(1, 2, 3), keepdim=True).sqrt()).clamp(-2.0, 2.0)
    y_air = _weights(tb, {"O2": 1.0, "N2": 3.76})
    y_fuel = _weights(tb, _fuel(mech))
    y_burnt = _weights(tb, {"H2O": 1.0, "N2": 2.0, "O2": 0.1, "OH": 1e-3, "H": 1e-4, "O": 1e-4, "HO2": 1e-5,
                            "H2O2": 1e-6, "CO2": 0.1, "HCO": 1e-6, "AR": 0.01, "HE": 0.01, "CO": 0.05, "H2": 0.05})
    z = (0.0144 if mech == "h2air9" else 0.08) * (1.0 + 0.4 * g[0])
    b = 0.01 * (1.0 + 0.4 * g[1])
    T = 1200.0 + 150.0 * g[2]
    col = lambda a: a.reshape(-1, 1, 1, 1)  # noqa: E731
    Y = (1.0 - b) * (z * col(y_fuel) + (1.0 - z) * col(y_air)) + b * col(y_burnt)
    rho = 101325.0 / ((col(_dev(tb.rgas)) * Y).sum(0) * T)
    e = _energy(tb, T, Y)
    w = torch.cat([rho * Y, rho * vel, (rho * (e + 0.5 * vel.square().sum(0)))[None]])
    return w, T


def _padded(a):
    """Periodic ghost layers on the last three axes."""
    for d in (-3, -2, -1):
        n = a.shape[d]
        a = a.index_select(a.dim() + d, torch.arange(-NG, n + NG, device=a.device) % n)
    return a


def _box_solver(case, numerics, seed):
    pkg, tb = package(), tables(case["mech"])
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    w, T = _turbulence(tb, case["mech"], (nz, ny, nx), seed)
    dx = 2.0e-3 * math.pi / 256
    s = pkg.solver.Solver(pkg.solver.HipBackend(DEV), tb, nx, ny, nz, NG, [nx * dx, ny * dx, nz * dx],
                          numerics=numerics, rho0=0.25, u0=230.0)
    s.w.copy_(_padded(w))
    s.w_aux[tb.n_species + 4].copy_(_padded(T))
    s.compute_aux()
    s.compute_dt(0.5)
    return s


def _premixed_requests(count, most, seed):
    """A burst of requests to the reactor server: from `most` premixed reactors down to a
    few, in turn of the two mechanisms."""
    pkg = package()
    mechs = {"h2": tables("h2air9"), "syngas": tables("keromnes14")}
    rng = np.random.default_rng(seed)
    out = []
    for rid in range(count):
        mech = ("h2", "syngas")[rid % 2]
        tb = mechs[mech]
        n = int(round(most ** (1.0 - (rid // 2 * 2) / count)))
        phi = np.exp(rng.uniform(math.log(0.3), math.log(3.0), n))
        y = pkg.serving.premixed(tb, phi, _fuel("h2air9" if mech == "h2" else "keromnes14"))
        out.append(dict(rid=rid, mech=mech, temperature=rng.uniform(900.0, 1800.0, n), pressure=np.full(n, 101325.0),
                        y=y, horizon=math.exp(rng.uniform(math.log(1e-5), math.log(4e-5)))))
    return mechs, out


def prepare(case, seed):
    pkg, kind = package(), case["kind"]
    if kind == "box":
        s = _box_solver(case, pkg.solver.Numerics(), seed)
        return dict(case=case, s=s)
    if kind == "les":
        num = pkg.solver.Numerics(enable_chemistry=2, rosenbrock_version=1, operator_splitting=2, **LES)
        s = _box_solver(case, num, seed)
        return dict(case=case, s=s, w0=s.w.clone())
    if kind == "tube":
        tb = tables("tube9")
        y = np.array([pkg.cases.SHOCK_TUBE_Y.get(n, 0.0) for n in tb.names])
        fp = pkg.cases.flow_params(tb, y, 0.072, 7173.0)
        num = pkg.solver.Numerics(sensor_threshold=-0.2, sensor_type=0, enable_chemistry=2, rosenbrock_version=2,
                                  operator_splitting=2)
        w, tg, _ = pkg.cases.shock_tube(tb, case["nx"], y, fp["rho0"], fp["p0"])
        # the seed's own tube: the driven gas and the mixture a little denser or thinner
        w = w * (1.0 + 0.02 * np.random.default_rng(seed).uniform(-1.0, 1.0))
        s = pkg.solver.Solver(pkg.solver.HipBackend(DEV), tb, case["nx"], 1, 1, NG, [0.12, 0.01, 0.01],
                              bctags=(8, 2, 0, 0, 0, 0), numerics=num, rho0=fp["rho0"], u0=fp["u0"], p0=fp["p0"])
        s.set_state(w, tg)
        s.compute_aux()
        for _ in range(12):                  # past the start: shock, contact and expansion on several cells
            s.compute_dt(0.5)
            s.advance()
        return dict(case=case, s=s, w0=s.w.clone())
    if kind == "layer":
        tb = tables("keromnes14")
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        w, tg, info = pkg.cases.mixing_layer(tb, nx, ny, nz, seed=seed)
        num = pkg.solver.Numerics() if case["form"] < 0 else pkg.solver.Numerics(
            enable_chemistry=2, operator_splitting=2, chem_batch_form=case["form"])
        s = pkg.solver.Solver(pkg.solver.HipBackend(DEV), tb, nx, ny, nz, NG, info["length"], numerics=num,
                              rho0=info["rho0"], u0=info["u0"])
        s.set_state(w, tg)
        s.compute_aux()
        duc = s.be.to_numpy(s.w_aux[tb.n_species + 8])[NG:-NG, NG:-NG, NG:-NG]
        num.sensor_threshold = pkg.cases.weno_threshold_for_fraction(duc, num.weno_scheme, 0.10)
        s.compute_dt(0.5)
        return dict(case=case, s=s, w0=s.w.clone())
    if kind in ("reactors", "tick"):
        tb, n, ns = tables(case["mech"]), case["n"], tables(case["mech"]).n_species
        gen = torch.Generator(device=DEV)
        gen.manual_seed(int(seed) % (1 << 62))
        uni = lambda a, b: a + (b - a) * torch.rand(n, dtype=torch.float64, device=DEV, generator=gen)  # noqa: E731
        w = torch.zeros((ns + 4, n), dtype=torch.float64, device=DEV)
        st = dict(case=case, R=pkg.reactors.ReactorBatchGPU(pkg.solver.HipBackend(DEV), tb))
        if kind == "reactors":
            T = torch.exp(uni(math.log(800.0), math.log(2500.0)))
            p = torch.exp(uni(math.log(0.5 * 101325.0), math.log(20.0 * 101325.0)))
            Y = -torch.log(torch.rand((ns, n), dtype=torch.float64, device=DEV, generator=gen).clamp_min(1e-300))
            Y = Y / Y.sum(0)                 # Dirichlet(1)
            rho = p / ((_dev(tb.rgas)[:, None] * Y).sum(0) * T)
            w[:ns] = rho * Y
            w[ns + 3] = rho * _energy(tb, T, Y)
            st.update(w=w, tg=T, first=torch.full_like(T, 1e-9), end=torch.full_like(T, 1e-6), pres=None)
            return st
        T = uni(900.0, 1800.0)
        phi = torch.exp(uni(math.log(0.3), math.log(3.0))).cpu().numpy()
        Y = _dev(pkg.serving.premixed(tb, phi, _fuel(case["mech"])).T)
        w[:ns] = Y
        w[ns + 3] = _energy(tb, T, Y) + (_dev(tb.rgas)[:, None] * Y).sum(0) * T
        hz = torch.exp(uni(math.log(1e-6), math.log(1e-4)))
        st.update(w=w, tg=T, first=torch.full_like(T, 1e-9), end=hz, pres=torch.full_like(T, 101325.0),
                  td=torch.zeros_like(T), dn=torch.zeros_like(T))
        return st
    mechs, reqs = _premixed_requests(case["requests"], case["most"], seed)
    srv = pkg.serving.ReactorServer(pkg.solver.HipBackend(DEV), mechs, hbm_bytes=1 << 24, slices=4, mixed=True,
                                    budget=case["budget"])
    return dict(case=case, srv=srv, reqs=reqs)


# ------------------------------------------------------------------------- one pass
def _field(s):
    n, ns = NG, s.ns
    w = s.w[:, n:-n, n:-n, n:-n]
    return {"rho_y": w[:ns], "rho_u": w[ns:ns + 3], "rho_e": w[ns + 3], "rhs_y": s.fl[:ns], "rhs_u": s.fl[ns:ns + 3],
            "rhs_e": s.fl[ns + 3]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "box":                        # the flow goes on from pass to pass
        s = state["s"]
        s.rk_sync(fused=case["fused"])
        return _field(s)
    if kind in ("les", "layer", "tube"):     # every pass is the same step: from the prepared field
        s = state["s"]
        s.w.copy_(state["w0"])
        if kind == "tube":
            s.compute_dt(0.5)
        if kind == "layer" and case["form"] < 0:
            s.rk_sync()
        else:
            s.advance()
        return _field(s)
    if kind == "reactors":
        w, tg = state["w"].clone(), state["tg"].clone()
        state["R"].integrate(w, tg, state["first"], state["end"], mixed=case["form"])
        return {"w": w, "t": tg}
    if kind == "tick":
        w, tg, td, dn = (state[k].clone() for k in ("w", "tg", "td", "dn"))
        state["R"].integrate(w, tg, state["first"], state["end"], mixed=case["form"], pressure=state["pres"],
                             t_done=td, dt_next=dn, maxsteps=case["budget"])
        return {"y": w[:-4], "h": w[-1], "t": tg, "t_done": td, "dt_next": dn}
    reqs = [package().serving.Request(**r) for r in state["reqs"]]
    state["srv"].run(reqs, realtime=False)
    return {"t": np.concatenate([r.t_final for r in reqs]), "y_h2": np.concatenate([r.y_final for r in reqs[0::2]]),
            "y_syngas": np.concatenate([r.y_final for r in reqs[1::2]]),
            "ignition": np.concatenate([r.ignition for r in reqs])}


# ------------------------------------------------------------------------- its floor
def work(case):
    """Bytes: the state in and out once per pass, for a field once per Runge-Kutta substep
    with the accumulator (each substep needs the whole field of the one before).  Flops: the
    terms of the scheme, and 13 right-hand sides of 90 flops a reaction per integrator step."""
    if case["kind"] in ("box", "les", "layer", "tube"):
        tb = tables(case["mech"])
        ns, nr, nv = tb.n_species, tb.nreactions, tb.n_species + 4
        cells = case["nx"] * case.get("ny", 1) * case.get("nz", 1)
        dims = 1 if case["kind"] == "tube" else 3
        per = 6 * ns * ns + 12 * ns * ns + dims * (20 * nv + 40 * ns) + 60 * ns + (90 * nr if case["kind"] == "box" or case.get("form", 0) < 0 else 0)
        flops = 3 * per * cells
        if case["kind"] != "box" and case.get("form", 0) >= 0:
            flops += 2 * (ns + 4) * 90 * nr * cells
        return {"bytes": 3 * 4 * nv * 8 * cells, "flops": flops}
    if case["kind"] == "serve":
        n, steps, ns, nr = 2 * case["most"], 400, 12, 29
    else:
        tb = tables(case["mech"])
        n, ns, nr = case["n"], tb.n_species, tb.nreactions
        steps = case["budget"] or 345
    return {"bytes": 2 * 8 * (ns + 5) * n, "flops": n * steps * (ns + 4) * 90 * nr}


# ------------------------------------------------------------------ the same in plain torch
class _Plain:
    """The RHS of the periodic box (KEEP central flux of sixth order with the split energy,
    staggered viscous and diffusive flux, cross terms, explicit chemistry) and the Wray RK3
    step in plain torch, on interior arrays (nv, nz, ny, nx)."""

    C = (0.75, -0.15, 1.0 / 60.0)

    def __init__(self, tb, dx):
        self.tb, self.dx, self.ns = tb, dx, tb.n_species

    @staticmethod
    def at(a, d, n):
        """a at the cell n further along axis d (0 x, 1 y, 2 z)."""
        return torch.roll(a, -n, dims=a.dim() - 1 - d)

    def aux(self, w, T):
        tb, ns = self.tb, self.ns
        ry = w[:ns].clamp_min(0.0)
        rho = ry.sum(0)
        Y = ry / rho
        u = w[ns:ns + 3] / rho
        e = w[ns + 3] / rho - 0.5 * u.square().sum(0)
        for _ in range(12):
            m = _range_of(tb, T)
            f, c = -e, torch.zeros_like(e)
            for s in range(ns):
                f = f + Y[s] * _poly(tb, tb.cv_coeff, T, s, m[s], True)
                c = c + Y[s] * _poly(tb, tb.cv_coeff, T, s, m[s], False)
            dT = f / c
            T = T - dT
            if float(dT.abs().max()) < 1e-11:
                break
        R = sum(float(tb.rgas[s]) * Y[s] for s in range(ns))
        return rho, Y, u, T, rho * R * T, R

    def rows(self, T):
        tb = self.tb
        it = ((T - tb.t_min_tab) / tb.dt_tab).floor().long().clamp(0, tb.num_t_tab - 1)
        return it, (T - (tb.t_min_tab + it * tb.dt_tab)) / tb.dt_tab

    def transport(self, rho, Y, T, p, R):
        tb, ns = self.tb, self.ns
        from_table = lambda col: col[it] + (col[it + 1] - col[it]) * ft  # noqa: E731
        it, ft = self.rows(T)
        W = package().mechanism.R_UNIV / R
        X = [Y[s] * W / float(tb.mw[s]) for s in range(ns)]
        lam = [from_table(_dev(tb.lambda_species[:, s])) for s in range(ns)]
        k = 0.5 * (sum(X[s] * lam[s] for s in range(ns)) + 1.0 / sum(X[s] / lam[s] for s in range(ns)))
        del lam
        mus = [from_table(_dev(tb.visc_species[:, s])) for s in range(ns)]
        mu = torch.zeros_like(T)
        for a in range(ns):
            den = torch.zeros_like(T)
            for b in range(ns):
                phi = (1.0 + torch.sqrt(mus[b] / mus[a]) * float(tb.mw[b] / tb.mw[a]) ** 0.25) ** 2
                den = den + Y[b] / float(tb.mw[b]) * phi / math.sqrt(1.0 + float(tb.mw[a] / tb.mw[b]))
            mu = mu + mus[a] * Y[a] / float(tb.mw[a]) / den
        mu = math.sqrt(8.0) * mu
        rd = torch.zeros_like(Y)
        for a in range(ns):
            den = torch.zeros_like(T)
            for b in range(ns):
                if b != a:
                    den = den + X[b] / from_table(_dev(tb.diffbin_species[:, a, b]))
            rd[a] = torch.where(den > 1e-15, (1.0 - Y[a]) / den * (tb.p0 / p * rho), torch.zeros_like(T))
        return mu, k, rd, W

    def chemistry(self, rho, Y, T, out):
        tb, ns = self.tb, self.ns
        it, ft = self.rows(T)
        c = [rho * Y[s] / float(tb.mw[s]) for s in range(ns)]
        RT = package().mechanism.R_UNIV * T
        arr = lambda r, q: float(tb.arr_a[r, q]) * T ** float(tb.arr_b[r, q]) * torch.exp(-float(tb.arr_ea[r, q]) / RT)  # noqa: E731
        for r in range(tb.nreactions):
            ty, kf, third = int(tb.reac_ty[r]), arr(r, 0), None
            if ty >= 1:
                third = sum(float(tb.tb_eff[r, s]) * c[s] for s in range(ns))
            if ty >= 2:
                kinf = arr(r, 1)
                pr = kf * third / kinf
                f = torch.ones_like(T)
                if ty == 3:
                    a, t3, t1, t2 = (float(tb.falloff_coeffs[r, q]) for q in range(4))
                    fc = (1.0 - a) * torch.exp(-T / t3) + a * torch.exp(-T / t1)
                    fc = torch.log10(fc + (torch.exp(-t2 / T) if t2 != -3.14 else 0.0))
                    x = torch.log10(pr) - 0.4 - 0.67 * fc
                    f = 10.0 ** (fc / (1.0 + (x / (0.75 - 1.27 * fc - 0.14 * x)) ** 2))
                kf = torch.where(pr < 1e-30, kf * third, kinf * (pr / (1.0 + pr)) * f) if ty == 3 else kinf * (pr / (1.0 + pr)) * f
            q1, q2 = torch.ones_like(T), torch.ones_like(T)
            for s in range(ns):
                if tb.r_coeffs[r, s]:
                    q1 = q1 * c[s] ** float(tb.r_coeffs[r, s])
                if tb.p_coeffs[r, s]:
                    q2 = q2 * c[s] ** float(tb.p_coeffs[r, s])
            q = kf * q1
            if int(tb.isRev[r]) == 1:
                kc = _dev(tb.kc_tab[:, r])
                q = q - kf / (kc[it] + (kc[it + 1] - kc[it]) * ft) * q2
            q = q * third if ty == 1 else q
            for s in range(ns):
                net = float(tb.p_coeffs[r, s] - tb.r_coeffs[r, s])
                if net:
                    out[s] -= net * q * float(tb.mw[s])

    def rhs(self, w, T):
        tb, ns, at, dx = self.tb, self.ns, self.at, self.dx
        rho, Y, u, T, p, R = self.aux(w, T)
        mu, k, rd, W = self.transport(rho, Y, T, p, R)
        e = w[ns + 3] / rho - 0.5 * u.square().sum(0)
        m = _range_of(tb, T)
        out = torch.zeros_like(w)
        grad = lambda a, d: sum(self.C[l - 1] * (at(a, d, l) - at(a, d, -l)) for l in (1, 2, 3)) / dx  # noqa: E731
        for d in range(3):
            fc = torch.zeros_like(w)
            for l in (1, 2, 3):
                for q in range(l):
                    pair = lambda a: at(a, d, -q) + at(a, d, l - q)  # noqa: E731
                    un = 0.25 * self.C[l - 1] * pair(rho) * pair(u[d])
                    for s in range(ns):
                        fc[s] += un * pair(Y[s])
                    for c in range(3):
                        fc[ns + c] += un * pair(u[c])
                    fc[ns + d] += self.C[l - 1] * pair(p)
                    fc[ns + 3] += un * (pair(e) + sum(at(u[c], d, -q) * at(u[c], d, l - q) for c in range(3)))
                    fc[ns + 3] += self.C[l - 1] * (at(u[d], d, -q) * at(p, d, l - q) + at(u[d], d, l - q) * at(p, d, -q))
            mf, kf = 0.5 * (mu + at(mu, d, 1)) / dx, 0.5 * (k + at(k, d, 1)) / dx
            ke = 0.5 * u.square().sum(0)
            for c in range(3):
                fc[ns + c] -= mf * (at(u[c], d, 1) - u[c])
            fc[ns + 3] -= kf * (at(T, d, 1) - T) + mf * (at(ke, d, 1) - ke)
            Wp = at(W, d, 1)
            wf = 0.5 * (Wp + W) / (Wp * W) / dx
            jump = [0.5 * (rd[s] + at(rd[s], d, 1)) * (at(Y[s], d, 1) * Wp - Y[s] * W) * wf for s in range(ns)]
            total = sum(jump)
            for s in range(ns):
                sig = 0.5 * (Y[s] + at(Y[s], d, 1)) * total - jump[s]
                h = _poly(tb, tb.cp_coeff, T, s, m[s], True)
                fc[s] += sig
                fc[ns + 3] += sig * 0.5 * (h + at(h, d, 1))
            del jump, total
            out += (fc - at(fc, d, -1)) / dx
            del fc
        g = [[grad(u[c], d) for c in range(3)] for d in range(3)]          # g[d][c] = du_c/dx_d
        div3 = (g[0][0] + g[1][1] + g[2][2]) / 3.0
        gmu, gdiv = [grad(mu, d) for d in range(3)], [grad(div3, d) for d in range(3)]
        S = [[g[c][d] - (2.0 * div3 if c == d else 0.0) for d in range(3)] for c in range(3)]
        sig = [sum(gmu[d] * S[c][d] for d in range(3)) + mu * gdiv[c] for c in range(3)]
        heat = sum(S[c][d] * g[d][c] for c in range(3) for d in range(3)) * mu
        for c in range(3):
            out[ns + c] -= sig[c]
        out[ns + 3] -= sum(sig[c] * u[c] for c in range(3)) + heat
        self.chemistry(rho, Y, T, out)
        return out, T

    def step(self, w, T, dt):
        fl = torch.zeros_like(w)
        for rho_k, gam_k in zip((0.0, -17.0 / 60.0, -5.0 / 12.0), (8.0 / 15.0, 5.0 / 12.0, 3.0 / 4.0)):
            old = fl
            fl, T = self.rhs(w, T)
            w = w - rho_k * dt * old - gam_k * dt * fl
            del old
        return w, fl


def exact(case, seed):
    """The RK3 step of the periodic boxes in plain torch.  The others have no such value: what
    an adaptive integrator returns is its own step sequence's (some hundreds of steps of
    thousands of operations each, minutes in plain torch), and so are the LES, shock-tube and
    Strang steps that contain one; the WENO fluxes of the mixing layer jump with the
    sensor's last bit."""
    if case["kind"] != "box":
        return None
    s = _box_solver(case, package().solver.Numerics(), seed)
    inner = lambda a: a[..., NG:-NG, NG:-NG, NG:-NG].clone()  # noqa: E731
    w, T, dt, ns = inner(s.w), inner(s.w_aux[s.ns + 4]), s.dt, s.ns
    del s
    torch.cuda.empty_cache()
    w, fl = _Plain(tables(case["mech"]), 2.0e-3 * math.pi / 256).step(w, T, dt)
    return {"rho_y": w[:ns], "rho_u": w[ns:ns + 3], "rho_e": w[ns + 3], "rhs_y": fl[:ns], "rhs_u": fl[ns:ns + 3],
            "rhs_e": fl[ns + 3]}
