"""Timed cases of the framework's public entry points.

Each case is a dict with a "kind"; `listed()` holds one or two cases per kind at
the sizes users run, `draw()` more of the same ranges.  The kinds:

  point     PNJL.solve at one (T, mu, xi): the interactive call, all latency
  default   a DefaultSeed grid scan (host arrays in and out)
  stable    a MultiSeed grid scan: the stable phase of a phase diagram
  chains    the scan driver's continuity chains along T (p 12, t 6)
  branches  dual-branch scans: hadron and quark branches along mu per line
  learned   the learned-seed scan of a large grid resident in HBM
  pi_grid   Pi(k0, k) on whole grids for a set of equilibrium points
  pi_batch  single Pi queries (both channels, with and without a width)
  props     D_S / D_P of scattering processes, device-resident
  masses    meson pole masses over a (T, mu) grid
  derivs    implicit thermodynamic derivatives, orders 1 and 2
  train     Adam steps of the learned seed's network (forward and backward)

Every input is drawn from the seed: the grids are shifted by a fraction of
their spacing.  DefaultSeed scans stay on the sides of the phase diagram
(T below 110 MeV at mu below 250 MeV, or T above 190 MeV) where the solver's
path to the root does not hang on the last bit of a node sum (between them
about one point in two thousand reaches another of its roots when the sums
are added in another order); there the stable and learned scans (argmin Omega
over the candidate roots) cover the transition, the learned one from T = 100
MeV (below, at the spinodals, one point in a million does the same).  Equilibrium states used as inputs are rounded to the six
decimals of the scan files, so that they are the same inputs whatever solver
produced them.
"""
import math

import numpy as np
import torch

from julia_relaxtime_amd import _lib, dual_branch, pnjl, propagators, surrogate, thermo_derivatives
from julia_relaxtime_amd import polarization as pol

HB = 197.327
FIELDS = ("x", "omega", "pressure", "rho_norm", "entropy", "energy", "masses", "n_q", "n_qbar", "converged")
XIS = (-0.4, -0.2, 0.0, 0.2, 0.4)
LEARNING_RATE = 5e-5     # a quarter of the training schedule's last phase: the loss curve does not amplify rounding


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one equilibrium state at the reference defaults (p 64, t 8)
        dict(name="point", kind="point", T=85.0, mu=120.0, xi=0.2, p=64, t=8),
        # the 32 x 32 isotropic scan of the benchmark, quark-gluon side
        dict(name="default_32x32", kind="default", side="qgp", nT=32, nmu=32, nxi=1, p=64, t=8),
        # the 64 x 64 x 9 anisotropic scan of the benchmark
        dict(name="stable_64x64x9", kind="stable", nT=64, nmu=64, nxi=9, p=64, t=4),
        # the scan driver's default grid: T 50-200 step 10, mu_B 0-1200 step 60, four xi
        dict(name="chains_driver", kind="chains", nT=16, nmu=21, nxi=4, p=12, t=6),
        # dual-branch lines around the first-order transition (p 24, t 8)
        dict(name="branches_45x111", kind="branches", lines=45, nmu=111, p=24, t=8),
        # the benchmark's default workload: 256 x 256 x 17 points from the learned seed
        dict(name="learned_256x256x17", kind="learned", nT=256, nmu=256, nxi=17, p=64, t=4),
        # the benchmark's polarization grid: 256 points x 3 pairs x 2 channels x 128 x 64
        dict(name="pi_grid_256x128x64", kind="pi_grid", npts=256, nk0=128, nk=64),
        # loose Pi queries as a pole search or a scattering integral makes them, an odd number
        dict(name="pi_batch_4999", kind="pi_batch", n=4999),
        # propagators of all table channels (a quarter of the benchmark's batch)
        dict(name="props_262144", kind="props", n=262144),
        # pole masses of all eight mesons on a 48 x 48 slice
        dict(name="masses_48x48", kind="masses", nT=48, nmu=48),
        # transport inputs along a medium scan: derivatives at 5000 states
        dict(name="derivs_5000", kind="derivs", n=5000, p=64, t=4),
        # steps of the learned seed's training at the benchmark's batch, at a fine-tuning rate
        dict(name="train_batch8192", kind="train", n=20000, batch=8192, steps=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("point", "default", "stable", "chains", "branches", "learned", "pi_grid", "pi_batch", "props",
                       "masses", "derivs", "train"))
    if kind == "point":
        if rng.random() < 0.5:
            T, mu = rng.uniform(30.0, 110.0), rng.uniform(5.0, 245.0)
        else:
            T, mu = rng.uniform(190.0, 290.0), rng.uniform(5.0, 440.0)
        return dict(kind=kind, T=round(T, 3), mu=round(mu, 3), xi=rng.choice(XIS), p=rng.choice((24, 48, 64)),
                    t=rng.choice((4, 6, 8)))
    if kind == "default":
        return dict(kind=kind, side=rng.choice(("qgp", "hadron")), nT=_log(rng, 3, 60), nmu=_log(rng, 3, 60),
                    nxi=rng.choice((1, 2, 3)), p=rng.choice((24, 48, 64)), t=rng.choice((4, 6, 8)))
    if kind == "stable":
        return dict(kind=kind, nT=_log(rng, 4, 64), nmu=_log(rng, 4, 64), nxi=rng.choice((1, 3, 5, 9)),
                    p=rng.choice((24, 48, 64)), t=rng.choice((4, 6)))
    if kind == "chains":
        return dict(kind=kind, nT=_log(rng, 4, 40), nmu=_log(rng, 2, 60), nxi=rng.choice((1, 2, 3, 4)),
                    p=rng.choice((12, 24)), t=rng.choice((6, 8)))
    if kind == "branches":
        return dict(kind=kind, lines=_log(rng, 2, 120), nmu=_log(rng, 20, 160), p=rng.choice((16, 24)), t=8)
    if kind == "learned":
        return dict(kind=kind, nT=_log(rng, 40, 256), nmu=_log(rng, 40, 256), nxi=rng.choice((3, 5, 9, 17)), p=64, t=4)
    if kind == "pi_grid":
        return dict(kind=kind, npts=_log(rng, 1, 200), nk0=_log(rng, 5, 110), nk=_log(rng, 3, 60))
    if kind == "pi_batch":
        return dict(kind=kind, n=_log(rng, 1, 60000))
    if kind == "props":
        return dict(kind=kind, n=_log(rng, 100, 400000))
    if kind == "masses":
        return dict(kind=kind, nT=_log(rng, 4, 64), nmu=_log(rng, 4, 64))
    if kind == "derivs":
        return dict(kind=kind, n=_log(rng, 10, 40000), p=rng.choice((24, 48, 64)), t=rng.choice((4, 6)))
    return dict(kind=kind, n=_log(rng, 5000, 40000), batch=rng.choice((2048, 4096, 8192)), steps=_log(rng, 8, 32))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _axis(rng, lo, hi, n):
    """n points in [lo, hi], equally spaced, shifted by a random part of the spacing."""
    h = (hi - lo) / n
    return lo + h * (np.arange(n) + rng.uniform(0.05, 0.95))


def _grid(rng, nT, nmu, nxi, T_range, mu_range):
    xi = {1: [0.0], 2: [0.0, 0.3], 3: [-0.3, 0.0, 0.3]}.get(nxi, np.linspace(-0.4, 0.4, nxi))
    T, mu, x = np.meshgrid(_axis(rng, *T_range, nT), _axis(rng, *mu_range, nmu), np.asarray(xi, float), indexing="ij")
    return T.ravel() / HB, mu.ravel() / HB, np.round(x.ravel(), 6)


def _states(rng, n, T_range=(40.0, 290.0), mu_range=(5.0, 440.0), xis=XIS):
    """n stable equilibrium states (T, mu, xi, x) rounded as in the scan files."""
    T, mu = rng.uniform(*T_range, n) / HB, rng.uniform(*mu_range, n) / HB
    xi = rng.choice(xis, n)
    r = pnjl.solve_batch(pnjl.FixedMu(), T, mu, xi=xi, seed_strategy=pnjl.MultiSeed(), p_num=64, t_num=4, iterations=40)
    return T, mu, xi, np.round(r["x"], 6)


def _masses(x):
    P = _lib.default_params()
    m = [P.m_ud0 - 4 * P.G * x[:, 0] + 2 * P.K * x[:, 1] * x[:, 2], P.m_s0 - 4 * P.G * x[:, 2] + 2 * P.K * x[:, 0] * x[:, 1]]
    return np.round(m[0], 6), np.round(m[1], 6)


def _quark_A(T, mu, m_u, m_s, Phi, Phib):
    """A(m_u), A(m_s) on GL(0, 20, 16), rounded."""
    xp, wp = np.polynomial.legendre.leggauss(16)
    xp, wp = 10.0 * xp + 10.0, 10.0 * wp
    a = np.concatenate([np.stack([m, mu, T, Phi, Phib], 1) for m in (m_u, m_s)])
    return np.round(pol.A_batch(a, xp, wp), 8).reshape(2, -1)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    k = case["kind"]
    if k == "point":
        return dict(case, T_fm=(case["T"] + rng.uniform(-2, 2)) / HB, mu_fm=(case["mu"] + rng.uniform(-2, 2)) / HB)
    if k in ("default", "stable"):
        box = ((50.0, 300.0), (0.0, 400.0)) if k == "stable" else \
            (((190.0, 300.0), (0.0, 400.0)) if case["side"] == "qgp" else ((20.0, 110.0), (0.0, 250.0)))
        T, mu, xi = _grid(rng, case["nT"], case["nmu"], case["nxi"], *box)
        return dict(case, grid=(T, mu, xi))
    if k == "chains":
        T = _axis(rng, 50.0, 200.0, case["nT"]) / HB
        mu = _axis(rng, 0.0, 400.0, case["nmu"]) / HB
        xi = np.array([0.0, 0.2, 0.4, -0.2])[:case["nxi"]]
        X, M, TT = np.meshgrid(xi, mu, T, indexing="ij")
        return dict(case, grid=(TT.ravel(), M.ravel(), X.ravel()))
    if k == "branches":
        T = np.tile(_axis(rng, 45.0, 140.0, -(-case["lines"] // 3)), 3)[:case["lines"]]
        xi = np.repeat([0.0, 0.2, 0.4], -(-case["lines"] // 3))[:case["lines"]]
        return dict(case, T=T, xi=xi, mu=_axis(rng, 200.0, 420.0, case["nmu"]))
    if k == "learned":
        ctx = _lib.Context(0)
        opts = _lib.default_opts(max_iter=40, ftol=1e-10, surrogate_judge=_lib.JUDGE_OMEGA)
        model, _ = surrogate.learned_seed(ctx, opts=_lib.default_opts(max_iter=40, ftol=1e-10))
        # the launch geometry the autotuner picks for this workload
        ctx.set_launch_cfg(lanes_per_point=8, chunk=1, waves_per_cu=16, tail_lanes_per_point=16)
        T, mu, xi = _grid(rng, case["nT"], case["nmu"], case["nxi"], (100.0, 300.0), (0.0, 450.0))
        g = [torch.tensor(a, device="cuda") for a in (T, mu, xi)]
        n = T.size
        out = {f: torch.empty((n, w) if w > 1 else (n,), device="cuda",
                              dtype=torch.float64 if dt == np.float64 else torch.int32) for f, w, dt in _lib.OUT_FIELDS}
        return dict(case, ctx=ctx, opts=opts, model=model, grid=g, out=out, seeds=torch.empty((n, 5), dtype=torch.float64,
                                                                                             device="cuda"))
    if k == "pi_grid":
        T, mu, xi, x = _states(rng, case["npts"])
        m_u, m_s = _masses(x)
        pts = np.stack([T, mu, xi, m_u, m_s, x[:, 3], x[:, 4]], 1)
        k0, kk = np.linspace(0.0, 4.0, case["nk0"]), np.linspace(0.0, 3.0, case["nk"])
        dev = [torch.tensor(a, device="cuda") for a in (pts, k0, kk)]
        shape = (case["npts"], 3, 2, case["nk0"], case["nk"])
        return dict(case, pts=dev[0], k0=dev[1], kk=dev[2],
                    out=tuple(torch.empty(shape, dtype=torch.float64, device="cuda") for _ in range(2)))
    if k == "pi_batch":
        return dict(case, q=_pi_queries(rng, case["n"]))
    if k == "props":
        n = case["n"]
        T, mu, xi, x = _states(rng, 256)
        m_u, m_s = _masses(x)
        A = _quark_A(T, mu, m_u, m_s, x[:, 3], x[:, 4])
        pc = [(propagators.PROCESS_ID[p], propagators.CHANNEL_ID[c]) for p in propagators.PROCESSES
              for c in propagators.process_channels(p)]
        sel, i = rng.integers(0, len(pc), n), rng.integers(0, 256, n)
        q = np.zeros(n, dtype=propagators.PROP_QUERY_DTYPE)
        q["process"], q["channel"] = np.array([c[0] for c in pc])[sel], np.array([c[1] for c in pc])[sel]
        q["k0"], q["k"] = rng.uniform(0.0, 4.0, n), rng.uniform(0.02, 3.0, n)
        for f, v in dict(T=T, mu_u=mu, mu_s=mu, xi=xi, m_u=m_u, m_s=m_s, Phi=x[:, 3], Phib=x[:, 4], A_u=A[0],
                         A_s=A[1]).items():
            q[f] = v[i]
        return dict(case, q=torch.from_numpy(q.view(np.uint8).copy()).cuda(),
                    out=torch.empty((n, 4), dtype=torch.float64, device="cuda"))
    if k == "masses":
        T, mu, xi = _grid(rng, case["nT"], case["nmu"], 1, (30.0, 290.0), (0.0, 400.0))
        r = pnjl.solve_batch(pnjl.FixedMu(), T, mu, xi=xi, seed_strategy=pnjl.MultiSeed(), p_num=64, t_num=4, iterations=40)
        x = np.round(r["x"], 6)
        m_u, m_s = _masses(x)
        A = _quark_A(T, mu, m_u, m_s, x[:, 3], x[:, 4])
        rep = lambda v: np.repeat(v, 8)  # noqa: E731
        return dict(case, q=propagators.make_mass_queries(np.tile(np.arange(8), T.size), rep(T), rep(x[:, 3]), rep(x[:, 4]),
                                                          0.0, rep(m_u), rep(m_s), rep(mu), rep(mu), rep(A[0]), rep(A[1])))
    if k == "derivs":
        T, mu, xi, x = _states(rng, case["n"], T_range=(90.0, 290.0))
        return dict(case, grid=(T, mu, xi), x=x)
    # train
    T, mu, xi, x = _states(rng, case["n"], T_range=(20.0, 300.0), mu_range=(0.0, 450.0))
    xi = rng.uniform(-0.4, 0.4, case["n"])   # the inputs' spread over the training box
    init = surrogate.Surrogate(0, init_seed=4)
    init.fit_output_scaling(x)
    return dict(case, data=(T, mu, xi, x), model=init, start=init.params)


def _pi_queries(rng, n):
    """Queries of all forms: the three quark pairs (num_s 0, 1, 2), P and S,
    with and without a width, at rest and moving, isotropic and not."""
    m = min(n, 512)
    T, mu, xi, x = (np.resize(a, (n,) + a.shape[1:]) for a in _states(rng, m))
    m_u, m_s = _masses(x)
    A_u, A_s = _quark_A(T, mu, m_u, m_s, x[:, 3], x[:, 4])
    pair = rng.integers(0, 3, n)
    pick = lambda u, s, c: np.where(pair == c, s, u)  # noqa: E731
    q = np.zeros(n, dtype=pol.QUERY_DTYPE)
    q["channel"] = rng.integers(1, 3, n)
    q["num_s"] = pair
    q["width"] = rng.random(n) < 0.5
    q["gamma"] = np.where(q["width"] == 1, np.round(rng.uniform(0.0, 1.0, n), 4), 0.0)
    q["k0"] = np.round(rng.uniform(0.05, 4.0, n), 4)
    q["k"] = np.where(rng.random(n) < 0.25, 0.0, np.round(rng.uniform(0.05, 3.0, n), 4))
    q["m1"], q["m2"] = pick(m_u, m_s, 2), np.where(pair == 0, m_u, m_s)
    q["A1"], q["A2"] = pick(A_u, A_s, 2), np.where(pair == 0, A_u, A_s)
    q["mu1"] = q["mu2"] = mu
    q["T"], q["xi"], q["Phi"], q["Phib"] = T, xi, x[:, 3], x[:, 4]
    return q


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    k = s["kind"]
    if k == "point":
        r = pnjl.solve(pnjl.FixedMu(), s["T_fm"], s["mu_fm"], xi=s["xi"], p_num=s["p"], t_num=s["t"])
        return dict(x=r.x_state, omega=r.omega, pressure=r.pressure, rho_norm=r.rho_norm, entropy=r.entropy,
                    energy=r.energy, masses=r.masses, n_q=r.n_q, n_qbar=r.n_qbar, converged=r.converged)
    if k in ("default", "stable", "chains"):
        T, mu, xi = s["grid"]
        if k == "default":
            r = pnjl.solve_batch(pnjl.FixedMu(), T, mu, xi=xi, p_num=s["p"], t_num=s["t"])
        elif k == "stable":
            r = pnjl.solve_batch(pnjl.FixedMu(), T, mu, xi=xi, seed_strategy=pnjl.MultiSeed(), p_num=s["p"], t_num=s["t"],
                                 iterations=40)
        else:
            r = pnjl.solve_batch(pnjl.FixedMu(), T, mu, xi=xi, seed_strategy=pnjl.PhaseAwareContinuitySeed(),
                                 chain_len=s["nT"], p_num=s["p"], t_num=s["t"], iterations=40)
        return {f: r[f] for f in FIELDS}
    if k == "branches":
        res = dual_branch.run_dual_branch_scan_batch(s["T"], s["mu"], s["xi"], p_num=s["p"], t_num=s["t"])
        return {"%s_%s" % (b, f): np.stack([r[b][f] for r in res]) for b in ("hadron", "quark", "physical")
                for f in ("x", "omega", "rho_norm", "entropy", "masses", "valid")}
    if k == "learned":
        T, mu, xi = s["grid"]
        seeds = s["model"].infer(T, mu, xi, out=s["seeds"], sync=False)
        r = s["ctx"].solve_batch(T, mu, xi, policy=_lib.SEED_SURROGATE, seed=seeds, p_num=s["p"], t_num=s["t"],
                                 opts=s["opts"], out=s["out"])
        return {f: r[f] for f in FIELDS}
    if k == "pi_grid":
        return list(pol.polarization_grid(s["pts"], s["k0"], s["kk"], out=s["out"]))
    if k == "pi_batch":
        return list(pol.polarization_batch(s["q"]))
    if k == "props":
        return propagators.propagator_by_channel_device(s["q"], s["out"])
    if k == "masses":
        r = propagators.meson_mass_batch(s["q"])
        # a search that stops without a pole leaves no mass
        ok = r["converged"]
        return dict(mass=np.where(ok, r["mass"], np.nan), gamma=np.where(ok, r["gamma"], np.nan), converged=ok,
                    exception=r["exception"])
    if k == "derivs":
        T, mu, xi = s["grid"]
        a = thermo_derivatives.thermo_derivatives_batch(T, mu, xi=xi, roots=s["x"], p_num=s["p"], t_num=s["t"])
        b = thermo_derivatives.implicit_derivatives2_batch(T, mu, xi=xi, roots=s["x"], p_num=s["p"], t_num=s["t"])
        return dict(first=a, second=b)
    # train: from the same start each pass
    T, mu, xi, x = s["data"]
    s["model"].params = s["start"]
    loss = s["model"].train(T, mu, xi, x, steps=s["steps"], batch=s["batch"], lr=LEARNING_RATE)
    return dict(loss=loss, params=s["model"].params)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
NODE = 178           # FP64 operations of one node and flavour (Omega, gradient, Hessian terms)
OUT_BYTES = 8 * (5 + 5 + 3 + 3 + 3 + 1) + 4 * 5


def work(case):
    k = case["kind"]
    nx = case.get("nxi", 1)
    # angle nodes matter at xi != 0 only
    t_eff = case.get("t", 4) if k != "point" else (case["t"] if case["xi"] else 1)
    if k in ("default", "stable", "chains", "learned"):
        n = case["nT"] * case["nmu"] * nx
        iso = 1.0 if nx == 1 else 1.0 / nx
        t_eff = iso + (1.0 - iso) * case["t"]
        # Newton passes per point: a start, three or four steps and the check; six starts for the stable scan
        passes = dict(default=6, stable=36, chains=5, learned=5)[k]
        return dict(bytes=n * (24 + OUT_BYTES), flops=2.0 * n * passes * case["p"] * t_eff * NODE)
    if k == "point":
        return dict(bytes=24 + OUT_BYTES, flops=2.0 * 6 * case["p"] * t_eff * NODE)
    if k == "branches":
        n = 2 * case["lines"] * case["nmu"]
        return dict(bytes=n * (24 + OUT_BYTES), flops=2.0 * n * 4 * case["p"] * case["t"] * NODE)
    if k == "pi_grid":
        n = case["npts"] * 3 * case["nk0"] * case["nk"]
        return dict(bytes=n * 32.0 + case["npts"] * 56, flops=n * 2 * 43286.0)
    if k == "pi_batch":
        return dict(bytes=case["n"] * (16 + 13 * 8 + 16.0), flops=case["n"] * 2 * 43286.0)
    if k == "props":
        return dict(bytes=case["n"] * (112 + 32.0), flops=case["n"] * 119772.0)
    if k == "masses":
        n = 8 * case["nT"] * case["nmu"]
        return dict(bytes=n * (136 + 48.0), flops=n * 822180.0)
    if k == "derivs":
        n = case["n"]
        return dict(bytes=n * 8.0 * (2 * 8 + 36 + 48), flops=2.0 * n * case["p"] * case["t"] * (260 + 900))
    # train: 3-128-128-128-4, forward and the two products of the backward
    par = 34052
    return dict(bytes=case["n"] * 64.0 + 3 * 4 * par, flops=case["steps"] * case["batch"] * par * 6.0)


def tolerance(case):
    return TOL[case["kind"]]


# Each is four times or more what the outputs move by when the inputs move by an
# ulp or the node sums are added in another order (measured beside it).
TOL = {
    # the solver stops at |F| < 1e-9 or |dx| < 1e-9, so x carries the last step of its
    # path to the root: 1.7e-10 (largest 1.2e-8, next to the critical end point)
    "point": dict(rel=2e-9, max=2e-7),
    "default": dict(rel=2e-9, max=2e-7),
    "stable": dict(rel=2e-9, max=2e-7),
    "chains": dict(rel=2e-9, max=2e-7),
    "branches": dict(rel=2e-9, max=2e-7),
    "learned": dict(rel=2e-9, max=2e-7),
    "pi_grid": dict(rel=1e-11, max=1e-8),     # 9e-14, largest 2e-10 next to a threshold
    "pi_batch": dict(rel=1e-11, max=1e-8),
    "props": dict(rel=2e-8, max=1e-6),        # 2.3e-9: the poles of D amplify Pi's rounding
    "masses": dict(rel=1e-9, max=1e-7),       # 6e-12
    "derivs": dict(rel=2e-9, max=2e-7),       # 2.7e-10 (d mu_B / dT at constant s / n)
    "train": dict(rel=3e-2, max=0.5),         # 1e-2 in the loss from 1e-7 in the targets: bf16 products
}


# ---------------------------------------------------------------------------
# the same numbers from plain torch in 64 bits
# ---------------------------------------------------------------------------
EXACT_POINTS = 1500       # gap equations
EXACT_CELLS = 300000      # Pi values


def exact(case, seed):
    k = case["kind"]
    if k in ("point", "default", "stable"):
        s = prepare(case, seed)
        g = s["grid"] if k != "point" else tuple(np.array([v]) for v in (s["T_fm"], s["mu_fm"], float(s["xi"])))
        if g[0].size > EXACT_POINTS:
            return None
        r = _stable_roots(*g, case["p"], case["t"])
        if k == "point":
            r = {f: (v[0] if v.ndim > 1 else float(v[0])) for f, v in r.items()}
        return dict(r, converged=None)
    if k == "pi_grid":
        if case["npts"] * 3 * case["nk0"] * case["nk"] > EXACT_CELLS:
            return None
        s = prepare(case, seed)
        return _pi_grid_exact(s["pts"], s["k0"], s["kk"])
    if k == "pi_batch":
        if case["n"] > EXACT_CELLS:
            return None
        return _pi_batch_exact(prepare(case, seed)["q"])
    if k == "derivs":
        if case["n"] > 8192:
            return None
        s = prepare(case, seed)
        return _derivs_exact(s["x"], *s["grid"], case["p"], case["t"])
    # chains and branches follow the whole solver policy, the pole search its
    # iterates; the propagators' Pi values are pi_batch's, and training runs in
    # 16-bit products: no value of their own to state here
    return None


def _gl(a, b, n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (b - a) * x + 0.5 * (b + a), 0.5 * (b - a) * w


class _Gap:
    """Omega(x, T, mu, xi) of the 2+1-flavour PNJL model on p x t nodes."""

    def __init__(self, p, t, dev="cuda"):
        P = _lib.default_params()
        self.c = {f: getattr(P, f) for f in ("Lambda", "G", "K", "m_ud0", "m_s0", "T0", "a0", "a1", "a2", "b3", "rho0")}
        px, pw = _gl(0.0, 10.0, p)
        tx, tw = _gl(0.0, 1.0, t)
        C = (pw[:, None] * 2.0 * tw[None, :]) * px[:, None] ** 2 / (2 * np.pi) ** 2
        mk = lambda a: torch.tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        self.p2, self.cc, self.C = mk(np.repeat(px ** 2, t)), mk(np.tile(tx ** 2, p)), mk(C.ravel())

    def masses(self, x):
        c = self.c
        u, d, s = x[:, 0], x[:, 1], x[:, 2]
        return torch.stack([c["m_ud0"] - 4 * c["G"] * u + 2 * c["K"] * d * s, c["m_ud0"] - 4 * c["G"] * d + 2 * c["K"] * u * s,
                            c["m_s0"] - 4 * c["G"] * s + 2 * c["K"] * u * d], 1)

    def _ab(self, M, T, mu, xi):
        E = torch.sqrt(self.p2 * (1 + xi[:, None] * self.cc) + M[:, None] ** 2)
        return (mu[:, None] - E) / T[:, None], -(E + mu[:, None]) / T[:, None]

    def omega(self, x, T, mu, xi):
        c = self.c
        Phi, Phib = x[:, 3], x[:, 4]
        M = self.masses(x)
        chi = 2 * c["G"] * (x[:, 0] ** 2 + x[:, 1] ** 2 + x[:, 2] ** 2) - 4 * c["K"] * x[:, 0] * x[:, 1] * x[:, 2]
        Tr = c["T0"] / T
        Ta, Tb = c["a0"] + c["a1"] * Tr + c["a2"] * Tr ** 2, c["b3"] * Tr ** 3
        PP = Phi * Phib
        v = 1 - 6 * PP + 4 * (Phib ** 3 + Phi ** 3) - 3 * PP ** 2
        om = chi + T ** 4 * (-0.5 * Ta * PP + Tb * torch.log(torch.clamp(v, min=1e-16)))
        L = c["Lambda"]
        for i in range(3):
            Mi = M[:, i]
            m2 = Mi ** 2
            s = torch.sqrt(L * L + m2)
            I = (L * s * (2 * L * L + m2) - m2 * m2 * torch.log((L + s) / Mi.abs())) / (16 * np.pi ** 2)
            S = 0.0
            for a, c1, c2 in zip(self._ab(Mi, T, mu, xi), (Phi, Phib), (Phib, Phi)):
                pos = a > 0
                e = torch.exp(-a.abs())
                z = torch.where(pos, e ** 3 + 3 * (c1[:, None] * e ** 2 + c2[:, None] * e) + 1,
                                1 + 3 * (c1[:, None] * e + c2[:, None] * e ** 2) + e ** 3)
                S = S + torch.log(torch.clamp(z, min=1e-16)) + torch.where(pos, 3 * a, torch.zeros_like(a))
            om = om - 6 * I - 2 * T * (S * self.C).sum(1)
        return om

    def densities(self, x, T, mu, xi):
        M = self.masses(x)
        nq, nqb = [], []
        for i in range(3):
            for a, c1, c2, o in zip(self._ab(M[:, i], T, mu, xi), (x[:, 3], x[:, 4]), (x[:, 4], x[:, 3]), (nq, nqb)):
                e = torch.exp(-a.abs())
                pos = a > 0
                n1, n2, n3 = torch.where(pos, e ** 2, e), torch.where(pos, e, e ** 2), torch.where(pos, torch.ones_like(e), e ** 3)
                n0 = torch.where(pos, e ** 3, torch.ones_like(e))
                f = (c1[:, None] * n1 + 2 * c2[:, None] * n2 + n3) / (n0 + 3 * c1[:, None] * n1 + 3 * c2[:, None] * n2 + n3)
                o.append(6 * (f * self.C).sum(1))
        return torch.stack(nq, 1), torch.stack(nqb, 1)

    def newton(self, x, T, mu, xi, steps=40):
        """Damped Newton on dOmega/dx = 0 (steps cut at 0.15): the states and their residuals"""
        x, res = x.clone(), torch.full_like(T, float("inf"))
        on = torch.arange(T.numel(), device=T.device)       # rows still moving
        for _ in range(steps):
            F, H = _hessian(self.omega, x[on].requires_grad_(True), T[on], mu[on], xi[on])
            dx = torch.nan_to_num(torch.linalg.solve_ex(H, -F[:, :, None])[0][:, :, 0])
            big = dx.abs().amax(1, keepdim=True)
            x[on] += dx * torch.clamp(0.15 / big.clamp(min=1e-300), max=1.0)
            res[on] = F.abs().amax(1)
            on = on[~(big[:, 0] < 1e-12)]
            if not on.numel():
                break
        return x, res


def _hessian(fn, x, *rest):
    """gradient and Hessian of fn(x, ...) per row"""
    F, = torch.autograd.grad(fn(x, *rest).sum(), x, create_graph=True)
    H = torch.stack([torch.autograd.grad(F[:, i].sum(), x, retain_graph=True)[0] for i in range(x.shape[1])], 1)
    return F.detach(), H.detach()


SEEDS = [[-1.84329, -1.84329, -2.22701, 1.0e-5, 4.0e-5], [-0.73192, -0.73192, -1.79539, 0.60532, 0.60532],
         [-0.50, -0.50, -1.20, 1e-3, 1e-3], [-0.50, -0.50, -1.20, 0.80, 0.80], [-0.30, -0.30, -0.90, 0.90, 0.90],
         [-1.3647, -1.3647, -2.14502, 0.10594, 0.15569], [-0.21695, -0.21695, -2.01372, 0.18601, 0.22333]]


def _stable_roots(T, mu, xi, p, t, chunk=1024):
    """The root of lowest Omega among those that Newton reaches from the seeds, and its thermodynamics."""
    gap = _Gap(p, t)
    rows = []
    for c in range(0, T.size, chunk):
        Tc, mc, xc = (torch.tensor(a[c:c + chunk], device="cuda") for a in (T, mu, xi))
        best, bom = torch.full((Tc.numel(), 5), float("nan"), device="cuda", dtype=torch.float64), torch.full_like(Tc, float("inf"))
        for sd in SEEDS:
            x, res = gap.newton(torch.tensor([sd] * Tc.numel(), device="cuda", dtype=torch.float64), Tc, mc, xc)
            om = gap.omega(x, Tc, mc, xc)
            ok = (res < 1e-8) & (x[:, 3] >= -1e-8) & (x[:, 3] <= 1) & (x[:, 4] >= -1e-8) & (x[:, 4] <= 1) & \
                (gap.masses(x) > 0).all(1) & torch.isfinite(om) & (om < bom)
            best[ok], bom[ok] = x[ok], om[ok]
        Tg = Tc.clone().requires_grad_(True)
        s, = torch.autograd.grad(-gap.omega(best, Tg, mc, xc).sum(), Tg)
        nq, nqb = gap.densities(best, Tc, mc, xc)
        rho = (nq - nqb).sum(1)
        rows.append(dict(x=best, omega=bom, pressure=-bom, rho_norm=rho / (3 * gap.c["rho0"]), entropy=s,
                         energy=bom + mc * rho + Tc * s, masses=gap.masses(best), n_q=nq, n_qbar=nqb))
    return {f: torch.cat([r[f] for r in rows]).cpu().numpy() for f in rows[0]}


def _derivs_exact(x, T, mu, xi, p, t, chunk=512):
    """x_a = -H^-1 F_a and x_ab = -H^-1 d_b(H x_a + F_a), by automatic differentiation."""
    gap, rows = _Gap(p, t), []
    for c in range(0, T.size, chunk):
        xc, Tc, mc, xic = (torch.tensor(a[c:c + chunk], device="cuda") for a in (x, T, mu, xi))
        z = torch.cat([xc, Tc[:, None], mc[:, None]], 1).requires_grad_(True)
        fn = lambda z: gap.omega(z[:, :5], z[:, 5], z[:, 6], xic)  # noqa: E731
        F, H = _hessian(fn, z)
        solve = lambda b: torch.linalg.solve(H[:, :5, :5], -b[:, :, None])[:, :, 0]  # noqa: E731
        w = []
        for a in (5, 6):
            e = torch.zeros_like(F)
            e[:, a] = 1.0
            e[:, :5] = solve(H[:, :5, a])
            w.append(e)
        second = {}
        for name, a, b in (("d2x_dT2", 0, 0), ("d2x_dTdmu", 0, 1), ("d2x_dmu2", 1, 1)):
            g, = torch.autograd.grad(fn(z).sum(), z, create_graph=True)
            g, = torch.autograd.grad((g * w[a]).sum(), z, create_graph=True)
            g, = torch.autograd.grad((g * w[b]).sum(), z)
            second[name] = solve(g[:, :5])
        rows.append(dict(first=dict(pressure=-fn(z).detach(), entropy=-F[:, 5], dP_dmu=-F[:, 6]),
                         second=dict(second, x=xc, dx_dT=w[0][:, :5], dx_dmu=w[1][:, :5])))
    return {o: {f: torch.cat([r[o][f] for r in rows]).cpu().numpy() for f in rows[0][o]} for o in ("first", "second")}


# ---- Pi: the fixed quadrature of the one-loop integrals, a whole batch at once ----
_EPS = 1e-12


def _rules():
    r = {}
    for n in (16, 32):
        x, w = np.polynomial.legendre.leggauss(n)
        u, ia = (x + 1) / 2, 1 / 0.35
        r["gl%d" % n] = (x, w)
        # x = a + len t(u), weight w t'(u) len: clustered at the left or the right end
        r["left%d" % n] = (u ** ia, w * ia * u ** (ia - 1) / 2)
        r["right%d" % n] = (1 - (1 - u) ** ia, w * ia * (1 - u) ** (ia - 1) / 2)
    tk = np.arange(-16, 17) * 0.15
    s = np.pi / 2 * np.sinh(tk)
    r["both"] = ((1 + np.tanh(s)) / 2, 0.15 * np.pi / 4 * np.cosh(tk) / np.cosh(s) ** 2)
    return r


class _Pi:
    """B0 and its first-order anisotropic correction for rows of
    (m, m', mu, T, Phi, Phibar, xi); Lambda the cutoff."""

    def __init__(self):
        self.L = _lib.default_params().Lambda
        self.R = {k: tuple(torch.tensor(v, device="cuda") for v in w) for k, w in _rules().items()}

    def segment(self, f, rows, a, b, rule):
        """integral of f(E, *rows) over [a, b] where b > a, else 0; non-finite nodes count 0"""
        out = torch.zeros_like(a)
        on = torch.isfinite(a) & torch.isfinite(b) & (b > a)
        if on.any():
            t, w = self.R[rule]
            sub = [r[on][:, None] for r in rows]
            ln = (b - a)[on][:, None]
            v = f(a[on][:, None] + ln * t, *sub)
            out[on] = torch.where(torch.isfinite(v), v * w * ln, torch.zeros_like(v)).sum(1)
        return out

    def dist(self, plus, E, mu, T, c1, c2):
        """f+(E), or f+(-E) = 1 - f-(E)"""
        e = torch.exp(-(E - mu) / T if plus else -(E + mu) / T).clamp(1e-200, 1e200)
        u, v = (c1, c2) if plus else (c2, c1)
        f = (u * e + 2 * v * e ** 2 + e ** 3) / (1 + 3 * u * e + 3 * v * e ** 2 + e ** 3)
        return f if plus else 1 - f

    def cumulative(self, plus, E, mu, T, c1, c2):
        e = torch.exp(-(E - mu) / T if plus else -(E + mu) / T).clamp(1e-200, 1e200)
        u, v = (c1, c2) if plus else (c2, c1)
        g = -T * torch.log((1 + 3 * u * e + 3 * v * e ** 2 + e ** 3).clamp(min=1e-300)) / 3
        return g if plus else E - g

    @staticmethod
    def cuts(lam, k, m, mp, Emin, Emax):
        """[E1, E2] of the piecewise quadrature and the (up to two) intervals of the imaginary part"""
        nan, inf = torch.full_like(lam, float("nan")), float("inf")
        a = lam ** 2 - k ** 2
        flat = a.abs() < _EPS
        A = a + m ** 2 - mp ** 2
        disc = A ** 2 - 4 * m ** 2 * a
        sq = torch.sqrt(disc)
        r1, r2 = (lam * A - k * sq) / (-2 * a), (lam * A + k * sq) / (-2 * a)
        lo, hi = torch.minimum(r1, r2), torch.maximum(r1, r2)
        good = ~flat & (disc >= 0) & (hi - lo >= _EPS)
        iv = []
        # timelike: between the roots
        c1, c2 = torch.maximum(lo, Emin), torch.minimum(hi, Emax)
        tl = good & (a > 0) & (hi > Emin) & (lo < Emax) & (c2 > c1)
        # spacelike: outside the roots
        b1 = torch.minimum(lo, Emax)
        s1 = good & (a < 0) & (lo > Emin) & (b1 > Emin)
        b2 = torch.maximum(hi, Emin)
        s2 = good & (a < 0) & (hi < Emax) & (Emax > b2)
        m2d = mp ** 2 - m ** 2
        Ec = m2d / (4 * lam) + lam * m ** 2 / m2d
        fl = flat & (lam > 0) & (mp > m) & (Ec < Emax)
        E1 = torch.where(tl, c1, torch.where(s1 & s2, b1, torch.where(s1, Emin, torch.where(s2, b2, torch.where(
            fl, torch.maximum(Ec, Emin), nan)))))
        E2 = torch.where(tl, c2, torch.where(s1 & s2, b2, torch.where(s1, b1, torch.where(s2 | fl, Emax, nan))))
        iv.append((torch.where(tl, c1, torch.where(s1, Emin, torch.where(s2, b2, torch.where(fl, E1, nan)))),
                   torch.where(tl, c2, torch.where(s1, b1, torch.where(s2 | fl, Emax, nan)))))
        iv.append((torch.where(s1 & s2, b2, nan), torch.where(s1 & s2, Emax, nan)))
        return E1, E2, iv, inf

    def term(self, plus, lam, k, m, mp, mu, T, c1, c2):
        """B~0(lam, k) of one sign"""
        Emin, Emax = m, torch.sqrt(m ** 2 + self.L ** 2)
        re, im = torch.zeros_like(lam), torch.zeros_like(lam)
        mv = k.abs() >= 1e-9
        if mv.any():
            g = [v[mv] for v in (lam, k, m, mp, mu, T, c1, c2)]
            r, i = self.moving(plus, *g, Emin[mv], Emax[mv])
            re[mv], im[mv] = r, i
        if (~mv).any():
            g = [v[~mv] for v in (lam, m, mp, mu, T, c1, c2)]
            r, i = self.rest(plus, *g, Emin[~mv], Emax[~mv])
            re[~mv], im[~mv] = r, i
        return re, im

    def moving(self, plus, lam, k, m, mp, mu, T, c1, c2, Emin, Emax):
        def f(E, lam, k, m, mp, mu, T, c1, c2):
            p = torch.sqrt(E * E - m * m)
            com = (lam + E) ** 2 - mp ** 2
            num, den = com - (p - k) ** 2, com - (p + k) ** 2
            skip = (num.abs() < _EPS) & (den.abs() < _EPS)
            den = torch.where(den.abs() < _EPS, torch.where(den < 0, -_EPS, _EPS), den)
            v = self.dist(plus, E, mu, T, c1, c2) * torch.log((num / den).abs().clamp(min=1e-300))
            return torch.where(skip, torch.zeros_like(v), v)

        rows = (lam, k, m, mp, mu, T, c1, c2)
        E1, E2, iv, _ = self.cuts(lam, k, m, mp, Emin, Emax)
        cut = torch.isfinite(E1)
        end = torch.where(cut, Emin, Emax)          # no cut: one rule over the whole range
        re = self.segment(f, rows, Emin, torch.where(cut, Emin, Emax), "left16")
        re = re + self.segment(f, rows, Emin, torch.where(cut, E1, end), "right32") * cut
        re = re + self.segment(f, rows, E1, E2, "both") + self.segment(f, rows, E2, torch.where(cut, Emax, E2), "left16")
        im = torch.zeros_like(lam)
        for a, b in iv:
            d = self.cumulative(plus, b, mu, T, c1, c2) - self.cumulative(plus, a, mu, T, c1, c2)
            im = im + torch.where(torch.isfinite(a), d, torch.zeros_like(d))
        return re / k, im * np.pi * torch.sign(lam) / k

    def rest(self, plus, lam, m, mp, mu, T, c1, c2, Emin, Emax):
        dt = (lam ** 2 + m ** 2 - mp ** 2) / 2
        E0 = -dt / lam
        tol = 1e-8 * E0.abs().clamp(min=1.0)
        has = torch.isfinite(E0) & (E0 > Emin - tol) & (E0 < Emax + tol)
        num = lambda E, m, mu, T, c1, c2: torch.nan_to_num(  # noqa: E731
            torch.sqrt(E * E - m * m) * self.dist(plus, E, mu, T, c1, c2), nan=0.0)

        def pole(E, lam, m, dt, mu, T, c1, c2):
            den = lam * E + dt
            v = num(E, m, mu, T, c1, c2) / den
            return torch.where(den.abs() < _EPS, torch.zeros_like(v), v)

        rows = (lam, m, dt, mu, T, c1, c2)
        f0 = num(E0, m, mu, T, c1, c2)
        etol = 1e-10 * (Emax - Emin).clamp(min=1.0)
        edge = has & (((E0 - Emin).abs() <= etol) | ((Emax - E0).abs() <= etol))
        gap = torch.maximum(1e-6 * (Emax - Emin), 64 * torch.abs(torch.nextafter(E0.abs(), E0.abs() * 2 + 1) - E0.abs()))
        no = torch.full_like(lam, float("nan"))
        plain = self.segment(pole, rows, torch.where(has, no, Emin), Emax, "left16")
        split = self.segment(pole, rows, torch.where(edge, Emin, no), torch.maximum(Emin, E0 - gap), "left16") + \
            self.segment(pole, rows, torch.where(edge, torch.minimum(Emax, E0 + gap), no), Emax, "left16")

        def regular(E, m, mu, T, c1, c2, E0, f0):
            return (num(E, m, mu, T, c1, c2) - f0) / (E - E0)

        pv = self.segment(regular, (m, mu, T, c1, c2, E0, f0), torch.where(has & ~edge, Emin, no), Emax, "left32")
        pv = (pv + f0 * (torch.log((Emax - E0).abs()) - torch.log((Emin - E0).abs()))) / lam
        re = 2 * torch.where(~has, plain, torch.where(edge, split, pv))
        im = torch.where(has, 2 * np.pi * f0 / lam, 0.0 / lam)
        return re, im

    def coef(self, plus, p, m, mu, T, c1, c2, xi):
        """first-order coefficient of cos^2: xi p^2 / (2 E) df/dE"""
        E = torch.sqrt(p * p + m * m)
        e = torch.exp(-(E - mu) / T if plus else -(E + mu) / T).clamp(1e-200, 1e200)
        u, v = (c1, c2) if plus else (c2, c1)
        num, den = u * e + 2 * v * e ** 2 + e ** 3, 1 + 3 * u * e + 3 * v * e ** 2 + e ** 3
        dnum, dden = -(u * e + 4 * v * e ** 2 + 3 * e ** 3), -3 * num
        return 0.5 * xi * p * p / E * (dnum * den - num * dden) / den ** 2 / T

    def corr_term(self, plus, lam, k, m, mp, mu, T, c1, c2, xi):
        Emin, Emax = m, torch.sqrt(m ** 2 + self.L ** 2)
        re, im = torch.zeros_like(lam), torch.zeros_like(lam)
        mv = k > 1e-9
        if mv.any():
            r, i = self.corr_moving(plus, *[v[mv] for v in (lam, k, m, mp, mu, T, c1, c2, xi, Emin, Emax)])
            re[mv], im[mv] = r, i
        if (~mv).any():
            r, i = self.corr_rest(plus, *[v[~mv] for v in (lam, m, mp, mu, T, c1, c2, xi, Emin, Emax)])
            re[~mv], im[~mv] = r, i
        return re, im

    def corr_rest(self, plus, lam, m, mp, mu, T, c1, c2, xi, Emin, Emax):
        cE, dc = 2 * lam, lam ** 2 + m ** 2 - mp ** 2
        E0 = -dc / cE
        has = torch.isfinite(E0) & (E0 >= Emin) & (E0 <= Emax)

        def numer(E, m, mu, T, c1, c2, xi):
            p = torch.sqrt(E * E - m * m)
            return 4.0 / 3.0 * p * self.coef(plus, p, m, mu, T, c1, c2, xi)

        A0 = torch.where(has, numer(E0, m, mu, T, c1, c2, xi), torch.zeros_like(lam))
        x, w = self.R["gl32"]
        E = ((Emax - Emin)[:, None] * x + (Emax + Emin)[:, None]) / 2
        col = lambda v: v[:, None]  # noqa: E731
        v = (numer(E, *[col(q) for q in (m, mu, T, c1, c2, xi)]) - A0[:, None]) / (cE[:, None] * E + dc[:, None])
        s = (torch.where(torch.isfinite(v), v, torch.zeros_like(v)) * w).sum(1) * (Emax - Emin) / 2
        lg = A0 / cE * (torch.log((cE * Emax + dc).abs()) - torch.log((cE * Emin + dc).abs()))
        return s + torch.where(has, lg, torch.zeros_like(lg)), torch.where(has, np.pi * A0 / cE, torch.zeros_like(A0))

    def corr_moving(self, plus, lam, k, m, mp, mu, T, c1, c2, xi, Emin, Emax):
        def pieces(E, lam, k, m, mp):
            p = torch.sqrt(E * E - m * m)
            return p, 2 * p * k, lam ** 2 + 2 * lam * E + m ** 2 - mp ** 2 - k ** 2

        def real(E, lam, k, m, mp, mu, T, c1, c2, xi):
            p, cx, dc = pieces(E, lam, k, m, mp)
            tool = -2 * dc / cx ** 2 + dc ** 2 / cx ** 3 * torch.log(((cx + dc) / (cx - dc)).abs())
            return 2 * p * tool * self.coef(plus, p, m, mu, T, c1, c2, xi)

        def imag(E, lam, k, m, mp, mu, T, c1, c2, xi):
            p, cx, dc = pieces(E, lam, k, m, mp)
            return 2 * p * np.pi * dc ** 2 / cx ** 3 * self.coef(plus, p, m, mu, T, c1, c2, xi)

        rows = (lam, k, m, mp, mu, T, c1, c2, xi)
        # breakpoints: the roots of A + B and A - B inside the range
        C = lam ** 2 + m ** 2 - mp ** 2 - k ** 2
        a, b, c = k ** 2 - lam ** 2, -lam * C, -(k ** 2 * m ** 2 + C ** 2 / 4)
        D = b * b - 4 * a * c
        sD = torch.sqrt(D)
        nan = torch.full_like(lam, float("nan"))
        lin = a.abs() < 1e-14
        cand = [torch.where(lin, torch.where(b.abs() < 1e-14, nan, -c / b), (-b - sD) / (2 * a)),
                torch.where(lin, nan, (-b + sD) / (2 * a))]
        roots = []
        for E in cand:
            p, A, B = pieces(E, lam, k, m, mp)
            ok = (E >= m) & (E <= Emax) & (((A + B).abs() < 1e-10) | ((A - B).abs() < 1e-10))
            roots.append(torch.where(ok, E, torch.full_like(E, float("inf"))))
        r1, r2 = torch.minimum(*roots), torch.maximum(*roots)
        r2 = torch.where(r1 == r2, torch.full_like(r2, float("inf")), r2)
        n = torch.isfinite(r1).int() + torch.isfinite(r2).int()
        d = (1e-8 * (Emax - Emin)).clamp(min=1e-10)
        re = self.segment(real, rows, torch.where(n == 0, Emin, nan), Emax, "left16")
        wide = lambda x, y: y > x + 1e-16  # noqa: E731
        # the intervals between the roots; the one-interval rule where the others are empty
        ends = [(Emin, r1 - d), (r1 + d, torch.where(n == 2, r2 - d, Emax)), (torch.where(n == 2, r2 + d, nan), Emax)]
        live = torch.stack([(n > 0) & torch.isfinite(x) & torch.isfinite(y) & wide(x, y) for x, y in ends])
        cnt = live.sum(0)
        before = torch.zeros_like(cnt)
        for (x, y), on in zip(ends, live):
            first, last = before == 0, before == cnt - 1
            for rule, sel in (("both", on & ((cnt == 1) | (~first & ~last))), ("right32", on & (cnt > 1) & first),
                              ("left16", on & (cnt > 1) & last & ~first)):
                re = re + self.segment(real, rows, torch.where(sel, x, nan), y, rule)
            before = before + on.int()
        im = torch.zeros_like(lam)
        x, w = self.R["gl16"]
        for lo, hi in self.cuts(lam, k, m, mp, Emin, Emax)[2]:
            on = torch.isfinite(lo)
            if on.any():
                h, ctr = ((hi - lo) / 2)[on][:, None], ((hi + lo) / 2)[on][:, None]
                v = imag(ctr + h * x, *[r[on][:, None] for r in rows])
                im[on] += (torch.where(torch.isfinite(v), v, torch.zeros_like(v)) * w * h).sum(1)
        return re, im * torch.sign(lam)

    def b0(self, lam, k, m1, mu1, m2, mu2, T, c1, c2, xi):
        re = im = 0.0
        for plus, l, a, b, mu in ((True, -lam, m1, m2, mu1), (False, lam, m1, m2, mu1), (True, lam, m2, m1, mu2),
                                  (False, -lam, m2, m1, mu2)):
            r, i = self.term(plus, l, k, a, b, mu, T, c1, c2)
            s = 1.0 if plus else -1.0
            re, im = re + s * r, im + s * i
            on = xi.abs() > _EPS
            if on.any():
                r, i = self.corr_term(plus, *[v[on] for v in (l, k, a, b, mu, T, c1, c2, xi)])
                re, im = re.clone(), im.clone()
                re[on], im[on] = re[on] + r, im[on] + i
        return re, im

    def value(self, chan, num_s, width, k0, gamma, k, m1, m2, mu1, mu2, T, c1, c2, xi, A12):
        lam = k0 + mu1 - mu2
        br, bi = self.b0(lam, k, m1, mu1, m2, mu2, T, c1, c2, xi)
        sym = num_s == 1
        if sym.any():
            g = [v[sym] for v in (k, m1, mu1, m2, mu2, T, c1, c2, xi)]
            r, i = self.b0((-k0 + mu1 - mu2)[sym], *g)
            br[sym], bi[sym] = 0.5 * (br[sym] + r), 0.5 * (bi[sym] + i)
        pref = k ** 2 - lam ** 2 + torch.where(chan == 1, (m1 - m2) ** 2, (m1 + m2) ** 2)
        g2 = torch.where(width == 1, gamma, torch.zeros_like(gamma))
        pref = pref + g2 ** 2 / 4
        fac = -3.0 / (8 * np.pi ** 2)
        return fac * (A12 + pref * br - g2 * lam * bi), fac * (pref * bi + g2 * lam * br)


def _pi_batch_exact(q, chunk=20000):
    pi, out = _Pi(), []
    for c in range(0, q.size, chunk):
        g = {f: torch.tensor(np.ascontiguousarray(q[f][c:c + chunk]), device="cuda") for f in q.dtype.names}
        out.append(pi.value(g["channel"], g["num_s"], g["width"], g["k0"], g["gamma"], g["k"], g["m1"], g["m2"], g["mu1"],
                            g["mu2"], g["T"], g["Phi"], g["Phib"], g["xi"], g["A1"] + g["A2"]))
    return [torch.cat([o[i] for o in out]).cpu().numpy() for i in range(2)]


def _A_aniso(m, mu, T, c1, c2, xi, L, np_=64, nc=4):
    (px, pw), (cx, cw) = _gl(0.0, 10.0, np_), np.polynomial.legendre.leggauss(nc)
    mk = lambda a: torch.tensor(a, device="cuda")  # noqa: E731
    p, w = mk(np.repeat(px, nc)), mk(np.repeat(pw * px ** 2, nc) * np.tile(cw, np_))
    x2 = mk(np.tile(cx ** 2, np_))
    col = lambda v: v[:, None]  # noqa: E731
    E0, E = torch.sqrt(p * p + col(m) ** 2), torch.sqrt(p * p * (1 + col(xi) * x2) + col(m) ** 2)
    f = 0.0
    for s, u, v in ((-1.0, c1, c2), (1.0, c2, c1)):
        e = torch.exp(-(E + s * col(mu)) / col(T)).clamp(1e-200, 1e200)
        f = f + (col(u) * e + 2 * col(v) * e ** 2 + e ** 3) / (1 + 3 * col(u) * e + 3 * col(v) * e ** 2 + e ** 3)
    s = torch.sqrt(L * L + m * m)
    return 2 * (w / E0 * f).sum(1) - 2 * (L * s - m * m * torch.log((L + s) / m))


def _pi_grid_exact(pts, k0, kk):
    pi, out = _Pi(), []
    T, mu, xi, mu_, ms_, c1, c2 = (pts[:, i] for i in range(7))
    A = [_A_aniso(m, mu, T, c1, c2, xi, pi.L) for m in (mu_, ms_)]
    K0, K = (v.reshape(-1) for v in torch.meshgrid(k0, kk, indexing="ij"))
    for i in range(pts.shape[0]):
        for pair, (a, b) in enumerate(((0, 0), (0, 1), (1, 1))):
            m = (mu_, ms_)
            e = lambda v: v[i].expand_as(K0)  # noqa: E731
            one = torch.ones_like(K0)
            res = [pi.value(ch * one, pair * one, 0 * one, K0, 0 * one, K, e(m[a]), e(m[b]), e(mu), e(mu), e(T), e(c1), e(c2),
                            e(xi), (A[a] + A[b])[i]) for ch in (1, 2)]
            out.append(torch.stack([torch.stack(r) for r in res]))
    v = torch.stack(out).reshape(pts.shape[0], 3, 2, 2, k0.numel(), kk.numel())
    return [v[:, :, :, j].contiguous() for j in range(2)]
