"""GPU parity of the anisotropic one-loop polarization (libpnjl_hip.so via
its C ABI) against the oracle's restatement of the reference quadrature,
on seeded random queries covering k = 0 / k > 0, poles, cuts, xi = 0 and
xi != 0, the three flavour pairs and both channels; and the hipGraph grid
(replayed, with other GPU work between replays).

Tolerance: 1e-9 relative to max(|Pi|, 1e-3 |Pi|_typ) -- both sides run the
same breakpoints and rules in unfused IEEE arithmetic; differences come from
last-bit exp/log results amplified by principal-value cancellation.  The
reference's singular lambda = k = 0 values (NaN or infinite) must match as
such."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _queries(n, seed=1):
    rng = np.random.default_rng(seed)
    k = rng.uniform(0, 3, n)
    k[rng.random(n) < 0.2] = 0.0
    xi = rng.uniform(-0.4, 0.4, n)
    xi[rng.random(n) < 0.3] = 0.0
    m1 = rng.uniform(0.01, 2.0, n)
    m2 = np.where(rng.random(n) < 0.3, m1, rng.uniform(0.01, 2.0, n))
    mu1 = rng.uniform(0, 2.3, n)
    mu2 = np.where(rng.random(n) < 0.5, mu1, rng.uniform(0, 2.3, n))
    cols = dict(channel=rng.choice([1, 2], n), num_s=rng.choice([0, 1, 2], n), width=(rng.random(n) < 0.2).astype(int),
                k0=rng.uniform(0, 4, n), gamma=rng.uniform(0, 0.5, n), k=k, m1=m1, m2=m2, mu1=mu1, mu2=mu2,
                T=rng.uniform(0.1, 1.5, n), Phi=rng.uniform(0, 1, n), Phib=rng.uniform(0, 1, n), xi=xi,
                A1=rng.uniform(-3, 0, n), A2=rng.uniform(-3, 0, n))
    return cols


def _close(g, o, rtol=1e-9):
    scale = np.maximum(np.abs(o), 1e-3 * np.nanmedian(np.abs(o)))
    both_nan = np.isnan(g) & np.isnan(o)
    with np.errstate(invalid="ignore"):
        return both_nan | (g == o) | (np.abs(g - o) <= rtol * scale)


def test_polarization_batch_matches_oracle(gpu_ctx, oracle):
    from julia_relaxtime_amd import polarization as P
    cols = _queries(3000)
    q = np.zeros(3000, dtype=P.QUERY_DTYPE)
    for f, v in cols.items():
        q[f] = v
    re, im = P.polarization_batch(q)
    oq = oracle.pol_queries(**cols)
    ore, oim = oracle.polarization_batch(oq)
    ok = _close(re, ore) & _close(im, oim)
    bad = np.flatnonzero(~ok)
    assert ok.all(), [(int(i), re[i], ore[i], im[i], oim[i]) for i in bad[:5]]
    assert np.isfinite(ore).mean() > 0.99


@pytest.mark.parametrize("n", [1, 2, 4096, 4097, 32769, 196609])
def test_lane_split_does_not_change_results(gpu_ctx, n):
    """A value does not depend on how many lanes its batch gives it: the lanes
    of a group add their terms in the one-lane order, bit for bit (sizes on
    both sides of each change of the split; 196 609 queries run on one lane
    each).  Queries of all forms, k = 0 and k > 0, equal and unequal masses and
    chemical potentials, and one with NaN and one with infinite inputs."""
    from julia_relaxtime_amd import polarization as P
    cols = _queries(512, 3)
    q = np.zeros(512, dtype=P.QUERY_DTYPE)
    for f, v in cols.items():
        q[f] = v
    q["mu1"][7] = np.nan
    q["k0"][9] = np.inf
    q["T"][11] = 1e-3
    ref = P.polarization_batch(np.resize(q, 200000))
    re, im = P.polarization_batch(np.resize(q, n))
    for g, r in ((re, ref[0]), (im, ref[1])):
        assert np.array_equal(g.view(np.int64), np.resize(r[:512], n).view(np.int64)) or \
            np.array_equal(g, np.resize(r[:512], n), equal_nan=True)


def test_B0_and_correction_batches_match_oracle(gpu_ctx, oracle):
    from julia_relaxtime_amd import polarization as P
    rng = np.random.default_rng(4)
    n = 1500
    lam = rng.uniform(-4, 4, n)
    k = np.where(rng.random(n) < 0.25, 0.0, rng.uniform(0, 3, n))
    m1, m2 = rng.uniform(0.01, 2, n), rng.uniform(0.01, 2, n)
    mu1, mu2 = rng.uniform(0, 2.3, n), rng.uniform(0, 2.3, n)
    T, Phi, Phib, xi = rng.uniform(0.1, 1.5, n), rng.uniform(0, 1, n), rng.uniform(0, 1, n), rng.uniform(-0.4, 0.4, n)
    re, im = P.B0_batch(np.stack([lam, k, m1, mu1, m2, mu2, T, Phi, Phib], 1))
    o = np.array([oracle.B0(*a) for a in zip(lam, k, m1, mu1, m2, mu2, T, Phi, Phib)])
    assert (_close(re, o[:, 0]) & _close(im, o[:, 1])).all()
    re, im = P.B0_correction_batch(np.stack([lam, k, m1, m2, mu1, mu2, T, Phi, Phib, xi], 1))
    o = np.array([oracle.B0_correction(*a) for a in zip(lam, k, m1, m2, mu1, mu2, T, Phi, Phib, xi)])
    assert (_close(re, o[:, 0]) & _close(im, o[:, 1])).all()


def test_A_batches_match_oracle(gpu_ctx, oracle):
    from julia_relaxtime_amd import polarization as P
    rng = np.random.default_rng(6)
    n = 400
    a = np.stack([rng.uniform(0, 2, n), rng.uniform(0, 2.3, n), rng.uniform(0.1, 1.5, n), rng.uniform(0, 1, n),
                  rng.uniform(0, 1, n), rng.uniform(-0.4, 0.4, n)], 1)
    xp, wp = np.polynomial.legendre.leggauss(64)
    xp, wp = 5 * (xp + 1), 5 * wp
    xc, wc = np.polynomial.legendre.leggauss(4)
    g = P.A_batch(a[:, :5], xp, wp)
    o = np.array([oracle.A(*r, xp, wp) for r in a[:, :5]])
    assert np.all(np.abs(g - o) <= 1e-12 * np.maximum(1, np.abs(o)))
    g = P.A_batch(a, xp, wp, xc, wc)
    o = np.array([oracle.A_aniso(*r, xp, wp, xc, wc) for r in a])
    assert np.all(np.abs(g - o) <= 1e-12 * np.maximum(1, np.abs(o)))


def _grid_oracle(oracle, pts, k0, k, npn=64, nc=4):
    xp, wp = np.polynomial.legendre.leggauss(npn)
    xp, wp = 5 * (xp + 1), 5 * wp
    xc, wc = np.polynomial.legendre.leggauss(nc)
    out = np.zeros((len(pts), 3, 2, k0.size, k.size), dtype=complex)
    for i, p in enumerate(pts):
        Au = oracle.A_aniso(p["m_u"], p["mu"], p["T"], p["Phi"], p["Phib"], p["xi"], xp, wp, xc, wc)
        As = oracle.A_aniso(p["m_s"], p["mu"], p["T"], p["Phi"], p["Phib"], p["xi"], xp, wp, xc, wc)
        for pair, (m1, m2, A1, A2) in enumerate(((p["m_u"], p["m_u"], Au, Au), (p["m_u"], p["m_s"], Au, As),
                                                 (p["m_s"], p["m_s"], As, As))):
            for c, ch in enumerate((1, 2)):
                for a, kk0 in enumerate(k0):
                    for b, kk in enumerate(k):
                        r = oracle.polarization(ch, kk0, kk, m1, m2, p["mu"], p["mu"], p["T"], p["Phi"], p["Phib"],
                                                p["xi"], A1, A2, pair)
                        out[i, pair, c, a, b] = complex(*r)
    return out


def test_polarization_grid_graph_replays_match_oracle(gpu_ctx, oracle):
    import torch
    from julia_relaxtime_amd import polarization as P
    rng = np.random.default_rng(9)
    k0 = np.linspace(0, 4, 6)
    k = np.linspace(0, 3, 5)

    def points(seed):
        r = np.random.default_rng(seed)
        p = np.zeros(3, dtype=P.POINT_DTYPE)
        p["T"], p["mu"], p["xi"] = r.uniform(0.2, 1.2, 3), r.uniform(0, 2, 3), [0.0, 0.3, -0.2]
        p["m_u"], p["m_s"] = r.uniform(0.02, 1.8, 3), r.uniform(0.5, 2.5, 3)
        p["Phi"], p["Phib"] = r.uniform(0, 1, 3), r.uniform(0, 1, 3)
        return p

    for rep, seed in enumerate((1, 1, 2, 1)):
        pts = points(seed)
        re, im = P.polarization_grid(pts, k0, k)
        # unrelated eager GPU work and a synchronisation between replays
        x = torch.randn(1 << 20, device="cuda", dtype=torch.float64)
        (x * 2).sum().item()
        o = _grid_oracle(oracle, pts, k0, k)
        assert _close(re, o.real).all() and _close(im, o.imag).all(), rep


def test_cache_semantics(gpu_ctx):
    from julia_relaxtime_amd import polarization as P
    P.reset_cache()
    args = ("P", 0.5, 0.3, 0.3, 0.5, 0.1, 0.1, 0.15, 0.3, 0.35, 0.2, -1.0, -1.2, 1)
    a = P.polarization_aniso_cached(*args)
    b = P.polarization_aniso_cached(*args)
    assert a == b
    near = list(args)
    near[1] = 0.5 * (1 + 2.0 ** -46)          # same 40-bit bucket: a hit, first value returned
    assert P.polarization_aniso_cached(*near) == a
    far = list(args)
    far[1] = 0.5 * (1 + 2.0 ** -30)
    P.polarization_aniso_cached(*far)
    s = P.get_cache_stats()
    assert (s["total_calls"], s["cache_hits"], s["cache_size"]) == (4, 2, 2)
    assert a == P.polarization_aniso(*args)
    with pytest.raises(ValueError):
        P.polarization_aniso("X", *args[1:])
