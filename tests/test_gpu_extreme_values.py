"""FP64 row passes at values where their shared-reciprocal arithmetic must
hand over to the general code: displacements far below the spacing (down to
subnormal), bonds whose length is the double just below a power of two times
the spacing (the one mantissa whose reciprocal the fast form does not round
correctly), particles on top of each other (|r| = 0), and huge or non-finite
displacements.  Every result equals the oracle's bit for bit (NaN where it
has NaN)."""
import numpy as np
import pytest

from cabanapd_amd import configs, engine
from cabanapd_amd._abi import make_desc
from tests.parity import ctx, pair, say

pytestmark = pytest.mark.gpu

N = 9
H = 1.0 / 64.0  # a power of two: bond vectors along the axes are exact


def workload(kind, seed, wild):
    x, vol, _ = configs.grid_node_centred(N, H)
    rng = np.random.default_rng(seed)
    n = x.shape[0]
    sizes = np.array([0.0, 5e-324, 1e-310, 1e-200, 1e-40, 2.0 ** -59, 2.0 ** -58, 1e-9, 1e-5])
    u = rng.choice(sizes, size=(n, 3)) * rng.choice([-1.0, 1.0], size=(n, 3))
    u[rng.random(n) < 0.4] = 0.0
    if wild:
        c = (N // 2) * (1 + N + N * N)
        u[c] = [-H, 0.0, 0.0]              # onto its neighbour
        u[c + 1 + N] = [H, 0.0, 1e-200]    # onto the next one but for a tiny offset
        u[3] = [1e180, 0.0, 0.0]
        u[N * N * N - 4] = [np.inf, 1.0, 0.0]
    kw = dict(horizon=3.01 * H, K=2e9, dt=1e-9)
    model = "PMB"
    frac = kind in ("pmb_fracture", "lps_fracture", "epp", "materials")
    if frac:
        kw.update(fracture=True, G0=0.5)
    if kind.startswith("lps"):
        model = "LPS"
        kw.update(G=1.1e9, influence=1 if kind == "lps_influence1" else 0)
    if kind == "epp":
        kw.update(mechanics="epp", sigma_y=1e5)
    if kind == "heat":
        kw.update(thermal="dynamic", alpha=1e-5, temp0=0.0, kappa=1.0, cp=1.0, thermal_subcycle=1)
    w = configs._base(make_desc(model, **kw), x, vol, 1000.0, "extreme_" + kind, H, 2)
    w["u"] = u
    if kind == "heat":
        w["temperature"] = rng.choice([0.0, 1e-320, 1e-200, 1e-20, 1.0, 30.0], size=n)
    if kind == "materials":
        w["materials"] = ([(2e9, 1.1e9, 0.5), (5e9, 2e9, 2.0)], (rng.random(n) < 0.5).astype(np.int32))
    return w


def same(a, b, what):
    a, b = np.asarray(a), np.asarray(b)
    bad = (a != b) & ~(np.isnan(a) & np.isnan(b))
    assert not bad.any(), f"{what}: {int(bad.sum())} values differ"


@pytest.mark.parametrize("wild", [False, True])
@pytest.mark.parametrize("kind", ["pmb", "pmb_fracture", "lps", "lps_influence1", "lps_fracture", "epp", "materials",
                                  "heat"])
def test_extreme_displacements_match_oracle(kind, wild):
    say(f"case: {kind}, {N}^3 FP64, tiny to subnormal displacements, wild={wild}")
    w = workload(kind, 17, wild)
    g, o = pair(w)
    assert "Rows" in g.kernel_name(0)
    for fld in ("f", "W"):
        same(g.get(fld), o.get(fld), fld + " at init")
    g.compute_stress()
    o.compute_stress()
    same(g.get("stress"), o.get("stress"), "stress")
    g.step(2)
    o.step(2)
    for fld in ("u", "v", "f") + (("m", "theta") if kind.startswith("lps") else ()) + (
            ("temperature",) if kind == "heat" else ()):
        same(g.get(fld), o.get(fld), fld)
    assert np.array_equal(g.bonds()[2], o.bonds()[2])
    g.close()


@pytest.mark.parametrize("kind", ["pmb", "pmb_fracture", "lps", "lps_influence1", "lps_fracture", "epp", "epp_tiny",
                                  "materials", "heat"])
def test_fading_displacements_match_oracle(kind):
    """A front's tail: displacements (and temperatures) that fade from 1e-7 of
    the spacing through both sides of the limit of the fast form (2^-400 = 4e-121
    at most) to subnormal, one component far smaller than the others; with
    epp_tiny a yield stretch below the fast form's range."""
    say(f"case: {kind}, {N}^3 FP64, displacements fading over 300 powers of ten")
    w = workload("epp" if kind == "epp_tiny" else kind, 5, False)
    rng = np.random.default_rng(8)
    n = w["x"].shape[0]
    fade = 10.0 ** -np.interp(np.arange(n), [0, n // 3, n - 1], [9, 130, 322])
    scale = rng.choice([1.0, 1e-3, 1e-60, 0.0], size=(n, 3), p=[0.5, 0.2, 0.2, 0.1])
    w["u"] = rng.uniform(-1, 1, size=(n, 3)) * fade[:, None] * scale
    w["u"][:, 0] += 1e-6 * H * rng.uniform(-1, 1, size=n)  # every bond along x carries force
    if kind == "epp_tiny":
        w["desc"].sigma_y = 1e-290
    if kind == "heat":
        w["temperature"] = rng.uniform(-1, 1, size=n) * fade[::-1]
    g, o = pair(w)
    for fld in ("f", "W"):
        same(g.get(fld), o.get(fld), fld + " at init")
    g.compute_stress()
    o.compute_stress()
    same(g.get("stress"), o.get("stress"), "stress")
    g.step(3)
    o.step(3)
    for fld in ("u", "v", "f") + (("m", "theta") if kind.startswith("lps") else ()) + (
            ("temperature",) if kind == "heat" else ()):
        same(g.get(fld), o.get(fld), fld)
    assert np.array_equal(g.bonds()[2], o.bonds()[2])
    g.close()


@pytest.mark.parametrize("model", ["PMB", "LPS"])
def test_fading_displacements_keep_the_fast_rows(model):
    """Small values that a front leaves ahead of it (down to 1e-100) in rows
    that carry force do not send them through the general code: the force pass
    takes the time that it takes without them (evaluating the rows twice took
    1.6 times as long)."""
    h = 5e-4
    x, vol, _ = configs.grid_cell_centred([0, 0, 0], [64 * h, 64 * h, 64 * h], (64, 64, 64))
    kw = dict(horizon=3.01 * h, K=4.3e10, dt=1e-9, fracture=True, G0=3.8e3)
    if model == "LPS":
        kw.update(G=2.9e10, influence=0)
    w = configs._base(make_desc(model, **kw), x, vol, 2440.0, "fading", h, 25)
    n = x.shape[0]
    rng = np.random.default_rng(2)
    full = rng.uniform(-1, 1, size=(n, 3)) * 1e-6 * h
    tails = full.copy()
    tails[:, 1:] *= 10.0 ** -rng.uniform(40, 90, size=(n, 1))
    s = engine.Spec(ctx(), w["desc"], n)
    best = {}
    for name, u in (("full", full), ("tails", tails)):
        w["u"] = u
        configs.upload(s, w)
        configs.setup(s, w)
        best[name] = np.inf
        for _ in range(5):
            s.timing(True)
            s.compute_force()
            best[name] = min(best[name], s.kernel_time(0)[0])
        s.timing(False)
    say(f"case: {model}, {n} particles, force pass {best['full']:.4f} ms, with tails {best['tails']:.4f} ms")
    assert best["tails"] < 1.25 * best["full"]
    s.close()


@pytest.mark.parametrize("where", ["current", "reference", "both"])
@pytest.mark.parametrize("model", ["PMB", "LPS"])
def test_lengths_near_powers_of_two_match_oracle(model, where):
    """Bond lengths (current, reference) within 16 ulp of powers of two, where
    a reciprocal's last bit is the hardest: roots and quotients of 3e6 bonds
    through the shared reciprocals, the oracle's bits."""
    n_side = 29
    ulp = 2.0 ** -58  # of the doubles from 1/64 on; half as much below
    x, vol, _ = configs.grid_node_centred(n_side, H)
    n = x.shape[0]
    rng = np.random.default_rng(11)
    u = rng.uniform(-1, 1, size=(n, 3)) * 1e-9 * H
    if where in ("current", "both"):
        u[:, 0] = rng.integers(-16, 17, size=n) * ulp / 2
    else:
        u[:, 0] += rng.uniform(-1, 1, size=n) * 1e-4 * H
    if where in ("reference", "both"):
        x[:, 0] += rng.integers(-8, 9, size=n) * np.spacing(np.maximum(x[:, 0], H))
    kw = dict(horizon=3.01 * H, K=2e9, dt=1e-9)
    if model == "LPS":
        kw.update(G=1.1e9, influence=0)
    w = configs._base(make_desc(model, **kw), x, vol, 1000.0, "near_powers", H, 2)
    w["u"] = u
    g, o = pair(w)
    say(f"case: {model}, {where} lengths near powers of two, {n} particles, {g.bond_stats()[0]} bonds, "
        f"{g.kernel_name(0)}")
    assert "Rows" in g.kernel_name(0)
    for fld in ("f", "W") + (("m", "theta") if model == "LPS" else ()):
        same(g.get(fld), o.get(fld), fld + " at init")
    g.compute_stress()
    o.compute_stress()
    same(g.get("stress"), o.get("stress"), "stress")
    g.step(2)
    o.step(2)
    for fld in ("u", "v", "f"):
        same(g.get(fld), o.get(fld), fld)
    g.close()
