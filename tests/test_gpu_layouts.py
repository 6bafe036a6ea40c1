"""Bond layouts chosen by the build against the compact form: the same bonds
and, in FP64, the same bits."""
import numpy as np
import pytest

from cabanapd_amd import configs, engine
from cabanapd_amd._abi import PDK_BONDS_COMPACT, make_desc
from tests.parity import ctx, rel_err, say

pytestmark = pytest.mark.gpu


def run(w, precision, layout, steps=25):
    d = type(w["desc"]).from_buffer_copy(w["desc"])
    d.precision = precision
    d.bond_layout = layout
    s = engine.Spec(ctx(), d, w["x"].shape[0])
    configs.upload(s, w)
    configs.setup(s, w)
    s.step(steps)
    out = dict(bonds=s.bonds(), u=s.get("u"), v=s.get("v"), f=s.get("f"), layout=s.layout(), name=s.kernel_name(0))
    s.close()
    return out


def same(a, b, precision):
    for k in range(3):
        assert np.array_equal(a["bonds"][k], b["bonds"][k])
    for fld in ("u", "v", "f"):
        if precision == 0:
            assert np.array_equal(a[fld], b[fld]), fld
        else:
            assert rel_err(a[fld], b[fld]) <= 1e-6, fld


def box(model, dims, m, fracture, h=5e-4, seed=3):
    x, vol, _ = configs.grid_cell_centred([0, 0, 0], [h * k for k in dims], dims)
    kw = dict(horizon=m * h + 1e-10, K=4.3e10, dt=3e-8)
    if fracture:
        kw.update(fracture=True, G0=3.8)
    if model == "LPS":
        kw.update(G=2.9e10, influence=0)
    w = configs._base(make_desc(model, **kw), x, vol, 2440.0, "box", h, 25)
    rng = np.random.default_rng(seed)
    w["u"] = rng.uniform(-1, 1, size=x.shape) * 2e-4 * h
    w["v"] = rng.uniform(-1, 1, size=x.shape) * 3.0
    return w


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("m", [1, 2, 3])
@pytest.mark.parametrize("model", ["PMB", "LPS"])
def test_whole_number_horizons_take_stencil_slots(model, m, precision):
    """Horizons of m spacings (+ 1e-10): lattice vectors lie on the cutoff."""
    say(f"case: {model} 17x10x4, horizon {m} h + 1e-10, precision {precision}: slots vs compact")
    w = box(model, (17, 10, 4), m, True)
    a = run(w, precision, 0)
    b = run(w, precision, PDK_BONDS_COMPACT)
    assert a["layout"]["stencil_slots"] and not b["layout"]["stencil_slots"]
    assert (a["bonds"][2] == 0).any()
    same(a, b, precision)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["pmb", "lps", "epp", "materials", "thermal"])
def test_split_slices_match_gathers(kind, precision):
    """Specimens of few slices share each slice's rows among the waves of a
    block (8 up to 256 slices, 4 up to a limit, then one wave per slice):
    the gathers' bits on both sides of the lines, a part-filled last slice
    and one slice alone included."""
    for dims in ((4, 5, 3), (9, 9, 9), (16, 32, 32), (17, 31, 32), (32, 33, 66), (41, 41, 41), (44, 51, 73)):
        w = box("LPS" if kind in ("lps", "materials") else "PMB", dims, 3.01, True)
        d = w["desc"]
        n = w["x"].shape[0]
        rng = np.random.default_rng(5)
        if kind == "epp":
            d.mechanics, d.sigma_y = 1, 2.5e7
        if kind == "thermal":
            d.thermal, d.alpha, d.temp0 = 1, 1e-6, 20.0
            w["temperature"] = 20.0 + 40.0 * rng.random(n)
        if kind == "materials":
            w["materials"] = ([(4.3e10, 2.9e10, 3.8), (8e10, 5e10, 38.0)], (rng.random(n) < 0.4).astype(np.int32))
        d.precision = precision
        out = []
        for variant in (0, 4):
            s = engine.Spec(ctx(), d, n)
            configs.upload(s, w)
            configs.setup(s, w)
            s.set_tuning(variant)
            s.step(4)
            out.append([s.get("u"), s.get("v"), s.get("f"), s.bonds()[2], s.kernel_name(0)])
            s.close()
        say(f"case: {kind} {dims} precision {precision}: {(n + 63) // 64} slices, {out[0][4]} vs {out[1][4]}")
        assert "Rows" in out[0][4] and "Rows" not in out[1][4]
        for a, b in zip(out[0][:4], out[1][:4]):
            assert np.array_equal(a, b)
