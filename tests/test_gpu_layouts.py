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
