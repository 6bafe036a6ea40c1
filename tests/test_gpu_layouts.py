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


def cut(w, dims, keep):
    """Keep the particles of a box (x fastest) where keep(i, j, k)."""
    k, j, i = np.meshgrid(*(np.arange(d) for d in dims[::-1]), indexing="ij")
    m = keep(i.ravel(), j.ravel(), k.ravel())
    for key in ("x", "vol", "rho", "u", "v"):
        w[key] = np.ascontiguousarray(w[key][m])
    return w


SHAPES = {
    "hole": ((40, 31, 6), lambda i, j, k: (i - 20) ** 2 + (j - 13) ** 2 > 49),
    "waist": ((251, 17, 5), lambda i, j, k: np.abs(j - 8) <= np.where(np.abs(i - 125) < 50, 3, 8)),
    "random": ((23, 19, 11), lambda i, j, k: np.random.default_rng(3).random(i.size) < 0.8),
    "sparse": ((25, 25, 9), lambda i, j, k: np.random.default_rng(4).random(i.size) < 0.2),
    "corner": ((33, 20, 12), lambda i, j, k: ~((i > 15) & (j > 8))),
    "comb": ((64, 20, 6), lambda i, j, k: (j % 5 > 1) | (i % 9 == 0)),
    "steps": ((150, 12, 4), lambda i, j, k: i < np.where(j < 6, 9, 150)),
}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["pmb", "pmb_elastic", "lps", "lps_elastic", "epp", "materials", "thermal"])
def test_missing_sites_match_compact(kind, precision):
    """Lattices with missing sites on row windows, one wave per slice and
    split, against the compact form and against the gathers over the same
    layout: the same bonds, bits (FP64) and output passes.  (steps, comb: windows
    longer than the passes stage; the build keeps the compact form.)"""
    big = ((120, 81, 20), lambda i, j, k: (i - 60) ** 2 + (j - 30) ** 2 > 400)
    for name, (dims, keep) in dict(SHAPES, big=big).items():
        w = box("LPS" if kind in ("lps", "lps_elastic", "materials") else "PMB", dims, 3.01,
                kind not in ("pmb_elastic", "lps_elastic", "thermal"))
        cut(w, dims, keep)
        d = w["desc"]
        n = w["x"].shape[0]
        rng = np.random.default_rng(6)
        if kind == "epp":
            d.mechanics, d.sigma_y = 1, 2.5e7
        if kind == "thermal":
            d.thermal, d.alpha, d.temp0, d.kappa, d.cp, d.thermal_subcycle = 2, 1e-6, 20.0, 10.0, 1.0, 2
            w["temperature"] = 20.0 + 40.0 * rng.random(n)
        if kind == "materials":
            w["materials"] = ([(4.3e10, 2.9e10, 3.8), (8e10, 5e10, 38.0)], (rng.random(n) < 0.4).astype(np.int32))
        d.precision = precision
        out = []
        for layout, variant in ((0, None), (PDK_BONDS_COMPACT, None), (0, 4)):
            d.bond_layout = layout
            s = engine.Spec(ctx(), d, n)
            configs.upload(s, w)
            configs.setup(s, w)
            if variant is not None:
                s.set_tuning(variant)
            s.step(5)
            s.compute_energy()
            s.compute_stress()
            out.append(dict(bonds=s.bonds(), name=s.kernel_name(0), lay=s.layout(),
                            **{f: s.get(f) for f in ("u", "v", "f", "W", "stress")}))
            s.close()
        say(f"case: {kind} {name} precision {precision}: {n} particles, {out[0]['name']}")
        assert ("Rows" in out[0]["name"]) == (name not in ("steps", "comb"))
        assert not out[0]["lay"]["stencil_slots"]
        for o in out[1:]:
            for b in range(3):
                assert np.array_equal(out[0]["bonds"][b], o["bonds"][b])
            for f in ("u", "v", "f", "W", "stress"):
                if precision == 0 or o is out[2]:
                    assert np.array_equal(out[0][f], o[f], equal_nan=True), f
                else:
                    assert rel_err(np.nan_to_num(out[0][f]), np.nan_to_num(o[f])) <= 1e-6, f


@pytest.mark.parametrize("precision", [0, 1])
def test_missing_sites_in_the_batch(precision):
    """Specimens with missing sites beside full ones in one batch: each as alone."""
    ws = []
    for name in ("hole", "corner", "random"):
        dims, keep = SHAPES[name]
        ws.append(cut(box("PMB", dims, 3.01, True), dims, keep))
    ws.append(box("PMB", (20, 21, 9), 3.01, True))
    ws.append(cut(box("LPS", (21, 20, 9), 3.01, True), (21, 20, 9), lambda i, j, k: i + j > 6))
    specs, alone = [], []
    for w in ws:
        w["desc"].precision = precision
        pair = []
        for _ in range(2):
            s = engine.Spec(ctx(), w["desc"], w["x"].shape[0])
            configs.upload(s, w)
            configs.setup(s, w)
            pair.append(s)
        pair[1].step(12)
        alone.append([pair[1].get(f) for f in ("u", "v", "f")])
        pair[1].close()
        specs.append(pair[0])
    for s in specs:
        ctx().submit(s, 12)
    ctx().progress()
    for s, ref in zip(specs, alone):
        for f, r in zip(("u", "v", "f"), ref):
            assert np.array_equal(s.get(f), r, equal_nan=True)
        s.close()


@pytest.mark.parametrize("shape", ["hole", "whole horizon"])
def test_tight_budgets_keep_the_compact_form(shape):
    """Where the HBM budget holds the compact form but not both forms at
    once, the build keeps the compact one instead of failing."""
    if shape == "hole":
        dims, keep = SHAPES["hole"]
        w = cut(box("PMB", dims, 3.01, True), dims, keep)
    else:
        w = box("PMB", (40, 31, 6), 3, True)
    n = w["x"].shape[0]

    def build(budget, layout):
        d = type(w["desc"]).from_buffer_copy(w["desc"])
        d.bond_layout = layout
        with engine.Context(0, budget) as c:
            s = None
            try:
                s = engine.Spec(c, d, n)
                configs.upload(s, w)
                configs.setup(s, w)
                s.step(3)
                return s.get("u"), s.kernel_name(0)
            except engine.PdkError:
                return None
            finally:
                if s is not None:
                    s.close()

    seen = set()
    for budget in np.geomspace(4e6, 4e7, 40).astype(int):
        compact, auto = build(int(budget), PDK_BONDS_COMPACT), build(int(budget), 0)
        if compact is None:
            continue
        assert auto is not None, f"budget {budget}"
        assert np.array_equal(auto[0], compact[0])
        seen.add("Rows" in auto[1])
    say(f"case: {shape}: row windows chosen over the budgets: {sorted(seen)}")
    assert seen == {False, True}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("model", ["PMB", "LPS"])
def test_kernel_names_tell_the_instance(model, precision):
    """Waves per slice and missing sites are part of the reported names: 8 up
    to 256 slices, 4 above, 1 on large specimens."""
    hole = lambda i, j, k: (i - 16) ** 2 + (j - 15) ** 2 > 49
    for dims, keep, waves in (((16, 32, 32), None, 8), ((17, 31, 32), None, 4), ((60, 60, 60), None, 1),
                              ((33, 30, 10), hole, 8), ((33, 30, 33), hole, 4), ((60, 60, 60), hole, 1)):
        w = box(model, dims, 3.01, True)
        if keep:
            cut(w, dims, keep)
        w["desc"].precision = precision
        s = engine.Spec(ctx(), w["desc"], w["x"].shape[0])
        configs.upload(s, w)
        configs.setup(s, w)
        tail = f"{waves}, {'true' if keep else 'false'}"
        m = {"PMB": 0, "LPS": 1}[model]
        say(f"case: {model} {dims} precision {precision}: {s.kernel_name(0)} {s.kernel_name(1)}")
        assert s.kernel_name(0) == f"kForceRows<{m}, true, {precision}, false, {tail}, {5 if waves > 1 else 1}>"
        if model == "LPS":
            assert s.kernel_name(1) == f"kLpsStateRows<true, {precision}, false, {tail}>"
        s.close()


def waves_of(s):
    return int(s.kernel_name(0).split("<")[1].split(",")[4])


LINES = {  # (kind, rows of a 1.5-spacing horizon, missing sites): four waves up to, FP64 and mixed
    ("pmb", False, False): (2560, 1024), ("pmb", True, False): (1536, 768), ("pmb", False, True): (1536, 1280),
    ("lps", False, False): (2560, 1536), ("lps", True, False): (1536, 1024), ("lps", False, True): (1792, 1024),
    ("materials", True, False): (1536, 1024), ("thermal", False, False): (1792, 1280),
    ("thermal", True, True): (768, 512), ("epp", False, True): (1792, 1536), ("epp", True, False): (1792, 1536),
}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind,short,hole", list(LINES))
def test_lines_of_split_launches(kind, short, hole, precision):
    """The size up to which four waves share a slice depends on the rows, the
    form and the precision: on both sides of each line, the gathers' bits."""
    line = LINES[kind, short, hole][precision]
    for slices, waves in ((line, 4), (line + 1, 1)):
        # layers of 8 x 8 = 64 particles; with a hole wider ones, cut off after
        # so many particles
        dims = (33, 32, slices // 14 + 2) if hole else (8, 8, slices)
        w = box("LPS" if kind in ("lps", "materials") else "PMB", dims, 1.5 if short else 3.01, True)
        if hole:
            cut(w, dims, lambda i, j, k: (i - 16) ** 2 + (j - 15) ** 2 > 36)
            for key in ("x", "vol", "rho", "u", "v"):
                w[key] = np.ascontiguousarray(w[key][:64 * slices])
        d = w["desc"]
        n = w["x"].shape[0]
        assert n == 64 * slices
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
        for variant in (None, 4):
            s = engine.Spec(ctx(), d, n)
            configs.upload(s, w)
            configs.setup(s, w)
            if variant is None:
                say(f"case: {kind} {slices} slices precision {precision}: {s.kernel_name(0)}")
                assert waves_of(s) == waves
            else:
                s.set_tuning(variant)
            s.step(3)
            out.append([s.get("u"), s.get("v"), s.get("f"), s.bonds()[2]])
            s.close()
        for a, b in zip(*out):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("shape,kind", [("hole", "epp"), ("whole horizon", "epp"), ("sparse", "epp"), ("sparse", "pmb"),
                                        ("hole", "pmb")])
def test_tight_budgets_hold_the_whole_run(shape, kind):
    """Wherever the HBM budget holds build, steps, stress and downloads over
    the compact form, the form that the build chooses gets through them too:
    the plastic stretches of its slots and the buffers of later calls count."""
    if shape == "whole horizon":
        w = box("PMB", (40, 31, 6), 3, True)
    else:
        dims, keep = SHAPES["hole"] if shape == "hole" else (
            (60, 50, 20), lambda i, j, k: np.random.default_rng(4).random(i.size) < 0.2)
        w = cut(box("PMB", dims, 3.01, True), dims, keep)
    d = type(w["desc"]).from_buffer_copy(w["desc"])
    if kind == "epp":
        d.mechanics, d.sigma_y = 1, 2.5e7
    n = w["x"].shape[0]

    def run(budget, layout):
        d.bond_layout = layout
        with engine.Context(0, budget) as c:
            s = None
            try:
                s = engine.Spec(c, d, n)
                configs.upload(s, w)
                configs.setup(s, w)
                s.step(3)
                s.compute_stress()
                s.set_body_force(np.zeros((n, 3)))
                return s.get("u"), s.get("stress"), s.kernel_name(0)
            except engine.PdkError:
                return None
            finally:
                if s is not None:
                    s.close()

    seen = set()
    for budget in np.geomspace(3e6, 6e7, 60).astype(int):
        compact, auto = run(int(budget), PDK_BONDS_COMPACT), run(int(budget), 0)
        if compact is None:
            continue
        assert auto is not None, f"budget {budget}"
        assert np.array_equal(auto[0], compact[0]) and np.array_equal(auto[1], compact[1], equal_nan=True)
        seen.add("Rows" in auto[2])
    say(f"case: {shape} {kind}, {n} particles: row windows chosen over the budgets: {sorted(seen)}")
    assert seen == {False, True}


@pytest.mark.parametrize("kind", ["pmb", "lps", "epp", "whole horizon"])
def test_copy_state_between_the_forms_memory_left(kind):
    """Two identical specimens of which the second finds no room for the slot
    form: state is copied both ways (broken bonds, plastic stretches), and each
    goes on with the other's bits.  Layouts asked for differently stay refused."""
    dims, keep = SHAPES["hole"]
    w = box("LPS" if kind == "lps" else "PMB", dims, 3 if kind == "whole horizon" else 3.01, True)
    if kind != "whole horizon":
        cut(w, dims, keep)
    d = w["desc"]
    if kind == "epp":
        d.mechanics, d.sigma_y = 1, 2.5e7
    n = w["x"].shape[0]

    def made(c, layout=0):
        d.bond_layout = layout
        s = engine.Spec(c, d, n)
        configs.upload(s, w)
        configs.setup(s, w)
        return s

    with engine.Context(0) as c:
        a = made(c)
        one = c.bytes_in_use()
        b = made(c, PDK_BONDS_COMPACT)
        two = c.bytes_in_use()
        assert "Rows" in a.kernel_name(0) and "Rows" not in b.kernel_name(0)
        with pytest.raises(engine.PdkError):
            b.copy_state_from(a)
        a.close()
        b.close()
    with engine.Context(0, two + 150 * n) as c:
        a, b = made(c), made(c)
        say(f"case: {kind}, {n} particles: {one} and {two - one} B; {a.kernel_name(0)} and {b.kernel_name(0)}")
        assert "Rows" in a.kernel_name(0) and "Rows" not in b.kernel_name(0)
        for src, dst in ((a, b), (b, a)):
            src.step(6)
            dst.copy_state_from(src)
            for k in range(3):
                assert np.array_equal(src.bonds()[k], dst.bonds()[k])
            assert (src.bonds()[2] == 0).any()
            src.step(5)
            dst.step(5)
            for f in ("u", "v", "f"):
                assert np.array_equal(src.get(f), dst.get(f)), f
            src.step(2)
        a.close()
        b.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_row_windows_can_be_chosen_on_missing_sites(precision):
    """Every pass that pdk_autotune may choose can be set, the row windows of a
    lattice with missing sites as well, before and after the gathers; a
    specimen in the compact form still refuses them."""
    dims, keep = SHAPES["hole"]
    w = cut(box("PMB", dims, 3.01, True), dims, keep)
    w["desc"].precision = precision
    out, names = [], []
    for tune in ((), (4,), (4, 0), (0,)):
        s = engine.Spec(ctx(), w["desc"], w["x"].shape[0])
        configs.upload(s, w)
        configs.setup(s, w)
        for t in tune:
            s.set_tuning(t)
        s.step(6)
        out.append([s.get(f) for f in ("u", "v", "f")])
        names.append(s.kernel_name(0))
        best = s.autotune()
        s.set_tuning(best)
        s.close()
    say(f"case: missing sites, precision {precision}: {names}")
    assert names[2] == names[3] == names[0] and "Rows" in names[0] and "Rows" not in names[1]
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)
    w["desc"].bond_layout = PDK_BONDS_COMPACT
    s = engine.Spec(ctx(), w["desc"], w["x"].shape[0])
    configs.upload(s, w)
    configs.setup(s, w)
    with pytest.raises(engine.PdkError):
        s.set_tuning(0)
    s.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_spec_bytes_hold_the_forms_tables(precision):
    """What a specimen reports to hold differs between the forms by what its
    context has in use."""
    dims, keep = SHAPES["hole"]
    for w in (cut(box("PMB", dims, 3.01, True), dims, keep), box("PMB", (40, 31, 6), 3, True)):
        d = w["desc"]
        d.precision = precision
        held, used = [], []
        for layout in (0, PDK_BONDS_COMPACT):
            d.bond_layout = layout
            with engine.Context(0) as c:
                s = engine.Spec(c, d, w["x"].shape[0])
                configs.upload(s, w)
                configs.setup(s, w)
                held.append(s.bytes())
                used.append(c.bytes_in_use())
                s.close()
        say(f"case: precision {precision}, {w['x'].shape[0]} particles: held {held}, in use {used}")
        assert held[0] != held[1]
        assert abs((held[0] - held[1]) - (used[0] - used[1])) <= 4096


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind,most", [("pmb", (1.75, 2.4)), ("lps", (2.1, np.inf)), ("epp", (1.4, 1.4)),
                                       ("heat", (1.4, 1.4))])
def test_sparse_lattices_take_the_faster_form(kind, most, precision):
    """Large boxes with sites missing at random: the slot form where its slots
    with a bond are at most so many per row of the compact form, the compact
    form beyond (its row passes would run with few lanes live); the same bits."""
    dims = (60, 60, 40)
    seen = set()
    for fill in (0.2, 0.45, 0.6, 0.75):
        w = box("LPS" if kind == "lps" else "PMB", dims, 3.01, kind != "heat")
        cut(w, dims, lambda i, j, k: np.random.default_rng(9).random(i.size) < fill)
        d = w["desc"]
        n = w["x"].shape[0]
        if kind == "epp":
            d.mechanics, d.sigma_y = 1, 2.5e7
        if kind == "heat":
            d.thermal, d.alpha, d.temp0, d.kappa, d.cp, d.thermal_subcycle = 2, 1e-6, 20.0, 10.0, 1.0, 2
            w["temperature"] = 20.0 + 40.0 * np.random.default_rng(6).random(n)
        d.precision = precision
        out = []
        for layout in (0, PDK_BONDS_COMPACT):
            d.bond_layout = layout
            s = engine.Spec(ctx(), d, n)
            configs.upload(s, w)
            configs.setup(s, w)
            s.step(3)
            out.append(s.bonds() + (s.get("u"), s.kernel_name(0)))
            s.close()
        slices = (n + 63) // 64
        cnt = np.pad(np.diff(out[0][0]), (0, slices * 64 - n)).reshape(slices, 64)
        ratio = 122 * slices / cnt.max(1).sum()  # every slot has a bond in some lane here
        rows = "Rows" in out[0][4]
        say(f"case: {kind} precision {precision} fill {fill}: {slices} slices, {ratio:.2f} slots a row, {out[0][4]}")
        assert rows == (ratio <= most[precision])
        seen.add(rows)
        for b in range(3):
            assert np.array_equal(out[0][b], out[1][b])
        if precision == 0:
            assert np.array_equal(out[0][3], out[1][3])
        else:
            assert rel_err(out[0][3], out[1][3]) <= 1e-6
    assert True in seen
