"""The one-launch half-step (update, CPML slabs, TFSF and lumped corrections,
probes) against a launch per correction, which the parity tests hold to the
oracle bitwise: the same bits in FP64 and in FP32, whose sums every kernel writes
out alike."""

import ctypes

import numpy as np
import pytest

from oracle import RefSim
from xfdtd_core_amd import native
from xfdtd_core_amd import spec as S

pytestmark = pytest.mark.gpu
FIELDS = ("EX", "EY", "EZ", "HX", "HY", "HZ")


def _box(n, pml=6, faces=("XN", "XP", "YN", "YP", "ZN", "ZP"), tfsf=True):
    """n cells including the CPML: a lossy sphere, an inductor and a dipole,
    a TFSF box and probes on both sides of it."""
    dl = 1e-3
    inner = [m - 2 * pml for m in n]
    s = S.Simulation(dl, dl, dl, 0.9)
    size = S.Vector(*[m * dl for m in inner])
    s.addObject(S.Object("domain", S.Cube(S.Vector(0, 0, 0), size), S.Material.createAir()))
    mid = [m / 2 * dl for m in inner]
    s.addObject(S.Object("ball", S.Sphere(S.Vector(*mid), 3 * dl),
                         S.Material("m", S.ElectroMagneticProperty(3.0, 1.0, 0.02, 0.0))))
    cell = [m // 2 * dl for m in inner]
    s.addObject(S.Inductor("l", S.Cube(S.Vector(cell[0] - 2 * dl, cell[1], cell[2]), S.Vector(0, 0, 2 * dl)), "Z",
                           1e-9))
    s.addObject(S.CurrentSource("d", S.Cube(S.Vector(*cell), S.Vector(0, 0, dl)), "ZP", 1e12,
                                S.Waveform.gaussian(20e-12, 40e-12)))
    if tfsf:
        s.addWaveformSource(S.TFSF3D(pml + 2, pml + 2, pml + 2, 0.7, 0.4, 0.3, S.Waveform.gaussian(20e-12, 40e-12)))
    for f in faces:
        s.addBoundary(S.PML(pml, f))
    for q, (c, comp) in enumerate(((0, "EZ"), (1, "HY"), (2, "EX"))):
        at = [min(3 + 2 * c, m - 2) * dl for m in inner]
        s.addMonitor(S.FieldTimeMonitor(f"p{q}", S.Cube(S.Vector(*at), S.Vector(dl, dl, dl)), "", comp))
    return s.spec()


def _run(monkeypatch, spec, precision, steps, on, chunk=None, z_inside=False):
    monkeypatch.setenv("XFD_CPML_INSWEEP", "1" if on else "0")
    if z_inside:  # the default: long FP32 rows correct z first, in the sweeps or in the one launch
        monkeypatch.delenv("XFD_CPML_ZFUSED", raising=False)
    else:
        monkeypatch.setenv("XFD_CPML_ZFUSED", "0")
    if chunk:
        monkeypatch.setenv("XFD_ICHUNK", str(chunk))
    sim = native.Simulation(spec, precision)
    sim.init(steps)
    assert sim.cpml_fused() == (4 if on else 2 if z_inside else 0)
    return sim


def _compare(a, b, precision, label):
    for f in FIELDS:
        x, y = a.field(f), b.field(f)
        assert np.abs(y).max() > 0
        np.testing.assert_array_equal(x, y, err_msg=f"{label} {precision} {f}")


# nz around the 64- and 128-lane tiles, ny off the 4-row tile, nx off the chunk
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n,chunk", [((23, 22, 63), None), ((24, 25, 65), 3), ((21, 23, 128), 4),
                                     ((22, 21, 129), 1), ((30, 26, 24), 64)])
def test_half_step_matches_separate_launches(monkeypatch, n, chunk, precision):
    spec, steps = _box(n), 50
    a = _run(monkeypatch, spec, precision, steps, True, chunk)
    b = _run(monkeypatch, spec, precision, steps, False, chunk)
    for sim in (a, b):
        sim.advance(0, 20)
        sim.advance(20, steps - 20)
        sim.finish()
    _compare(a, b, precision, f"{n} {chunk}")
    for m in range(a.monitor_count()):
        for x, y in zip(a.monitor_records(m), b.monitor_records(m)):
            np.testing.assert_array_equal(x, y)


# FP32 rows of three k-tiles and up: the z corrections precede the x and y ones
@pytest.mark.parametrize("faces", [("XN", "XP", "YN", "YP", "ZN", "ZP"), ("ZN", "ZP", "YP", "YN", "XN", "XP"),
                                   ("YN", "ZP", "XP", "XN")])
def test_half_step_order_of_long_fp32_rows(monkeypatch, faces):
    spec, steps = _box((22, 21, 140), faces=faces, tfsf=len(faces) == 6), 60
    a = _run(monkeypatch, spec, "f32", steps, True, z_inside=True)
    b = _run(monkeypatch, spec, "f32", steps, False, z_inside=True)
    for sim in (a, b):
        sim.advance(0, steps)
        sim.finish()
    _compare(a, b, "f32", str(faces))


# the slabs' order decides which correction a point of two slabs adds first
@pytest.mark.parametrize("faces", [("ZN", "ZP", "YP", "YN", "XN", "XP"), ("YN", "XP", "XN"), ("ZP",), ()])
def test_half_step_slab_orders(monkeypatch, faces):
    spec, steps = _box((26, 24, 30), faces=faces, tfsf=len(faces) == 6), 40
    a = _run(monkeypatch, spec, "f64", steps, True)
    b = _run(monkeypatch, spec, "f64", steps, False)
    for sim in (a, b):
        sim.advance(0, steps)
        sim.finish()
    _compare(a, b, "f64", str(faces))


def test_half_step_refuses_interleaved_slabs(monkeypatch):
    """Slabs whose axes interleave in boundary order have no order per axis
    pair: they keep a launch each."""
    monkeypatch.setenv("XFD_CPML_INSWEEP", "1")
    sim = native.Simulation(_box((26, 24, 30), faces=("XN", "YN", "ZN", "XP", "YP", "ZP")), "f64")
    sim.init(2)
    assert sim.cpml_fused() == 0


def test_half_step_far_planes(monkeypatch):
    """Values written on the far planes take their slab corrections."""
    spec, steps = _box((26, 24, 30)), 30
    runs = []
    for on in (True, False):
        sim = _run(monkeypatch, spec, "f64", steps, on)
        ctx, L = sim.device_context(), native.load_library()
        sim.advance(0, 5)
        rng = np.random.default_rng(3)
        for q, ext in ((0, (26, 25, 31)), (5, (26, 24, 31)), (2, (27, 25, 30))):
            v = np.ascontiguousarray(rng.standard_normal(ext))
            assert L.xfd_write_field(ctypes.c_void_p(ctx), q, v.ctypes.data) == 0
        sim.advance(5, steps - 5)
        sim.finish()
        runs.append(sim)
    _compare(*runs, "f64", "far planes")
    assert np.abs(runs[0].field("EX")[:, :, -1]).max() > 0


def _plane(nx, ny, faces=("XN", "XP", "YN", "YP"), pml=6, tfsf=12):
    """A 2D grid of nx x ny cells including the CPML: a lossy cylinder in a
    plane wave, probes and a movie."""
    inf, dl = float("inf"), 1e-3
    inner = [nx - sum(pml for f in faces if f[0] == "X"), ny - sum(pml for f in faces if f[0] == "Y")]
    s = S.Simulation(dl, dl, 1.0, 0.9)
    size = [m * dl for m in inner]
    s.addObject(S.Object("domain", S.Cube(S.Vector(0, 0, -inf), S.Vector(*size, inf)), S.Material.createAir()))
    s.addObject(S.Object("rod", S.Cylinder(S.Vector(size[0] / 2, size[1] / 2, -inf), 4 * dl, inf, "Z"),
                         S.Material("m", S.ElectroMagneticProperty(3.0, 1.0, 0.02, 0.0))))
    s.addWaveformSource(S.TFSF2D(tfsf, tfsf, 0.6, S.Waveform.gaussian(20e-12, 60e-12)))
    for f in faces:
        s.addBoundary(S.PML(pml, f))
    for q, (at, comp) in enumerate((((1, 1), "EZ"), ((inner[0] // 2, inner[1] // 2), "HX"),
                                    ((inner[0] - 1, inner[1] - 1), "EZ"))):
        s.addMonitor(S.FieldTimeMonitor(f"p{q}", S.Cube(S.Vector(at[0] * dl, at[1] * dl, -inf), S.Vector(dl, dl, inf)),
                                        "", comp))
    s.addMonitor(S.MovieMonitor(S.FieldMonitor(S.Cube(S.Vector(0, 0, -inf), S.Vector(*size, inf)), "EZ"), 9, "movie",
                                ""))
    return s.spec()


# ny around the 64 lanes, nx around the 4 wavefronts and their rows, slab orders
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,chunk,faces", [(37, 63, None, ("XN", "XP", "YN", "YP")),
                                               (33, 65, 3, ("YP", "YN", "XP", "XN")), (40, 128, 16, ("YN", "XP")),
                                               (64, 33, 1, ())])
def test_plane_half_step(monkeypatch, nx, ny, chunk, faces, precision):
    spec, steps = _plane(nx, ny, faces), 120
    runs = []
    for on in (True, False):
        sim = _run(monkeypatch, spec, precision, steps, on, chunk)
        sim.advance(0, 50)
        sim.advance(50, steps - 50)
        sim.finish()
        runs.append(sim)
    a, b = runs
    for f in FIELDS:
        np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
    for m in range(a.monitor_count()):
        for x, y in zip(a.monitor_records(m), b.monitor_records(m)):
            np.testing.assert_array_equal(x, y)
    assert np.abs(b.field("EZ")).max() > 0


def test_plane_half_step_after_writes(monkeypatch):
    """A field that no longer stays zero takes a 2D grid off the one launch."""
    spec, steps = _plane(40, 44), 40
    runs = []
    for on in (True, False):
        sim = _run(monkeypatch, spec, "f64", steps, on)
        sim.advance(0, 10)
        rng = np.random.default_rng(5)
        for q, ext in ((2, (41, 45, 1)), (5, (40, 44, 2))):
            v = np.ascontiguousarray(rng.standard_normal(ext))
            assert native.load_library().xfd_write_field(ctypes.c_void_p(sim.device_context()), q, v.ctypes.data) == 0
        sim.advance(10, steps - 10)
        sim.finish()
        runs.append(sim)
    _te = [np.abs(runs[0].field(f) - runs[1].field(f)).max() for f in FIELDS]
    assert _te == [0] * 6


@pytest.mark.parametrize("on", [True, False])
def test_fp32_keeps_the_field_product_unrounded(monkeypatch, on):
    """E = s E + a d with s != 1: the product s E, the larger one, is not rounded
    by itself, so one step is within the one rounding of its result (half a unit
    in the last place) and that of a d (2^-24 of it)."""
    monkeypatch.setenv("XFD_CPML_INSWEEP", "1" if on else "0")
    n, rng = (9, 11, 70), np.random.default_rng(1)
    ext = {c: tuple(m + (1 if (q != "xyz".index(c[0]) if c[1] == "e" else q == "xyz".index(c[0])) else 0)
                    for q, m in enumerate(n)) for c in ("xe", "ye", "ze", "xh", "yh", "zh")}
    f32 = lambda v: v.astype(np.float32).astype(np.float64)  # noqa: E731
    coeffs = {name: np.full(ext[name[2] + name[1]], 1.0 if name[1] == name[3] else 0.0) for name in native.COEFF_NAMES}
    s, a = (f32(rng.choice(v, ext["xe"])) for v in ((0.7, 0.9, 0.99), (0.013, 0.021)))
    coeffs["cexe"], coeffs["cexhy"] = s, a
    ctx = native.Context(coeffs, "f32")
    e, h = f32(rng.standard_normal(ext["xe"])), f32(rng.standard_normal(ext["yh"]))
    ctx.write("EX", e)
    ctx.write("HY", h)
    ctx.step(0, 1)
    got = ctx.read("EX")[:, 1:-1, 1:-1]
    ad = a[:, 1:-1, 1:-1] * f32(np.diff(h, axis=2))[:, 1:-1]
    want = s[:, 1:-1, 1:-1] * e[:, 1:-1, 1:-1] + ad
    unit = np.spacing(np.maximum(np.abs(got), np.abs(want)).astype(np.float32))
    assert (np.abs(got - want) <= 0.5 * unit + 2.0**-24 * np.abs(ad)).all()
    assert np.abs(got - e[:, 1:-1, 1:-1]).max() > 0


def _poles(kind, n):
    """A material of n poles; the modified Lorentz scheme also where kinds mix."""
    w = [2e10 * (1 + 0.7 * p) for p in range(n)]
    if kind == "drude":
        return S.DrudeMedium.makeDrudeMedium("d", 2.0, [0.6 * v for v in w], [1e9 * (1 + p) for p in range(n)])
    if kind == "debye":
        return S.DebyeMedium.makeDebyeMedium("d", 2.0, [3.0 + p for p in range(n)], [1e-11 * (1 + p) for p in range(n)])
    return S.LorentzMedium.makeMLorentz("d", 2.0, [0.4 * v * v for v in w], [2e9] * n, [v * v for v in w],
                                        [2e9 * (1 + p) for p in range(n)], [1.0] * n)


# room for two poles, for four, and the loop over more
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("kind", ["drude", "debye", "lorentz"])
def test_dispersive_half_step(monkeypatch, kind, n):
    """A dispersive block in a driven box: FP64 the oracle's bits, and in both
    precisions those of a launch per correction, of all of them or of the E
    half-step's alone (the arrangement of large grids)."""
    dl, pml, inner, steps = 1e-3, 5, (14, 13, 60), 60
    s = S.Simulation(dl, dl, dl, 0.9)
    s.addObject(S.Object("domain", S.Cube(S.Vector(0, 0, 0), S.Vector(*[m * dl for m in inner])),
                         S.Material.createAir()))
    s.addObject(S.Object("block", S.Cube(S.Vector(0, 4 * dl, 10 * dl), S.Vector(14 * dl, 5 * dl, 30 * dl)),
                         _poles(kind, n)))
    s.addObject(S.CurrentSource("i", S.Cube(S.Vector(7 * dl, 2 * dl, 9 * dl), S.Vector(0, 0, dl)), "ZP", 1e3,
                                S.Waveform.gaussian(10e-12, 20e-12)))
    for f in ("XN", "XP", "YN", "YP", "ZN", "ZP"):
        s.addBoundary(S.PML(pml, f))
    spec = s.spec()
    ref = RefSim(spec)
    ref.run(steps)
    for precision in ("f64", "f32"):
        a = _run(monkeypatch, spec, precision, steps, True)
        b = _run(monkeypatch, spec, precision, steps, False)
        for sim in (a, b):
            sim.advance(0, steps)
            sim.finish()
        _compare(a, b, precision, f"{kind} {n}")
        with monkeypatch.context() as m:
            m.setenv("XFD_ADE_E", "apart")
            e = _run(m, spec, precision, steps, True)
            e.set_profiling(True)
            e.advance(0, steps)
            e.finish()
            launches = {k: v[0] for k, v in e.kernel_stats().items()}
            assert launches.get("cpml_h", 0) == 0 and launches["cpml_e"] > 0
        _compare(e, b, precision, f"{kind} {n} E apart")
        if precision == "f64":
            for f in FIELDS:
                np.testing.assert_array_equal(a.field(f), ref.field(f), err_msg=f)


# where the one launch loses: FP32 rows of whole 128-lane tiles past 128 MiB
@pytest.mark.parametrize("n,mode", [((130, 130, 256), 0), ((130, 130, 250), 4), ((64, 64, 128), 4)])
def test_large_dispersive_grids_keep_separate_launches(n, mode):
    dl = 1e-3
    s = S.Simulation(dl, dl, dl, 0.9)
    s.addObject(S.Object("domain", S.Cube(S.Vector(0, 0, 0), S.Vector(*[m * dl for m in n])), S.Material.createAir()))
    s.addObject(S.Object("block", S.Cube(S.Vector(0, 0, 0), S.Vector(9 * dl, 9 * dl, 9 * dl)), _poles("debye", 1)))
    sim = native.Simulation(s.spec(), "f32")
    sim.init(1)
    assert sim.cpml_fused() == mode


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("layout", ["classed", "wide", "dense"])
def test_half_step_coefficient_layouts(monkeypatch, layout, precision):
    """16-bit class ids, 32-bit ones (80000 distinct triples a component) and
    dense coefficients: the bits of a launch per correction."""
    n, rng = (70, 66, 75), np.random.default_rng(2)
    monkeypatch.setenv("XFD_COEF_MODE", "dense" if layout == "dense" else "")
    classes = 80000 if layout == "wide" else 50
    coeffs = {}
    for name in native.COEFF_NAMES:
        c, e = "xyz".index(name[2]), name[1] == "e"
        ext = tuple(m + (1 if (q == c) != e else 0) for q, m in enumerate(n))
        if len(name) == 4:  # the component's own coefficient comes first
            ids = rng.integers(0, classes, ext)
        lo, hi = (0.7, 1.0) if len(name) == 4 else (-0.3, 0.3)
        coeffs[name] = rng.uniform(lo, hi, classes)[ids]
    start = None
    out = []
    for on in (True, False):
        monkeypatch.setenv("XFD_CPML_INSWEEP", "1" if on else "0")
        ctx = native.Context(coeffs, precision)
        mode = ctypes.c_int32()
        assert native.load_library().xfd_cpml_fused(ctx._h, ctypes.byref(mode)) == 0 and mode.value == (4 if on else 0)
        assert ctx.coef_layout()[0] == (layout != "dense")
        assert (max(ctx.coef_layout()[1]) > 65535) == (layout == "wide")
        start = start or {f: rng.standard_normal(ctx.extent(f)) for f in FIELDS}
        for f in FIELDS:
            ctx.write(f, start[f])
        ctx.step(0, 6)
        out.append({f: ctx.read(f) for f in FIELDS})
        ctx.close()
    for f in FIELDS:
        np.testing.assert_array_equal(out[0][f], out[1][f], err_msg=f)
        assert np.isfinite(out[0][f]).all()
