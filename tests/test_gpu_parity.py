"""GPU parity: the HIP path against the oracle and against closed forms.

FP64 runs compare the device results with the oracle on the same inputs:
relative L2 <= 1e-12 per field / frame (the bar for summation order), and the
tests also report how many values are bitwise equal (the FP64 kernels are
built without FMA contraction, so equality is expected).  FP32 runs state
their error against the FP64 oracle.
"""

import sys

import numpy as np
import pytest

import eigenmode as em
from oracle import RefSim, rel_l2
from xfdtd_core_amd import native, scenarios
from xfdtd_core_amd import spec as S

pytestmark = pytest.mark.gpu

FIELDS = ("EX", "EY", "EZ", "HX", "HY", "HZ")
TOL_F64 = 1e-12
ETA0 = 376.730313668


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("field", ["EZ", "EX", "EY"])
def test_capi_cavity_eigenmode(field):
    """Drives xfd_create/xfd_write_field/xfd_step directly with the oracle's
    coefficients: GPU == oracle bitwise and == the closed form."""
    say(f"[gpu] cavity eigenmode {field}")
    n, dl = (24, 20, 16), (1e-3, 1.2e-3, 0.9e-3)
    steps = 150
    ref = RefSim(em.cavity_spec(n, dl))
    ref.init(steps)
    coeffs = {c: ref.coeff(c) for c in native.COEFF_NAMES}
    e0, _, _ = em.mode(field, n)
    ctx = native.Context(coeffs, "f64")
    ctx.write(field, e0)
    ctx.step(0, steps)
    gpu = {f: ctx.read(f) for f in FIELDS}
    ref.write_field(field, e0)
    ref.loop()
    for f in FIELDS:
        np.testing.assert_array_equal(gpu[f], ref.field(f), err_msg=f)
    g = em.growth(field, n, dl, ref.dt, steps)
    np.testing.assert_allclose(gpu[field], g * e0, rtol=0, atol=2e-12 * np.abs(e0).max())


def _compare_run(spec, steps, threads, label, precision="f64", classed=True):
    say(f"[gpu] {label}: oracle {steps} steps")
    ref = RefSim(spec, threads=threads)
    ref.run(steps)
    say(f"[gpu] {label}: device {precision}")
    dev = native.Simulation(spec, precision)
    dev.run(steps)
    assert dev.coef_classed() == classed, "coefficient layout"
    out = {}
    for f in FIELDS:
        a, b = dev.field(f), ref.field(f)
        out[f] = (rel_l2(a, b), float(np.mean(a == b)))
    for m in range(dev.monitor_count()):
        ra, rb = dev.monitor_records(m), ref.monitor_records(m)
        assert len(ra) == len(rb), (m, len(ra), len(rb))
        errs = [rel_l2(x, y) for x, y in zip(ra, rb)]
        eq = [float(np.mean(x == y)) for x, y in zip(ra, rb)]
        out[f"monitor{m}"] = (max(errs) if errs else 0.0, min(eq) if eq else 1.0)
    for k, (e, q) in out.items():
        say(f"  {label} {k}: rel_l2={e:.3e} bitwise_fraction={q:.6f}")
    return out


def test_readme_sphere_fp64_full_run():
    """README example (63^3, TFSF, 6 CPML slabs, Ex movie), 2000 steps:
    every movie frame and final field within 1e-12 of the oracle.  The oracle
    runs as one domain: with several threads the reference's CPML E
    correction of a negative-side slab also writes the first plane of the
    next thread's task, concurrently with that thread's own correctors
    (simulation.cpp:424-435 describes the hazard), so only the one-domain
    order is deterministic."""
    out = _compare_run(scenarios.dielectric_sphere().spec(), 2000, (1, 1, 1), "readme")
    for k, (e, _) in out.items():
        assert e <= TOL_F64, (k, e)


def test_inhomogeneous_box_fp64():
    """Scaled inhomogeneous box: spheres, centred current source, CPML,
    six-field snapshots and Ez probes."""
    sp = scenarios.inhomogeneous_box(n_total=48, pml=6, n_spheres=6, r_cells=(3, 7), seed=11,
                                     snapshot_interval=100).spec()
    out = _compare_run(sp, 300, (1, 1, 1), "box48")
    for k, (e, _) in out.items():
        assert e <= TOL_F64, (k, e)


def test_inhomogeneous_box_dense_coefficients_fp64(monkeypatch):
    """The same box with the 18 dense coefficient arrays on the device
    (XFD_COEF_MODE=dense) instead of per-cell class ids."""
    monkeypatch.setenv("XFD_COEF_MODE", "dense")
    sp = scenarios.inhomogeneous_box(n_total=48, pml=6, n_spheres=6, r_cells=(3, 7), seed=11,
                                     snapshot_interval=100).spec()
    out = _compare_run(sp, 300, (1, 1, 1), "box48-dense", classed=False)
    for k, (e, _) in out.items():
        assert e <= TOL_F64, (k, e)


def test_capi_coefficient_classes_match_dense(monkeypatch):
    """Random per-cell coefficients drawn from a few values: the classed and
    the dense device layouts give identical fields."""
    say("[gpu] class ids vs dense arrays")
    rng = np.random.default_rng(5)
    n = (20, 18, 70)
    ref = RefSim(em.cavity_spec(n, (1e-3, 1e-3, 1e-3)))
    ref.init(10)
    coeffs = {}
    for c in native.COEFF_NAMES:
        base = ref.coeff(c)
        scale = rng.choice(np.array([1.0, 0.97, 1.01, 0.5]), size=base.shape)
        coeffs[c] = base * scale
    e0 = rng.standard_normal((n[0] + 1, n[1] + 1, n[2]))
    out = {}
    for mode in ("classed", "dense"):
        if mode == "dense":
            monkeypatch.setenv("XFD_COEF_MODE", "dense")
        ctx = native.Context(coeffs, "f64")
        classed, classes = ctx.coef_layout()
        assert classed == (mode == "classed"), mode
        if classed:
            for q in range(6):
                trip = np.stack([coeffs[native.COEFF_NAMES[3 * q + r]].ravel() for r in range(3)], -1)
                assert classes[q] == np.unique(trip, axis=0).shape[0], (q, classes)
        ctx.write("EZ", e0)
        ctx.step(0, 40)
        out[mode] = {f: ctx.read(f) for f in FIELDS}
        ctx.close()
    for f in FIELDS:
        np.testing.assert_array_equal(out["classed"][f], out["dense"][f], err_msg=f)


def test_lumped_oblique_tfsf_fp64():
    from test_precompute_parity import _lumped_box

    sp = _lumped_box().spec()
    out = _compare_run(sp, 250, (1, 1, 1), "lumped")
    for k, (e, _) in out.items():
        assert e <= TOL_F64, (k, e)


@pytest.mark.filterwarnings("ignore:Mean of empty slice:RuntimeWarning")
@pytest.mark.filterwarnings("ignore:invalid value encountered:RuntimeWarning")
def test_circuit_elements_fp64():
    """Capacitors, inductors (per-edge current state on the device), PEC
    planes, a resistor and a voltage source beside a lossy sphere and CPML."""
    from test_precompute_parity import _circuit_box

    sp = _circuit_box()
    sp.addMonitor(S.MovieMonitor(S.FieldMonitor(S.Cube(S.Vector(-0.010, -0.011, 0.0), S.Vector(0.020, 0.022, 0.001)),
                                                "EZ"), 25, "ez_xy", ""))
    # a zero-thickness box records empty frames, as in the reference
    sp.addMonitor(S.MovieMonitor(S.FieldMonitor(S.Cube(S.Vector(-0.010, -0.011, 0.0), S.Vector(0.020, 0.022, 0.0)),
                                                "EY"), 50, "ey_empty", ""))
    out = _compare_run(sp.spec(), 300, (1, 1, 1), "circuit")
    for k, (e, _) in out.items():
        assert e <= TOL_F64, (k, e)


DISPERSIVE = {
    "mixed": dict(n_total=48, kinds=("drude", "debye", "lorentz", "mlorentz")),
    "drude_only": dict(n_total=40, kinds=("drude",)),
    "debye_only": dict(n_total=40, kinds=("debye", "debye")),
}


@pytest.mark.parametrize("case", sorted(DISPERSIVE))
def test_dispersive_ade_fp64(case):
    """ADE dispersion on the device (per-cell material ids, pole currents):
    the mixed scene runs the modified-Lorentz scheme, the others the
    Drude-only and Debye-only schemes; TFSF, resistor and voltage source in
    the same box."""
    kw = DISPERSIVE[case]
    sp = scenarios.dispersive_slabs(pml=5, slab=6, gap=2, tfsf_offset=7, snapshot_interval=100, **kw).spec()
    out = _compare_run(sp, 300, (1, 1, 1), f"ade-{case}")
    for k, (e, _) in out.items():
        assert e <= TOL_F64, (k, e)


def _compare_nf2ff(dev, ref, nf, label):
    """Accumulated surface currents, potentials and power of NF2FF 0."""
    theta = np.linspace(0.1, np.pi - 0.1, 17)
    worst = 0.0
    for f in range(nf):
        for d in range(6):
            for w in range(4):
                a, b = dev.nf2ff_current(0, f, d, w), ref.nf2ff_current(0, f, d, w)
                assert a.shape == b.shape
                if b.size:
                    worst = max(worst, rel_l2(a, b))
        for a_pot in (True, False):
            for th_comp in (True, False):
                a = dev.nf2ff_potential(0, f, a_pot, th_comp, theta, 0.4)
                b = ref.nf2ff_potential(0, f, a_pot, th_comp, theta, 0.4)
                worst = max(worst, rel_l2(a, b))
        pa, pb = dev.nf2ff_power(0, f), ref.nf2ff_power(0, f)
        worst = max(worst, abs(pa - pb) / abs(pb))
    say(f"  {label} nf2ff worst relative L2: {worst:.3e}")
    return worst


def test_nf2ff_dipole_fp64():
    """NF2FF running DFT on the device (FP64 accumulators, the per-frequency
    repeat): surface currents, far-field potentials and radiated power of a
    radiating dipole equal the oracle's."""
    from test_oracle_nf2ff import STEPS, _dipole

    sp = _dipole([6e9, 9e9])
    say("[gpu] nf2ff dipole: oracle")
    ref = RefSim(sp)
    ref.run(STEPS)
    say("[gpu] nf2ff dipole: device")
    dev = native.Simulation(sp, "f64")
    dev.run(STEPS)
    for f in FIELDS:
        assert rel_l2(dev.field(f), ref.field(f)) <= TOL_F64, f
    assert _compare_nf2ff(dev, ref, 2, "dipole") <= TOL_F64


def test_nf2ff_plain_dft_fp64():
    """The non-repeating DFT option on the device equals the oracle's."""
    from test_oracle_nf2ff import _dipole

    sp = _dipole([6e9, 9e9], plain=True)
    ref = RefSim(sp)
    ref.run(300)
    dev = native.Simulation(sp, "f64")
    dev.run(300)
    assert _compare_nf2ff(dev, ref, 2, "plain-dft") <= TOL_F64


def test_nf2ff_dispersive_box_fp64():
    """NF2FF (8 frequencies, 5-40 GHz) around the dispersive, lumped and
    TFSF-driven box."""
    sp = scenarios.dispersive_slabs(n_total=48, pml=5, slab=6, gap=2, tfsf_offset=7, nf2ff_distance=6).spec()
    say("[gpu] nf2ff dispersive: oracle")
    ref = RefSim(sp)
    ref.run(200)
    say("[gpu] nf2ff dispersive: device")
    dev = native.Simulation(sp, "f64")
    dev.run(200)
    assert _compare_nf2ff(dev, ref, 8, "dispersive") <= TOL_F64


def test_fp32_error_against_fp64_oracle():
    """FP32 fields and updates against the FP64 oracle on the scaled box.

    Stated figures: per snapshot frame the relative L2 of the E and H groups
    with the frame's own norm and with the run's peak norm, and the relative
    L2 of each probe series.  Bounds: while the pulse is in the box (step
    100) the plain relative L2 is <= 1e-5; every frame and the final fields
    are within 1e-5 of the run's peak norm; probe series within 1e-4.  The
    late frames' own-norm figures (up to ~1e-3) are printed, not bounded:
    the field has decayed about a thousandfold by then while the FP32
    residue stays at ~1e-7 of the peak."""
    from xfdtd_core_amd import accuracy

    sp = scenarios.inhomogeneous_box(n_total=48, pml=6, n_spheres=6, r_cells=(3, 7), seed=11,
                                     snapshot_interval=100).spec()
    steps = 300
    say("[gpu] box48-f32: oracle")
    ref = RefSim(sp, threads=(1, 1, 1))
    ref.run(steps)
    say("[gpu] box48-f32: device f32")
    dev = native.Simulation(sp, "f32")
    dev.run(steps)
    snaps_d = {f: dev.monitor_records(i) for i, f in enumerate(FIELDS)}
    snaps_r = {f: ref.monitor_records(i) for i, f in enumerate(FIELDS)}
    frames = accuracy.snapshot_errors(snaps_d, snaps_r, [100 * k for k in range(len(snaps_r["EX"]))])
    frames = [r for r in frames if r["E"]["own"] is not None and r["H"]["own"] is not None]
    for r in frames:
        say(f"  step {r['step']}: E own {r['E']['own']:.2e} peak {r['E']['peak']:.2e} | "
            f"H own {r['H']['own']:.2e} peak {r['H']['peak']:.2e}")
    peaks = {g: max(np.sqrt(sum(float(np.sum(snaps_r[f][i] ** 2)) for f in fl))
                    for i in range(len(snaps_r["EX"])))
             for g, fl in accuracy.GROUPS.items()}
    final = {}
    for g, fl in accuracy.GROUPS.items():
        d = np.sqrt(sum(float(np.sum((dev.field(f) - ref.field(f)) ** 2)) for f in fl))
        n = np.sqrt(sum(float(np.sum(ref.field(f) ** 2)) for f in fl))
        final[g] = (d / n, d / peaks[g])
        say(f"  final {g}: own {final[g][0]:.2e} peak {final[g][1]:.2e}")
    probes = [accuracy.series_error(dev.monitor_records(m)[0][1], ref.monitor_records(m)[0][1])
              for m in range(len(FIELDS), dev.monitor_count())]
    probes = [p for p in probes if p is not None]
    assert probes
    say(f"  probes: max relative L2 {max(probes):.2e}")
    at100 = [r for r in frames if r["step"] == 100][0]
    assert at100["E"]["own"] <= 1e-5 and at100["H"]["own"] <= 1e-5, at100
    for r in frames:
        assert r["E"]["peak"] <= 1e-5 and r["H"]["peak"] <= 1e-5, r
    for g in final:
        assert final[g][1] <= 1e-5, (g, final[g])
    assert max(probes) <= 1e-4


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_cpml_inside_sweeps_matches_separate_launches(monkeypatch, precision):
    """The Yee sweeps with the CPML corrections applied in the same pass give
    the separate-launch results: bitwise in FP64, and in FP32 within the
    contraction freedom of the compiler.  Cases where a record lands in a
    slab or ADE is present keep the separate launches."""
    sp = scenarios.inhomogeneous_box(n_total=48, pml=8, n_spheres=6, r_cells=(3, 7), seed=5).spec()
    say(f"[gpu] fused CPML vs separate {precision}")
    monkeypatch.setenv("XFD_STEP_FUSED", "0")
    monkeypatch.setenv("XFD_CPML_INSWEEP", "0")
    monkeypatch.setenv("XFD_CPML_FUSED", "1")
    fused = native.Simulation(sp, precision)
    fused.run(200)
    assert fused.cpml_fused()
    monkeypatch.setenv("XFD_CPML_FUSED", "0")
    monkeypatch.setenv("XFD_CPML_ZFUSED", "0")
    sep = native.Simulation(sp, precision)
    sep.run(200)
    assert sep.cpml_fused() == 0
    for f in FIELDS:
        a, b = fused.field(f), sep.field(f)
        if precision == "f64":
            np.testing.assert_array_equal(a, b, err_msg=f)
        else:
            # contraction differences grow while the field decays; the FP32
            # accuracy target (1e-4) bounds them
            assert rel_l2(a, b) < 1e-4, (f, rel_l2(a, b))
    monkeypatch.setenv("XFD_CPML_FUSED", "1")
    disp = native.Simulation(scenarios.dispersive_slabs(n_total=40, pml=6, slab=6, gap=2, tfsf_offset=9,
                                                        lumped=False).spec(), precision)
    disp.init(2)
    assert disp.cpml_fused() == 0


def _tall_box(nz_total, pml=8, n_xy=24):
    """A vacuum box of n_xy x n_xy x nz_total cells including the CPML."""
    dl = 1e-3
    s = S.Simulation(dl, dl, dl, 0.9)
    n_in = [n_xy - 2 * pml, n_xy - 2 * pml, nz_total - 2 * pml]
    s.addObject(S.Object("domain", S.Cube(S.Vector(*[-a * dl / 2 for a in n_in]), S.Vector(*[a * dl for a in n_in])),
                         S.Material.createAir()))
    for d in ("XN", "XP", "YN", "YP", "ZN", "ZP"):
        s.addBoundary(S.PML(pml, d))
    return s.spec()


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_z_cpml_inside_sweeps(monkeypatch, precision):
    """The sweeps apply the z CPML slabs: FP32 by default when a k-row spans
    at least 3 sweep tiles, the whole slab; FP64 only when forced, and only
    where no x/y slab corrects the point (the frame follows the x/y slabs in
    a launch of its own, keeping the reference's order).  Forced on a 48^3
    box, where one wavefront holds lanes of both z slabs: FP64 equals the
    all-separate run and the oracle bitwise; FP32 is as close to FP64 as the
    separate run.  Contexts with ADE keep separate slabs."""
    sp = scenarios.inhomogeneous_box(n_total=48, pml=8, n_spheres=6, r_cells=(3, 7), seed=5).spec()
    say(f"[gpu] z CPML inside the sweeps vs separate {precision}")
    monkeypatch.setenv("XFD_STEP_FUSED", "0")
    monkeypatch.setenv("XFD_CPML_INSWEEP", "0")
    monkeypatch.delenv("XFD_CPML_FUSED", raising=False)
    monkeypatch.delenv("XFD_CPML_ZFUSED", raising=False)
    for nz, want in ((128, 0), (129, 2 if precision == "f32" else 0)):  # 2 and 3 tiles of 64 k-lanes
        tall = native.Simulation(_tall_box(nz), precision)
        tall.init(2)
        assert tall.cpml_fused() == want, (nz, tall.cpml_fused())
        tall.close()
    auto = native.Simulation(sp, precision)
    auto.init(2)
    assert auto.cpml_fused() == 0
    auto.close()
    monkeypatch.setenv("XFD_CPML_ZFUSED", "1")
    zf = native.Simulation(sp, precision)
    zf.run(200)
    assert zf.cpml_fused() == 2
    monkeypatch.setenv("XFD_CPML_ZFUSED", "0")
    sep = native.Simulation(sp, precision)
    sep.run(200)
    assert sep.cpml_fused() == 0
    if precision == "f64":
        ref = RefSim(sp)
        ref.run(200)
        for f in FIELDS:
            np.testing.assert_array_equal(zf.field(f), sep.field(f), err_msg=f)
            np.testing.assert_array_equal(zf.field(f), ref.field(f), err_msg=f)
    else:
        monkeypatch.setenv("XFD_CPML_ZFUSED", "0")
        ref = native.Simulation(sp, "f64")
        ref.run(200)

        def layers(x):  # the z slabs' 8 layers at both ends
            return np.concatenate([x[:, :, :9].ravel(), x[:, :, -9:].ravel()])

        for f in FIELDS:
            a, b, r = zf.field(f), sep.field(f), ref.field(f)
            d, e_sep, e_zf = rel_l2(a, b), rel_l2(b, r), rel_l2(a, r)
            l_sep, l_zf = rel_l2(layers(b), layers(r)), rel_l2(layers(a), layers(r))
            say(f"  {f}: z-fused vs separate {d:.2e}; vs f64: separate {e_sep:.2e}, z-fused {e_zf:.2e}; "
                f"z layers: separate {l_sep:.2e}, z-fused {l_zf:.2e}")
            assert d < 1e-4, (f, d)
            assert e_zf <= 2 * e_sep + 1e-6, (f, e_zf, e_sep)
            assert l_zf <= 2 * l_sep + 1e-6, (f, l_zf, l_sep)
    monkeypatch.setenv("XFD_CPML_ZFUSED", "1")
    disp = native.Simulation(scenarios.dispersive_slabs(n_total=40, pml=6, slab=6, gap=2, tfsf_offset=9,
                                                        lumped=False).spec(), precision)
    disp.init(2)
    assert disp.cpml_fused() == 0


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_sweep_tile_128_by_2(monkeypatch, precision):
    """The plain and z-in-sweep Yee sweeps take 128 k-lanes x 2 j-rows where
    nz is a multiple of 128 and 64 x 4 elsewhere (XFD_SWEEP_TILE forces
    either).  Every point's arithmetic is the same under both tiles, so they
    give the same bits: a 128^3 box (128 x 2 by default; FP64 also equal to
    the oracle) and a 96^3 box forced to 128 x 2 (every row one full and one
    half-idle wavefront), each against 64 x 4, with the z CPML slabs as
    separate launches and inside the sweeps."""
    steps = 60
    monkeypatch.setenv("XFD_STEP_FUSED", "0")
    monkeypatch.setenv("XFD_CPML_INSWEEP", "0")
    monkeypatch.delenv("XFD_CPML_FUSED", raising=False)
    for n, forced in ((128, None), (96, "128")):
        sp = scenarios.inhomogeneous_box(n_total=n, pml=8, n_spheres=6, r_cells=(3, 9), seed=11).spec()
        for zf in ("0", "1"):
            monkeypatch.setenv("XFD_CPML_ZFUSED", zf)
            say(f"[gpu] sweep tile 128 x 2 vs 64 x 4, {n}^3 {precision}, z slabs {'inside' if zf == '1' else 'apart'}")
            if forced:
                monkeypatch.setenv("XFD_SWEEP_TILE", forced)
            else:
                monkeypatch.delenv("XFD_SWEEP_TILE", raising=False)
            a = native.Simulation(sp, precision)
            a.run(steps)
            assert a.cpml_fused() == (2 if zf == "1" else 0)
            monkeypatch.setenv("XFD_SWEEP_TILE", "64")
            b = native.Simulation(sp, precision)
            b.run(steps)
            for f in FIELDS:
                np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f"{n} {zf} {f}")
            assert np.abs(a.field("EZ")).max() > 0
            if precision == "f64" and n == 128 and zf == "0":
                ref = RefSim(sp)
                ref.run(steps)
                for f in FIELDS:
                    np.testing.assert_array_equal(a.field(f), ref.field(f), err_msg=f"oracle {f}")
            a.close()
            b.close()


@pytest.mark.parametrize("kinds", [("drude", "debye", "lorentz", "mlorentz"), ("drude",), ("debye",)],
                         ids=["mlorentz", "drude", "debye"])
def test_dispersive_sweep_tile_128_by_2(monkeypatch, kinds):
    """The dispersive E sweep (k_update_e_ade, each of its three schemes)
    takes the plain sweeps' tile: 128 x 2 on a 128^3 box by default, the same
    bits as 64 x 4 in FP64 and FP32."""
    steps = 60
    monkeypatch.delenv("XFD_CPML_ZFUSED", raising=False)
    sp = scenarios.dispersive_slabs(n_total=128, pml=8, slab=16, gap=4, tfsf_offset=12, kinds=kinds,
                                    lumped=False).spec()
    for precision in ("f64", "f32"):
        say(f"[gpu] dispersive sweep tile 128 x 2 vs 64 x 4, {'+'.join(kinds)} {precision}")
        monkeypatch.delenv("XFD_SWEEP_TILE", raising=False)
        a = native.Simulation(sp, precision)
        a.run(steps)
        monkeypatch.setenv("XFD_SWEEP_TILE", "64")
        b = native.Simulation(sp, precision)
        b.run(steps)
        for f in FIELDS:
            np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f"{precision} {f}")
        assert np.abs(a.field("EZ")).max() > 0 or np.abs(a.field("EX")).max() > 0
        a.close()
        b.close()


def test_far_field_on_device_matches_host(monkeypatch):
    """The far-field potentials summed on the GPU (xfd_nf2ff_far_field) equal
    the host sums over the same currents, for a theta cut and a phi cut
    (measured against the largest potential of the cut: the cross-polarised
    ones are cancellations of much larger terms)."""
    from test_oracle_nf2ff import _dipole

    dev = native.Simulation(_dipole([6e9, 9e9]), "f64")
    dev.run(300)
    theta = np.linspace(0.0, np.pi, 37)
    phi = np.linspace(0.0, 2 * np.pi, 25)
    combos = [(a, t) for a in (True, False) for t in (True, False)]
    for f in range(2):
        for th, ph in ((theta, 0.7), (1.1, phi)):
            monkeypatch.delenv("XFD_FARFIELD", raising=False)
            g = [dev.nf2ff_potential(0, f, a, t, th, ph) for a, t in combos]
            monkeypatch.setenv("XFD_FARFIELD", "host")
            h = [dev.nf2ff_potential(0, f, a, t, th, ph) for a, t in combos]
            scale = max(np.abs(x).max() for x in h)
            assert scale > 0
            for gi, hi in zip(g, h):
                assert np.abs(gi - hi).max() <= 1e-12 * scale


NET_FREQS = [1e9, 2.5e9, 4e9, 6e9]


def _line_monitor_spec(network_dir=None):
    """A 50-ohm voltage source and a 50-ohm resistor (6-cell z gaps) in a
    CPML box, with a voltage and a current monitor on each and a voltage
    monitor across a 2 x 3 x 4 block along y.  With `network_dir` (a path,
    or "" for no files), also a two-port network: port 1 (source) on the
    voltage source, port 2 on the resistor."""
    dl = 1e-3
    s = S.Simulation(dl, dl, dl, 0.9)
    half = 12 * dl
    s.addObject(S.Object("domain", S.Cube(S.Vector(-half, -half, -half), S.Vector(2 * half, 2 * half, 2 * half)),
                         S.Material.createAir()))
    tau = 15 * dl / 6e8
    src = S.Cube(S.Vector(-3 * dl, 0.0, -3 * dl), S.Vector(0.0, 0.0, 6 * dl))
    res = S.Cube(S.Vector(4 * dl, 0.0, -3 * dl), S.Vector(0.0, 0.0, 6 * dl))
    s.addObject(S.VoltageSource("v1", src, "ZP", 50.0, S.Waveform.gaussian(tau, 4.5 * tau, 1.0)))
    s.addObject(S.Resistor("r1", res, "Z", 50.0))
    for d in ("XN", "XP", "YN", "YP", "ZN", "ZP"):
        s.addBoundary(S.PML(6, d))
    mons = [S.VoltageMonitor("v_src", src, "ZP"), S.CurrentMonitor("i_src", src, "ZP"),
            S.VoltageMonitor("v_res", res, "ZN"), S.CurrentMonitor("i_res", res, "ZN"),
            S.VoltageMonitor("v_blk", S.Cube(S.Vector(-dl, -2 * dl, dl), S.Vector(2 * dl, 3 * dl, 4 * dl)), "YP"),
            S.CurrentMonitor("i_blk", S.Cube(S.Vector(-dl, -2 * dl, dl), S.Vector(2 * dl, 3 * dl, 4 * dl)), "XN")]
    for m in mons:
        s.addMonitor(m)
    if network_dir is not None:
        s.addNetwork(S.Network([S.Port(1, True, 50.0, mons[1], mons[0]), S.Port(2, False, 50.0, mons[3], mons[2])],
                               NET_FREQS, network_dir))
    return s.spec()


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_voltage_current_monitors(precision):
    """VoltageMonitor / CurrentMonitor series on the device equal the
    oracle's: bitwise in FP64; FP32 within 1e-4 of each series' peak."""
    sp = _line_monitor_spec()
    steps = 400
    ref = RefSim(sp)
    ref.run(steps)
    dev = native.Simulation(sp, precision)
    dev.run(steps)
    assert dev.monitor_count() == 6
    for m in range(6):
        a, b = dev.monitor_records(m)[0], ref.monitor_records(m)[0]
        assert a.shape == b.shape == (2, steps)
        np.testing.assert_array_equal(a[0], b[0])  # times
        assert np.abs(b[1]).max() > 0, m
        if precision == "f64":
            np.testing.assert_array_equal(a[1], b[1], err_msg=f"monitor {m}")
        else:
            err = np.abs(a[1] - b[1]).max() / np.abs(b[1]).max()
            say(f"  monitor {m}: fp32 error {err:.2e} of the peak")
            assert err < 1e-4, (m, err)


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_network_s_parameters(tmp_path, precision):
    """Network::output on the device-recorded port series: S11 and S21 of a
    two-port (source, resistor) equal the oracle's bitwise in FP64 (same
    recordings, same host transform); FP32 within 1e-3.  The product writes
    s11.npy / s21.npy (complex128) and frequencies.npy."""
    out = tmp_path / precision
    sp = _line_monitor_spec(str(out))
    steps = 400
    say(f"[gpu] network S-parameters {precision}")
    ref = RefSim(_line_monitor_spec(""))
    ref.run(steps)
    want = ref.network_s(0, (11, 21), len(NET_FREQS))
    dev = native.Simulation(sp, precision)
    dev.run(steps)
    assert dev.network_count() == 1
    got = dev.network_output(0)
    assert sorted(got) == [11, 21]
    for k in (11, 21):
        if precision == "f64":
            np.testing.assert_array_equal(got[k], want[k], err_msg=f"s{k}")
        else:
            err = np.abs(got[k] - want[k]).max()
            say(f"  s{k}: fp32 error {err:.2e} (|S| up to {np.abs(want[k]).max():.3f})")
            assert err < 1e-3, (k, err)
        np.testing.assert_array_equal(np.load(out / f"s{k}.npy"), got[k])
    np.testing.assert_array_equal(np.load(out / "frequencies.npy"), np.array(NET_FREQS))
    assert np.abs(want[11]).max() > 0.1 and np.abs(want[21]).max() > 1e-4  # |S21| ~ 1e-3 here


@pytest.mark.parametrize("precision,merge", [("f64", False), ("f64", True), ("f32", False)])
def test_time_domain_nf2ff(tmp_path, monkeypatch, precision, merge):
    """Time-domain NF2FF on the device (per-cell bins, then each bin summed
    in the reference's cell order: fixed runs, or with XFD_TDNF_MERGE=1 the
    merge of the delay buckets that the general case needs): every surface
    potential and the far field equal the oracle's in FP64; FP32 within 1e-4
    of the far field's co-polarised peak.  The far-field .npy files carry
    the same values."""
    from test_oracle_nf2ff_td import STEPS, dipole_td

    if merge:
        monkeypatch.setenv("XFD_TDNF_MERGE", "1")
    else:
        monkeypatch.delenv("XFD_TDNF_MERGE", raising=False)
    theta, phi = np.pi / 3, 1.1
    say(f"[gpu] time-domain NF2FF {precision}{' merging bins' if merge else ''}")
    ref = RefSim(dipole_td(theta, phi))
    ref.run(STEPS)
    out = tmp_path / precision
    dev = native.Simulation(dipole_td(theta, phi, str(out)), precision)
    dev.run(STEPS)
    far = dev.nf2ff_td_far_field(0)
    want = ref.nf2ff_td_far_field(0)
    assert far.shape == want.shape
    if precision == "f64":
        for d in range(6):
            for w in range(4):
                a, b = dev.nf2ff_td_potential(0, d, w), ref.nf2ff_td_potential(0, d, w)
                assert np.abs(b).max() > 0, (d, w)
                err = rel_l2(a, b)
                say(f"  surface {d} potential {w}: rel_l2 {err:.2e}, bitwise {np.mean(a == b):.4f}")
                assert err <= TOL_F64, (d, w, err)
        for w in range(4):
            assert rel_l2(far[w], want[w]) <= TOL_F64, w
    else:
        peak = np.abs(ETA0 * want[0] + want[3]).max()
        err = max(np.abs(far[w] - want[w]).max() * (ETA0 if w < 2 else 1.0) for w in range(4)) / peak
        say(f"  fp32 far-field error {err:.2e} of the co-polarised peak")
        assert err < 1e-4, err
    for w, name in enumerate(("w_theta", "w_phi", "u_theta", "u_phi")):
        np.testing.assert_array_equal(np.load(out / f"{name}.npy"), far[w])


@pytest.mark.parametrize("single_pass", [False, True])
def test_profiling_selected_kernel_classes(monkeypatch, single_pass):
    """HIP-event timing can be limited to chosen kernel classes: only those
    classes report launches, and with every class the counts match the
    launches of the steps (two sweeps and three slab launches per half-step,
    the two slabs of each axis sharing one, or six with XFD_CPML_PAIR=0; or
    one single-pass launch per step)."""
    sp = scenarios.inhomogeneous_box(n_total=40, pml=6, n_spheres=3, r_cells=(3, 5), seed=3).spec()
    say(f"[gpu] profiling selected kernel classes (single pass: {single_pass})")
    if single_pass:
        monkeypatch.setenv("XFD_STEP_FUSED", "1")
        sim = native.Simulation(sp, "f64")
        sim.init(40)
        assert sim.cpml_fused() == 3
        sim.set_profiling(True, classes=["step"])
        sim.advance(0, 20)
        st = sim.kernel_stats()
        assert st["step"][0] == 20 and st["step"][1] > 0
        assert all(v[0] == 0 for k, v in st.items() if k != "step"), st
        sim.set_profiling(True)
        sim.advance(20, 20)
        st = sim.kernel_stats()
        assert st["step"][0] == 20 and st["records_e"][0] == 20, st
        assert st["update_e"][0] == st["update_h"][0] == st["cpml_e"][0] == st["cpml_h"][0] == 0, st
        return
    monkeypatch.setenv("XFD_STEP_FUSED", "0")
    sim = native.Simulation(sp, "f64")
    sim.init(40)
    sim.set_profiling(True, classes=["update_e"])
    sim.advance(0, 20)
    st = sim.kernel_stats()
    assert st["update_e"][0] == 20 and st["update_e"][1] > 0
    assert all(v[0] == 0 for k, v in st.items() if k != "update_e"), st
    sim.set_profiling(True)
    sim.advance(20, 20)
    st = sim.kernel_stats()
    assert st["update_e"][0] == 20 and st["update_h"][0] == 20 and st["cpml_e"][0] == 20 * 3, st
    monkeypatch.setenv("XFD_CPML_PAIR", "0")
    sim.init(20)
    sim.set_profiling(True)
    sim.advance(0, 20)
    st = sim.kernel_stats()
    assert st["cpml_e"][0] == 20 * 6 and st["cpml_h"][0] == 20 * 6, st


def test_full_size_box_is_repeatable_and_linear():
    """The 384^3 inhomogeneous box (64 spheres, 12-cell CPML, the measured
    workload) at full size, through properties that hold at any size: two
    runs give bitwise the same fields (no race in any launch), FP64 and FP32;
    and doubling the waveform amplitude multiplies every FP64 field by 4.
    Each step is linear in the source current, and the reference's current
    source applies the amplitude twice: in the waveform's values
    (waveform.cpp:31) and in its amplitude factor (current_source.cpp:63).
    Scaling by a power of 2 is exact; values in the denormal range at the
    edge of the light cone may round differently, hence the 1e-14 bound
    instead of equality."""
    base = scenarios.inhomogeneous_box(monitors=False).spec()

    def spec(amplitude):  # the waveform amplitude is the source line's last token
        lines = base.splitlines()
        src = [n for n, ln in enumerate(lines) if ln.startswith("current_source ")]
        assert len(src) == 1 and lines[src[0]].split()[-1] == "1.0"
        lines[src[0]] = " ".join(lines[src[0]].split()[:-1] + [repr(amplitude)])
        return "\n".join(lines) + "\n"

    steps = 150
    for precision in ("f64", "f32"):
        say(f"[gpu] 384^3 box, {steps} steps, {precision}: repeatability" + (" and linearity" if precision == "f64" else ""))
        runs = []
        for amp in ((1.0, 1.0, 2.0) if precision == "f64" else (1.0, 1.0)):
            sim = native.Simulation(spec(amp), precision)
            sim.run(steps)
            runs.append(sim)
        for f in FIELDS:
            a, b = runs[0].field(f), runs[1].field(f)
            assert np.abs(a).max() > 0, f
            np.testing.assert_array_equal(a, b, err_msg=f)
            if precision == "f64":
                c = runs[2].field(f)
                e = np.linalg.norm(c - 4 * a) / np.linalg.norm(4 * a)
                say(f"  {f}: doubled-amplitude residue {e:.1e}, exact in {np.mean(c == 4 * a):.6f} of the points")
                assert e < 1e-14, (f, e)
            del a, b
        for sim in runs:
            sim.close()


def test_full_size_dispersive_box_is_repeatable():
    """The 256^3 dispersive + lumped box (Drude, Debye, Lorentz and modified
    Lorentz slabs, TFSF plane wave, lumped elements; the measured workload)
    at full size: two FP64 runs give bitwise the same fields, so the ADE,
    record and CPML launches carry no race at this size."""
    sp = scenarios.dispersive_slabs().spec()
    steps = 200
    say(f"[gpu] 256^3 dispersive box, {steps} steps, f64: repeatability")
    runs = []
    for _ in range(2):
        sim = native.Simulation(sp, "f64")
        sim.run(steps)
        runs.append(sim)
    for f in FIELDS:
        a, b = runs[0].field(f), runs[1].field(f)
        assert np.abs(a).max() > 0, f
        np.testing.assert_array_equal(a, b, err_msg=f)
    for sim in runs:
        sim.close()


FP32_ADE = {
    # the modified-Lorentz scheme with the specified stiff Drude pole
    # (wp = 1.37e16 rad/s, wp dt ~ 1e4), the Lorentz pair and a1 != 0 modified
    # Lorentz; the Debye slab is left out (b2 = 0 breaks that scheme's
    # stability condition, and its fields grow without bound in FP64 too)
    "mlorentz_stiff_drude": dict(n_total=48, kinds=("drude", "lorentz", "mlorentz")),
    # the Drude-only scheme (its first-order update is bounded only for a
    # smaller plasma frequency)
    "drude_only": dict(n_total=40, kinds=("drude",), drude_wp=1.9e11),
    "debye_only": dict(n_total=40, kinds=("debye", "debye")),
}


@pytest.mark.parametrize("case", sorted(FP32_ADE))
def test_fp32_ade_against_fp64_oracle(case):
    """k_update_e_ade<float>: FP32 fields, pole currents and previous E on
    the device against the FP64 oracle, with TFSF, the lumped resistor and
    voltage source, and (mixed case) an 8-frequency NF2FF in the box.

    Stated and bounded (1e-4, the FP32 accuracy target): the field state
    (E and eta0 H together) at steps 150 and 300, the far-field potentials
    (each against the largest of the four at its frequency) and the radiated
    power at every frequency."""
    kw = dict(FP32_ADE[case])
    nf = case == "mlorentz_stiff_drude"
    sp = scenarios.dispersive_slabs(pml=5, slab=6, gap=2, tfsf_offset=7, nf2ff_distance=6 if nf else 0,
                                    **kw).spec()
    say(f"[gpu] fp32 ade {case}: oracle and device")
    errs = {}
    for steps in (150, 300):
        ref = RefSim(sp)
        ref.run(steps)
        dev = native.Simulation(sp, "f32")
        dev.run(steps)
        num = den = 0.0
        for f in FIELDS:
            w = ETA0 if f[0] == "H" else 1.0
            a, b = dev.field(f) * w, ref.field(f) * w
            assert np.isfinite(a).all(), f
            num += float(np.sum((a - b) ** 2))
            den += float(np.sum(b ** 2))
        errs[f"fields@{steps}"] = float(np.sqrt(num / den))
        if nf and steps == 300:
            theta = np.linspace(0.1, np.pi - 0.1, 17)
            pot = pw = 0.0
            for fq in range(8):
                pa = [dev.nf2ff_potential(0, fq, ap, tc, theta, 0.4) for ap in (True, False) for tc in (True, False)]
                pb = [ref.nf2ff_potential(0, fq, ap, tc, theta, 0.4) for ap in (True, False) for tc in (True, False)]
                scale = max(float(np.abs(x).max()) for x in pb)
                pot = max([pot] + [float(np.abs(x - y).max()) / scale for x, y in zip(pa, pb)])
                pw = max(pw, abs(dev.nf2ff_power(0, fq) / ref.nf2ff_power(0, fq) - 1))
            errs["far_field"] = pot
            errs["power"] = pw
        dev.close()
    say("  " + ", ".join(f"{k} {v:.2e}" for k, v in errs.items()))
    for k, v in errs.items():
        assert v <= 1e-4, (case, k, v)


def test_full_size_fp64_matches_oracle():
    """The 384^3 measured workload at full size in FP64 against the oracle
    (100 steps, all six fields and the 32 probe series): the GPU FP64 run the
    benchmark uses as the FP32 error reference equals the oracle at this
    size, not only on the scaled boxes."""
    sp = scenarios.inhomogeneous_box(snapshot_interval=500).spec()
    steps = 100
    say(f"[gpu] 384^3 box, {steps} FP64 steps: device")
    dev = native.Simulation(sp, "f64")
    dev.run(steps)
    say("[gpu] 384^3 box: oracle (16 threads along x)")
    ref = RefSim(sp, threads=(16, 1, 1))
    ref.run(steps)
    worst = 0.0
    for f in FIELDS:
        a, b = dev.field(f), ref.field(f)
        assert np.abs(b).max() > 0, f
        e = rel_l2(a, b)
        say(f"  {f}: relative L2 {e:.2e}, bitwise equal in {np.mean(a == b):.6f} of the points")
        worst = max(worst, e)
        del a, b
    assert dev.monitor_count() == len(FIELDS) + 32
    for m in range(len(FIELDS), dev.monitor_count()):
        a, b = dev.monitor_records(m)[0][1], ref.monitor_records(m)[0][1]
        np.testing.assert_array_equal(a, b)
    assert worst <= TOL_F64, worst
    dev.close()


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("chunk", [4, 7, 1])
def test_single_pass_step(monkeypatch, precision, chunk):
    """The single-pass step (one launch per step: H, its CPML, E, its CPML;
    two field sets) against the two Yee sweeps with separate slab launches,
    on a 136^3 box (three k-tiles of 64 lanes, the last partial) with random
    spheres, the current-source dipole, six-field snapshots and probes, and
    several i-chunks (planes per work-item: 7 does not divide the grid, 1
    recomputes every plane's i-1 neighbour).  FP64: every field, frame and probe equal to the separate
    launches and to the oracle; FP32: as close to the FP64 result as the
    separate launches' FP32 run (contraction choices differ between the two
    FP32 kernels, so the two FP32 runs agree to ~1e-5, not bitwise)."""
    sp = scenarios.inhomogeneous_box(n_total=136, pml=9, n_spheres=12, r_cells=(4, 14), seed=11,
                                     snapshot_interval=40, probes=(2, 2, 2)).spec()
    steps = 120
    say(f"[gpu] single-pass step {precision} chunk {chunk}")
    monkeypatch.setenv("XFD_STEP_FUSED", "1")
    monkeypatch.setenv("XFD_STEP_CHUNK", str(chunk))
    one = native.Simulation(sp, precision)
    one.run(steps)
    assert one.cpml_fused() == 3
    monkeypatch.setenv("XFD_STEP_FUSED", "0")
    monkeypatch.setenv("XFD_CPML_ZFUSED", "0")
    monkeypatch.setenv("XFD_CPML_INSWEEP", "0")
    sep = native.Simulation(sp, precision)
    sep.run(steps)
    assert sep.cpml_fused() == 0
    if precision == "f32":
        r64 = native.Simulation(sp, "f64")
        r64.run(steps)
    for f in FIELDS:
        a, b = one.field(f), sep.field(f)
        if precision == "f64":
            np.testing.assert_array_equal(a, b, err_msg=f)
        else:
            r = r64.field(f)
            e_one, e_sep = rel_l2(a, r), rel_l2(b, r)
            say(f"  {f}: single pass vs f64 {e_one:.2e}, separate vs f64 {e_sep:.2e}, between {rel_l2(a, b):.2e}")
            assert rel_l2(a, b) < 1e-4 and e_one <= 2 * e_sep + 1e-6, (f, e_one, e_sep)
    for m in range(one.monitor_count()):
        for q, (a, b) in enumerate(zip(one.monitor_records(m), sep.monitor_records(m))):
            if precision == "f64":
                np.testing.assert_array_equal(a, b, err_msg=f"monitor {m}")
            elif np.abs(b).max() > 0:
                r = r64.monitor_records(m)[q]
                assert rel_l2(a, r) <= 2 * rel_l2(b, r) + 1e-6, (m, rel_l2(a, r), rel_l2(b, r))
    if precision == "f64" and chunk == 4:
        say("[gpu] single-pass step: oracle")
        ref = RefSim(sp, threads=(8, 1, 1))
        ref.run(steps)
        for f in FIELDS:
            np.testing.assert_array_equal(one.field(f), ref.field(f), err_msg=f)
        for m in range(one.monitor_count()):
            for a, b in zip(one.monitor_records(m), ref.monitor_records(m)):
                np.testing.assert_array_equal(a, b, err_msg=f"monitor {m}")


def test_single_pass_step_field_io(monkeypatch):
    """xfd_read_field / xfd_write_field around an odd number of single-pass
    steps (the second field set current): a cavity mode stepped 31 times
    equals the oracle; the state read back, Ez doubled and written, stepped
    30 more times equals the oracle started from that state, bitwise."""
    monkeypatch.setenv("XFD_STEP_FUSED", "1")
    n, dl = (24, 20, 16), (1e-3, 1.2e-3, 0.9e-3)
    ref = RefSim(em.cavity_spec(n, dl))
    ref.init(31)
    coeffs = {c: ref.coeff(c) for c in native.COEFF_NAMES}
    e0, _, _ = em.mode("EZ", n)
    ctx = native.Context(coeffs, "f64")
    ctx.write("EZ", e0)
    ref.write_field("EZ", e0)
    ctx.step(0, 31)
    ref.loop()
    state = {}
    for f in FIELDS:
        state[f] = ctx.read(f)
        np.testing.assert_array_equal(state[f], ref.field(f), err_msg=f)
    state["EZ"] = 2 * state["EZ"]
    ctx.write("EZ", state["EZ"])
    ctx.step(31, 30)
    ref2 = RefSim(em.cavity_spec(n, dl))
    ref2.init(30)
    for f in FIELDS:
        ref2.write_field(f, state[f])
    ref2.loop()
    for f in FIELDS:
        np.testing.assert_array_equal(ctx.read(f), ref2.field(f), err_msg=f)


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_all_slabs_inside_sweeps(monkeypatch, precision):
    """Every CPML slab applied inside the two Yee sweeps (XFD_CPML_INSWEEP=1,
    where no record lands in a slab and no ADE is present; the far grid
    planes in k_cpml_faces) against the separate slab launches, on a 136^3 box (three
    k-tiles, the last partial, with lanes of both z slabs) and on the README
    scenario (TFSF records outside the slabs).  FP64: every field and
    recording equal to the separate launches, and the README case equal to
    the oracle; FP32: as close to FP64 as the separate launches."""
    cases = {
        "box": (scenarios.inhomogeneous_box(n_total=136, pml=9, n_spheres=12, r_cells=(4, 14), seed=11,
                                            snapshot_interval=40, probes=(2, 2, 2)).spec(), 120),
        "readme": (scenarios.dielectric_sphere().spec(), 300),
    }
    for name, (sp, steps) in cases.items():
        say(f"[gpu] all slabs inside the sweeps: {name} {precision}")
        monkeypatch.setenv("XFD_CPML_INSWEEP", "1")
        ins = native.Simulation(sp, precision)
        ins.run(steps)
        assert ins.cpml_fused() == 4
        monkeypatch.setenv("XFD_CPML_INSWEEP", "0")
        monkeypatch.setenv("XFD_CPML_ZFUSED", "0")
        sep = native.Simulation(sp, precision)
        sep.run(steps)
        assert sep.cpml_fused() == 0
        if precision == "f32":
            r64 = native.Simulation(sp, "f64")
            r64.run(steps)
        for f in FIELDS:
            a, b = ins.field(f), sep.field(f)
            if precision == "f64":
                np.testing.assert_array_equal(a, b, err_msg=f"{name} {f}")
            else:
                r = r64.field(f)
                e_in, e_sep = rel_l2(a, r), rel_l2(b, r)
                say(f"  {name} {f}: in-sweep vs f64 {e_in:.2e}, separate vs f64 {e_sep:.2e}")
                assert e_in <= 2 * e_sep + 1e-6, (name, f, e_in, e_sep)
        for m in range(ins.monitor_count()):
            for q, (a, b) in enumerate(zip(ins.monitor_records(m), sep.monitor_records(m))):
                if precision == "f64":
                    np.testing.assert_array_equal(a, b, err_msg=f"{name} monitor {m}")
        if precision == "f64" and name == "readme":
            ref = RefSim(sp)
            ref.run(steps)
            for f in FIELDS:
                np.testing.assert_array_equal(ins.field(f), ref.field(f), err_msg=f)
        monkeypatch.delenv("XFD_CPML_ZFUSED", raising=False)



def test_staged_recordings(monkeypatch):
    """Recordings staged to pinned host memory at their cadence (two device
    frame slots, copies on a second stream) equal the same recordings kept on
    the device, bitwise: movies of six-field 136^3 frames every 10 steps
    (staged by default: 20 MB frames), stepped in several calls, and the
    README movie forced into staging (XFD_STAGE=1), whose frames also equal
    the oracle's."""
    big = scenarios.inhomogeneous_box(n_total=136, pml=9, n_spheres=8, r_cells=(4, 12), seed=3,
                                      snapshot_interval=10, probes=(1, 1, 1)).spec()
    readme = scenarios.dielectric_sphere().spec()
    for name, sp, steps, force in (("box", big, 95, None), ("readme", readme, 400, "1")):
        say(f"[gpu] staged recordings: {name}")
        runs = {}
        for mode in (force or "", "0"):
            if mode:
                monkeypatch.setenv("XFD_STAGE", mode)
            else:
                monkeypatch.delenv("XFD_STAGE", raising=False)
            sim = native.Simulation(sp, "f64")
            sim.init(steps)
            for t0 in range(0, steps, 37):  # several calls, frames across their ends
                sim.advance(t0, min(37, steps - t0))
            sim.finish()
            runs[mode or "default"] = [sim.monitor_records(m) for m in range(sim.monitor_count())]
            sim.close()
        a, b = list(runs.values())
        nframes = 0
        for ra, rb in zip(a, b):
            assert len(ra) == len(rb)
            for x, y in zip(ra, rb):
                np.testing.assert_array_equal(x, y)
                nframes += 1
        say(f"  {name}: {nframes} recordings equal")
        if name == "readme":
            ref = RefSim(sp)
            ref.run(steps)
            for x, y in zip(a[0], ref.monitor_records(0)):
                np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("dim", [3, 1])
def test_lumped_elements_at_the_far_planes_fp64(dim):
    """Elements that reach a box's last nodes, and elements on a line, whose
    cross section is one cell: the nodes on a far plane take no correction."""
    dl, inf = 1e-3, float("inf")
    wave = S.Waveform.gaussian(10e-12, 20e-12)
    s = S.Simulation(dl, dl, dl, 0.9)
    n = [12 * dl, 10 * dl, 20 * dl]
    lo, size = (S.Vector(0, 0, 0), S.Vector(*n)) if dim == 3 else (S.Vector(-inf, -inf, 0), S.Vector(inf, inf, n[2]))
    s.addObject(S.Object("domain", S.Cube(lo, size), S.Material.createAir()))

    def box(i, j, k, di, dj, dk):
        if dim == 1:
            return S.Cube(S.Vector(-inf, -inf, k * dl), S.Vector(inf, inf, dk * dl))
        return S.Cube(S.Vector(i * dl, j * dl, k * dl), S.Vector(di * dl, dj * dl, dk * dl))

    s.addObject(S.CurrentSource("i", box(4, 7, 9, 2, 3, 2), "XP", 2.0, wave))     # to the far y plane
    s.addObject(S.VoltageSource("v", box(4, 2, 15, 2, 2, 5), "XP", 50.0, wave))   # to the far z plane
    s.addObject(S.Inductor("l", box(4, 4, 5, 2, 6, 1), "X", 1e-9))
    s.addObject(S.Resistor("r", box(4, 8, 12, 2, 2, 1), "X", 75.0))
    sp, steps = s.spec(), 80
    ref, dev = RefSim(sp), native.Simulation(sp, "f64")
    ref.run(steps)
    dev.run(steps)
    for f in FIELDS:
        np.testing.assert_array_equal(dev.field(f), ref.field(f), err_msg=f)
    assert np.abs(ref.field("EX")).max() > 0
