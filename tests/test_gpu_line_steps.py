"""1D grids stepped many times per launch against a launch per correction,
which the low-dimension tests hold to the oracle: the same bits in FP64 and FP32."""

import numpy as np
import pytest

from oracle import RefSim
from xfdtd_core_amd import native
from xfdtd_core_amd import spec as S

pytestmark = pytest.mark.gpu
INF = float("inf")


def _line(nz, tfsf=5, pml=8, faces=("ZN", "ZP"), movie=True, driven=()):
    """A line of nz cells and its CPML: a lossy slab, a plane wave, probes; a
    movie whose frames end a launch every 7 steps; `driven`: lumped elements by
    kind and cell count, 12 cells in."""
    dl = 1e-3
    s = S.Simulation(dl, dl, dl, 0.9)
    s.addObject(S.Object("domain", S.Cube(S.Vector(-INF, -INF, 0.0), S.Vector(INF, INF, nz * dl)),
                         S.Material.createAir()))
    lo = round(0.5 * nz) * dl
    s.addObject(S.Object("slab", S.Cube(S.Vector(-INF, -INF, lo), S.Vector(INF, INF, 0.2 * nz * dl)),
                         S.Material("m", S.ElectroMagneticProperty(3.0, 1.0, 0.02, 0.0))))
    s.addWaveformSource(S.TFSF1D(tfsf, True, S.Waveform.gaussian(20e-12, 60e-12)))
    wave = S.Waveform.gaussian(20e-12, 60e-12)
    for kind, cells in driven:
        at = S.Cube(S.Vector(-INF, -INF, 12 * dl), S.Vector(INF, INF, cells * dl))
        s.addObject({"current": lambda: S.CurrentSource("i", at, "XP", 1.0, wave),
                     "voltage": lambda: S.VoltageSource("v", at, "XP", 50.0, wave),
                     "inductor": lambda: S.Inductor("l", at, "X", 1e-9)}[kind]())
    for f in faces:
        s.addBoundary(S.PML(pml, f))
    for q, (at, comp) in enumerate(((1, "EX"), (nz // 2, "HY"), (nz - 2, "EX"))):
        cell = S.Cube(S.Vector(-INF, -INF, at * dl), S.Vector(INF, INF, dl))
        s.addMonitor(S.FieldTimeMonitor(f"p{q}", cell, "", comp))
    if movie:
        s.addMonitor(S.MovieMonitor(S.FieldMonitor(S.Cube(S.Vector(-INF, -INF, 0.0), S.Vector(INF, INF, nz * dl)),
                                                   "EX"), 7, "movie", ""))
    return s.spec()


def _compare(monkeypatch, spec, precision, steps, cuts, fast=True):
    sims = []
    for on in (True, False):
        if on:
            monkeypatch.delenv("XFD_STEP_FUSED", raising=False)
        else:
            monkeypatch.setenv("XFD_STEP_FUSED", "0")
        sim = native.Simulation(spec, precision)
        sim.init(steps)
        sim.set_profiling(True)
        for t0, t1 in zip(cuts[:-1], cuts[1:]):
            sim.advance(t0, t1 - t0)
        assert (sim.kernel_stats()["update_h"][0] == 0) == (on and fast)
        sim.finish()
        sims.append(sim)
    a, b = sims
    for f in ("EX", "EY", "EZ", "HX", "HY", "HZ"):
        np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
    for m in range(a.monitor_count()):
        for x, y in zip(a.monitor_records(m), b.monitor_records(m)):
            np.testing.assert_array_equal(x, y)
    assert np.abs(b.field("EX")).max() > 0
    return a


# 64, 1024, 2048 and 4096 nodes are the edges of the work-items and their
# cells; a TFSF face in a CPML layer keeps the separate launches
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("nz,tfsf,faces", [(30, 12, ("ZN", "ZP")), (47, 5, ("ZP", "ZN")), (48, 12, ("ZP",)),
                                           (1008, 20, ("ZN", "ZP")), (2031, 12, ("ZN", "ZP")),
                                           (4080, 12, ("ZN", "ZP")), (8000, 12, ("ZN", "ZP")), (200, 6, ())])
def test_line_steps_match_separate_launches(monkeypatch, nz, tfsf, faces, precision):
    _compare(monkeypatch, _line(nz, tfsf, faces=faces), precision, 260, (0, 1, 150, 260),
             fast=tfsf > 8 or not faces)


# no frames: whole stretches per launch.  64 steps fill the addends in LDS once,
# 4096 are a launch's most; 1, 2, 4 and 8 cells per work-item
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("nz,cuts", [(47, (0, 64, 129, 333)), (47, (0, 4096 + 77)), (1500, (0, 333)),
                                     (3000, (0, 190, 333)), (8000, (0, 333))])
def test_long_launches_match_separate_launches(monkeypatch, nz, cuts, precision):
    _compare(monkeypatch, _line(nz, 12, movie=False), precision, cuts[-1], cuts)


# sources and inductors on the line, with and without a plane wave's records on
# the same work-items; more than 32 corrected points have no addends ahead
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("nz,driven", [(47, (("current", 6),)), (47, (("voltage", 2), ("inductor", 3))),
                                       (300, (("inductor", 5),)), (300, (("current", 20),)),
                                       (300, (("current", 40),))])
def test_driven_lines_match_separate_launches(monkeypatch, nz, driven, precision):
    spec = _line(nz, 12, movie=False, driven=driven)
    sim = _compare(monkeypatch, spec, precision, 333, (0, 100, 333))
    if precision == "f64":
        ref = RefSim(spec)
        ref.run(333)
        for f in ("EX", "HY", "HZ"):
            np.testing.assert_array_equal(sim.field(f), ref.field(f), err_msg=f)


def test_device_bytes_count_the_lists_of_a_path(monkeypatch):
    """What a 1D grid stepped many times per launch holds beyond separate
    launches is counted: the addends of its TFSF corrections, 4096 steps of doubles each, and its lists."""
    held = []
    for env in ("0", None):
        monkeypatch.setenv("XFD_STEP_FUSED", env) if env else monkeypatch.delenv("XFD_STEP_FUSED", raising=False)
        sim = native.Simulation(_line(200, 12), "f64")
        sim.init(4)
        held.append(sim.device_bytes())
    assert held[1] - held[0] >= 3 * 4096 * 8
