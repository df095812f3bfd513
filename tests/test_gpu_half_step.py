"""The cache-resident form of the FAST half steps (kh_half.hpp) against the pml_*
kernels (KH_PML_KERNELS=1) on the device: the same operations on the same
values, so fields, monitors and fluxes are equal bit for bit (tolerance 0).
Every comparison asserts which kernels ran (update_form): half_kernel in one run
and not in the other, but for a field group without any sigma, which steps with
the inner kernels in both and is compared as such.

Sizes around the kernel's edges: rows of an odd number of cells, of one wave
(128 cells), one less and one more, rows that start inside a wave, a last
block that is nearly empty, one-cell axes, no sigma = 0 cells at all; PML on
some axes, on none; 2D; wrapped axes in every combination with real and
complex fields; H and E sources of every form; odd and even numbers of steps,
as graphs and one by one.
"""
import math

import numpy as np
import pytest

import khronos_hip as kh
from khronos_hip.boundaries import PML, Bloch, Periodic

pytestmark = pytest.mark.gpu

COMPS = [kh.Ex, kh.Ey, kh.Ez, kh.Hx, kh.Hy, kh.Hz]


def _pulse(f=1.0):
    return kh.GaussianPulseSource(fcen=f, fwidth=1.5)


def _build(n, precision, bcs=None, pml=(3, 3, 3), sources="point", eps="lut", media=None, monitors=True, res=10):
    rng = np.random.default_rng(11)
    cell = [v / res for v in n]
    pmls = [[v / res for v in (p if isinstance(p, tuple) else (p, p))] for p in pml]
    pt = [0.07 * c for c in cell]
    if n[2] == 0:
        pmls, pt[2] = pmls[:2], 0.0
    U = lambda comp, c, size=(0.0, 0.0, 0.0): kh.UniformSource(  # noqa: E731
        time_profile=_pulse(), component=comp, center=list(c), size=list(size), amplitude=1.0)
    src = {"point": [U(kh.Ez(), pt)],
           "plane": [U(kh.Ez(), [pt[0], 0.0, 0.0], (0.0, 0.9 * cell[1], 0.9 * cell[2])), U(kh.Hy(), pt)],
           "two": [U(kh.Ez(), pt), U(kh.Ez(), pt), U(kh.Hx(), [-v for v in pt])],
           "clash": [U(kh.Hy(), pt), U(kh.Hy(), pt)]}.get(sources)
    if sources == "wave":
        kx, ky = (bcs[a][0].k if bcs and isinstance(bcs[a][0], Bloch) else 0.0 for a in (0, 1))
        k = 2 * math.pi
        src = [kh.PlaneWaveSource(time_profile=_pulse(), center=[0.0, 0.0, -0.1 * cell[2]],
                                  size=[math.inf, math.inf, 0.0], k_vector=[-kx / k, -ky / k, 0.9])]
    geo = []
    if eps == "lut":
        geo = [kh.Object(kh.Box([0.0, 0.1 * cell[1], 0.0], [0.5 * cell[0], 0.3 * cell[1], 9.0]), kh.Material(ε=4.0)),
               kh.Object(kh.Box([0.0] * 3, [99.0] * 3), kh.Material(ε=1.7))]
    elif eps == "array":
        for _ in range(300):
            c = [float(rng.uniform(-0.5, 0.5)) * v for v in cell]
            geo.append(kh.Object(kh.Box(c, [0.35, 0.35, 0.35]), kh.Material(ε=float(rng.uniform(1.2, 9.0)))))
    if media:
        geo.insert(0, kh.Object(kh.Sphere([0.0] * 3, 0.3 * min(v for v in cell if v)),
                                kh.Material(ε=2.0, chi3=0.5, susceptibilities=[
                                    kh.LorentzianSusceptibility(1.1, 0.1, 0.6)])))
    mons = []
    if monitors:
        mons = [kh.DFTMonitor(component=c(), center=[0.0] * 3, size=[cell[0], cell[1], 0.0], frequencies=[0.8, 1.1],
                              decimation=3) for c in (kh.Ez, kh.Hx)]
        mons.append(kh.DFTMonitor(component=kh.Ez(), center=[0.0] * 3, size=[0.5, 0.0, 0.0], frequencies=[0.9]))
    return kh.Simulation(cell_size=cell, resolution=res, sources=src, geometry=geo, monitors=mons, boundaries=pmls,
                         boundary_conditions=bcs, precision=precision)


def _state(sim):
    return [sim.read_field(C()) for C in COMPS] + [sim.engine.read_dft(i) for i in range(len(sim.spec.dfts))]


def _groups_with_sigma(sim):
    """Bit 0 (H), bit 1 (E): some sigma the kernels read is not zero."""
    sig = sim.spec.sigma or {}
    return sum(1 << bit for bit, key in enumerate("BD")
               if any(s is not None and np.any(np.asarray(s)[0:2 * n:2]) for s, n in zip(sig.get(key, ()), sim.spec.N)))


def _compare(monkeypatch, runs, half=None, build=_build, **kw):
    out = []
    for split in ("1", "0"):
        monkeypatch.setenv("KH_PML_KERNELS", split)
        sim = build(**kw)
        got = []
        for n in runs:
            sim.step(n)
            got += _state(sim)
        out.append(got)
        want = 0 if split == "1" else _groups_with_sigma(sim) if half is None else half
        assert sim.engine.update_form() == want
        sim.engine.close()
    assert any(np.abs(a).max() > 0 for a in out[0])
    for a, b in zip(*out):
        assert np.array_equal(a, b), np.abs(a - b).max()


per, pml_ = [Periodic(), Periodic()], [PML(), PML()]


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("n", [(13, 9, 11), (128, 5, 6), (127, 7, 5), (129, 6, 4), (64, 8, 7), (1, 12, 9), (20, 1, 1),
                               (258, 3, 8), (40, 33, 28)])
def test_sizes(monkeypatch, n, precision):
    _compare(monkeypatch, [1, 2, 20], n=n, precision=precision, pml=tuple(min(3, v // 3) for v in n))


@pytest.mark.parametrize("kw", [
    dict(pml=(0, 0, 0)), dict(pml=(4, 0, 0)), dict(pml=(0, 4, 0)), dict(pml=(0, 0, 4)), dict(pml=(7, 7, 7)),
    dict(eps="none"), dict(eps="array"), dict(sources="plane"), dict(sources="two"), dict(sources="clash"),
    dict(media=True), dict(monitors=False, sources="plane"), dict(n=(37, 26, 0)), dict(n=(37, 26, 0), sources="two"),
], ids=lambda kw: "-".join(f"{k}={v}" for k, v in kw.items()).replace(" ", ""))
@pytest.mark.parametrize("precision", ["f32", "f64"])
def test_forms(monkeypatch, kw, precision):
    _compare(monkeypatch, [17, 33, 1], **{**dict(n=(35, 22, 19), precision=precision), **kw})


@pytest.mark.parametrize("bloch", [False, True])
@pytest.mark.parametrize("axes", ["x", "y", "z", "xy", "yz", "xz", "xyz"])
@pytest.mark.parametrize("sources", ["point", "two", "wave"])
@pytest.mark.parametrize("n,precision", [((20, 13, 12), "f32"), ((21, 12, 13), "f32"), ((129, 6, 9), "f32"),
                                         ((20, 13, 12), "f64"), ((21, 12, 13), "f64")])
def test_wrapped_axes(monkeypatch, n, precision, sources, axes, bloch):
    bcs = [([Bloch(k=0.7 + a)] * 2 if bloch and "xyz"[a] in axes[:2] else per) if "xyz"[a] in axes else pml_
           for a in range(3)]
    _compare(monkeypatch, [16, 5, 1], n=n, precision=precision, bcs=bcs, sources=sources, media=(n[0] == 20),
             pml=tuple(0 if "xyz"[a] in axes else 2 for a in range(3)))


def _conductor(group, precision, bloch):
    """A block with material conductivity of one field group only."""
    mat = kh.Material(ε=2.0, σD=1.3) if group == "E" else kh.Material(ε=2.0, σB=0.8)
    src = [kh.UniformSource(time_profile=_pulse(), component=c(), center=[0.3, -0.2, 0.1], size=[0.0] * 3)
           for c in (kh.Ez, kh.Hx)]
    bcs = [[Bloch(k=0.7)] * 2, pml_, pml_] if bloch else None
    mon = kh.DFTMonitor(component=kh.Ez(), center=[0.0] * 3, size=[1.0, 0.8, 0.0], frequencies=[0.8, 1.1])
    return kh.Simulation(cell_size=[2.1, 1.4, 1.6], resolution=10, sources=src, monitors=[mon],
                         geometry=[kh.Object(kh.Box([0.2, 0.0, 0.0], [0.8, 0.7, 0.5]), mat)],
                         boundaries=[[0.0 if bloch else 0.3] * 2, [0.3] * 2, [0.3] * 2], boundary_conditions=bcs,
                         precision=precision)


@pytest.mark.parametrize("bloch", [False, True])
@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("group,half", [("E", 1), ("H", 2)])
def test_conductivity_in_one_group(monkeypatch, group, half, precision, bloch):
    """The conductive group keeps the pml kernels and their C stage, the other
    steps with half_kernel."""
    _compare(monkeypatch, [17, 20, 1], half=half, build=_conductor, group=group, precision=precision, bloch=bloch)


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("side", [(4, 0), (0, 4)], ids=["low", "high"])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_inner_box_with_one_slab(monkeypatch, axis, side, precision):
    """KH_INNER=1 with PML on one side of one axis: an inner box and one slab.
    The slab is not the whole grid, so half_kernel must leave it alone."""
    monkeypatch.setenv("KH_INNER", "1")
    _compare(monkeypatch, [1, 2, 20], half=0, n=(20, 12, 16), precision=precision,
             pml=tuple(side if a == axis else 0 for a in range(3)))


@pytest.mark.parametrize("n,precision,pml,pole,form", [
    ((40, 30, 20), "f32", 5, False, 3),
    # the same 168^3 state (400 MB of arrays): thin PML, thick PML
    ((168, 168, 168), "f32", 10, False, 3), ((168, 168, 168), "f32", 24, False, 0),
    # 144^3: the material pass's arrays count, the padding of rows does not
    ((144, 144, 144), "f32", 10, False, 3), ((144, 144, 144), "f32", 10, True, 0),
    ((144, 144, 144), "f64", 10, False, 3), ((192, 192, 192), "f32", 10, False, 0),
], ids=str)
def test_line_between_the_forms(n, precision, pml, pole, form):
    """half_kernel runs where a step touches at most 195 MB: fields, stages in
    the PML and the material pass's box, without the rows' padding."""
    cell = [v / 20 for v in n]
    sus = [kh.LorentzianSusceptibility(1.1, 0.1, 0.6)] if pole else []
    geo = [kh.Object(kh.Box([0.0] * 3, [0.95 * v for v in cell]), kh.Material(ε=2.0, susceptibilities=sus))]
    src = kh.UniformSource(time_profile=_pulse(), component=kh.Ez(), center=[0.0] * 3, size=[0.0] * 3)
    sim = kh.Simulation(cell_size=cell, resolution=20, sources=[src], geometry=geo if pole else [],
                        boundaries=[[pml / 20] * 2] * 3, precision=precision, setup_precision="f64")
    sim.step(1)
    assert sim.engine.update_form() == form
    sim.engine.close()


def test_contexts_in_flight_share_the_line(monkeypatch):
    """Two 144^3 float states, about 102 MB a step each: one alone steps with
    half_kernel, both at once with the pml kernels, chosen anew by every call.
    A run that changes form between steps and graphs gives the same bits."""
    kw = dict(n=(144, 144, 144), precision="f32", pml=(10, 10, 10), eps="none", res=20)
    monkeypatch.setenv("KH_PML_KERNELS", "1")
    ref = _build(**kw)
    ref.step(83)
    want = _state(ref)
    assert ref.engine.update_form() == 0
    ref.engine.close()
    monkeypatch.delenv("KH_PML_KERNELS")
    a, b = _build(**kw), _build(**kw)
    forms = []
    a.step(16)                        # alone
    forms.append(a.engine.update_form())
    b.step(33)                        # beside a's steps
    forms.append(b.engine.update_form())
    a.engine.sync()
    b.step(17)                        # a has finished
    forms.append(b.engine.update_form())
    a.step(35)                        # beside b's
    forms.append(a.engine.update_form())
    got_b = b.read_field(kh.Ez())     # waits for b
    a.step(32)
    forms.append(a.engine.update_form())
    b.engine.close()                  # a is in flight, b is gone
    a.step(0)
    assert forms == [3, 0, 3, 0, 3] and np.abs(got_b).max() > 0
    for x, y in zip(want, _state(a)):
        assert np.array_equal(x, y)
    a.engine.close()


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("scale,form", [(1.0, 3), (-0.5, 0), (1e9, 0), (math.nan, 0)], ids=str)
def test_sigma_outside_the_quotients_range(monkeypatch, scale, form, precision):
    """half_kernel's quotients hold for 0 <= sigma <= 2^20; any other profile (as
    kh_create takes it) steps with the pml kernels."""
    import khronos_hip.boundaries as bnd
    plain = bnd.compute_sigma
    monkeypatch.setattr(bnd, "compute_sigma", lambda *a: plain(*a) * a[-1](scale))
    sim = _build((20, 14, 13), precision)
    sim.step(2)
    assert sim.engine.update_form() == form
    sim.engine.close()


@pytest.mark.parametrize("precision", ["f32", "f64"])
def test_values_the_quotients_special_case(monkeypatch, precision):
    """Zeros of both signs, infinities, NaN, the largest and the smallest numbers
    and values around the guard for tiny ones, written into the fields of a grid
    that is all PML: the same values, and NaN in the same places."""
    dt, guard = (np.float32, -100) if precision == "f32" else (np.float64, -960)
    info = np.finfo(dt)
    special = [0.0, -0.0, info.smallest_subnormal, info.tiny, 2.0 ** guard, np.nextafter(dt(2.0 ** guard), dt(0)),
               1.5 * 2.0 ** guard, -(2.0 ** (guard - 1)), 2.0 ** (guard + 1), 1.0]
    for wild in ([], [info.max, -info.max], [np.inf], [np.nan, -np.inf, info.max]):
        out = []
        for split in ("1", "0"):
            monkeypatch.setenv("KH_PML_KERNELS", split)
            sim = _build((21, 14, 13), precision, pml=(7, 7, 7), monitors=False)
            rng = np.random.default_rng(7)
            sim.step(1)
            for code in range(6):
                shape = sim.engine.field_shape(code)
                v = rng.choice(np.array(special + [-x for x in special], dt), size=shape)
                for k, x in enumerate(wild):
                    v[3 + 4 * k, 5, 6] = x
                sim.engine.write_field(code, v)
            got = []
            for n in (1, 1, 3):
                sim.step(n)
                got += _state(sim)
            out.append(got)
            assert sim.engine.update_form() == (3 if split == "0" else 0)
            sim.engine.close()
        for a, b in zip(*out):
            assert np.array_equal(a, b, equal_nan=True)
            assert np.array_equal(np.signbit(a[a == 0]), np.signbit(b[a == 0]))


def test_written_ghosts_reset_and_single_steps(monkeypatch):
    """Fields written from the host (ghosts included), single steps and graphs,
    and a reset in between."""
    out = []
    for split in ("1", "0"):
        monkeypatch.setenv("KH_PML_KERNELS", split)
        sim = _build((22, 15, 14), "f32")
        rng = np.random.default_rng(3)
        sim.step(3)
        for code in range(6):
            sim.engine.write_field(code, rng.standard_normal(sim.engine.field_shape(code)))
        got = []
        for n in (1, 1, 1, 20, 1, 33):
            sim.step(n)
            got += _state(sim)
        kh.reset_fields(sim)
        for n in (1, 18, 1, 1):
            sim.step(n)
            got += _state(sim)
        out.append(got)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
