"""The material pass's read-ahead of its first two poles against poles it reads
one by one: splitting a cell's poles over more of them changes neither the
sum's order nor a value when the extra poles are zero at the front or the back.

Adding a pole whose sigma is zero everywhere but in one far cell adds an exact
0 to fPD at every other cell; so the fields of a run with that pole put first,
last, or left out are equal bit for bit (tolerance 0) as long as nothing has
reached the far cell, while the real poles move from the read-ahead slots to
the loop behind them.  1, 2 and 3 real poles, with and without chi3, real and
complex fields, both precisions, FAST and EXACT.
"""
import numpy as np
import pytest

import khronos_hip as kh
from khronos_hip.boundaries import PML, Bloch

pytestmark = pytest.mark.gpu


def _run(npole, front, back, precision, mode, bloch, chi3):
    cell = [1.7, 1.5, 2.3]
    real = [kh.LorentzianSusceptibility(0.9 + 0.2 * k, 0.1, 0.4 + 0.1 * k) for k in range(npole)]
    # poles are told apart by omega and gamma: these belong to the far object only
    far = [kh.LorentzianSusceptibility(2.0 + 0.1 * k, 0.05, 0.3) for k in range(front + back)]
    near_obj = kh.Object(kh.Sphere([0.0, 0.0, 0.3], 0.45),
                         kh.Material(ε=2.0, chi3=0.5 if chi3 else 0.0, susceptibilities=real))
    far_objs = [kh.Object(kh.Sphere([0.0, 0.0, -1.05], 0.11), kh.Material(ε=1.0, susceptibilities=[f])) for f in far]
    geo = far_objs[:front] + [near_obj] + far_objs[front:]
    bcs = [[Bloch(1.3), Bloch(1.3)], [PML(), PML()], [PML(), PML()]] if bloch else None
    src = kh.UniformSource(time_profile=kh.GaussianPulseSource(fcen=1.0, fwidth=1.5), component=kh.Ez(),
                           center=[0.1, 0.0, 0.7], size=[0.0] * 3, amplitude=3.0)
    sim = kh.Simulation(cell_size=cell, resolution=10, sources=[src], geometry=geo, mode=mode, precision=precision,
                        boundaries=[[0.0, 0.0] if bloch else [0.3, 0.3], [0.3, 0.3], [0.0, 0.0]],
                        boundary_conditions=bcs)
    sim.step(13)  # the source is 17 cells from the far object
    out = [sim.read_field(C()) for C in (kh.Ex, kh.Ey, kh.Ez, kh.Hx, kh.Hy, kh.Hz)]
    n = len(sim.spec.poles)
    sim.engine.close()
    return out, n


@pytest.mark.parametrize("bloch", [False, True])
@pytest.mark.parametrize("precision,mode,chi3", [("f64", "fast", False), ("f32", "fast", True), ("f32", "exact", True)])
@pytest.mark.parametrize("npole", [1, 2, 3])
def test_pole_slots(npole, precision, mode, chi3, bloch):
    base, n0 = _run(npole, 0, 0, precision, mode, bloch, chi3)
    assert n0 == npole and np.abs(base[2]).max() > 0
    for front, back in ((1, 0), (2, 0), (0, 2)):
        got, n = _run(npole, front, back, precision, mode, bloch, chi3)
        assert n == npole + front + back
        for a, b in zip(base, got):
            assert np.array_equal(a, b), np.abs(a - b).max()


def _layers(order, npole, precision, mode, bloch, rewrite):
    """Boxes side by side, box k with pole k alone, and one with every pole."""
    poles = [kh.LorentzianSusceptibility(0.9 + 0.2 * k, 0.1, 0.4 + 0.1 * k) for k in range(npole)]
    box = lambda k: kh.Box([0.0, 0.0, -0.55 + 0.3 * k], [0.9, 0.8, 0.29])  # noqa: E731
    geo = [kh.Object(box(k), kh.Material(ε=2.0, susceptibilities=[poles[k]])) for k in order]
    geo.append(kh.Object(box(npole), kh.Material(ε=1.5, chi3=0.5, susceptibilities=poles)))
    bcs = [[Bloch(1.3), Bloch(1.3)], [PML(), PML()], [PML(), PML()]] if bloch else None
    src = kh.UniformSource(time_profile=kh.GaussianPulseSource(fcen=1.0, fwidth=1.5), component=kh.Ez(),
                           center=[0.1, 0.0, -0.1], size=[0.0] * 3, amplitude=3.0)
    sim = kh.Simulation(cell_size=[1.7, 1.5, 2.3], resolution=10, sources=[src], geometry=geo, mode=mode,
                        precision=precision, boundary_conditions=bcs,
                        boundaries=[[0.0, 0.0] if bloch else [0.3, 0.3], [0.3, 0.3], [0.3, 0.3]])
    sim.step(20)
    if rewrite:
        for k in range(npole):
            sim.engine.write_pole(k, 0, 0, sim.engine.read_pole(k, 0, 0))
    sim.step(41)
    out = [sim.read_field(C()) for C in (kh.Ex, kh.Ey, kh.Ez, kh.Hx, kh.Hy, kh.Hz)]
    sim.engine.close()
    return out


@pytest.mark.parametrize("bloch", [False, True])
@pytest.mark.parametrize("precision,mode", [("f64", "fast"), ("f32", "fast"), ("f32", "exact")])
@pytest.mark.parametrize("npole", [1, 2, 3])
def test_poles_a_cell_does_not_have(npole, precision, mode, bloch):
    """A pole is read ahead only in the cells that have it.  A cell of one pole
    gives the same fields whichever slot that pole has, the cells of all poles
    add them (two additions in any order, or the slots' order kept), and
    writing a polarization back as it is makes the pass read every pole in
    every cell: equal bit for bit (tolerance 0)."""
    kw = dict(npole=npole, precision=precision, mode=mode, bloch=bloch)
    base = _layers(range(npole), rewrite=False, **kw)
    assert np.abs(base[2]).max() > 0
    others = [_layers(range(npole), rewrite=True, **kw)]
    if npole == 2:
        others.append(_layers((1, 0), rewrite=False, **kw))
    for got in others:
        for a, b in zip(base, got):
            assert np.array_equal(a, b), np.abs(a - b).max()
