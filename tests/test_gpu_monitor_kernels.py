"""The DFT accumulation kernel's frequency groups (eight to a lane) and the flux
sums' shares of a plane.

DFT: a monitor's frequencies are independent of each other, so an accumulator
that holds nf of them equals, bit for bit (tolerance 0), accumulators of one
frequency each: nf on both sides of one and two groups, real and complex
fields, float32 and float64 accumulators; monitors of several lengths and
decimations in one launch, periods past the longest graph included (there the
kernel itself leaves out the monitors that are not due).

Flux: against the host's correctly rounded sum over the same accumulators.
Each of n products of the device's sum has at most 8 roundings, the sum itself
n, so |device - host| <= (n + 8) u sum(|E1 H2| + |E2 H1|) dA, u = 2^-53.
Planes of less than one block, of one share (512 cells) and one more row, and
of several shares; 1 and 20 frequencies; each normal axis.
"""
import numpy as np
import pytest

import khronos_hip as kh
from khronos_hip.boundaries import PML, Bloch
from khronos_hip.monitors import flux_from_dft

pytestmark = pytest.mark.gpu

FREQS = [0.7 + 0.04 * k for k in range(17)]


def _sim(mons, cell=(1.9, 1.3, 1.1), precision="f32", accum="f64", bloch=False):
    src = [kh.UniformSource(time_profile=kh.GaussianPulseSource(fcen=1.0, fwidth=1.5), component=c(),
                            center=[0.21 * cell[0], 0.13 * cell[1], 0.1 * cell[2]], size=[0.0] * 3, amplitude=1.0)
           for c in (kh.Ez, kh.Hx)]
    bcs = [[Bloch(1.3), Bloch(1.3)], [PML(), PML()], [PML(), PML()]] if bloch else None
    return kh.Simulation(cell_size=list(cell), resolution=10, sources=src, monitors=mons,
                         boundaries=[[0.0, 0.0] if bloch else [0.3, 0.3], [0.3, 0.3], [0.3, 0.3]],
                         boundary_conditions=bcs, precision=precision, dft_accum=accum)


def _dfts(mons, steps, **kw):
    sim = _sim(mons, **kw)
    for n in steps:
        sim.step(n)
    out = [sim.engine.read_dft(i) for i in range(len(sim.spec.dfts))]
    sim.engine.close()
    return out


def _mon(comp, freqs, dec, size=(1.9, 1.3, 0.0)):
    return kh.DFTMonitor(component=comp(), center=[0.0] * 3, size=list(size), frequencies=list(freqs), decimation=dec)


@pytest.mark.parametrize("precision,accum,bloch", [("f32", "f64", False), ("f32", "f32", False),
                                                   ("f64", "f64", False), ("f32", "f64", True)])
@pytest.mark.parametrize("nf", [1, 7, 8, 9, 16, 17])
def test_frequencies_stand_alone(nf, precision, accum, bloch):
    kw = dict(precision=precision, accum=accum, bloch=bloch)
    comps = (kh.Hy, kh.Ez)
    many = _dfts([_mon(c, FREQS[:nf], 2) for c in comps], (33,), **kw)
    ones = _dfts([_mon(c, [f], 2) for c in comps for f in (FREQS[0], FREQS[nf // 2], FREQS[nf - 1])], (33,), **kw)
    for i in range(len(comps)):
        assert np.abs(many[i]).max() > 0 and many[i].shape[-1] == nf
        for j, k in enumerate((0, nf // 2, nf - 1)):
            assert np.array_equal(many[i][..., k], ones[3 * i + j][..., 0])


@pytest.mark.parametrize("decs", [(1, 3, 5), (1, 7, 300)])
def test_monitors_of_one_launch(decs):
    mons = lambda: [_mon(kh.Hy, FREQS[:n], d, s)  # noqa: E731
                    for n, d, s in zip((3, 17, 8), decs, ((1.9, 1.3, 0.0), (0.3, 0.0, 0.0), (1.9, 1.3, 1.1)))]
    steps = (33, 1, 270)
    together = _dfts(mons(), steps)
    for i in range(3):
        alone = _dfts([mons()[i]], steps)[0]
        assert np.abs(alone).max() > 0 and np.array_equal(together[i], alone)


@pytest.mark.parametrize("nf", [1, 20])
@pytest.mark.parametrize("cell,axis", [((1.3, 1.1, 1.2), 0), ((1.2, 2.0, 2.4), 0), ((3.2, 1.4, 1.6), 1),
                                       ((3.3, 1.5, 1.2), 2), ((7.7, 6.1, 1.2), 2)])
def test_flux_shares(cell, axis, nf):
    size = [0.0 if a == axis else 2 * v for a, v in enumerate(cell)]
    mon = kh.FluxMonitor(center=[0.03] * 3, size=size, frequencies=[0.8 + 0.02 * k for k in range(nf)])
    sim = _sim([mon], cell=cell)
    sim.step(70)
    md = mon.monitor_data
    tang = md.tangential_E_monitors + md.tangential_H_monitors
    acc = [sim.read_dft(m.monitor_data) for m in tang]
    want = flux_from_dft(md, *acc, [m.monitor_data.gv for m in tang])
    got = kh.get_flux(mon)
    again = kh.get_flux(mon)
    sim.engine.close()
    assert np.abs(want).max() > 0 and np.array_equal(got, again)
    lens = [max(np.prod(a.shape[:3]) // max(a.shape[axis], 1), 1) for a in acc]
    amp = [np.abs(np.asarray(a, np.complex128)).sum(axis=axis).reshape(-1, nf) for a in acc]
    n = min(lens)
    # sum |a||b| <= |a|_2 |b|_2, whatever cells the planes share
    s = sum(np.linalg.norm(amp[i], axis=0) * np.linalg.norm(amp[j], axis=0) for i, j in ((0, 3), (1, 2)))
    assert np.all(np.abs(got - want) <= (n + 8) * 2.0**-53 * s * 0.1 * 0.1)
