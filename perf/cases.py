"""Performance cases of khronos_hip: the simulations its users run, small to large.

A case is a dict of plain values; ``prepare`` builds what a user's program
holds before the run (the Simulation with its device context, or the
optimisation problem), ``run`` is one whole pass through the public entry
points and returns what the run is for (DFT fields, fluxes, gradients, far
fields), ``work`` the bytes the pass cannot do without and ``exact`` the same
outputs in float64 from a plain torch Yee solver.

Kinds:
  fdtd      a time-domain run from zero fields: ``scene`` is what is in the
            cell, ``monitor`` what is recorded, ``loop`` how it is stopped
            ("steps": a known end time, "decay": the DFT-decay callback
            with a minimum run time, asked after every step)
  gradient  objective and design gradient of the 2D bend (time-reversed adjoint)
  farfield  near-to-far projection of a recorded surface

Scenes: "vacuum"; "solids" (1-3 boxes or spheres, the serving requests);
"smooth" (the same, anisotropic subpixel smoothing); "strip" (silicon strip
waveguide, planar Gaussian source); "drude" (a Drude + Lorentz sphere, real
fields); "lattice" (Bloch-periodic x/y, cylinders with two Lorentz poles and
chi3, plane-wave source, complex fields).
"""
import math
import os
import sys

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "khronos.jl_amd"))

import khronos_hip as kh  # noqa: E402
from khronos_hip import workloads  # noqa: E402
from khronos_hip.boundaries import PML, Bloch  # noqa: E402
from khronos_hip.smoothing import AnisotropicSmoothing  # noqa: E402

LATTICE_W0 = (0.9, 1.3)
LATTICE_GAMMA = 0.05


def _fdtd(name, nx, ny, nz, precision, steps, scene, monitor, n_freq, resolution=20, pml=10, loop="steps",
          snapshot=True):
    return {"name": name, "kind": "fdtd", "nx": nx, "ny": ny, "nz": nz, "precision": precision, "steps": steps,
            "scene": scene, "monitor": monitor, "n_freq": n_freq, "resolution": resolution, "pml": pml, "loop": loop,
            "snapshot": snapshot}


def listed():
    return [
        # a 2D study (nz = 0), the smallest thing a user runs: launches and latency only
        _fdtd("planar_2d_f64", 96, 81, 0, "f64", 400, "solids", "plane", 3, pml=12),
        # run(until=stop_when_dft_decayed()): one step per callback, on a small cell
        _fdtd("decay_loop_48_f32", 48, 45, 40, "f32", 300, "solids", "plane", 5, pml=8, loop="decay"),
        # the plain double-precision point dipole: 80^3, a 5-frequency DFT plane, 500 steps
        _fdtd("dipole_80_f64", 80, 80, 80, "f64", 500, "vacuum", "plane", 5),
        # a small serving request: 64^3, a 20-frequency flux plane, 1000 steps
        _fdtd("request_64_f32", 64, 64, 64, "f32", 1000, "solids", "flux", 20),
        # a serving request of a ragged size
        _fdtd("request_ragged_f32", 131, 117, 101, "f32", 500, "solids", "flux", 20),
        # the largest serving grid: the GPU's bandwidth is the limit
        _fdtd("request_256_f32", 256, 256, 256, "f32", 300, "solids", "flux", 20, snapshot=False),
        # smoothed materials with more distinct values than a byte can index
        _fdtd("smooth_spheres_f32", 160, 145, 120, "f32", 400, "smooth", "flux", 20),
        # the headline workload: the strip waveguide, two flux planes at 50 frequencies
        _fdtd("strip_f32", 384, 192, 160, "f32", 400, "strip", "flux", 50, pml=12, snapshot=False),
        # dispersive metal in double precision: poles, real fields
        _fdtd("drude_96_f64", 96, 75, 64, "f64", 300, "drude", "plane", 9),
        # the periodic dispersive metasurface: Bloch phases, complex fields, poles and chi3
        _fdtd("lattice_c32", 128, 128, 192, "f32", 160, "lattice", "flux", 100, resolution=32, pml=16,
              snapshot=False),
        # inverse design: objective and gradient of the 400 x 400 bend, 120 x 120 parameters
        {"name": "bend_gradient_f32", "kind": "gradient", "n_design": 120, "resolution": 40, "steps": 1000,
         "every": 100, "precision": "f32"},
        # radiation pattern: a recorded surface projected to a hemisphere of directions
        {"name": "farfield_128", "kind": "farfield", "nx": 128, "ny": 120, "n_theta": 46, "n_phi": 37, "n_freq": 5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["planar", "loop", "vacuum", "solids", "solids", "smooth", "strip", "drude", "lattice",
                       "gradient", "farfield"])
    prec = rng.choice(["f32", "f64"])
    if kind == "gradient":
        return {"kind": "gradient", "n_design": rng.randint(30, 120), "resolution": 40,
                "steps": rng.randint(300, 1000), "every": rng.choice([50, 100]), "precision": prec}
    if kind == "farfield":
        return {"kind": "farfield", "nx": rng.randint(40, 128), "ny": rng.randint(40, 120),
                "n_theta": rng.randint(8, 46), "n_phi": rng.randint(8, 37), "n_freq": rng.randint(1, 5)}
    if kind == "planar":
        return _fdtd("", rng.randint(60, 300), rng.randint(60, 300), 0, prec, rng.randint(100, 600), "solids", "plane",
                     rng.randint(1, 9), pml=rng.randint(8, 14)) | {"name": "drawn planar"}
    if kind == "loop":
        return _fdtd("drawn loop", rng.randint(32, 64), rng.randint(32, 64), rng.randint(32, 64), prec,
                     rng.randint(100, 300), "solids", "plane", rng.randint(1, 9), pml=8, loop="decay")
    if kind == "lattice":
        n = 32 * rng.randint(2, 4)
        return _fdtd("drawn lattice", n, n, rng.randint(80, 192), "f32", rng.randint(120, 160), "lattice", "flux",
                     rng.randint(5, 100), resolution=32, pml=16, snapshot=False)
    hi = {"vacuum": 100, "solids": 256, "smooth": 160, "strip": 160, "drude": 96}[kind]
    n = [_log(rng, 48, hi) for _ in range(3)]
    if kind == "strip":
        n[0] = min(384, 2 * n[0])
    cells = n[0] * n[1] * n[2]
    top = 2.0e9 if prec == "f32" else 1.0e9
    steps = max(40, min(rng.randint(100, 1000), int(top / cells)))
    return _fdtd("drawn " + kind, n[0], n[1], n[2], prec, steps, kind, rng.choice(["plane", "flux"]),
                 rng.randint(1, 50), pml=rng.randint(8, 12), snapshot=cells < 3_000_000)


# ------------------------------------------------------------------ scenes
def _scene(case, seed):
    """Plain numbers of a case's set-up, shared by the framework's run and the float64 solver."""
    r = np.random.default_rng([int(seed), 77])
    res = case["resolution"]
    two_d = case["nz"] == 0
    n = (case["nx"], case["ny"], case["nz"])
    cell = [v / res for v in n]
    pml = case["pml"] / res
    half = [c / 2 - pml for c in cell]
    s = {"cell": cell, "n": n, "res": res, "pml": pml, "objects": [], "poles": [], "fcen": 1.0, "fwidth": 0.5,
         "bloch": None, "dt": 0.5 / res}
    scene = case["scene"]
    u = lambda lo, hi: float(r.uniform(lo, hi))  # noqa: E731
    if scene in ("solids", "smooth"):
        for _ in range(int(r.integers(1, 4))):
            eps = u(1.5, 12.0)
            c = [u(-0.25, 0.25) * v for v in cell]
            if two_d:
                c[2] = 0.0
            if r.random() < 0.5:
                size = [u(0.1, 0.3) * v for v in cell]
                if two_d:
                    size[2] = 1.0
                s["objects"].append(("box", c, size, eps))
            else:
                s["objects"].append(("sphere", c, u(0.08, 0.15) * min(v for v in cell if v), eps))
    elif scene == "strip":
        s["fcen"], s["fwidth"] = 1 / 1.55, 0.5
        w, h = u(0.45, 0.55), u(0.2, 0.24)
        s["objects"] = [("box", [0.0, 0.0, 0.0], [2 * cell[0], w, h], 12.1),
                        ("box", [0.0, 0.0, 0.0], [2 * v for v in cell], 2.085)]
    elif scene == "drude":
        c = [u(-0.1, 0.1) * v for v in cell]
        rad = u(0.15, 0.22) * min(cell)
        s["objects"] = [("sphere", c, rad, u(1.5, 3.0))]
        s["poles"] = [(0.0, u(0.02, 0.1), [u(20.0, 60.0)]), (u(0.9, 1.4), 0.05, [u(0.3, 1.0)])]
    elif scene == "lattice":
        lx, ly = case["nx"] // 32, case["ny"] // 32
        s["bloch"] = (u(-math.pi, math.pi), u(-math.pi, math.pi))
        sig = ([], [])
        for i in range(lx):
            for j in range(ly):
                c = [-cell[0] / 2 + i + 0.5, -cell[1] / 2 + j + 0.5, 0.0]
                s["objects"].append(("cylinder", c, u(0.2, 0.4), 0.5, 2.0))
                for q in sig:
                    q.append(u(0.5, 2.0))
        s["poles"] = [(w0, LATTICE_GAMMA, q) for w0, q in zip(LATTICE_W0, sig)]
        s["chi3"] = 1e-3
    f, w = s["fcen"], s["fwidth"]
    s["freqs"] = [float(v) for v in np.linspace(f - w / 4, f + w / 4, case["n_freq"])]
    jit = [u(-0.45, 0.45) / res for _ in range(3)]  # sources and monitors lie anywhere between grid points
    if two_d:
        jit[2] = 0.0
    if scene == "strip":
        s["source"] = {"kind": "gauss", "comp": "Ez", "center": [-half[0] * 0.8 + jit[0], 0.0, 0.0],
                       "size": [0.0, 1.8 * half[1] + jit[1] / 4, 1.7 * half[2] + jit[2] / 4], "waist": 1.0}
        planes = [-0.6 * half[0] + jit[1], -0.35 * half[0] + jit[2]]
        s["flux"] = [([x, 0.0, 0.0], [0.0, 1.8 * half[1] + jit[0] / 4, 1.7 * half[2] + jit[1] / 4]) for x in planes]
    elif scene == "lattice":
        k = 2 * math.pi * f
        kx, ky = s["bloch"]
        kv = [-kx / k, -ky / k, math.sqrt(max(0.0, 1 - (kx * kx + ky * ky) / (k * k)))]
        s["source"] = {"kind": "wave", "center": [0.0, 0.0, -0.5 + jit[2]], "k": kv}
        s["flux"] = [([0.0, 0.0, 0.45 + jit[0]], [cell[0], cell[1], 0.0])]
    else:
        s["source"] = {"kind": "point", "comp": "Ez", "center": [j + 0.1 * h for j, h in zip(jit, half)]}
        if two_d:
            s["source"]["center"][2] = 0.0
        s["flux"] = [([0.55 * half[0] + jit[1], 0.0, 0.0], [0.0, 2 * half[1] - abs(jit[0]), 2 * half[2] - abs(jit[2])])]
    s["plane"] = ([0.0, 0.0, jit[1] if not two_d else 0.0],
                  [cell[0] - 0.3 / res, cell[1] - 0.3 / res, 0.0])
    return s


def _simulation(case, s):
    geo = []
    for i, o in enumerate(s["objects"]):
        sus = [kh.LorentzianSusceptibility(w0, g, q[i]) for w0, g, q in s["poles"] if i < len(q)]
        mat = kh.Material(ε=o[-1], chi3=s.get("chi3"), susceptibilities=sus)
        if o[0] == "box":
            shape = kh.Box(o[1], o[2])
        elif o[0] == "sphere":
            shape = kh.Sphere(o[1], o[2])
        else:
            shape = kh.Cylinder(o[1], o[2], o[3], axis=2)
        geo.append(kh.Object(shape, mat))
    tp = kh.GaussianPulseSource(fcen=s["fcen"], fwidth=s["fwidth"])
    q = s["source"]
    if q["kind"] == "point":
        src = kh.UniformSource(time_profile=tp, component=kh.Ez(), center=q["center"], size=[0.0, 0.0, 0.0])
    elif q["kind"] == "gauss":
        src = kh.GaussianProfileSource(time_profile=tp, component=kh.Ez(), center=q["center"], size=q["size"],
                                       waist=q["waist"])
    else:
        src = kh.PlaneWaveSource(time_profile=tp, center=q["center"], size=[math.inf, math.inf, 0.0], k_vector=q["k"])
    if case["monitor"] == "plane":
        mons = [kh.DFTMonitor(component=kh.Ez(), center=s["plane"][0], size=s["plane"][1], frequencies=s["freqs"])]
    else:
        mons = [kh.FluxMonitor(center=c, size=z, frequencies=s["freqs"]) for c, z in s["flux"]]
    pml = s["pml"]
    kw = {}
    if s["bloch"]:
        kx, ky = s["bloch"]
        kw["boundary_conditions"] = [[Bloch(k=kx), Bloch(k=kx)], [Bloch(k=ky), Bloch(k=ky)], [PML(), PML()]]
        bnd = [[0.0, 0.0], [0.0, 0.0], [pml, pml]]
    else:
        bnd = [[pml, pml]] * (2 if case["nz"] == 0 else 3)
    if case["scene"] == "smooth":
        kw["subpixel_smoothing"] = AnisotropicSmoothing()
    if case["scene"] in ("smooth", "strip"):
        kw["raster"] = "device"
    sim = kh.Simulation(cell_size=s["cell"], resolution=s["res"], sources=[src], geometry=geo, monitors=mons,
                        boundaries=bnd, precision=case["precision"], setup_precision="f64", **kw)
    assert (sim.Nx, sim.Ny, sim.Nz) == s["n"], (sim.Nx, sim.Ny, sim.Nz, s["n"])
    return sim, mons


def _bend(case):
    opt, _ = workloads.adjoint_bend(precision=case["precision"], setup_precision="f64", n_design=case["n_design"],
                                    resolution=case["resolution"], steps=case["steps"],
                                    checkpoint_every=case["every"])
    return opt


def _surface(case, seed):
    """The far-field case's recording run: a small source box under a z-normal surface."""
    r = np.random.default_rng([int(seed), 78])
    res, pad, nz = 32, 12, 48
    n = (case["nx"] + 2 * pad, case["ny"] + 2 * pad, nz)
    u = lambda lo, hi: float(r.uniform(lo, hi))  # noqa: E731
    s = {"cell": [v / res for v in n], "n": n, "res": res, "pml": pad / res, "objects": [], "poles": [],
         "fcen": 1.0, "fwidth": 0.5, "bloch": None, "dt": 0.5 / res,
         "freqs": [float(v) for v in np.linspace(0.9, 1.1, case["n_freq"])],
         "source": {"kind": "point", "comp": "Ez", "center": [u(-0.4, 0.4), u(-0.4, 0.4), u(-0.1, 0.05)]}}
    s["flux"] = [([0.0, 0.0, 0.25 + u(0.1, 0.4) / res],
                  [(case["nx"] - 1.3) / res, (case["ny"] - 1.3) / res, 0.0])]
    s["theta"] = [float(v) for v in np.radians(np.linspace(1.0, 89.0, case["n_theta"]))]
    s["phi"] = [float(v) for v in np.radians(np.linspace(0.0, 351.0, case["n_phi"]))]
    s["obs_r"] = 200.0
    return s


SURFACE_STEPS = 160


# ------------------------------------------------------------------ protocol
def prepare(case, seed):
    if case["kind"] == "gradient":
        opt = _bend(case)
        rho = np.random.default_rng([int(seed), 79]).random(case["n_design"] ** 2)
        return {"case": case, "opt": opt, "rho": rho}
    if case["kind"] == "farfield":
        s = _surface(case, seed)
        mon = kh.Near2FarMonitor(center=s["flux"][0][0], size=s["flux"][0][1], frequencies=s["freqs"],
                                 theta=s["theta"], phi=s["phi"], r=s["obs_r"])
        src = kh.UniformSource(time_profile=kh.GaussianPulseSource(fcen=1.0, fwidth=0.5), component=kh.Ez(),
                               center=s["source"]["center"], size=[0.0, 0.0, 0.0])
        sim = kh.Simulation(cell_size=s["cell"], resolution=s["res"], boundaries=[[s["pml"]] * 2] * 3,
                            sources=[src], monitors=[mon], precision="f32", setup_precision="f64")
        kh.run(sim, until=(SURFACE_STEPS - 0.5) * sim.dt_n)
        return {"case": case, "sim": sim, "mon": mon}
    sim, mons = _simulation(case, _scene(case, seed))
    sim.prepare()
    return {"case": case, "sim": sim, "mons": mons}


def run(state):
    case = state["case"]
    if case["kind"] == "gradient":
        f0, g = state["opt"](state["rho"])
        return {"objective": f0, "gradient": g}
    if case["kind"] == "farfield":
        return {"far": kh.compute_far_field(state["mon"])}
    sim = state["sim"]
    kh.reset_fields(sim)
    until = (case["steps"] - 0.5) * sim.dt_n
    if case["loop"] == "decay":
        kh.run(sim, until=kh.stop_when_dft_decayed(minimum_runtime=until, maximum_runtime=until))
    else:
        kh.run(sim, until=until)
    if case["monitor"] == "plane":
        out = {"dft": [m.monitor_data.fields for m in state["mons"]]}
    else:
        out = {"flux": [kh.get_flux(m) for m in state["mons"]]}
    if case["snapshot"]:
        out["ez"] = sim.read_field(kh.Ez())
    return out


def work(case):
    """Per step: each field of a cell read and written once, PML auxiliaries of
    the shell likewise, a byte of material index per component where there are
    materials; two flops per difference and update term."""
    if case["kind"] == "farfield":
        evals = 4.0 * case["nx"] * case["ny"] * case["n_theta"] * case["n_phi"] * case["n_freq"]
        return {"bytes": 4 * 16.0 * case["nx"] * case["ny"] * case["n_freq"], "flops": 130.0 * evals}
    if case["kind"] == "gradient":
        n = case["n_design"] + 7 * case["resolution"]
        cells, s, passes = n * n, 4 if case["precision"] == "f32" else 8, 3  # forward, re-run, walk back
        return {"bytes": float(passes * case["steps"] * cells * 12 * s), "flops": float(passes * case["steps"] * cells * 60)}
    n = [case["nx"], case["ny"], max(1, case["nz"])]
    cells = n[0] * n[1] * n[2]
    s = 4 if case["precision"] == "f32" else 8
    parts = 2 if case["scene"] == "lattice" else 1
    axes = [2] if case["scene"] == "lattice" else ([0, 1] if case["nz"] == 0 else [0, 1, 2])
    shell = sum(2 * case["pml"] / n[a] for a in axes) * cells  # cell-axis pairs with a PML stage
    per = 12 * cells * s * parts + 8 * shell * s * parts
    per += 3 * cells * (4 if case["scene"] == "smooth" else 0 if case["scene"] == "vacuum" else 1)
    return {"bytes": float(case["steps"] * per), "flops": float(case["steps"] * cells * parts * 60)}


# ------------------------------------------------------------------ float64 solver
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


COMPS = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")


def _spacing(s):
    return s["cell"][0] / s["n"][0]


def _origin(s, comp):
    """Position of grid index 1 of a component, per axis (a 2D cell has z = 0 only)."""
    a0, el, d = COMPS.index(comp) % 3, comp[0] == "E", _spacing(s)
    out = []
    for a in range(3):
        shifted = (a != a0) if el else (a == a0)
        out.append(-s["cell"][a] / 2 + d / 2 + (-d / 2 if shifted else 0.0))
    return out


def _span(s, comp, center, size):
    """First and last grid index per axis of a volume snapped outwards to the grid."""
    org, d = _origin(s, comp), _spacing(s)
    lo, hi = [], []
    for a in range(3):
        if s["n"][a] == 0:
            lo.append(1), hi.append(1)
            continue
        top = -org[a]
        p0 = min(max(center[a] - size[a] / 2, org[a]), top)
        p1 = min(max(center[a] + size[a] / 2, org[a]), top)
        lo.append(int(math.floor((p0 - org[a]) / d + 1)))
        hi.append(int(math.ceil((p1 - org[a]) / d + 1)))
    return lo, hi


def _coords(s, comp, lo, hi):
    org, d = _origin(s, comp), _spacing(s)
    return [np.array([0.0]) if s["n"][a] == 0 else org[a] + (np.arange(lo[a], hi[a] + 1) - 1) * d for a in range(3)]


def _inside(o, X, Y, Z):
    c = o[1]
    if o[0] == "box":
        return (abs(X - c[0]) <= o[2][0] / 2) & (abs(Y - c[1]) <= o[2][1] / 2) & (abs(Z - c[2]) <= o[2][2] / 2)
    if o[0] == "sphere":
        return (X - c[0]) ** 2 + (Y - c[1]) ** 2 + (Z - c[2]) ** 2 <= o[2] ** 2
    return ((X - c[0]) ** 2 + (Y - c[1]) ** 2 <= o[2] ** 2) & (abs(Z - c[2]) <= o[3] / 2)


def _weight(p, c, size, d):
    """How much of a source of extent ``size`` a grid point at p carries."""
    lo, hi = c - size / 2, c + size / 2
    if size == 0.0:
        return max(0.0, 1 - abs(p - c) / d)
    if p <= lo - d or p >= hi + d:
        return 0.0
    if p < lo:
        return 0.5 * (1 - (lo - p) / d) ** 2
    if p - lo < d:
        return 1 - 0.5 * (1 - (p - lo) / d) ** 2
    if p > hi:
        return 0.5 * (1 - (p - hi) / d) ** 2
    if hi - p < d:
        return 1 - 0.5 * (1 - (hi - p) / d) ** 2
    return 1.0


def _source_terms(s):
    """[(component, first index, amplitude array)]"""
    q, d = s["source"], _spacing(s)
    if q["kind"] == "wave":
        k = 2 * math.pi * s["fcen"]
        kv = np.asarray(q["k"]) / np.linalg.norm(q["k"])
        nv = np.array([0.0, 0.0, 1.0])
        pol = np.cross(nv, kv)
        je, jm = np.cross(nv, np.cross(kv, pol)), -np.cross(nv, pol)
        terms = [(c, v) for c, v in (("Ex", je[0]), ("Ey", je[1]), ("Hx", jm[0]), ("Hy", jm[1])) if v != 0.0]
        center, size = q["center"], [1e9, 1e9, 0.0]
    else:
        terms, center, size = [(q["comp"], 1.0)], q["center"], q.get("size", [0.0, 0.0, 0.0])
    out = []
    for comp, scale in terms:
        lo, hi = _span(s, comp, center, size)
        x = _coords(s, comp, lo, hi)
        f = []
        for a in range(3):
            if s["n"][a] == 0 or size[a] > 1e8:
                w = np.ones(len(x[a]), dtype=complex)
            else:
                w = np.array([_weight(p, center[a], size[a], d) for p in x[a]], dtype=complex)
            if q["kind"] == "wave":
                w = w * np.exp(-1j * k * kv[a] * x[a])
            elif q["kind"] == "gauss" and size[a] != 0.0:
                w = w * np.exp(-((x[a] - center[a]) ** 2) / q["waist"] ** 2)
            f.append(w)
        if q["kind"] == "wave" and len(x[2]) == 1:
            f[2] = np.ones(1, dtype=complex)
        out.append((comp, lo, scale * f[0][:, None, None] * f[1][None, :, None] * f[2][None, None, :]))
    return out


def _pulse(s):
    """(f(t), last time it is on) of the Gaussian pulse."""
    width = 1.0 / s["fwidth"]
    cut = width * 5.0
    peak = round(cut / 2 * s["fcen"]) / s["fcen"]

    def f(t):
        tt = t - peak
        if tt > cut:
            return 0j
        return math.exp(-tt * tt / (2 * width * width)) * complex(math.cos(2 * math.pi * s["fcen"] * tt),
                                                                   -math.sin(2 * math.pi * s["fcen"] * tt))
    return f, cut, s["fcen"] + math.sqrt(-2 * math.log(1e-7)) / (width * math.pi) / 2


def _sigma(n, d, dt, thick):
    """PML profile at the samples of grid index 1..n."""
    out = np.zeros(n)
    if thick > 0:
        u0 = -math.log(1e-15) / (4 * thick / 3) * 0.5 * dt
        total = (2 * n + 1) * d / 2
        for i in range(1, n + 1):
            pos = (2 * i - 1) * d / 2
            for depth in (thick - pos, thick - (total - pos)):
                if depth > 0:
                    out[i - 1] = u0 * (depth / thick) ** 2
                    break
    return out


class _Yee:
    """The whole-grid Yee + PML recurrences in float64 (complex128 with Bloch sides).

    Arrays hold grid indices 0..N+1; U, T (= D or B) and W are the PML's curl,
    flux and material stages."""

    def __init__(self, s):
        self.s, dev = s, _dev()
        self.n = n = [max(1, v) for v in s["n"]]
        self.d = [math.inf if s["n"][a] == 0 else _spacing(s) for a in range(3)]
        self.dt = s["dt"]
        self.cx = s["bloch"] is not None
        self.dtype = torch.complex128 if self.cx else torch.float64
        z = lambda: torch.zeros([v + 2 for v in n], dtype=self.dtype, device=dev)  # noqa: E731
        zi = lambda: torch.zeros(n, dtype=self.dtype, device=dev)  # noqa: E731
        self.F = {c: z() for c in COMPS}
        self.U, self.T, self.W = ({c: zi() for c in COMPS} for _ in range(3))
        self.sig = []
        for a in range(3):
            thick = 0.0 if s["n"][a] == 0 or (self.cx and a < 2) else s["pml"]
            shape = [1, 1, 1]
            shape[a] = n[a]
            self.sig.append(torch.tensor(_sigma(n[a], self.d[a], self.dt, thick) if thick else np.zeros(n[a]),
                                         device=dev).reshape(shape))
        self.phase = []
        for a in range(2 if self.cx else 0):
            x = s["bloch"][a] * s["cell"][a]
            self.phase.append(complex(math.cos(x), math.sin(x)))
        self._materials(dev)
        self.src = [(c, lo, torch.tensor(amp, device=dev)) for c, lo, amp in _source_terms(s)]

    def _grid(self, comp, n, dev):
        x = _coords(self.s, comp, [1, 1, 1], n)
        return [torch.tensor(v, device=dev).reshape([-1 if b == a else 1 for b in range(3)])
                for a, v in enumerate(x)]

    def _materials(self, dev):
        s, n = self.s, self.n
        self.m = {}
        for c in COMPS[:3]:
            # the staggered extent, one longer off the component's axis
            cnt = [v + (0 if b == COMPS.index(c) else 1) for b, v in enumerate(n)]
            X = self._grid(c, cnt, dev)
            e = torch.ones(cnt, dtype=torch.float64, device=dev)
            for o in reversed(s["objects"]):
                e = torch.where(_inside(o, *X), 1.0 / o[-1], e)
            self.m[c] = e
        for c in COMPS[3:]:
            self.m[c] = 1.0
        self.poles, self.P = [], {c: 0.0 for c in COMPS[:3]}
        chi1 = torch.zeros(n, dtype=torch.float64, device=dev)
        X = self._grid("Ex", n, dev)
        for w0, gam, q in s["poles"]:
            sg = torch.zeros(n, dtype=torch.float64, device=dev)
            for i, o in reversed(list(enumerate(s["objects"]))):
                if i < len(q):
                    sg = torch.where(_inside(o, *X), q[i], sg)
            for a in range(3):
                if self.cx and a < 2:
                    continue
                edge = s["cell"][a] / 2 - s["pml"]
                sg = torch.where((X[a] < -edge) | (X[a] > edge), 0.0, sg)
            gd = gam * math.pi * self.dt
            w2 = (2 * math.pi * w0 * self.dt) ** 2
            drive = w2 if w0 else gam * 2 * math.pi * self.dt ** 2
            chi1 += sg * drive / (1 + gd) / 2
            zi = {c: torch.zeros(n, dtype=self.dtype, device=dev) for c in COMPS[:3]}
            self.poles.append([sg, 1 / (1 + gd), 1 - gd, 2 - w2, drive, zi, {c: v.clone() for c, v in zi.items()}])
        if s["poles"]:
            for c in COMPS[:3]:
                # the correction runs along the flat column-major index of both arrays
                e = self.m[c].permute(2, 1, 0).contiguous().reshape(-1)
                x = chi1.permute(2, 1, 0).contiguous().reshape(-1)
                e[:x.numel()] = e[:x.numel()] / (1 + e[:x.numel()] * x)
                cnt = self.m[c].shape
                self.m[c] = e.reshape(cnt[2], cnt[1], cnt[0]).permute(2, 1, 0)
        for c in COMPS[:3]:
            self.m[c] = self.m[c][:n[0], :n[1], :n[2]].contiguous()
        self.chi3 = None
        if s.get("chi3"):
            # painted on the cell centres
            d = _spacing(s)
            C = [torch.tensor(-s["cell"][a] / 2 + d / 2 + np.arange(n[a]) * d, device=dev).reshape(
                [-1 if b == a else 1 for b in range(3)]) for a in range(3)]
            self.chi3 = torch.zeros(n, dtype=torch.float64, device=dev)
            for o in s["objects"]:
                self.chi3 = torch.where(_inside(o, *C), s["chi3"], self.chi3)

    def _diff(self, comp, axis, sign):
        """Forward (+1) or backward (-1) difference of a component on indices 1..N."""
        n, F = self.n, self.F[comp]
        core = [slice(1, n[a] + 1) for a in range(3)]
        off = list(core)
        off[axis] = slice(1 + sign, n[axis] + 1 + sign)
        return sign * (F[tuple(off)] - F[tuple(core)]) / self.d[axis]

    def _half(self, group, signal):
        other, sign = ("E", 1) if group == "H" else ("H", -1)
        for a, ax in enumerate("xyz"):
            o, nx, pv = a, (a + 1) % 3, (a + 2) % 3
            c = group + ax
            curl = self._diff(other + "xyz"[nx], pv, sign) - self._diff(other + "xyz"[pv], nx, sign)
            K = self.dt * (curl if group == "H" else -curl)
            U, T, W, F = self.U[c], self.T[c], self.W[c], self.F[c]
            Un = ((1 - self.sig[nx]) * U + K) / (1 + self.sig[nx])
            T.mul_(1 - self.sig[pv]).add_(Un).sub_(U).div_(1 + self.sig[pv])
            self.U[c] = Un
            net = T.clone()
            for comp, lo, amp in self.src:
                if comp == c and signal is not None:
                    v = signal.real * amp.real - signal.imag * amp.imag
                    end = [min(lo[b] - 1 + v.shape[b], self.n[b]) for b in range(3)]
                    b0 = [max(lo[b] - 1, 0) for b in range(3)]
                    net[b0[0]:end[0], b0[1]:end[1], b0[2]:end[2]] += v[
                        b0[0] - lo[0] + 1:end[0] - lo[0] + 1, b0[1] - lo[1] + 1:end[1] - lo[1] + 1,
                        b0[2] - lo[2] + 1:end[2] - lo[2] + 1]
            if group == "E" and self.poles:
                net = net - self.P[c]
            Wn = self.m[c] * net
            core = F[1:-1, 1:-1, 1:-1]
            so = self.sig[o]
            core.copy_(torch.where(so == 0, Wn, core + (1 + so) * Wn - (1 - so) * W))
            self.W[c] = Wn
        for a, ph in enumerate(self.phase):
            for ax in "xyz":
                F = self.F[group + ax].movedim(a, 0)
                F[0, 1:-1, 1:-1] = F[-2, 1:-1, 1:-1] * ph.conjugate()
                F[-1, 1:-1, 1:-1] = F[1, 1:-1, 1:-1] * ph

    def _media(self):
        if not self.poles:
            return
        E = {c: self.F[c][1:-1, 1:-1, 1:-1] for c in COMPS[:3]}
        if self.chi3 is not None:
            corr = 1 / (1 + self.chi3 * sum((v * v.conj()).real for v in E.values()))
            for v in E.values():
                v.mul_(corr)
        self.P = {c: 0.0 for c in E}
        for p in self.poles:
            sg, gi, g1, cp, drive, P, Pp = p
            for c in E:
                new = gi * (cp * P[c] - g1 * Pp[c] + drive * sg * E[c])
                Pp[c], P[c] = P[c], new
                self.P[c] = self.P[c] + new

    def run(self, steps, mons):
        """mons: [(component, lo, hi, freqs)] -> DFT arrays (nx, ny, nz, n_freq)."""
        f, cut, fmax = _pulse(self.s)
        dec = max(1, int(math.floor(1 / (2 * fmax * self.dt))))
        acc = [0.0] * len(mons)

        def record(group, t):
            for i, (c, lo, hi, fr) in enumerate(mons):
                if c[0] != group:
                    continue
                v = self.F[c][lo[0]:hi[0] + 1, lo[1]:hi[1] + 1, lo[2]:hi[2] + 1]
                short = [hi[b] + 1 - lo[b] - v.shape[b] for b in (2, 1, 0)]  # past the last ghost: zero
                v = torch.nn.functional.pad(v, [x for b in short for x in (0, b)])
                w = torch.tensor(np.exp(1j * np.asarray(fr) * 2 * math.pi * t) * self.dt, device=v.device)
                acc[i] = acc[i] + v[..., None] * w

        for k in range(steps):
            t = k * self.dt
            on = t <= cut
            self._half("H", f(t) if on else None)
            if k % dec == 0:
                record("H", t)
            self._half("E", f(t + self.dt / 2) if on else None)
            self._media()
            if k % dec == 0:
                record("E", t + self.dt / 2)
        return acc


def _flux_mons(s, center, size):
    na = [i for i, v in enumerate(size) if v == 0.0][0]
    t = [a for a in range(3) if a != na]
    comps = ["E" + "xyz"[t[0]], "E" + "xyz"[t[1]], "H" + "xyz"[t[0]], "H" + "xyz"[t[1]]]
    return na, [(c, *_span(s, c, center, size), s["freqs"]) for c in comps]


def _plane_of(na, v, n1, n2):
    """Normal average of a recorded plane, cut to n1 x n2 samples: (n1, n2, n_freq)."""
    v = v.movedim(na, 0)
    v = (v[0] + v[1]) / 2 if v.shape[0] >= 2 else v[0]
    return v[:n1, :n2]


def _planes(s, na, mons, acc):
    t = [a for a in range(3) if a != na]
    n1 = min(m[2][t[0]] - m[1][t[0]] + 1 for m in mons)
    n2 = min(m[2][t[1]] - m[1][t[1]] + 1 for m in mons)
    return [_plane_of(na, v, n1, n2) for v in acc]


def _snapshot(case, y):
    """Ez as the framework's arrays hold it: one more plane past the staggered extent."""
    return {"ez": torch.nn.functional.pad(y.F["Ez"], (0, 0, 0, 1, 0, 1)).cpu()} if case["snapshot"] else {}


def _exact_fdtd(case, seed):
    if case["scene"] == "smooth":
        return None  # subpixel smoothing has no closed form here
    s = _scene(case, seed)
    y = _Yee(s)
    if case["monitor"] == "plane":
        acc = y.run(case["steps"], [("Ez", *_span(s, "Ez", *s["plane"]), s["freqs"])])
        return {"dft": [v.cpu() for v in acc], **_snapshot(case, y)}
    groups = [_flux_mons(s, c, z) for c, z in s["flux"]]
    acc = y.run(case["steps"], [m for _, g in groups for m in g])
    out = []
    for i, (na, g) in enumerate(groups):
        e1, e2, h1, h2 = _planes(s, na, g, acc[4 * i:4 * i + 4])
        dA = 1.0
        for a in range(3):
            if a != na and s["n"][a]:
                dA *= _spacing(s)
        out.append((e1 * h2.conj() - e2 * h1.conj()).real.sum(dim=(0, 1)).cpu() * dA)
    return {"flux": out, **_snapshot(case, y)}


def _exact_farfield(case, seed):
    s = _surface(case, seed)
    na, mons = _flux_mons(s, *s["flux"][0])
    acc = _planes(s, na, mons, _Yee(s).run(SURFACE_STEPS, mons))
    dev, d = _dev(), _spacing(s)
    n1, n2 = acc[0].shape[:2]
    th, ph = torch.tensor(s["theta"], dtype=torch.float64), torch.tensor(s["phi"], dtype=torch.float64)
    P, T = torch.meshgrid(ph, th, indexing="ij")
    T, P = T.reshape(-1), P.reshape(-1)
    obs = (s["obs_r"] * torch.stack([T.sin() * P.cos(), T.sin() * P.sin(), T.cos()], 1)).to(dev)
    out = torch.zeros(obs.shape[0], 6, case["n_freq"], dtype=torch.complex128, device=dev)
    # currents J = -n x H, M = n x E on z = const: (recorded plane, current's component, its sign)
    for q, pol, electric, sign in ((3, 0, True, 1.0), (2, 1, True, -1.0), (1, 0, False, -1.0), (0, 1, False, 1.0)):
        comp, lo = mons[q][0], mons[q][1]
        org = _origin(s, comp)
        x = org[0] + (lo[0] - 1 + torch.arange(n1, dtype=torch.float64, device=dev)) * d
        y = org[1] + (lo[1] - 1 + torch.arange(n2, dtype=torch.float64, device=dev)) * d
        z = org[2] + (lo[2] - 1) * d
        pts = torch.stack([x[:, None].expand(n1, n2), y[None, :].expand(n1, n2), torch.full((n1, n2), z, device=dev,
                          dtype=torch.float64)], -1).reshape(-1, 3)
        cur = acc[q].reshape(n1 * n2, -1) * (sign * d * d)
        p = torch.zeros(3, dtype=torch.float64, device=dev)
        p[pol] = 1.0
        step = max(1, 4_000_000 // pts.shape[0])
        for o in range(0, obs.shape[0], step):
            rv = obs[o:o + step, None, :] - pts[None]
            r = rv.square().sum(-1).sqrt()
            rh = rv / r[..., None]
            pd = rh[..., pol]
            cr = torch.linalg.cross(rh, p.expand_as(rh))
            for k, freq in enumerate(s["freqs"]):
                kk = 2 * math.pi * freq
                kr = kk * r
                e = torch.polar(kk / (4 * math.pi * r), kr + math.pi / 2) * cur[None, :, k]
                i1, i2 = torch.complex(torch.zeros_like(kr), -1 / kr), -1 / (kr * kr)
                t1, t2, t3 = 1 - i1 + i2, (-1 + 3 * i1 - 3 * i2) * pd, 1 - i1
                for j in range(3):
                    par = (e * (t1 * p[j] + t2 * rh[..., j])).sum(1)
                    crs = (e * t3 * cr[..., j]).sum(1)
                    out[o:o + step, j if electric else 3 + j, k] += par
                    out[o:o + step, 3 + j if electric else j, k] += crs if electric else -crs
    return {"far": out.cpu()}


def _exact_gradient(case, seed):
    """The bend's Ez/Hx/Hy recurrences in float64 with torch autograd over every step."""
    res, nd, steps = case["resolution"], case["n_design"], case["steps"]
    design, wg, pad, pml = nd / res, 0.5, 2.0, 1.0
    side = design + 2 * pad + 2 * pml + 2 * wg
    n = int(math.floor(side * res))
    d = side / n
    dev = _dev()
    s = {"cell": [side, side, 0.0], "n": (n, n, 0), "pml": pml, "objects": [
        ("box", [-(design / 2 + pad + wg / 2), 0.0, 0.0], [pad + wg + pml, wg, 1.0], 12.1),
        ("box", [0.0, design / 2 + pad + wg / 2, 0.0], [wg, pad + wg + pml, 1.0], 12.1),
        ("box", [0.0, 0.0, 0.0], [side + 1, side + 1, 1.0], 2.085)], "poles": [], "fcen": 0.625, "fwidth": 0.5,
        "bloch": None, "dt": 0.5 * d, "source": {"kind": "gauss", "comp": "Ez", "waist": 1e30,
                                                   "center": [-(design / 2 + pad), 0.0, 0.0], "size": [0.0, wg, 0.0]}}
    y = _Yee(s)
    m0 = y.m["Ez"][:, :, 0]
    rho = torch.tensor(np.random.default_rng([int(seed), 79]).random(nd * nd), device=dev, requires_grad=True)
    # bilinear design map on the Ez points inside the region, clamped at its edge
    lo, hi = _span(s, "Ez", [0.0, 0.0, 0.0], [design, design, 0.0])
    X = _coords(s, "Ez", lo, hi)
    idx, wt = [], []
    for a in range(2):
        gx = np.linspace(-design / 2, design / 2, nd)
        f = np.clip((X[a] - gx[0]) / (gx[1] - gx[0]), 0.0, nd - 1.0)
        i = np.minimum(np.floor(f).astype(int), nd - 2)
        idx.append(torch.tensor(i, device=dev)), wt.append(torch.tensor(f - i, device=dev))
    R = rho.reshape(nd, nd).T  # x first: parameters run along x fastest
    (i, j), (u, v) = idx, (wt[0][:, None], wt[1][None, :])
    r = ((1 - u) * (1 - v) * R[i][:, j] + u * (1 - v) * R[i + 1][:, j] + (1 - u) * v * R[i][:, j + 1]
         + u * v * R[i + 1][:, j + 1])
    m = m0.clone()
    m[lo[0] - 1:hi[0], lo[1] - 1:hi[1]] = 1.0 / (2.085 + r * (12.1 - 2.085))
    mlo, mhi = _span(s, "Ez", [0.0, design / 2 + pad, 0.0], [2 * wg, 0.0, 0.0])
    f, cut, _ = _pulse(s)
    sx, sy = y.sig[0][:, :, 0], y.sig[1][:, :, 0]
    dt, zero = s["dt"], torch.zeros(n, n, dtype=torch.float64, device=dev)
    _, slo, amp = y.src[0]
    S = zero.clone()
    S[slo[0] - 1:slo[0] - 1 + amp.shape[0], slo[1] - 1:slo[1] - 1 + amp.shape[1]] = amp.real[:, :, 0]
    S2 = zero.clone()
    S2[slo[0] - 1:slo[0] - 1 + amp.shape[0], slo[1] - 1:slo[1] - 1 + amp.shape[1]] = amp.imag[:, :, 0]
    freqs = np.array([0.55, 0.625, 0.7])
    pad2 = torch.nn.functional.pad

    def block(k0, k1, m, hx, hy, ez, ux, wx, wy, tz, uz, acc):
        for k in range(k0, k1):
            # Hx: own x, next y; Hy: own y, prev x (next z has no PML); Ez: next x, prev y
            kx = -dt / d * (pad2(ez, (0, 1))[:, 1:] - ez)
            un = ((1 - sy) * ux + kx) / (1 + sy)
            wn = wx + un - ux
            hx = hx + (1 + sx) * wn - (1 - sx) * wx
            ux, wx = un, wn
            ky = dt / d * (pad2(ez, (0, 0, 0, 1))[1:] - ez)
            wn = ((1 - sx) * wy + ky) / (1 + sx)
            hy = hy + (1 + sy) * wn - (1 - sy) * wy
            wy = wn
            kz = dt / d * ((hy - pad2(hy, (0, 0, 1, 0))[:-1]) - (hx - pad2(hx, (1, 0))[:, :-1]))
            un = ((1 - sx) * uz + kz) / (1 + sx)
            tz = ((1 - sy) * tz + un - uz) / (1 + sy)
            uz = un
            t = k * dt
            q = f(t + dt / 2) if t <= cut else 0j
            ez = m * (tz + (q.real * S - q.imag * S2))
            w = np.exp(2j * math.pi * freqs * (t + dt / 2)) * dt
            line = ez[mlo[0] - 1:mhi[0], mlo[1] - 1:mhi[1]]
            acc = acc + line[..., None] * torch.tensor(w, device=dev)
        return hx, hy, ez, ux, wx, wy, tz, uz, acc

    state = (zero,) * 8 + (torch.zeros(mhi[0] - mlo[0] + 1, mhi[1] - mlo[1] + 1, 3, dtype=torch.complex128, device=dev),)
    for k0 in range(0, steps + 1, 50):
        state = checkpoint(block, k0, min(steps + 1, k0 + 50), m, *state, use_reentrant=False)
    J = state[-1].abs().square().sum()
    J.backward()
    return {"objective": float(J.detach()), "gradient": rho.grad.cpu()[:, None]}


def exact(case, seed):
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed)
    if case["kind"] == "farfield":
        return _exact_farfield(case, seed)
    return _exact_fdtd(case, seed)
