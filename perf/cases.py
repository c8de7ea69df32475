"""Timed cases of the adaptive shallow-water step, called as a flood model's
program calls it: a scenario is loaded from its .par and rasters, stepped, and
its state read back.

A pass takes a number of time steps and then reads what the step produced: the
simulated time and step, the tree (its significance mask and leaf count) and
every flow coefficient of the hierarchy, into host buffers that the program
keeps. Passes go on from where
the last one ended, as a simulation does.

The scenarios are this repository's own kinds, written in the formats it
reads:

  dam      circular dam break on a flat, frictionless 50 m square with closed
           walls (nearly everything wet, few leaves: the launches count)
  valley   rough bed (Gaussian random field) with a west-east slope and
           Manning friction, water standing in the low ground, a QVAR inflow
           on the west border and a FREE east border (dense leaves)
  urban    flat plain with rectangular blocks, a wet northern strip, point
           sources and closed walls (sparse leaves); `wet` is the strip's
           share of the domain, from the first minutes of a flood (1/16) to
           the hours where it covers the plain
  ensemble several valley scenarios of different sizes stepped together

Rasters have a fixed number of decimals, as survey products do. All outputs
are reproducible bit for bit, so the cases are compared exactly.
"""
from __future__ import annotations

import ctypes
import os
import shutil
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "gpu-mwdg2_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "gpu-mwdg2_amd"))

import mwdg2  # noqa: E402

COEFS = {"mwdg2": ("eta0", "eta1x", "eta1y", "qx0", "qx1x", "qx1y", "qy0", "qy1x", "qy1y"),
         "hwfv1": ("eta0", "qx0", "qy0")}


def listed():
    return [
        # a small basin stepped on its own: every launch and single-group pass shows
        dict(name="dam 64 hwfv1 f32", kind="dam", xsz=64, ysz=64, solver="hwfv1", prec="f32", steps=128),
        # the dam-break benchmark of the repository (256 x 256, FP64)
        dict(name="dam 256 mwdg2 f64", kind="dam", xsz=256, ysz=256, solver="mwdg2", prec="f64", steps=128),
        # the wet/dry hydrograph grid in each solver and precision that users run
        dict(name="valley 1024 mwdg2 f32", kind="valley", xsz=1024, ysz=1024, solver="mwdg2", prec="f32", steps=128,
             wet=0.1),
        dict(name="valley 1024 mwdg2 f64", kind="valley", xsz=1024, ysz=1024, solver="mwdg2", prec="f64", steps=96,
             wet=0.1),
        # a survey raster that is no power of two, first-order solver
        dict(name="valley 1403x987 hwfv1 f32", kind="valley", xsz=1403, ysz=987, solver="hwfv1", prec="f32",
             steps=128, wet=0.3),
        # one resolution everywhere (epsilon 0): no tree rebuild after the first step
        dict(name="valley 700x650 uniform f64", kind="valley", xsz=700, ysz=650, solver="mwdg2", prec="f64",
             steps=96, wet=0.5, eps=0.0),
        # slope limiter on
        dict(name="valley 512 limited f32", kind="valley", xsz=512, ysz=512, solver="mwdg2", prec="f32", steps=96,
             wet=0.5, limiter=True),
        # later in a flood: most of the plain under moving water
        dict(name="urban 1733x1291 flood f32", kind="urban", xsz=1733, ysz=1291, solver="mwdg2", prec="f32",
             steps=128, wet=0.7),
        # the headline benchmark: the 4096 x 4096 plain in its first minutes, FP32 and FP64
        dict(name="urban 4096 mwdg2 f32", kind="urban", xsz=4096, ysz=4096, solver="mwdg2", prec="f32", steps=200,
             wet=0.0625),
        dict(name="urban 4096 mwdg2 f64", kind="urban", xsz=4096, ysz=4096, solver="mwdg2", prec="f64", steps=160,
             wet=0.0625),
        # the learned step (network trained on the run's own first steps)
        dict(name="urban 2048 learned f32", kind="urban", xsz=2048, ysz=2048, solver="mwdg2", prec="f32", steps=128,
             wet=0.0625, learned=True),
        # scenarios of an ensemble, 256 to 1024 cells a side
        dict(name="ensemble 12 f32", kind="ensemble", members=12, lo=256, hi=1024, solver="mwdg2", prec="f32",
             steps=48, wet=0.1),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["dam", "valley", "valley", "urban", "urban", "ensemble"])
    prec = rng.choice(["f32", "f32", "f64"])
    solver = rng.choice(["mwdg2", "mwdg2", "hwfv1"])
    if kind == "dam":
        n = 1 << rng.randint(6, 9)
        return dict(kind=kind, xsz=n, ysz=n, solver=solver, prec=prec, steps=rng.randint(64, 160))
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(3, 12), lo=_log(rng, 128, 400), hi=_log(rng, 400, 1024),
                    solver="mwdg2", prec=prec, steps=rng.randint(16, 40), wet=round(rng.uniform(0.02, 0.6), 3))
    top = 1300 if kind == "valley" else 2600
    xsz, ysz = _log(rng, 100, top), _log(rng, 100, top)
    case = dict(kind=kind, xsz=xsz, ysz=ysz, solver=solver, prec=prec, steps=rng.randint(32, 96),
                wet=round(rng.uniform(0.02, 0.8), 3))
    option = rng.random()
    if option < 0.12:
        case.update(eps=0.0, xsz=min(xsz, 1500), ysz=min(ysz, 1500))
    elif option < 0.3:
        case["eps"] = rng.choice([1e-4, 1e-2])
    elif option < 0.4 and solver == "mwdg2":
        case["limiter"] = True
    elif option < 0.5 and solver == "mwdg2":
        case["learned"] = True
    return case


# ---------------------------------------------------------------------------
# Scenario files
# ---------------------------------------------------------------------------
def _level(xsz, ysz):
    return max(2, (max(xsz, ysz) - 1).bit_length())


def _write_raster(path, a, digits, decimals, cell=1.0):
    """ESRI ASCII grid of non-negative numbers with a fixed number of digits;
    row 0 of `a` is the southern row (written last)."""
    nrows, ncols = a.shape
    v = torch.round(a.flip(0).double() * 10 ** decimals).to(torch.int64)
    width = digits + 1 + decimals + 1                          # digits, point, decimals, separator
    text = torch.full((nrows, ncols, width), 32, dtype=torch.uint8, device=a.device)
    for k in range(digits + decimals):
        at = width - 2 - k if k < decimals else width - 3 - k
        text[:, :, at] = (v // 10 ** k % 10 + 48).to(torch.uint8)
    text[:, :, digits] = ord(".")
    text[:, -1, -1] = 10
    with open(path, "wb") as f:
        f.write(f"ncols        {ncols}\nnrows        {nrows}\nxllcorner    0.0\nyllcorner    0.0\n"
                f"cellsize     {cell!r}\nNODATA_value -9999\n".encode())
        f.write(text.cpu().numpy().tobytes())


def _rough_bed(xsz, ysz, gen, dev):
    """Gaussian random field, power k^-3, 5 m standard deviation, above 0."""
    n = 1 << _level(xsz, ysz)
    w = torch.randn(n, n, generator=gen, device=dev, dtype=torch.float32)
    k = torch.fft.fftfreq(n, device=dev)
    k = torch.sqrt(k[None, :] ** 2 + k[:, None] ** 2)
    amp = torch.where(k > 0, k.clamp_min(1e-9) ** -1.5, torch.zeros_like(k))
    z = torch.fft.ifft2(torch.fft.fft2(w) * amp).real
    z = (z - z.mean()) * (5.0 / z.std())
    z = z[:ysz, :xsz]
    x = torch.arange(xsz, device=dev) + 0.5
    z = z + 0.001 * (xsz - x)[None, :]
    return z - z.min() + 1.0


def _par(d, case, extra):
    ent = ["test_case     0", case["solver"], f"max_ref_lvl   {_level(case['xsz'], case['ysz'])}",
           f"epsilon       {case.get('eps', 1e-3)!r}", "wall_height   1000", "initial_tstep 1",
           "sim_time      100000", "massint       100000", "saveint       100000", "DEMfile       case.dem",
           "startfile     case.start"] + extra
    if case.get("limiter"):
        ent += ["limitslopes   on", "tol_Krivo     1"]
    par = os.path.join(d, "case.par")
    with open(par, "w") as f:
        f.write("\n".join(ent) + "\n")
    return par


def _dam(d, case, gen, dev):
    n = case["xsz"]
    u = torch.rand(4, generator=gen, device=dev).tolist()
    c = (torch.arange(n, device=dev) + 0.5) * (50.0 / n)
    cx, cy, rad, hin = 15 + 20 * u[0], 15 + 20 * u[1], 1.5 + 2.5 * u[2], 1.5 + 2.0 * u[3]
    h = torch.where((c[None, :] - cx) ** 2 + (c[:, None] - cy) ** 2 < rad ** 2, hin, 0.5)
    _write_raster(os.path.join(d, "case.dem"), torch.zeros_like(h), 1, 2, 50.0 / n)
    _write_raster(os.path.join(d, "case.start"), h, 1, 2, 50.0 / n)
    return _par(d, case, ["cfl           0.33"])


def _valley(d, case, gen, dev):
    xsz, ysz = case["xsz"], case["ysz"]
    z = _rough_bed(xsz, ysz, gen, dev)
    # water below a surface that falls to the east, so it is on the move
    x = torch.arange(xsz, device=dev) + 0.5
    rel = z - 0.0005 * (xsz - x)[None, :]
    srt = rel.flatten().sort().values
    top = srt[min(srt.numel() - 1, int(case["wet"] * srt.numel()))]
    h = (top - rel).clamp_min(0.0)
    h = torch.where(h < 0.01, torch.zeros_like(h), h)
    _write_raster(os.path.join(d, "case.dem"), z, 2, 3)
    _write_raster(os.path.join(d, "case.start"), h, 2, 3)
    with open(os.path.join(d, "case.bci"), "w") as f:
        f.write(f"W 0 {float(ysz)!r} QVAR inflow\nE 0 {float(ysz)!r} FREE\n")
    with open(os.path.join(d, "case.bdy"), "w") as f:
        f.write(f"inflow\n3 seconds\n{50.0 / ysz!r} 0.0\n{100.0 / ysz!r} 600.0\n0.0 100000.0\n")
    return _par(d, case, ["fpfric        0.035", "bcifile       case.bci", "bdyfile       case.bdy"])


def _urban(d, case, gen, dev):
    xsz, ysz = case["xsz"], case["ysz"]
    u = torch.rand(1 << 18, generator=gen, device=dev).cpu().numpy()
    z = np.zeros((ysz, xsz), dtype=np.float32)
    occ = np.zeros((ysz, xsz), dtype=bool)
    side = max(8, min(40, min(xsz, ysz) // 4))
    covered, k = 0, 0
    while covered < 0.3 * xsz * ysz and k + 5 <= u.size:
        w, b = 8 + int(u[k] * (side - 7)), 8 + int(u[k + 1] * (side - 7))
        x0, y0 = int(u[k + 2] * (xsz - w)), int(u[k + 3] * (ysz - b))
        blk = occ[y0:y0 + b, x0:x0 + w]
        covered += blk.size - int(np.count_nonzero(blk))
        blk[:] = True
        z[y0:y0 + b, x0:x0 + w] = 5.0 + 15.0 * u[k + 4]
        k += 5
    strip = max(1, int(case["wet"] * ysz))
    h = np.zeros((ysz, xsz), dtype=np.float32)
    # the wet strip's surface falls to the south in steps of a few cm, so it is on the move
    h[ysz - strip:, :] = (1.0 + np.round(np.linspace(0.0, 1.0, strip), 1)).astype(np.float32)[:, None]
    h[occ] = 0.0
    _write_raster(os.path.join(d, "case.dem"), torch.from_numpy(z).to(dev), 2, 2)
    _write_raster(os.path.join(d, "case.start"), torch.from_numpy(h).to(dev), 1, 1)
    lines = []
    while len(lines) < 16 and k + 2 <= u.size:
        xi, yi = int(u[k] * xsz), int(u[k + 1] * ysz)
        k += 2
        if not occ[yi, xi]:
            lines.append(f"P {xi + 0.5!r} {yi + 0.5!r} QFIX 5.0")
    with open(os.path.join(d, "case.bci"), "w") as f:
        f.write("\n".join(lines) + "\n")
    return _par(d, case, ["fpfric        0.02", "bcifile       case.bci"])


def _load(case, seed):
    """The scenario written to files and loaded, as its program starts."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))
    d = tempfile.mkdtemp(prefix="mwdg2_case_")
    try:
        par = {"dam": _dam, "valley": _valley, "urban": _urban}[case["kind"]](d, case, gen, dev)
        return mwdg2.Simulation(par, case["prec"])
    finally:
        shutil.rmtree(d, ignore_errors=True)


# ---------------------------------------------------------------------------
# Passes
# ---------------------------------------------------------------------------
class _Reader:
    """Host buffers that one simulation's state is read into."""

    def __init__(self, sim, case):
        self.sim = sim
        pin = torch.cuda.is_available()
        real = torch.float32 if case["prec"] == "f32" else torch.float64
        level = sim.counters()["max_ref_lvl"]
        nodes = (4 ** (level + 1) - 1) // 3 + 3                # of the whole hierarchy
        self.names = ["A." + c for c in COEFS[case["solver"]]]
        self.coefs = torch.zeros(len(self.names), nodes, dtype=real, pin_memory=pin)
        self.tree = torch.zeros((4 ** level - 1) // 3 + 3, dtype=torch.uint8, pin_memory=pin)

    def _read(self, name, buf):
        rc = mwdg2.lib().mw_download(self.sim._h, name.encode(), buf.data_ptr(), buf.numel(),
                                     ctypes.byref(ctypes.c_longlong()))
        if rc != mwdg2.MW_OK:
            raise mwdg2.MWError(rc, mwdg2.lib().mw_last_error().decode())

    def read(self):
        c = self.sim.counters()
        self._read("sig", self.tree)
        for name, row in zip(self.names, self.coefs):
            self._read(name, row)
        return {"time": c["time"], "dt_next": c["dt_next"], "leaves": c["n_leaves"], "tree": self.tree,
                "coefs": self.coefs}


def _members(case):
    n = case["members"]
    for i in range(n):
        side = int(round(case["lo"] * (case["hi"] / case["lo"]) ** (i / max(1, n - 1))))
        yield dict(kind="valley", xsz=side, ysz=side - side // 7 * (i % 2), solver="mwdg2", prec=case["prec"],
                   wet=case["wet"])


def prepare(case, seed):
    if case["kind"] == "ensemble":
        sims = [_load(m, 1000 * seed + i) for i, m in enumerate(_members(case))]
        readers = [_Reader(s, case) for s in sims]
        return dict(steps=case["steps"], ensemble=mwdg2.Ensemble(sims), readers=readers)
    sim = _load(case, seed)
    state = dict(steps=case["steps"], sim=sim, readers=[_Reader(sim, case)])
    if case.get("learned"):
        net = mwdg2.Mlp(int(seed) + 1)
        net.record(sim, 24)
        net.build_labels(8)
        net.fit(2, 4096)
        sim.set_learned(net)
    else:
        sim.step(8)
    sim.sync()
    return state


def run(state):
    if "ensemble" in state:
        state["ensemble"].step(state["steps"])
        state["ensemble"].sync()
        return [r.read() for r in state["readers"]]
    state["sim"].step(state["steps"])
    return state["readers"][0].read()


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _leaves(case):
    """About how many leaves (of them wet) a scenario of this kind has."""
    cells = case["xsz"] * case["ysz"]
    if case.get("eps", 1e-3) == 0.0:
        return cells, case["wet"] * cells
    if case["kind"] == "dam":
        return min(cells, 9000), min(cells, 9000)
    if case["kind"] == "urban":
        return 0.3 * cells, 0.3 * cells * case["wet"]
    if case["xsz"] != case["ysz"] or case["xsz"] & (case["xsz"] - 1):
        cells *= 0.2       # the walls around the raster raise the maxima that the thresholds are relative to
    return cells, case["wet"] * cells


def work(case):
    """Per step: each leaf's flow and bed coefficients read once and its flow
    coefficients written once; about 1500 operations for each wet leaf and
    Runge-Kutta stage of MWDG2 and 250 for a wet leaf of HWFV1."""
    size = 4 if case["prec"] == "f32" else 8
    mw = case["solver"] == "mwdg2"
    nbytes = flops = 0.0
    for c in (_members(case) if case["kind"] == "ensemble" else [case]):
        leaves, wet = _leaves(c)
        nbytes += case["steps"] * leaves * size * (21 if mw else 7)
        flops += case["steps"] * wet * (3000 if mw else 250)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Every result of the step is defined to the last bit: each multiply and
    add rounds on its own in a stated order, and the reductions are minima
    and maxima. The step at a threshold turns a last-bit change into another
    tree, so nothing else compares."""
    return "exact"


def exact(case, seed):
    """None: the state after some dozens of adaptive steps has no plain
    64-bit restatement that runs in seconds; the compared bits stand for it."""
    return None
