"""The work whose speed is measured: what a program that uses this framework
has it do, through the public entry points (cardioid_amd.hip and the C ABI of
include/cardioid_hip.h).

Five kinds of case:
  sim        hip.Simulation: one anatomy advanced by some steps (10 to 20 ms of
             activity), then its Vm and activation times read (and, where few,
             its 19 states), as a program does at every snapshot
  batch      hip.Batch: a chunk of graph-replayed steps of the slabs in
             flight, then each one's Vm, activation and APD90 times, as the
             serving loop does when requests end
  reaction   the drop-in TT06Dev reaction over cells without diffusion: calc
             and integrator on device arrays
  diffusion  the drop-in FGR diffusion: updateLocalVoltage, then calc
  loop       a host program's time loop over the drop-in objects: stimulus,
             reactions, diffusion, integrator, sensor

exact() is the same model in plain torch, 64 bits throughout: the monodomain
step with TT06 kinetics (ten Tusscher and Panfilov 2006) by rational fits or
by the voltage functions themselves, and the 19-point finite-volume operator.
"""
import ctypes as C
import functools
import math
import os
import re

import numpy as np
import torch

from cardioid_amd import hip
from cardioid_amd import workloads as W

FIT_FILE = os.path.join(os.path.dirname(hip.__file__), "data", "tt06_fit_tol1e-4_mod1.data")
EMI = W.CELLTYPES_EMI


# ---------------------------------------------------------------------- cases

def listed():
    return [
        # a few hundred cells: unit-test anatomies, single-cell studies;
        # steps of a few microseconds, where latency and launches count
        dict(name="sim-504-fp64", kind="sim", shape="brick", nx=7, ny=8, nz=9, mode="fp64_fused",
             deck="fits", dt=0.02, steps=500, sensors=1),
        # the Niederer benchmark slab (3 x 7 x 20 mm at 0.2 mm)
        dict(name="sim-niederer-fp64", kind="sim", shape="niederer", nx=15, ny=35, nz=100,
             mode="fp64_fused", deck="fits", dt=0.01, steps=500, sensors=1),
        # the 64^3 all-tissue brick of the parity workload
        dict(name="sim-brick64-fma", kind="sim", shape="brick", nx=64, ny=64, nz=64,
             mode="fp64_fma", deck="fits", dt=0.02, steps=1000, sensors=1),
        # the shell anatomy beyond every cache (the headline workload's
        # generator at 160 x 160 x 320), in both fused precisions
        dict(name="sim-shell160-fma", kind="sim", shape="shell", nx=160, ny=160, nz=320,
             mode="fp64_fma", deck="fits", dt=0.02, steps=500, sensors=1),
        dict(name="sim-shell160-mixed", kind="sim", shape="shell", nx=160, ny=160, nz=320,
             mode="mixed_fused", deck="fits", dt=0.02, steps=500, sensors=1),
        # the reaction factory's default deck (tolerance 0, the exact functions)
        dict(name="sim-shell96-exact", kind="sim", shape="shell", nx=96, ny=96, nz=192,
             mode="fp64_fused", deck="exact", dt=0.02, steps=200, sensors=1),
        # the reference's loop over the drop-in objects
        dict(name="sim-shell96-unfused", kind="sim", shape="shell", nx=96, ny=96, nz=192,
             mode="fp64_unfused", deck="fits", dt=0.02, steps=200, sensors=1),
        # drug-screen requests in flight: one alone, and a dozen together
        dict(name="batch-1-mixed", kind="batch", slabs=1, dims_seed=5, lo=48, hi=64,
             mode="mixed_fused", deck="fits", dt=0.02, steps=500, graph=10),
        dict(name="batch-12-mixed", kind="batch", slabs=12, dims_seed=4, lo=32, hi=128,
             mode="mixed_fused", deck="fits", dt=0.02, steps=500, graph=10),
        # the drop-in objects driven from outside: one cell type's cells
        # through an index array, the diffusion on a ragged anatomy, and the
        # whole loop with the default deck on a small block of tissue
        dict(name="reaction-300k", kind="reaction", n=300_007, deck="fits", dt=0.02, steps=4),
        dict(name="diffusion-shell96", kind="diffusion", shape="shell", nx=96, ny=96, nz=192),
        dict(name="loop-9k-exact", kind="loop", shape="brick", nx=19, ny=21, nz=23, deck="exact",
             dt=0.02, steps=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_shape(rng, most):
    while True:
        if rng.random() < 0.6:
            shape, d = "brick", [_log_int(rng, 4, 112) for _ in range(3)]
        else:
            n = _log_int(rng, 20, 112)
            shape, d = "shell", [n, n + rng.randint(-2, 2), 2 * n + rng.randint(-5, 5)]
        if d[0] * d[1] * d[2] <= most:
            return dict(shape=shape, nx=d[0], ny=d[1], nz=d[2])


def draw(rng):
    kind = rng.choices(["sim", "batch", "reaction", "diffusion", "loop"], [9, 3, 3, 2, 3])[0]
    deck = "exact" if rng.random() < 0.25 else "fits"
    if kind == "sim":
        mode = rng.choice(["fp64_fused", "fp64_unfused"] if deck == "exact" else
                          ["fp64_fused", "fp64_fma", "mixed_fused", "mixed_fused", "fp64_unfused"])
        s = _draw_shape(rng, 1_500_000)
        return dict(kind="sim", **s, mode=mode, deck=deck, dt=rng.choice([0.01, 0.02, 0.02]),
                    steps=rng.randint(100, 400), sensors=rng.choice([1, 1, 3]))
    if kind == "batch":
        lo = _log_int(rng, 8, 48)
        return dict(kind="batch", slabs=_log_int(rng, 1, 14), dims_seed=rng.randint(0, 1 << 20),
                    lo=lo, hi=lo + rng.randint(1, 56), deck="fits",
                    mode=rng.choice(["mixed_fused", "mixed_fused", "fp64_fma"]), dt=0.02,
                    steps=rng.choice([100, 177, 400]), graph=rng.choice([0, 10, 10]))
    if kind == "reaction":
        return dict(kind="reaction", n=_log_int(rng, 1, 600_000), deck=deck, dt=0.02,
                    steps=rng.randint(2, 6))
    if kind == "diffusion":
        return dict(kind="diffusion", **_draw_shape(rng, 2_000_000))
    return dict(kind="loop", **_draw_shape(rng, 400_000), deck=deck, dt=0.02,
                steps=rng.randint(5, 20))


# --------------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=4)
def _shell(nx, ny, nz):
    return W.ellipsoid_shell(nx, ny, nz, seed=0)[0]


def _anatomy(case, rng):
    """The anatomy, its cell types and its stimuli; fibres (where they do not
    follow from the shape) and stimulus sites from the seed."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["shape"] == "niederer":
        a, _, _ = W.niederer(0.2)
        types = ["epiCellML"]
    elif case["shape"] == "shell":
        a, types = _shell(nx, ny, nz), EMI
    else:
        a = W.fibre_slab(nx, ny, nz, float(rng.uniform(-90.0, 90.0)))
        types = ["endoCellML"]
        if case["kind"] == "loop":      # three reactions, as a ventricular wall has
            a.celltype = ((a.gid % nx) * 3 // nx).astype(np.uint8)
            types = EMI
    x, y, z = a.tuples()
    stim = []
    for c in rng.choice(a.ncell, size=min(4, a.ncell), replace=False):
        h = 4
        stim.append(W.box_stimulus(int(x[c]) - h, int(x[c]) + h, int(y[c]) - h, int(y[c]) + h,
                                   int(z[c]) - h, int(z[c]) + h, vStim=float(rng.uniform(-52, -35)),
                                   duration=float(rng.uniform(0.5, 1.0))))
    return a, types, stim


def _scales(rng, n):
    """One set of drug scales (s_kr, s_cal, s_na) for the whole anatomy."""
    return np.tile(rng.uniform(0.3, 1.0, 3), (n, 1))


def _slab_inputs(case, seed):
    """Per slab of a batch: anatomy, scales, stimuli.  The dimensions belong
    to the case, everything else to the seed."""
    dims = np.random.default_rng(case["dims_seed"])
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["slabs"]):
        nx, ny, nz = (int(round(math.exp(dims.uniform(math.log(case["lo"]), math.log(case["hi"])))))
                      for _ in range(3))
        a = W.fibre_slab(nx, ny, nz, float(rng.uniform(-90.0, 90.0)))
        out.append((a, rng.uniform(0.0, 1.0, 3),
                    [W.box_stimulus(xMax=4, nx=nx, ny=ny, nz=nz,
                                    vStim=float(rng.uniform(-52, -40)))]))
    return out


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _p(t):
    return C.c_void_p(t.data_ptr())


class _Handles:
    """Drop-in objects of one program; freed with it."""

    def __init__(self):
        self.tt06, self.fgr, self.sensor = [], [], []

    def __del__(self):
        L = hip.lib()
        for h in self.tt06:
            L.cdh_tt06_destroy(h)
        for h in self.fgr:
            L.cdh_fgr_destroy(h)
        for h in self.sensor:
            L.cdh_activation_sensor_destroy(h)

    def reaction(self, name, n, deck, dt):
        fl, fm, fc = hip.read_fit_file(hip.DEFAULT_FIT_FILE).packed()
        p = hip.TT06Params(dt=dt, tolerance=0.0 if deck == "exact" else 1e-4, mod=1, fastGate=1,
                           fastNonGate=0, fit_l=hip.ptr(fl, hip.ip), fit_m=hip.ptr(fm, hip.ip),
                           fit_coef=hip.ptr(fc), celltype=hip.standard_celltype(name), s_kr=1.0,
                           s_cal=1.0, s_na=1.0)
        h = C.c_void_p()
        hip.check(hip.lib().cdh_tt06_create(C.byref(p), n, C.byref(h)), "cdh_tt06_create")
        self.tt06.append(h)
        return h

    def diffusion(self, a):
        gid = np.ascontiguousarray(a.gid, np.int64)
        tissue = np.ones(a.ncell, np.int32)
        sig = np.ascontiguousarray(a.sigma, np.float64).reshape(-1)
        p = hip.FGRParams(nx=a.nx, ny=a.ny, nz=a.nz, dx=a.dx, dy=a.dy, dz=a.dz,
                          diffusionScale=W.DIFFUSION_SCALE, nLocal=a.ncell, nRemote=0,
                          gid=hip.ptr(gid, hip.i64p), cellType=hip.ptr(tissue, hip.ip),
                          sigma=hip.ptr(sig))
        h = C.c_void_p()
        hip.check(hip.lib().cdh_fgr_create(C.byref(p), C.byref(h)), "cdh_fgr_create")
        self.fgr.append(h)
        return h


def _cells(seed, n):
    """Cells somewhere along the action potential: Vm, and the rest states of
    endocardial cells with their gates moved, [19][n]."""
    rng = np.random.default_rng(seed)
    V = rng.uniform(-88.0, 35.0, n)
    st = np.repeat(np.array(_TYPES["endoCellML"][7])[:, None], n, 1)
    st[1] = st[1] / _constants()["c9"] + V
    st[7:] = np.clip(st[7:] + rng.uniform(-0.2, 0.2, (12, n)), 0.0, 1.0)
    return V, st


def _field(seed, n):
    """A smooth-ish Vm with noise, as a front and its wake give the diffusion."""
    rng = np.random.default_rng(seed)
    k = rng.uniform(2.0, 9.0)
    return -30.0 + 55.0 * np.sin(np.linspace(0.0, k, n)) + rng.uniform(-2.0, 2.0, n)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "sim":
        a, types, stim = _anatomy(case, rng)
        sim = hip.Simulation(a, types, case["dt"], W.DIFFUSION_SCALE, stim, mode=case["mode"],
                             scales=_scales(rng, a.ncell), sensors=case["sensors"],
                             exact_functions=case["deck"] == "exact",
                             jhTauSmooth=1 if case["deck"] == "exact" else 0)
        sim.sync()
        return dict(kind=kind, sim=sim, steps=case["steps"], sensors=case["sensors"],
                    states=a.ncell <= 4096)
    if kind == "batch":
        slabs = [hip.Slab(a, ["endoCellML"], W.DIFFUSION_SCALE, stim, scales=sc)
                 for a, sc, stim in _slab_inputs(case, seed)]
        ext = [s.extent() for s in slabs]
        b = hip.Batch(case["dt"], sum(e[0] for e in ext), sum(e[1] for e in ext),
                      slab_capacity=len(slabs), mode=case["mode"], sensors=3)
        ids = [b.add(s) for s in slabs]
        b.set_graph(case["graph"])
        b.sync()
        return dict(kind=kind, batch=b, ids=ids, steps=case["steps"])
    d, own = _dev(), _Handles()
    if kind == "reaction":
        n = case["n"]
        V, st = _cells(seed, n)
        h = own.reaction("endoCellML", n, case["deck"], case["dt"])
        hip.check(hip.lib().cdh_tt06_set_state(h, hip.ptr(np.ascontiguousarray(st).reshape(-1))),
                  "cdh_tt06_set_state")
        # one cell type's cells, two of every three, of a wall of several types
        idx = torch.arange(n, dtype=torch.int32, device=d) * 3 // 2
        N = int(n * 3 // 2 + 2)
        Vm = torch.full((N,), -86.709, dtype=torch.float64, device=d)
        Vm[idx.long()] = torch.from_numpy(V).to(d)
        zero = torch.zeros(N, dtype=torch.float64, device=d)
        return dict(kind=kind, own=own, h=h, n=n, N=N, idx=idx, Vm=Vm, dVmR=torch.zeros_like(Vm),
                    zero=zero, dt=case["dt"], steps=case["steps"])
    a, types, stim = _anatomy(case, rng)
    n = a.ncell
    f = own.diffusion(a)
    if kind == "diffusion":
        Vm = torch.from_numpy(_field(seed, n)).to(d)
        return dict(kind=kind, own=own, f=f, Vm=Vm, dVm=torch.zeros_like(Vm))
    groups = [np.nonzero(a.celltype == t)[0].astype(np.int32) for t in range(len(types))]
    react = [(own.reaction(types[t], g.size, case["deck"], case["dt"]),
              torch.from_numpy(g).to(d), int(g.size)) for t, g in enumerate(groups) if g.size]
    Vm = torch.zeros(n, dtype=torch.float64, device=d)
    for h, idx, m in react:
        hip.check(hip.lib().cdh_tt06_initialize_membrane_voltage(h, _p(idx), m, _p(Vm), None),
                  "cdh_tt06_initialize_membrane_voltage")
    Vm += torch.from_numpy(_field(seed, n) + 30.0).to(d).clamp(min=0.0)
    x, y, z = a.tuples()
    lists = []
    for b in stim:
        m = ((x > b.xMin) & (x < b.xMax) & (y > b.yMin) & (y < b.yMax) & (z > b.zMin) & (z < b.zMax))
        lists.append((b, torch.from_numpy(np.nonzero(m)[0].astype(np.int32)).to(d)))
    s = C.c_void_p()
    hip.check(hip.lib().cdh_activation_sensor_create(n, -40.0, C.byref(s)), "sensor")
    own.sensor.append(s)
    z64 = [torch.zeros_like(Vm) for _ in range(3)]
    return dict(kind=kind, own=own, f=f, react=react, lists=lists, sensor=s, n=n, Vm=Vm,
                dVmR=z64[0], dVmD=z64[1], iStim=z64[2], time=0.0, dt=case["dt"],
                steps=case["steps"])


# ------------------------------------------------------------------- one pass

def run(state):
    L, kind = hip.lib(), state["kind"]
    if kind == "sim":
        sim = state["sim"]
        sim.run(state["steps"])
        out = {"vm": sim.vm(), "activation": sim.activation()[1]}
        if state["sensors"] & 2:
            out["t90"] = sim.t90()
        if state["states"]:
            out["state"] = sim.state()
        return out
    if kind == "batch":
        b = state["batch"]
        b.run(state["steps"])
        b.sync()
        return [{"vm": b.vm(i), "activation": b.activation(i)[1], "t90": b.t90(i)}
                for i in state["ids"]]
    if kind == "reaction":
        Vm, dVm, z = _p(state["Vm"]), _p(state["dVmR"]), _p(state["zero"])
        for _ in range(state["steps"]):
            hip.check(L.cdh_tt06_calc(state["h"], state["dt"], _p(state["idx"]), state["n"], Vm,
                                      None, dVm, None), "cdh_tt06_calc")
            hip.check(L.cdh_integrate(state["N"], state["dt"], Vm, dVm, z, z, None),
                      "cdh_integrate")
        return {"Vm": state["Vm"], "dVm": state["dVmR"]}
    if kind == "diffusion":
        hip.check(L.cdh_fgr_update_local_voltage(state["f"], _p(state["Vm"]), None), "update")
        hip.check(L.cdh_fgr_calc(state["f"], _p(state["dVm"]), None), "cdh_fgr_calc")
        return state["dVm"]
    n, dt = state["n"], state["dt"]
    Vm, dR, dD, iS = (_p(state[k]) for k in ("Vm", "dVmR", "dVmD", "iStim"))
    for _ in range(state["steps"]):
        hip.check(L.cdh_fill(n, 0.0, iS, None), "cdh_fill")
        for b, cells in state["lists"]:
            if b.phase <= state["time"] < b.phase + b.duration:
                hip.check(L.cdh_set_list(cells.numel(), _p(cells), b.amplitude, iS, None), "stim")
        for h, idx, m in state["react"]:
            hip.check(L.cdh_tt06_calc(h, dt, _p(idx), m, Vm, iS, dR, None), "cdh_tt06_calc")
        hip.check(L.cdh_fgr_update_local_voltage(state["f"], Vm, None), "update")
        hip.check(L.cdh_fgr_calc(state["f"], dD, None), "cdh_fgr_calc")
        hip.check(L.cdh_integrate(n, dt, Vm, dR, dD, iS, None), "cdh_integrate")
        state["time"] += dt
        hip.check(L.cdh_activation_sensor_eval(state["sensor"], state["time"], Vm, None), "sensor")
    return {"Vm": state["Vm"], "dVmR": state["dVmR"], "dVmD": state["dVmD"]}


# ----------------------------------------------------------------------- work

def _ncell(case):
    if case["kind"] == "reaction":
        return case["n"]
    if case["kind"] == "batch":
        dims = np.random.default_rng(case["dims_seed"])
        return sum(math.prod(int(round(math.exp(dims.uniform(math.log(case["lo"]),
                                                             math.log(case["hi"])))))
                             for _ in range(3)) for _ in range(case["slabs"]))
    if case["shape"] == "shell":
        return _shell(case["nx"], case["ny"], case["nz"]).ncell
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """Per cell and step.  Fused FP64: 19 states and Vm read and written
    (320), 18 float weights (72).  Mixed: 17 FP32 and 2 FP64 states and Vm
    (184), compact weights (37).  The drop-in stages each read their inputs
    and write their outputs once: reaction 304 + 16 + 4, scatter 20, stencil
    76 + 16, integrator 40, fill 8, sensor 8.  About 1,060 floating
    operations with the fits; the exact functions' 49 exponentials at some 25
    operations each make it about 2,000."""
    n, kind = _ncell(case), case["kind"]
    flops = 2000 if case.get("deck") == "exact" else 1060
    if kind == "diffusion":
        return {"bytes": 112 * n, "flops": 41 * n}
    steps = case["steps"]
    if kind == "reaction":
        return {"bytes": (324 * n + 40 * (n * 3 // 2 + 2)) * steps, "flops": (flops - 41) * n * steps}
    if kind == "loop" or case["mode"] == "fp64_unfused":
        per = 324 + 20 + 92 + 40 + 8 + 8
    else:
        per = 221 if case["mode"] == "mixed_fused" else 392
    return {"bytes": per * n * steps, "flops": flops * n * steps}


# --------------------------------------------------------------- 64-bit values

_STATES = ["Ca_i", "dVK_i", "Na_i", "Ca_ss", "Ca_SR", "R_prime", "fCass", "m", "h", "j", "Xr1",
           "Xr2", "Xs", "r", "d", "f", "f2", "jL", "s"]
# s gate form, P_NaK, g_Ks, g_Kr, g_to, g_NaL, rest Vm, rest states (K_i in slot 1)
_TYPES = {
    "endoCellML": (0, 2.724, 0.392, 0.153, 0.073, 0.0, -86.709,
                   [0.00013, 138.4, 10.355, 0.00036, 3.715, 0.9068, 0.9953, 0.00155, 0.7573,
                    0.7225, 0.00448, 0.476, 0.0087, 2.235e-8, 3.164e-5, 0.8009, 0.9778, 0.066,
                    0.3212]),
    "midCellML": (1, 2.724, 0.098, 0.153, 0.294, 0.0, -85.423,
                  [0.000153, 138.52, 10.132, 0.00042, 4.272, 0.8978, 0.9942, 0.00165, 0.749,
                   0.6788, 0.0165, 0.473, 0.0174, 2.347e-8, 3.288e-5, 0.7026, 0.9526, 0.066,
                   0.999998]),
    "epiCellML": (1, 2.724, 0.392, 0.153, 0.294, 0.0, -85.23,
                  [0.000126, 136.89, 8.604, 0.00036, 3.64, 0.9073, 0.9953, 0.00172, 0.7444,
                   0.7045, 0.00621, 0.4712, 0.0095, 2.42e-8, 3.373e-5, 0.7888, 0.9755, 0.066,
                   0.999998]),
}


@functools.lru_cache(maxsize=None)
def _constants():
    """The model's physical parameters and the combinations its currents use."""
    F, RT, Cm, Vc, Vsr, Vss = 96485.3415, 8314.472 * 310, 0.185, 0.016404, 0.001094, 0.00005468
    Ko, Nao, Cao = 5.4, 140.0, 2.0
    e = RT / F
    c9 = -Cm / (Vc * F)
    fca = 0.5 * 0.0000398 * F
    na3 = Nao ** 3
    return dict(e=e, c9=c9, ENa=e * math.log(Nao), EK=e * math.log(Ko),
                EKs=e * math.log(Ko + 0.03 * Nao), ECa=0.5 * e * math.log(Cao), Vc=Vc, Vsr=Vsr,
                Vss=Vss, f1=1 / e, f2=-2 * Ko / (Ko + 1),
                f3=(87.5 ** 3 + na3) * (1.38 + Cao) / (1000 * Cao), f6=na3 * 2.5 / Cao, f7=fca,
                f9=4 * Cao * fca, gK1=5.405 * math.sqrt(Ko / 5.4),
                c13=Cm / (2 * Vss * F * c9), c23=-0.0038 * Vc / (Vss * c9))


@functools.lru_cache(maxsize=None)
def _fits():
    """{name: (numerator, denominator)} and the names in the model's order."""
    with open(FIT_FILE) as fh:
        text = fh.read()
    got, order = {}, []
    for name, body in re.findall(r"(\w+)\s+FIT\s*\{(.*?)\}", text, re.S):
        kv = dict((w.strip() for w in x.split("=", 1)) for x in body.split(";") if "=" in x)
        if name == "functions":
            order = kv["functions"].split()
            continue
        m, c = int(kv["m"]), [float(v) for v in kv["coef"].split()]
        got[name] = (c[:m], c[m:])
    return got, order


def _poly(c, x):
    s = torch.full_like(x, c[-1])
    for a in reversed(c[:-1]):
        s = a + x * s
    return s


def _fit(i, x):
    got, order = _fits()
    num, den = got[order[i]]
    return _poly(num, x) / _poly(den, x) if len(den) > 1 else _poly(num, x)


def _sig(x):
    return 1.0 / (1.0 + torch.exp(x))


def _h_rate(V):
    e = torch.exp
    low = 0.057 * e(-(V + 80) / 6.8) + 2.7 * e(0.079 * V) + 310000.0 * e(0.3485 * V)
    return torch.where(V < -40, low, 0.77 / 0.13 * _sig((V + 10.66) / -11.1))


def _j_rate(V):
    e = torch.exp
    low = ((-25428.0 * e(0.2444 * V) - 6.948e-06 * e(-0.04391 * V)) * (V + 37.78)
           * _sig(0.311 * (V + 79.23)) + 0.02424 * e(-0.01052 * V) * _sig(-0.1378 * (V + 40.14)))
    return torch.where(V < -40, low, 0.6 * e(0.057 * V) * _sig(-0.1 * (V + 32)))


@functools.lru_cache(maxsize=None)
def _bridge(name):
    """The cubic that joins a rate's two branches smoothly on [x0, x1]."""
    rate, x0, x1 = {"h": (_h_rate, -64.20, -23.3), "j": (_j_rate, -48.85, -17.6)}[name]
    x = torch.tensor([x0, x1], dtype=torch.float64, requires_grad=True)
    p = rate(x)
    d = torch.autograd.grad(p.sum(), x)[0].tolist()
    p, w = p.tolist(), x1 - x0
    return (x0, x1, p[0], d[0], 3 * (p[1] - p[0]) / w ** 2 - (2 * d[0] + d[1]) / w,
            -2 * (p[1] - p[0]) / w ** 3 + (d[0] + d[1]) / w ** 2)


def _bridged(name, V):
    x0, x1, a, b, c, d = _bridge(name)
    x = V - x0
    return torch.where((V < x0) | (V > x1), {"h": _h_rate, "j": _j_rate}[name](V),
                       a + x * (b + x * (c + x * d)))


def _gates_exact(V):
    """(steady state, rate) of m h j Xr1 Xr2 Xs r d f f2 jL s0 s1."""
    e = torch.exp
    hj = _sig((V + 71.55) / 7.43) ** 2
    yield _sig((-56.86 - V) / 9.03) ** 2, 1 / (_sig((-60 - V) / 5) *
                                               (0.1 * _sig((V + 35) / 5) + 0.1 * _sig((V - 50) / 200)))
    yield hj, _bridged("h", V)
    yield hj, _bridged("j", V)
    yield _sig((-26 - V) / 7), (1 + e((-45 - V) / 10)) / 450 * (1 + e((V + 30) / 11.5)) / 6
    yield _sig((V + 88) / 24), (1 + e((-60 - V) / 20)) / 3 * (1 + e((V - 60) / 20)) / 1.12
    yield _sig((-5 - V) / 14), 1 / (1400 / torch.sqrt(1 + e((5 - V) / 6)) * _sig((V - 35) / 15) + 80)
    yield _sig((20 - V) / 6), 1 / (9.5 * e(-(V + 40) ** 2 / 1800) + 0.8)
    yield _sig((-8 - V) / 7.5), 1 / ((1.4 * _sig((-35 - V) / 13) + 0.25) * 1.4 * _sig((V + 5) / 5)
                                     + _sig((50 - V) / 20))
    yield _sig((V + 20) / 7), 1 / (1102.5 * e(-(V + 27) ** 2 / 225) + 200 * _sig((13 - V) / 10)
                                   + 180 * _sig((V + 30) / 10) + 20)
    yield 0.67 * _sig((V + 35) / 7) + 0.33, 1 / (562 * e(-(V + 27) ** 2 / 240)
                                                 + 31 * _sig((25 - V) / 10) + 80 * _sig((V + 30) / 10))
    yield e(-(V + 91) * 2 / 6.1), torch.full_like(V, 1 / 670)
    yield _sig((V + 28) / 5), 1 / (1000 * e(-(V + 67) ** 2 / 1000) + 8)
    yield _sig((V + 20) / 5), 1 / (85 * e(-(V + 45) ** 2 / 320) + 5 * _sig((V - 20) / 5) + 3)


def _voltage_exact(V):
    k, e = _constants(), torch.exp
    f1 = k["f1"]
    x = 2 * f1 * (V - 15)
    near = x * x < 1e-4
    xs = torch.where(near, torch.ones_like(x), x)
    odd, even = 0.5 * x, 1 + x * x / 12 - x ** 4 / 720
    e1, e5 = e(-f1 * V), e(0.35 * f1 * V)
    a = 1 / (k["f3"] * (1 + 0.1 * e5 * e1))
    return [k["f2"] / (1 + 0.1245 * e(-0.1 * f1 * V) + 0.0353 * e1), e5 * a, e5 * e1 * a * k["f6"],
            k["f7"] * torch.where(near, even + odd, xs / -torch.expm1(-xs)),
            k["f9"] * torch.where(near, even - odd, xs / torch.expm1(xs)),
            0.0146 * _sig((25 - V) / 5.98)]


def _k1_exact(v):
    e = torch.exp
    return _constants()["gK1"] / (1 + (3 * e(0.0002 * v + 0.02) + e(0.1 * v - 1)) * _sig(-0.5 * v)
                                  * (10 + 10 * e(0.06 * v - 12)))


class _Model:
    """Cells of one or more slabs: their states, parameters and neighbours."""

    def __init__(self, V, st, ct, types, scales, deck, dt, tail):
        d = V.device
        rows = torch.tensor([_TYPES[t][:7] for t in types], dtype=torch.float64, device=d)[ct]
        self.form1 = rows[:, 0] > 0
        self.PNaK, self.gKs, self.gKr, self.gto, self.gNaL = rows[:, 1:6].unbind(1)
        self.skr, self.scal, self.sna = scales
        self.V, self.s, self.deck, self.dt, self.moves = V, st, deck, dt, ~tail

    def react(self):
        """-Iion at the present Vm; the states move by dt."""
        k, s, V, dt, fits = _constants(), self.s, self.V, self.dt, self.deck == "fits"
        Ca, Na, Css, Csr, R, fC = s[0], s[2], s[3], s[4], s[5], s[6]
        fv = [_fit(i, V) for i in range(6)] if fits else _voltage_exact(V)
        c9, e, Vc, Vsr, Vss = k["c9"], k["e"], k["Vc"], k["Vsr"], k["Vss"]
        hill = lambda x: x / (1 + x)  # noqa: E731
        buf = lambda c, b, kk: hill((c + kk) ** 2 / (b * kk))  # noqa: E731
        dV3 = V + 0.5 * e * torch.log(Ca) - k["ECa"]
        INaCa = Na ** 3 * fv[1] - Ca * fv[2]
        IbCa, IpCa = 0.000592 * dV3, 0.1238 * hill(Ca / 0.0005)
        Iup = 0.006375 / c9 * hill((Ca / 0.00025) ** 2)
        Ileak, Ixfer = 0.00036 / c9 * (Csr - Ca), k["c23"] * (Css - Ca)
        Idelta, Isum = Ileak - Iup, IbCa + IpCa
        Ki = c9 * (s[1] - V)
        dV0 = V + e * torch.log(Ki) - k["EK"]
        dV1 = V + e * torch.log(Na) - k["ENa"]
        dV2 = V + e * torch.log(Ki + 0.03 * Na) - k["EKs"]
        fv6 = _fit(6, dV0) if fits else _k1_exact(dV0)
        m3 = s[7] ** 3
        INaK = self.PNaK * hill(Na / 40) * fv[0]
        INa = self.sna * 14.838 * m3 * s[8] * s[9] * dV1
        IKs = self.gKs * s[12] ** 2 * dV2
        iNa = 3 * INaCa - 1.5 * INaK + INa + 0.00029 * dV1 + self.gNaL * m3 * s[17] * dV1
        iK = (IKs + INaK + fv[5] * dV0 + fv6 * dV0 + self.gto * s[13] * s[18] * dV0
              + self.skr * self.gKr * s[10] * s[11] * dV0)
        tmp8 = 0.045 * (2.5 - 1.5 * hill((Csr / 1.5) ** 2)) / c9
        ICaL = self.scal * s[14] * s[15] * s[16] * fC * (fv[4] - Css * fv[3])
        O = Css ** 2 * R / (tmp8 * 0.06 / (0.15 * 0.045) * c9 + Css ** 2)
        Irel = 0.102 / c9 * O * (Csr - Css)
        dVR = -Isum - (iNa + iK - 2 * INaCa) + ICaL
        t1 = 1 / (1 + (20 * Css) ** 2)
        new = [Ca + dt * c9 * buf(Ca, 0.2, 0.001) * (0.5 * Isum - INaCa - Ixfer * Vss / Vc
                                                     + Idelta * Vsr / Vc),
               s[1] + dt * iK + dt * dVR, Na + dt * c9 * iNa,
               Css + dt * c9 * buf(Css, 0.4, 0.00025) * (Ixfer + Irel * Vsr / Vss + ICaL * k["c13"]),
               Csr - dt * c9 * buf(Csr, 10.0, 0.3) * (Idelta + Irel),
               R + dt * c9 * (0.005 / c9 - (tmp8 * Css + 0.005 / c9) * R),
               fC + dt * (0.6 * t1 + 0.4 - fC) / (80 * t1 + 2)]
        # the gates: m by Rush-Larsen (with the fits by its series of degree
        # 16), the others by one explicit step
        if fits:
            pairs = [(_fit(7 + 2 * q, V), _fit(8 + 2 * q, V)) for q in range(13)]
        else:
            pairs = list(_gates_exact(V))
        pairs[11] = tuple(torch.where(self.form1, b, a) for a, b in zip(pairs[11], pairs[12]))
        for q in range(12):
            mhu, rate = pairs[q]
            r = dt * rate
            if q == 0:
                r = (1 - 1 / _poly([1 / math.factorial(i) for i in range(17)], r) if fits
                     else -torch.expm1(-r))
            g = s[7 + q]
            g = g + r * (mhu - g)
            new.append(torch.where(self.moves, g, s[7 + q]) if fits else g)
        self.s = new
        return dVR


_NODES = [(0, 0, 0), (-1, 0, 0), (0, -1, 0), (1, 0, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1),
          (-1, -1, 0), (1, -1, 0), (1, 1, 0), (-1, 1, 0), (-1, 0, -1), (0, -1, -1), (1, 0, -1),
          (0, 1, -1), (-1, 0, 1), (0, -1, 1), (1, 0, 1), (0, 1, 1)]


class _Stencil:
    """The finite-volume diffusion operator of several anatomies, each in a
    box of its own with an empty margin."""

    def __init__(self, anatomies, dev):
        at, stride, base, sig = [], [], 0, []
        for a in anatomies:
            x, y, z = (torch.from_numpy(np.ascontiguousarray(v)).to(dev) + 1 for v in a.tuples())
            sx, sy = (a.ny + 2) * (a.nz + 2), a.nz + 2
            at.append(base + x * sx + y * sy + z)
            stride.append(torch.tensor([sx, sy, 1], device=dev).expand(a.ncell, 3))
            sig.append(torch.from_numpy(np.ascontiguousarray(a.sigma)).to(dev))
            base += (a.nx + 2) * sx
        self.at, st, sg = torch.cat(at), torch.cat(stride), torch.cat(sig)
        h = [anatomies[0].dx, anatomies[0].dy, anatomies[0].dz]
        self.box = torch.zeros(base, dtype=torch.float64, device=dev)
        tissue = torch.zeros(base, dtype=torch.bool, device=dev)
        tissue[self.at] = True
        cell = torch.zeros(base, dtype=torch.int64, device=dev)
        cell[self.at] = torch.arange(self.at.numel(), device=dev)

        def node(d):
            return self.at + d[0] * st[:, 0] + d[1] * st[:, 1] + d[2] * st[:, 2]

        where = [node(d) for d in _NODES]
        has = [tissue[i] for i in where]
        w = [torch.zeros(self.at.numel(), dtype=torch.float64, device=dev) for _ in _NODES]
        full = ((0, 1, 2), (1, 3, 4), (2, 4, 5))       # tensor components by row
        for ax in range(3):
            for sign in (-1, 1):
                step = [0, 0, 0]
                step[ax] = sign
                k = _NODES.index(tuple(step))
                mean = (sg + sg[cell[where[k]]]) / 2
                flux = [has[k] * sign / h[ax] * mean[:, full[ax][j]] for j in range(3)]
                # normal: difference across the face
                w[k] += sign * flux[ax] / h[ax]
                w[0] -= sign * flux[ax] / h[ax]
                # transverse: mean of the central differences of both cells,
                # where all four of their nodes are tissue
                for j in range(3):
                    if j == ax:
                        continue
                    four = []
                    for s2 in (-1, 1):
                        for off in (0, sign):
                            p = [0, 0, 0]
                            p[ax], p[j] = off, s2
                            four.append((s2, _NODES.index(tuple(p))))
                    ok = has[four[0][1]] & has[four[1][1]] & has[four[2][1]] & has[four[3][1]]
                    for s2, q in four:
                        w[q] += ok * flux[j] * (0.25 * s2 / h[j])
        self.w = [v.float().double() for v in w[1:]]
        self.where = where[1:]

    def apply(self, V):
        self.box[self.at] = V
        out = torch.zeros_like(V)
        for w, i in zip(self.w, self.where):
            out += w * (self.box[i] - V)
        return out * W.DIFFUSION_SCALE


def _tail(ct, ntypes):
    """The cells past the last whole four of their type: the fits' gate
    updates go four at a time and leave them as they are."""
    out = np.zeros(ct.size, bool)
    for t in range(ntypes):
        i = np.nonzero(ct == t)[0]
        out[i[4 * (i.size // 4):]] = True
    return out


def _rest(ct, types, dev):
    rows = torch.tensor([_TYPES[t][7] for t in types], dtype=torch.float64, device=dev)
    v0 = torch.tensor([_TYPES[t][6] for t in types], dtype=torch.float64, device=dev)
    V = v0[ct]
    st = [rows[:, q][ct] for q in range(19)]
    st[1] = st[1] / _constants()["c9"] + V
    return V, st


def exact(case, seed):
    kind, dev = case["kind"], _dev()
    n, steps = _ncell(case), case.get("steps", 1)
    if steps * (0.009 + 1.2e-8 * n) > 14.0 or (dev.type == "cpu" and n * steps > 200_000):
        return None
    rng = np.random.default_rng(seed)
    up = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)  # noqa: E731
    if kind == "reaction":
        V, st = _cells(seed, n)
        ct = torch.zeros(n, dtype=torch.int64, device=dev)
        M = _Model(up(V), [up(v) for v in st], ct, ["endoCellML"], (1.0, 1.0, 1.0), case["deck"],
                   case["dt"], up(_tail(np.zeros(n, int), 1)))
        for _ in range(steps):
            d = M.react()
            M.V = M.V + case["dt"] * d
        idx = torch.arange(n, device=dev) * 3 // 2
        Vm = torch.full((n * 3 // 2 + 2,), -86.709, dtype=torch.float64, device=dev)
        dVm = torch.zeros_like(Vm)
        Vm[idx], dVm[idx] = M.V, d
        return {"Vm": Vm, "dVm": dVm}
    if kind == "batch":
        slabs = _slab_inputs(case, seed)
        anatomies, types = [s[0] for s in slabs], ["endoCellML"]
        sc = np.concatenate([np.tile(s[1], (s[0].ncell, 1)) for s in slabs])
        tail = np.concatenate([_tail(a.celltype, 1) for a in anatomies])
        stims = [s[2] for s in slabs]
    else:
        a, types, stim = _anatomy(case, rng)
        anatomies, stims = [a], [stim]
        if kind == "diffusion":
            return _Stencil(anatomies, dev).apply(up(_field(seed, n)))
        sc = _scales(rng, n) if kind == "sim" else np.ones((n, 3))
        tail = _tail(a.celltype, len(types))
    ct = up(np.concatenate([a.celltype for a in anatomies]).astype(np.int64))
    V, st = _rest(ct, types, dev)
    if kind == "loop":
        V = V + up(_field(seed, n) + 30.0).clamp(min=0.0)
    M = _Model(V, st, ct, types, up(sc).unbind(1), case["deck"], case["dt"], up(tail))
    S = _Stencil(anatomies, dev)
    boxes = []                      # (stimulus, its cells), in the order they are applied
    for q in range(max(len(s) for s in stims)):
        for k, a in enumerate(anatomies):
            b = stims[k][q]
            x, y, z = a.tuples()
            inside = ((x > b.xMin) & (x < b.xMax) & (y > b.yMin) & (y < b.yMax) & (z > b.zMin)
                      & (z < b.zMax))
            pre = sum(v.ncell for v in anatomies[:k])
            boxes.append((b, up(np.nonzero(inside)[0] + pre)))
    t = 0.0
    for _ in range(steps):
        cur = torch.zeros_like(M.V)
        for b, cells in boxes:
            if b.phase <= t < b.phase + b.duration:
                cur[cells] = b.amplitude
        dR, dD = M.react(), S.apply(M.V)
        M.V = M.V + case["dt"] * (dR + dD + cur)
        t += case["dt"]
    if kind == "loop":
        return {"Vm": M.V, "dVmR": dR, "dVmD": dD}
    if kind == "sim":
        out = {"vm": M.V, "activation": None}
        if n <= 4096:
            out["state"] = torch.stack(M.s)
        return out
    return [{"vm": v, "activation": None, "t90": None}
            for v in M.V.split([a.ncell for a in anatomies])]
