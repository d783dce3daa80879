"""Timed work of this framework: what a program that uses it has it do, through
its public entry points, over the range of sizes it is used at.

The marker step (thermal and visco-elasto-plastic), the batched ensemble, passive
tracers under population control, the nodal step, the two nodal solves and the
learned guess's network.  Inputs follow ``fvmic2d_amd.workloads``: the grids,
nodal fields, materials and options are its own; the markers are drawn on the GPU,
cell by cell (the order ``fvm_markers_reorder`` leaves a store in), with its
distributions.  Device arrays belong to torch, so a pass hands back the state's
own buffers.

``exact`` computes the same outputs with plain torch in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

from fvmic2d_amd import abi, workloads
from fvmic2d_amd.host import VEP_PROJ, Ensemble, MarkerPath, initial_pressure_guess
from fvmic2d_amd.lib import Context, DeviceGrid, DeviceNodal, fvm_markers
from fvmic2d_amd.unet import Buf, UNet, to_bf16_bits

F64 = torch.float64
DEV = "cuda"
G = 10.0                # gravity of the learned guess's box
STEP = 0.1              # largest marker displacement of a step in cells (options' displacementStepLimit)
VEP_CARRIED = ("dsxx", "dsyy", "dsxy")   # nodal arrays a VEP step updates in place


# ------------------------------------------------------------------ the cases --
def listed():
    return [
        # the smallest whole step: the 51x51 isoviscous box at 16 markers a cell,
        # the reference's full projection set; a call is short, so launches count
        {"name": "thermal_51", "kind": "thermal", "n": 51, "nm": 4, "list": "all2"},
        # the ordinary single run: temperature-dependent viscosity, 17 projections
        # onto all four staggered node families, 1.44 M markers
        {"name": "thermal_201", "kind": "thermal", "n": 201, "nm": 6, "list": "tdep"},
        # markers carried by a given flow (no projections), with the reference's
        # per-step population control; 4 M markers, sizes that divide nothing
        {"name": "tracers_403", "kind": "tracers", "n": 403, "nm": 5},
        # the full visco-elasto-plastic step on a small grid periodic in x
        {"name": "vep_periodic_130x67", "kind": "vep", "nx": 130, "ny": 67, "nm": 4, "periodic": True},
        # the full visco-elasto-plastic subduction step, 8 M markers, 5 materials
        {"name": "vep_801x401", "kind": "vep", "nx": 801, "ny": 401, "nm": 5, "periodic": False},
        # a parameter sweep of small problems stepped together
        {"name": "ensemble_256_small", "kind": "ensemble", "count": 256, "nmin": 17, "nmax": 65, "sizes": 4},
        # the largest: 64 problems of 65..257 nodes a side, about 47 M markers
        {"name": "ensemble_64", "kind": "ensemble", "count": 64, "nmin": 65, "nmax": 257, "sizes": 4},
        # between the Stokes solve and the marker updates: solution retrieval,
        # nodal stresses and strain rates, displacement limit of the time step
        {"name": "nodal_801x401", "kind": "nodal", "nx": 801, "ny": 401},
        # the energy equation of a step: assembly and solve to 1e-12
        {"name": "energy_801x401", "kind": "energy", "nx": 801, "ny": 401, "graded": True},
        # the plain initial pressure guess at the learned guess's tolerance
        {"name": "pressure_257", "kind": "pressure", "nx": 257, "ny": 257, "graded": False},
        # one optimiser step of the learned guess's network (forward, loss,
        # backward, Adam) at its training size: 128x128, batch 8
        {"name": "unet_train_128", "kind": "unet_train", "size": 128, "batch": 8, "levels": 4, "base": 32},
        # one prediction, as the guess is made in a run: a single state of 256x256
        {"name": "unet_predict_256", "kind": "unet_predict", "size": 256, "batch": 1, "levels": 4, "base": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["thermal", "thermal", "tracers", "vep", "vep", "ensemble", "nodal", "energy", "pressure",
                       "unet_train", "unet_predict"])
    if kind == "thermal":
        return {"kind": kind, "n": _log_int(rng, 33, 513), "nm": rng.randint(4, 6), "list": rng.choice(["all2", "tdep"])}
    if kind == "tracers":
        return {"kind": kind, "n": _log_int(rng, 51, 513), "nm": rng.randint(4, 6)}
    if kind == "vep":
        return {"kind": kind, "nx": _log_int(rng, 65, 801), "ny": _log_int(rng, 49, 401), "nm": rng.randint(4, 5),
                "periodic": rng.random() < 0.4}
    if kind == "ensemble":
        count = _log_int(rng, 8, 256)
        nmin = _log_int(rng, 17, 65)
        nmax = max(nmin + 8, int(min(257, 257 * math.sqrt(48.0 / count), nmin * rng.uniform(1.5, 4.0))))
        return {"kind": kind, "count": count, "nmin": nmin, "nmax": nmax, "sizes": rng.randint(1, 10 ** 6)}
    if kind in ("nodal", "energy"):
        c = {"kind": kind, "nx": _log_int(rng, 65, 801), "ny": _log_int(rng, 49, 401)}
        return c if kind == "nodal" else dict(c, graded=rng.random() < 0.7)
    if kind == "pressure":
        return {"kind": kind, "nx": _log_int(rng, 65, 400), "ny": _log_int(rng, 65, 400), "graded": rng.random() < 0.5}
    levels = rng.randint(3, 4)
    size = 2 ** (levels - 1) * rng.randint(4, 16 if kind == "unet_train" else 32)
    return {"kind": kind, "size": size, "batch": rng.randint(1, 8), "levels": levels, "base": rng.choice([16, 32])}


# ------------------------------------------------- a problem on torch's memory --
_context = None


def context():
    """The process's one library context."""
    global _context
    if _context is None:
        _context = Context()
    return _context


class _Slot:
    """A device array of the caller's (a torch tensor) under DeviceArray's names."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


class Store:
    """fvm_markers over torch columns: one tensor per field."""

    def __init__(self, cols, n, capacity):
        self.cols = cols
        self.desc = fvm_markers()
        self.desc.nMark, self.desc.maxMark = n, capacity
        for name, t in cols.items():
            setattr(self.desc, name, t.data_ptr())

    ref = property(lambda self: ctypes.byref(self.desc))
    n = property(lambda self: self.desc.nMark)

    def col(self, name):
        return getattr(self.desc, name)


class Fields(DeviceNodal):
    """Named nodal arrays over torch tensors."""

    def __init__(self, tensors):
        self.tensors = tensors
        self.arrays = {k: _Slot(t) for k, t in tensors.items()}
        self.desc = abi.NodalArrays()
        for k, t in tensors.items():
            if k in abi.NODAL_NAMES:
                setattr(self.desc, k, t.data_ptr())


class Problem(MarkerPath):
    """A MarkerPath whose marker store and nodal arrays are the caller's."""

    def __init__(self, w, store, fields):
        self.w, self.ctx = w, context()
        self.grid = DeviceGrid(self.ctx, w)
        self.markers, self.nodal = store, fields
        self._tables = []
        self.proj_list = self.projection_list(w.projections) if isinstance(w.projections, list) else None


def _field_names(w):
    names = list(abi.NODAL_NAMES)
    if isinstance(w.projections, list):
        names += [p[4] for p in w.projections]
    if w.kind == "vep":
        names += VEP_PROJ
    return list(dict.fromkeys(names))


def _fields(w, names=None):
    t = {}
    for k in names or _field_names(w):
        a = w.nodal.get(k)
        t[k] = torch.zeros((w.NY, w.NX), dtype=F64, device=DEV) if a is None else \
            torch.as_tensor(np.ascontiguousarray(a), dtype=F64).to(DEV)
    return t


def _columns(n):
    c = {k: torch.zeros(n, dtype=F64, device=DEV) for k in abi.DCOLS}
    c.update({k: torch.zeros(n, dtype=torch.int32, device=DEV) for k in abi.ICOLS})
    c["cellX"].fill_(-1)
    c["cellY"].fill_(-1)
    return c


def _positions(w, nm, gen):
    """nm x nm jittered markers in every cell, cell after cell."""
    xs = torch.as_tensor(np.append(w.x, w.LX) if w.xperiodic else w.x, dtype=F64).to(DEV)
    ys = torch.as_tensor(w.y, dtype=F64).to(DEV)
    hx, hy = (xs[1:] - xs[:-1]) / nm, (ys[1:] - ys[:-1]) / nm
    sub = torch.arange(nm, dtype=F64, device=DEV) + 0.5
    n = hx.numel() * hy.numel() * nm * nm
    shape = (hy.numel(), hx.numel(), nm, nm)
    X = xs[:-1].view(1, -1, 1, 1) + hx.view(1, -1, 1, 1) * (sub.view(1, 1, 1, -1) + _uniform(gen, shape, -0.25, 0.25))
    Y = ys[:-1].view(-1, 1, 1, 1) + hy.view(-1, 1, 1, 1) * (sub.view(1, 1, -1, 1) + _uniform(gen, shape, -0.25, 0.25))
    return X.reshape(n), Y.reshape(n)


def _uniform(gen, shape, lo, hi):
    return lo + (hi - lo) * torch.rand(shape, dtype=F64, device=DEV, generator=gen)


def _normal(gen, n):
    return torch.randn(n, dtype=F64, device=DEV, generator=gen)


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _thermal_workload(n, which, seed, contrast=1e5):
    w = workloads.convection_tdep(seed=seed, N=n, NM=1, contrast=contrast)
    if which == "all2":
        w.projections = "all2"
        w.materials.QonR[0] = 0.0
    w.dt *= STEP / 0.5
    return w


def _thermal_markers(c, w, nm, gen):
    """Fill columns c (slices of the store) for one convection problem."""
    X, Y = _positions(w, nm, gen)
    c["X"].copy_(X)
    c["Y"].copy_(Y)
    prof = 0.5 * torch.erf(Y / 0.05) + 0.5 * (1.0 + torch.erf((Y - 1.0) / 0.05))
    c["T"].copy_(prof * (1.0 + 0.02 * _normal(gen, X.numel())))
    c["eta"].copy_(torch.exp(-w.materials.QonR[0] * c["T"]))
    c["mu"].fill_(1e99)


def _vep_workload(case, seed):
    if case["periodic"]:
        w = workloads.periodic_box("vep", NX=case["nx"], NY=case["ny"], NM=1, seed=seed)
    else:
        w = workloads.vep_subduction(seed=seed, NX=case["nx"], NY=case["ny"], NM=1)
    w.dt *= STEP / 0.5
    return w


def _vep_markers(c, w, nm, gen):
    X, Y = _positions(w, nm, gen)
    n = X.numel()
    c["X"].copy_(X)
    c["Y"].copy_(Y)
    d = Y + 1.5e3 * torch.sin(2.0 * math.pi * X / w.LX) + 5e2 * torch.sin(6.0 * math.pi * X / w.LX)
    mat = (d >= 1.0e4).int() + (d >= 3.0e4).int() + (d >= 6.0e4).int()
    slab = ((Y - (X - 0.6e5) * 0.8).abs() < 1.2e4) & (X > 0.6e5)
    mat = torch.where(slab, torch.full_like(mat, 4), mat)
    c["Mat"].copy_(mat)
    T = 273.0 + 1300.0 * (Y / w.LY).clamp(0, 1) * (1.0 + 0.01 * _normal(gen, n))
    c["T"].copy_(torch.where(slab & (T > 800.0), T - 400.0, T))
    eta0 = torch.tensor(list(w.materials.materialEta), dtype=F64, device=DEV)
    c["eta"].copy_(eta0[mat.long()] * torch.exp(0.1 * _normal(gen, n)))
    c["mu"].fill_(1e10)
    c["sxx"].copy_(1e7 * _normal(gen, n))
    c["syy"].copy_(-c["sxx"] + 1e6 * _normal(gen, n))
    c["sxy"].copy_(5e6 * _normal(gen, n))
    c["exx"].copy_(1e-15 * _normal(gen, n))
    c["eyy"].copy_(-c["exx"])
    c["exy"].copy_(1e-15 * _normal(gen, n))
    c["p"].copy_(3300.0 * 9.8 * Y * (1.0 + 0.05 * _normal(gen, n)))
    c["Eii"].copy_(_uniform(gen, (n,), 0.0, 1.5))


def _n_cells(w):
    return (w.NX - (0 if w.xperiodic else 1)) * (w.NY - 1)


def _members(case, seed):
    """(workload, markers per cell and axis, first marker, first node) of every
    instance of a sweep; the sizes follow from the case alone."""
    r = workloads.Rng(case["sizes"], 7)
    out, at, node = [], 0, 0
    for i in range(case["count"]):
        u = r.uniform(3)
        n = int(case["nmin"] + min(int(u[0] * (case["nmax"] - case["nmin"] + 1)), case["nmax"] - case["nmin"]))
        nm = 4 + min(int(u[1] * 3), 2)
        w = _thermal_workload(n, "tdep", 1000 * seed + i, 10.0 ** (2.0 + 4.0 * u[2]))
        out.append((w, nm, at, node))
        at += -(-_n_cells(w) * nm * nm // 32) * 32     # columns start on 256-byte lines
        node += -(-n * n // 32) * 32
    return out, at, node


def _ensemble_arrays(case, seed):
    """The sweep's workloads, marker columns and nodal arrays: one tensor per
    field over all instances, and each instance's views into them."""
    members, total, nodes = _members(case, seed)
    cols = _columns(total)
    gen = _generator(seed)
    names = ["vx", "vy", "wxy", "thisT"] + [p[4] for p in members[0][0].projections]
    flat = {k: torch.zeros(nodes, dtype=F64, device=DEV) for k in names}
    views = []
    for w, nm, at, node in members:
        n = _n_cells(w) * nm * nm
        c = {k: v[at:at + n] for k, v in cols.items()}
        _thermal_markers(c, w, nm, gen)
        nn = w.NX * w.NY
        f = {k: v[node:node + nn].view(w.NY, w.NX) for k, v in flat.items()}
        for k in ("vx", "vy", "wxy", "thisT"):
            f[k].copy_(torch.as_tensor(np.ascontiguousarray(w.nodal[k]), dtype=F64))
        views.append((w, c, f))
    return cols, flat, views


THERMAL_OUT = ("X", "Y", "VX", "VY", "T", "Tdot", "sxx", "syy", "sxy", "rho", "rhodot", "Eii", "wxy", "cellX", "cellY",
               "cpu")
VEP_OUT = THERMAL_OUT + ("eta", "mu", "p", "exx", "eyy", "exy", "strainRateResidual")
ALL2 = ("rho", "rhodot", "etaN", "etaS", "kThermal", "lastT", "Cp", "soxx", "soyy", "soxy", "muS", "muN")


def _list_names(w):
    return list(ALL2) if w.projections == "all2" else [p[4] for p in w.projections]


def _box(case):
    """The grid of a nodal solve: uniform or refined in a central band."""
    class Grid:
        pass
    g = Grid()
    g.NX, g.NY, g.LX, g.LY = case["nx"], case["ny"], 1.0, 1.0
    space = workloads.spacing_tanh_band if case["graded"] else workloads.spacing_uniform
    g.xp, g.xcp = workloads.pad_grid(space(g.NX, g.LX), g.LX)
    g.yp, g.ycp = workloads.pad_grid(space(g.NY, g.LY), g.LY)
    return g


def _blob_density(g, seed):
    """rho0 - drho B for a normalised sum of Gaussian blobs (the learned guess's states)."""
    r = np.random.default_rng(seed)
    X, Y = np.meshgrid(g.xp[2:g.NX + 2], g.yp[2:g.NY + 2])
    B = np.zeros_like(X)
    for _ in range(int(r.integers(4, 9))):
        cx, cy, s, a = r.uniform(0.1, 0.9), r.uniform(0.1, 0.9), r.uniform(0.05, 0.2), r.uniform(0.3, 1.0)
        B += a * np.exp(-((X - cx) ** 2 + (Y - cy) ** 2) / s ** 2)
    return torch.as_tensor(3300.0 - 100.0 * B / B.max(), dtype=F64).to(DEV)


class _View:
    """What torch wraps of a Buf; torch holds it, and it holds the Buf, whose
    memory is freed with the last of the two."""

    def __init__(self, buf, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": buf.shape, "typestr": typestr, "data": (buf.ptr, False), "version": 2}


def _as_tensor(buf, typestr):
    """A torch view of a Buf's device memory."""
    return torch.as_tensor(_View(buf, typestr), device=DEV)


def _net_inputs(case, seed):
    r = np.random.default_rng(seed)
    shape = (case["batch"], case["size"], case["size"])
    X = np.zeros(shape + (16,), np.float32)
    x = np.linspace(0.0, 1.0, case["size"], dtype=np.float32)
    for b in range(case["batch"]):      # smooth fields, as the scaled states are, with a little noise
        for c in range(5):
            k, l, p, q = r.uniform(0.5, 4.0), r.uniform(0.5, 4.0), *r.uniform(0, 6.28, 2)
            X[b, :, :, c] = np.sin(k * 3.14 * x + p)[:, None] * np.cos(l * 3.14 * x + q)[None, :]
    X[..., :5] += 0.05 * r.standard_normal(shape + (5,), dtype=np.float32)
    T = X[..., :3] * X[..., 1:4] + 0.1 * r.standard_normal(shape + (3,), dtype=np.float32)
    return to_bf16_bits(X), T.astype(np.float32)


ADAM = {"lr": 2e-3, "b1": 0.9, "b2": 0.999, "eps": 1e-8}
ADAM_STEPS = 1000       # a training run is resumed there: biases and moments are not zero


def _network(case, seed):
    """The network with the weights, biases and Adam moments of a run under way."""
    net = UNet(context(), levels=case["levels"], base=case["base"], seed=seed)
    r = np.random.default_rng(seed + 1)
    params = {k: (W, 0.05 * r.standard_normal(b.shape).astype(np.float32)) for k, (W, b) in net.params_numpy().items()}
    params["out"][1][3:] = 0.0      # the padded output channels
    net.load_params(params)
    moments = {}
    for k, e in net.p.items():
        for q in ("w", "b"):
            shape = e[q].shape
            m = 1e-3 * r.standard_normal(shape).astype(np.float32)
            v = 1e-4 * (1.0 + r.random(shape)).astype(np.float32)
            e["m" + q].set(m)
            e["v" + q].set(v)
            moments[k, q] = m, v
    net.adam_step = ADAM_STEPS
    return net, params, moments


# ---------------------------------------------------------------------- prepare --
def prepare(case, seed):
    kind, ctx = case["kind"], context()
    s = {"kind": kind, "ctx": ctx}
    if kind in ("thermal", "tracers"):
        w = _thermal_workload(case["n"], case.get("list", "all2"), seed)
        n = _n_cells(w) * case["nm"] ** 2
        capacity = n
        if kind == "tracers":
            w.options.NMX = w.options.NMY = case["nm"]
            quarter = max(1, case["nm"] ** 2 // 4)
            w.options.minMarkers, w.options.maxMarkers = max(1, quarter // 2), 2 * quarter
            # every quarter cell full or just refilled, and as many slots to spare
            capacity = 4 * (w.NX - 1) * (w.NY - 1) * (max(2 * quarter, (case["nm"] + 1) ** 2 // 4) + 1)
        cols = _columns(capacity)
        _thermal_markers({k: v[:n] for k, v in cols.items()}, w, case["nm"], _generator(seed))
        fields = _fields(w)
        s.update(path=Problem(w, Store(cols, n, capacity), Fields(fields)), cols=cols, fields=fields, seed=seed)
    elif kind == "vep":
        w = _vep_workload(case, seed)
        n = _n_cells(w) * case["nm"] ** 2
        cols = _columns(n)
        _vep_markers(cols, w, case["nm"], _generator(seed))
        fields = _fields(w)
        s.update(path=Problem(w, Store(cols, n, n), Fields(fields)), cols=cols, fields=fields,
                 solved={k: fields[k].clone() for k in VEP_CARRIED})
    elif kind == "ensemble":
        cols, flat, views = _ensemble_arrays(case, seed)
        paths = [Problem(w, Store(c, c["X"].numel(), c["X"].numel()),
                         Fields({**f, **{k: f["T_b"] for k in abi.NODAL_NAMES if k not in f}})) for w, c, f in views]
        torch.cuda.synchronize()
        e = Ensemble(paths)
        e.set_tuning(256, 4)    # what the autotuner picks on such sweeps
        e.capture()
        s.update(ensemble=e, cols=cols, flat=flat)
    elif kind == "nodal":
        w = workloads.nodal_box(case["nx"], case["ny"], seed=seed)
        fields = _fields(w)
        S = torch.stack([fields["vx"], fields["vy"], torch.randn(fields["vx"].shape, dtype=F64, device=DEV,
                                                                 generator=_generator(seed))], -1).contiguous()
        heat = torch.zeros_like(fields["vx"])
        empty = Store(_columns(1), 0, 1)
        s.update(path=Problem(w, empty, Fields(fields)), fields=fields, S=S, solved=S.clone(), heat=heat)
    elif kind == "energy":
        w = workloads.thermal_box(case["nx"], case["ny"], seed=seed, graded=case["graded"])
        fields = _fields(w)
        n = w.NX * w.NY
        heating = torch.as_tensor(w.nodal["heating"], dtype=F64).to(DEV)
        s.update(path=Problem(w, Store(_columns(1), 0, 1), Fields(fields)), fields=fields, heating=heating,
                 coef=torch.zeros(5 * n, dtype=F64, device=DEV), rhs=torch.zeros(n, dtype=F64, device=DEV),
                 T=torch.zeros(n, dtype=F64, device=DEV))
    elif kind == "pressure":
        g = _box(case)
        s.update(grid=DeviceGrid(ctx, g), rho=_blob_density(g, seed),
                 p=torch.zeros((g.NY, g.NX), dtype=F64, device=DEV))
    else:
        net, _, _ = _network(case, seed)
        X, T = _net_inputs(case, seed)
        dX = Buf(ctx, X.shape, np.uint16)
        dX.set(X)
        s.update(net=net, X=dX)
        if kind == "unet_train":
            dT = Buf(ctx, T.shape, np.float32)
            dT.set(T)
            s.update(T=dT, grads={k: (_as_tensor(e["gw"], "<f4"), _as_tensor(e["gb"], "<f4"))
                                  for k, e in net.p.items()},
                     weights={k: (_as_tensor(e["w"], "<f4"), _as_tensor(e["b"], "<f4")) for k, e in net.p.items()})
    torch.cuda.synchronize()
    return s


# -------------------------------------------------------------------------- run --
def _arrive(s, dst, src):
    """A host solve's result arriving in the array the next call reads."""
    s["ctx"].call("fvm_memcpy_dtod", dst.data_ptr(), src.data_ptr(), dst.numel() * dst.element_size())


def run(s):
    kind = s["kind"]
    if kind == "thermal":
        s["path"].step_thermal()
        return {**{k: s["cols"][k] for k in THERMAL_OUT}, "nodal": {k: s["fields"][k] for k in _list_names(s["path"].w)}}
    if kind == "tracers":
        path = s["path"]
        path.advect(path.w.dt)
        outside = path.find_marker_cells()
        added, removed = path.check_marker_density(s["seed"])
        return {**{k: s["cols"][k] for k in ("X", "Y", "VX", "VY", "T", "cellX", "cellY")},
                "counts": [path.markers.n, outside, added, removed]}
    if kind == "vep":
        for k in VEP_CARRIED:
            _arrive(s, s["fields"][k], s["solved"][k])
        yielding, residual = s["path"].step_vep()
        return {**{k: s["cols"][k] for k in VEP_OUT},
                "nodal": {k: s["fields"][k] for k in list(VEP_PROJ) + list(VEP_CARRIED)},
                "yielding": yielding, "residual": residual}
    if kind == "ensemble":
        s["ensemble"].launch()
        return {**{k: s["cols"][k] for k in THERMAL_OUT},
                "nodal": {k: v for k, v in s["flat"].items() if k not in ("vx", "vy", "wxy", "thisT")}}
    if kind == "nodal":
        path = s["path"]
        _arrive(s, s["S"], s["solved"])
        path.retrieve_solutions(_Slot(s["S"]), 1e3)
        path.nodal_stress_strain(path.w.dt, _Slot(s["heat"]))
        dt = path.limit_displacement_timestep(path.w.dt)
        return {"S": s["S"], "heat": s["heat"], "dt": dt, **{k: s["fields"][k] for k in NODAL_OUT}}
    if kind == "energy":
        path = s["path"]
        _arrive(s, s["rhs"], s["heating"])
        path.form_thermal_system(path.w.dt, False, _Slot(s["coef"]), _Slot(s["rhs"]))
        path.solve_thermal_system(_Slot(s["coef"]), _Slot(s["rhs"]), _Slot(s["T"]), rtol=1e-12)
        return {"coef": s["coef"], "rhs": s["rhs"], "T": s["T"]}
    if kind == "pressure":
        initial_pressure_guess(s["ctx"], s["grid"], _Slot(s["rho"]), G, rtol=1e-10, maxit=50000, p_out=_Slot(s["p"]))
        return s["p"]
    net = s["net"]
    out = net.forward(s["X"])
    if kind == "unet_predict":
        if "out" not in s:
            s["out"] = _as_tensor(out, "<f4")
        return s["out"]
    loss = net.loss(s["T"])
    net.backward()
    net.adam(**ADAM)
    return {"loss": loss, "grads": s["grads"], "weights": s["weights"]}


NODAL_OUT = ("vx", "vy", "p", "edotxx", "edotyy", "edotxy", "wxy", "soxx", "soyy", "soxy", "dsxx", "dsyy", "dsxy",
             "eii", "sii")


# ------------------------------------------------------------------------- work --
def work(case):
    """Bytes read and written once, and arithmetic, of one pass."""
    kind = case["kind"]
    if kind == "thermal" or kind == "tracers":
        markers, nodes = (case["n"] - 1) ** 2 * case["nm"] ** 2, case["n"] ** 2
        if kind == "tracers":   # X, Y, s, e, Eii, cells in; X, Y, VX, VY, wxy, s, Eii, cells out
            return {"bytes": 160 * markers + 24 * nodes, "flops": 450 * markers}
        # X, Y, T, eta, Mat, s, e, Eii in; cells, rho, rhodot, T, Tdot, X, Y, VX, VY, wxy, s, Eii out
        return {"bytes": 208 * markers + 8 * (4 + (12 if case["list"] == "all2" else 17)) * nodes, "flops": 700 * markers}
    if kind == "vep":
        markers = (case["nx"] - (0 if case["periodic"] else 1)) * (case["ny"] - 1) * case["nm"] ** 2
        return {"bytes": 280 * markers + 8 * 31 * case["nx"] * case["ny"], "flops": 1300 * markers}
    if kind == "ensemble":
        r = workloads.Rng(case["sizes"], 7)
        markers = nodes = 0
        for _ in range(case["count"]):
            u = r.uniform(3)
            n = int(case["nmin"] + min(int(u[0] * (case["nmax"] - case["nmin"] + 1)), case["nmax"] - case["nmin"]))
            markers += (n - 1) ** 2 * (4 + min(int(u[1] * 3), 2)) ** 2
            nodes += n * n
        return {"bytes": 208 * markers + 8 * 21 * nodes, "flops": 700 * markers}
    nodes = case.get("nx", 0) * case.get("ny", 0)
    if kind == "nodal":     # S, viscosities, moduli, stresses, density in; S.p, 15 nodal fields, heating out
        return {"bytes": 8 * (3 + 4 + 3 + 2 + 1 + 16) * nodes, "flops": 150 * nodes}
    if kind == "energy":
        return {"bytes": 8 * (6 + 5 + 1 + 1) * nodes, "flops": 60 * nodes}
    if kind == "pressure":
        return {"bytes": 16 * nodes, "flops": 60 * nodes}
    pixels, flops, weights = case["batch"] * case["size"] ** 2, 0, 0
    for _, K, ci, co, lvl in _layers(case):
        flops += 2 * K * K * ci * co * (pixels >> 2 * lvl)
        weights += K * K * ci * co
    if kind == "unet_train":    # forward, both gradients; weights and moments in and out
        return {"bytes": (16 * 2 + 3 * 4) * pixels + 28 * weights, "flops": 3 * flops}
    return {"bytes": (16 * 2 + 16 * 4) * pixels + 2 * weights, "flops": flops}


def _layers(case):
    """(name, kernel, channels in, channels out, level) of the network."""
    ch = [case["base"] * 2 ** i for i in range(case["levels"])]
    out, prev = [], 16
    for i, c in enumerate(ch):
        out += [("e%d_1" % i, 3, prev, c, i), ("e%d_2" % i, 3, c, c, i)]
        prev = c
    for i in range(case["levels"] - 2, -1, -1):
        out += [("d%d_1" % i, 3, ch[i + 1] + ch[i], ch[i], i), ("d%d_2" % i, 3, ch[i], ch[i], i)]
    return out + [("out", 1, ch[0], 16, 0)]


# ------------------------------------------------------------------------ exact --
class Exact:
    """The marker step in plain torch, one problem; m: columns, f: nodal arrays."""

    def __init__(self, w, m, f):
        self.w, self.m, self.f, self.per = w, m, f, bool(w.xperiodic)
        self.xp, self.yp, self.xcp, self.ycp = (torch.as_tensor(a, dtype=F64).to(DEV) for a in (w.xp, w.yp, w.xcp, w.ycp))
        self.mat = {k: torch.tensor(list(getattr(w.materials, "material" + k)), dtype=F64, device=DEV)
                    for k in ("Eta", "Rho", "Alpha", "Cp", "kThermal", "Mu", "Cohesion", "Friction")}

    # coordinates and ghosted arrays, index 0 at element 2
    def x(self, i): return self.xp[i + 2]
    def y(self, i): return self.yp[i + 2]
    def xc(self, i): return self.xcp[i + 2]
    def yc(self, i): return self.ycp[i + 2]

    def ghosted(self, a):
        p = torch.zeros((self.w.NY + 4, self.w.NX + 4), dtype=F64, device=DEV)
        p[2:-2, 2:-2] = a
        if self.per:
            p[2:-2, :2], p[2:-2, -2:] = a[:, -2:], a[:, :2]
        return p

    def owned(self, p):
        a = p[2:-2, 2:-2].clone()
        if self.per:
            a[:, -2:] += p[2:-2, :2]
            a[:, :2] += p[2:-2, -2:]
        return a

    def at(self, a, cy, cx):
        return self.ghosted(a)[cy + 2, cx + 2]

    def bilinear(self, a, cy, cx, mx, my):
        p = self.ghosted(a)
        return ((1 - mx) * (1 - my) * p[cy + 2, cx + 2] + (1 - mx) * my * p[cy + 3, cx + 2] +
                mx * (1 - my) * p[cy + 2, cx + 3] + mx * my * p[cy + 3, cx + 3])

    def scatter(self, terms):
        """Sum of (cy, cx, value) terms at the nodes; ghosts dropped or wrapped."""
        p = torch.zeros((self.w.NY + 4) * (self.w.NX + 4), dtype=F64, device=DEV)
        for cy, cx, v in terms:
            p.index_add_(0, (cy + 2) * (self.w.NX + 4) + cx + 2, v)
        return self.owned(p.view(self.w.NY + 4, -1))

    def locate(self):
        m, w = self.m, self.w
        xs = torch.as_tensor(np.append(w.x, w.LX) if self.per else w.x, dtype=F64).to(DEV)
        ys = torch.as_tensor(w.y, dtype=F64).to(DEV)
        inside = (m["X"] >= 0) & (m["Y"] >= 0) & (m["X"] <= w.LX) & (m["Y"] <= w.LY)
        cx = (torch.searchsorted(xs, m["X"], right=True) - 1).clamp(0, xs.numel() - 2)
        cy = (torch.searchsorted(ys, m["Y"], right=True) - 1).clamp(0, ys.numel() - 2)
        m["cellX"] = torch.where(inside, cx, -1).int()
        m["cellY"] = torch.where(inside, cy, -1).int()
        m["cpu"] = torch.zeros_like(m["cellX"])
        self.inside, self.cx, self.cy = inside, cx, cy
        self.quarter = (m["X"] >= self.xc(cx + 1)).long(), (m["Y"] >= self.yc(cy + 1)).long()

    def density(self):
        m = self.m
        k = m["Mat"].long()
        m["rho"] = torch.where(self.inside, -self.mat["Rho"][k] * self.mat["Alpha"][k] * m["T"], m["rho"])
        m["rhodot"] = torch.where(self.inside, torch.zeros_like(m["T"]), m["rhodot"])

    def family(self, sx, sy):
        """Lattice cell and fractions of node family (sx, sy)."""
        bx, by = self.quarter
        X, Y = self.m["X"], self.m["Y"]
        cx, cy = self.cx + (0 if sx == 0 else bx if sx == -1 else bx - 1), self.cy + (0 if sy == 0 else by if sy == -1 else by - 1)
        x = (lambda i: self.x(i)) if sx == 0 else (lambda i: self.xc(i)) if sx == -1 else (lambda i: self.xc(i + 1))
        y = (lambda i: self.y(i)) if sy == 0 else (lambda i: self.yc(i)) if sy == -1 else (lambda i: self.yc(i + 1))
        return cx, cy, (X - x(cx)) / (x(cx + 1) - x(cx)), (Y - y(cy)) / (y(cy + 1) - y(cy))

    def project(self, v, sx, sy, method=abi.ARITHMETIC):
        cx, cy, mx, my = self.family(sx, sy)
        on = self.inside.to(F64)
        if method == abi.ARITHMETIC:
            terms = [(cy, cx, (1 - mx) * (1 - my) * on), (cy, cx + 1, mx * (1 - my) * on),
                     (cy + 1, cx, (1 - mx) * my * on), (cy + 1, cx + 1, mx * my * on)]
        else:
            rx, ry = mx >= 0.5, my >= 0.5
            terms = [(cy + ry, cx + rx, torch.where(rx, mx, 1 - mx) * torch.where(ry, my, 1 - my) * on)]
        return self.scatter([(a, b, wt * v) for a, b, wt in terms]) / self.scatter(terms)

    def project_list(self):
        out, m = {}, self.m
        for src, sx, sy, method, name in self.w.projections:
            v = self.mat[src[4:]][m["Mat"].long()] if src.startswith("mat:") else m[src]
            out[name] = self.project(v, sx, sy, method)
        return out, {"lastT": "T_b", "rho": "rho_b", "Cp": "Cp_b", "kThermal": "k_b"}

    def project_all2(self):
        m, k = self.m, self.m["Mat"].long()
        L = abi.ARITHMETIC_LOCAL
        big = torch.full((self.w.NY, self.w.NX), 1e99, dtype=F64, device=DEV)
        return {"rho": self.project(m["rho"], 0, 0), "rhodot": torch.zeros_like(big),
                "etaN": self.project(m["eta"], -1, -1), "etaS": self.project(m["eta"], 0, 0), "muS": big, "muN": big,
                "kThermal": self.project(self.mat["kThermal"][k], 0, 0), "lastT": self.project(m["T"], 0, 0),
                "Cp": self.project(self.mat["Cp"][k], 0, 0), "soxx": self.project(m["sxx"], -1, -1, L),
                "soyy": self.project(m["syy"], -1, -1, L), "soxy": self.project(m["sxy"], 0, 0, L)}

    def subgrid_temperature(self, nodal, thisT, dt, d):
        m, (cx, cy, mx, my) = self.m, self.family(0, 0)
        Tm, rho, Cp, k = (self.bilinear(nodal[q], cy, cx, mx, my) for q in ("lastT", "rho", "Cp", "kThermal"))
        dx, dy = self.x(cx + 1) - self.x(cx), self.y(cy + 1) - self.y(cy)
        tau = Cp * (self.mat["Rho"][0] + rho) / k / (2.0 / (dx * dx) + 2.0 / (dy * dy))
        dT = (Tm - m["T"]) * (1.0 - torch.exp(-d * dt / tau))
        delta = thisT - nodal["lastT"] - self.project(dT, 0, 0)
        dtm = self.bilinear(delta, cy, cx, mx, my) + dT
        m["T"] = torch.where(self.inside, m["T"] + dtm, m["T"])
        m["Tdot"] = torch.where(self.inside, dtm / dt, m["Tdot"])

    def velocity(self, X, Y):
        w, bv = self.w, self.w.bv
        lo, hi = (-1, w.NX - 1) if self.per else (0, w.NX - 2)
        base = 2 + lo
        cx = torch.bucketize(X, self.xp[base:hi + 4].contiguous(), right=True) - 1 + lo
        cy = torch.bucketize(Y, self.yp[2:w.NY + 2].contiguous(), right=True) - 1
        cx, cy = cx.clamp(lo, hi), cy.clamp(0, w.NY - 2)
        vxY = torch.where(Y < self.yc(cy + 1), cy - 1, cy)
        vyX = torch.where(X < self.xc(cx + 1), cx - 1, cx)
        gx, gy = self.ghosted(self.f["vx"]), self.ghosted(self.f["vy"])
        if bv.mechBCTop.type[0] == 0:
            gx[1, :] = 2.0 * bv.mechBCTop.value[0] - gx[2, :]
        elif bv.mechBCTop.type[0] == 1:
            gx[1, :] = gx[2, :]
        if not self.per and bv.mechBCLeft.type[1] == 0:
            gy[:, 1] = 2.0 * bv.mechBCLeft.value[1] - gy[:, 2]
        elif not self.per and bv.mechBCLeft.type[1] == 1:
            gy[:, 1] = gy[:, 2]

        def mix(p, cy, cx, mx, my):
            return ((1 - mx) * (1 - my) * p[cy + 2, cx + 2] + (1 - mx) * my * p[cy + 3, cx + 2] +
                    mx * (1 - my) * p[cy + 2, cx + 3] + mx * my * p[cy + 3, cx + 3])
        mx, my = (X - self.x(cx)) / (self.x(cx + 1) - self.x(cx)), (Y - self.y(cy)) / (self.y(cy + 1) - self.y(cy))
        nx = (X - self.xc(vyX + 1)) / (self.xc(vyX + 2) - self.xc(vyX + 1))
        ny = (Y - self.yc(vxY + 1)) / (self.yc(vxY + 2) - self.yc(vxY + 1))
        return mix(gx, vxY, cx, mx, ny), mix(gy, cy, vyX, nx, my), mix(self.ghosted(self.f["wxy"]), cy, cx, mx, my)

    def advect(self, dt):
        m, w = self.m, self.w
        X, Y = m["X"], m["Y"]
        k1 = self.velocity(X, Y)
        k2 = self.velocity(X + dt / 2 * k1[0], Y + dt / 2 * k1[1])
        k3 = self.velocity(X + dt / 2 * k2[0], Y + dt / 2 * k2[1])
        k4 = self.velocity(X + dt * k3[0], Y + dt * k3[1])
        VX, VY, spin = ((a + 2 * b + 2 * c + d) / 6 for a, b, c, d in zip(k1, k2, k3, k4))
        sxx, syy, sxy = m["sxx"], m["syy"], m["sxy"]
        th = -spin * dt
        c, s = torch.cos(th), torch.sin(th)
        nX, nY = X + dt * VX, Y + dt * VY
        if self.per:
            nX = torch.where(nX > w.LX, nX - w.LX, torch.where(nX < 0, nX + w.LX, nX))
        new = {"VX": VX, "VY": VY, "wxy": spin, "X": nX, "Y": nY,
               "sxx": sxx * c * c + syy * s * s - sxy * torch.sin(2 * th),
               "syy": sxx * s * s + syy * c * c + sxy * torch.sin(2 * th),
               "sxy": 0.5 * (sxx - syy) * torch.sin(2 * th) + sxy * torch.cos(2 * th),
               "Eii": m["Eii"] + dt * torch.sqrt(0.5 * (m["exx"] ** 2 + m["eyy"] ** 2) + m["exy"] ** 2)}
        for k, v in new.items():
            m[k] = torch.where(self.inside, v, m[k])

    def step_thermal(self):
        w = self.w
        self.locate()
        self.density()
        if w.projections == "all2":
            nodal, names = self.project_all2(), {}
        else:
            nodal, names = self.project_list()
        th = {k: nodal[names.get(k, k)] for k in ("lastT", "rho", "Cp", "kThermal")}
        self.subgrid_temperature(th, self.f["thisT"], w.dt, w.options.subgridTemperatureDiffusivity)
        self.advect(w.dt)
        return nodal

    # --- the visco-elasto-plastic parts ---
    def yielding(self, dt):
        m, o, mt, k = self.m, self.w.options, self.w.materials, self.m["Mat"].long()

        def table(v):
            return torch.tensor(list(v), dtype=F64, device=DEV)[k]
        Z = m["eta"] / (m["mu"] * dt + m["eta"])
        sn = [m["s" + q] * Z + 2 * m["eta"] * m["e" + q] * (1 - Z) for q in ("xx", "yy", "xy")]
        sii = torch.sqrt(0.5 * (sn[0] ** 2 + sn[1] ** 2) + sn[2] ** 2)
        law = table(mt.hasEtaT)
        eta = self.mat["Eta"][k]
        eta = torch.where(law == 1, eta * torch.exp(table(mt.QonR) * (1.0 / m["T"] - 1.0 / table(mt.Tref))), eta)
        plast = table(mt.hasPlasticity)
        g0, g1 = table([mt.gamma[i][0] for i in range(8)]), table([mt.gamma[i][1] for i in range(8)])
        c0, c1 = table([mt.C[i][0] for i in range(8)]), table([mt.C[i][1] for i in range(8)])
        f0, f1 = (table([math.sin(mt.F[i][j] / 180.0 * math.pi) for i in range(8)]) for j in (0, 1))
        h = ((m["Eii"] - g0) / (g1 - g0)).clamp(0, 1)
        soft = plast == 2
        c = torch.where(soft, c0 + (c1 - c0) * h, self.mat["Cohesion"][k])
        f = torch.where(soft, f0 + (f1 - f0) * h, self.mat["Friction"][k])
        siy = (c + f * m["p"]).clamp(min=0.0)
        act = self.inside & (plast > 0)
        y = act & (sii > siy)
        e2 = torch.sqrt(0.5 * (m["exx"] ** 2 + m["eyy"] ** 2) + m["exy"] ** 2)
        ny = siy / 2.0 / e2
        ny = torch.where(ny / eta < o.fractionalEtamin, o.fractionalEtamin * eta, ny).clamp(o.etamin, o.etamax)
        s2 = torch.sqrt(0.5 * (m["sxx"] ** 2 + m["syy"] ** 2) + m["sxy"] ** 2)
        scale = torch.where(y & (s2 != 0), siy / s2, torch.ones_like(s2))
        old = m["eta"]
        new = torch.where(act, torch.where(y, ny, old), eta)   # a marker below yield keeps the viscosity it came with
        m["eta"] = torch.where(self.inside, new, old).clamp(o.etamin, o.etamax)
        m["mu"] = torch.where(self.inside, self.mat["Mu"][k], m["mu"])
        for q in ("sxx", "syy", "sxy"):
            m[q] = m[q] * scale
        return int(bool(y.any()))

    def centre(self, xmax_in, xmax):
        """Cell-centre cell and fractions, clamped to the interior (not a projection's)."""
        bx, by = self.quarter
        cx = torch.where(self.cx < xmax_in, self.cx + bx, self.cx).clamp(1, xmax)
        cy = torch.where(self.cy < self.w.NY - 1, self.cy + by, self.cy).clamp(1, self.w.NY - 2)
        X, Y = self.m["X"], self.m["Y"]
        return cx, cy, (X - self.xc(cx)) / (self.xc(cx + 1) - self.xc(cx)), (Y - self.yc(cy)) / (self.yc(cy + 1) - self.yc(cy))

    def corner(self, xmax):
        cx = self.cx.clamp(0, xmax)
        X, Y = self.m["X"], self.m["Y"]
        return cx, self.cy, (X - self.x(cx)) / (self.x(cx + 1) - self.x(cx)), \
            (Y - self.y(self.cy)) / (self.y(self.cy + 1) - self.y(self.cy))

    def update(self, name, v):
        self.m[name] = torch.where(self.inside, v, self.m[name])

    def step_vep(self):
        w, m, f, o = self.w, self.m, self.f, self.w.options
        NX, dt = w.NX, w.dt
        self.locate()
        self.density()
        y = self.yielding(dt)
        nodal = self.project_all2()
        upd = (NX, NX - 1) if self.per else (NX - 2, NX - 2)

        def at(names, loc):
            cx, cy, mx, my = loc
            return [self.bilinear(f[k], cy, cx, mx, my) for k in names]
        p, exx, sxx, syy, dxx, dyy = at(("p", "edotxx", "soxx", "soyy", "dsxx", "dsyy"), self.centre(*upd))
        spin, exy, sxy, dxy = at(("wxy", "edotxy", "soxy", "dsxy"), self.corner(upd[1]))
        e = [s / 2.0 / m["eta"] + d / 2.0 / dt / m["mu"] for s, d in ((sxx, dxx), (syy, dyy), (sxy, dxy))]
        for k, v in (("p", p), ("wxy", spin), ("exx", e[0]), ("eyy", e[1]), ("exy", e[2])):
            self.update(k, v)
        self.update("strainRateResidual", torch.sqrt((e[0] - exx) ** 2 + (e[2] - exy) ** 2))
        srr = self.project(m["strainRateResidual"], -1, -1)
        residual = self.residual(srr)
        # subgrid stress
        sd = 1.0 - torch.exp((-o.subgridStressDiffusivity * dt / (m["eta"] / m["mu"])).clamp(min=-30.0))
        cx, cy, mx, my = self.corner(NX - 2)
        dxy = (self.bilinear(f["soxy"], cy, cx, mx, my) - m["sxy"]) * sd
        lx, ly, nx, ny = self.centre(NX - 1, NX - 2)
        dxx = (self.bilinear(f["soxx"], ly, lx, nx, ny) - m["sxx"]) * sd
        dyy = (self.bilinear(f["soyy"], ly, lx, nx, ny) - m["syy"]) * sd
        for k, v in (("sxx", dxx), ("syy", dyy), ("sxy", dxy)):
            self.update(k, m[k] + v)
        cx, cy, mx, my = self.family(0, 0)
        on = self.inside.to(F64)
        wc = (1.0 - (0.5 - mx).abs()) * (1.0 - (0.5 - my).abs()) * on
        ties = []
        for rx, hx, ux in ((0, mx <= 0.5, 1 - mx), (1, mx >= 0.5, mx)):
            for ry, hy, uy in ((0, my <= 0.5, 1 - my), (1, my >= 0.5, my)):
                ties.append((cy + ry, cx + rx, ux * uy * (hx & hy).to(F64) * on))
        wn, ws = self.scatter([(cy + 1, cx + 1, wc)]), self.scatter(ties)
        ds = {"dsxx": f["dsxx"] - self.scatter([(cy + 1, cx + 1, wc * dxx)]) / wn,
              "dsyy": f["dsyy"] - self.scatter([(cy + 1, cx + 1, wc * dyy)]) / wn,
              "dsxy": f["dsxy"] - self.scatter([(a, b, t * dxy) for a, b, t in ties]) / ws}
        f.update(ds)
        # marker stress
        dxx, dyy = at(("dsxx", "dsyy"), self.centre(*upd))
        dxy, = at(("dsxy",), self.corner(upd[1]))
        for k, v in (("sxx", dxx), ("syy", dyy), ("sxy", dxy)):
            self.update(k, m[k] + v)
        self.subgrid_temperature(nodal, f["thisT"], dt, o.subgridTemperatureDiffusivity)
        self.advect(dt)
        return nodal, ds, y, residual

    def residual(self, srr):
        w = self.w
        area = (self.x(torch.arange(1, w.NX, device=DEV)) - self.x(torch.arange(w.NX - 1, device=DEV))).view(1, -1) * \
            (self.y(torch.arange(1, w.NY, device=DEV)) - self.y(torch.arange(w.NY - 1, device=DEV))).view(-1, 1)
        return float((srr[1:, 1:] * area).sum() / (w.LX * w.LY))


def _exact_thermal(case, seed):
    w = _thermal_workload(case["n"], case["list"], seed)
    cols = _columns(_n_cells(w) * case["nm"] ** 2)
    _thermal_markers(cols, w, case["nm"], _generator(seed))
    nodal = Exact(w, cols, _fields(w, ["vx", "vy", "wxy", "thisT"])).step_thermal()
    return {**{k: cols[k] for k in THERMAL_OUT}, "nodal": {k: nodal[k] for k in _list_names(w)}}


def _exact_ensemble(case, seed):
    cols, flat, views = _ensemble_arrays(case, seed)
    for w, c, f in views:
        m = dict(c)
        nodal = Exact(w, m, f).step_thermal()
        for k in THERMAL_OUT:
            c[k].copy_(m[k])
        for k, v in nodal.items():
            f[k].copy_(v)
    return {**{k: cols[k] for k in THERMAL_OUT},
            "nodal": {k: v for k, v in flat.items() if k not in ("vx", "vy", "wxy", "thisT")}}


def _exact_vep(case, seed):
    w = _vep_workload(case, seed)
    cols = _columns(_n_cells(w) * case["nm"] ** 2)
    _vep_markers(cols, w, case["nm"], _generator(seed))
    nodal, ds, y, residual = Exact(w, cols, _fields(w)).step_vep()
    return {**{k: cols[k] for k in VEP_OUT}, "nodal": {**{k: nodal[k[5:]] for k in VEP_PROJ}, **ds},
            "yielding": y, "residual": residual}


def _exact_nodal(case, seed):
    w = workloads.nodal_box(case["nx"], case["ny"], seed=seed)
    f = _fields(w)
    pr = torch.randn(f["vx"].shape, dtype=F64, device=DEV, generator=_generator(seed)) * 1e3
    vx, vy, dt = f["vx"], f["vy"], w.dt
    x, y, xc, yc = (torch.as_tensor(np.ascontiguousarray(a), dtype=F64).to(DEV) for a in (w.x, w.y, w.xc, w.yc))
    dx, dy = (x[1:] - x[:-1]).view(1, -1), (y[1:] - y[:-1]).view(-1, 1)
    out = {"S": torch.stack([vx, vy, pr], -1), "vx": vx, "vy": vy}
    p = pr.clone()
    p[1:, 1:] -= (pr[1, 1:] * dx[0] / w.LX).sum()
    out["p"] = p
    a, b = (vx[:-1, 1:] - vx[:-1, :-1]) / dx, (vy[1:, :-1] - vy[:-1, :-1]) / dy
    exx, eyy = torch.zeros_like(vx), torch.zeros_like(vx)
    exx[1:, 1:], eyy[1:, 1:] = a - (a + b) / 3.0, b - (a + b) / 3.0
    left = w.bv.mechBCLeft
    top = w.bv.mechBCTop
    vym = torch.cat([(2.0 * left.value[1] - vy[:, :1]) if left.type[1] == 0 else vy[:, :1], vy[:, :-1]], 1)
    vxm = torch.cat([(2.0 * top.value[0] - vx[:1]) if top.type[0] == 0 else vx[:1], vx[:-1]], 0)
    u, v = (vx - vxm) / (yc[1:] - yc[:-1]).view(-1, 1), (vy - vym) / (xc[1:] - xc[:-1]).view(1, -1)
    out["wxy"], exy = 0.5 * (u - v), 0.5 * (u + v)
    out.update(edotxx=exx, edotyy=eyy, edotxy=exy)
    new = {}
    for q, e, node in (("xx", exx, "N"), ("yy", eyy, "N"), ("xy", exy, "S")):
        Z = f["eta" + node] / (f["eta" + node] + dt * f["mu" + node])
        new[q] = Z * f["so" + q] + f["eta" + node] * 2.0 * (1.0 - Z) * e
        out["so" + q], out["ds" + q] = new[q], new[q] - f["so" + q]

    def four(a):
        return (a[1:-1, 1:-1] + a[2:, 1:-1] + a[1:-1, 2:] + a[2:, 2:]) / 8.0

    def inner(v):
        z = torch.zeros_like(vx)
        z[1:-1, 1:-1] = v
        return z
    mid = (slice(1, -1), slice(1, -1))
    out["heat"] = inner(four(new["xx"] ** 2 / f["etaN"]) + four(new["yy"] ** 2 / f["etaN"]) +
                        (new["xy"] ** 2 / f["etaS"])[mid])
    out["eii"] = inner(torch.sqrt(four(exx ** 2) + four(eyy ** 2) + (exy ** 2)[mid]))
    out["sii"] = inner(torch.sqrt(four(new["xx"] ** 2) + four(new["yy"] ** 2) + (new["xy"] ** 2)[mid]))

    def least(h, n):
        return torch.cat([h[:1], torch.minimum(h[:-1], h[1:]), h[-1:]])
    lim, k = dt, w.options.displacementStepLimit
    for vel, h in ((vx, least(dx[0], w.NX).view(1, -1)), (vy, least(dy[:, 0], w.NY).view(-1, 1))):
        c = h / vel.abs() * k
        lim = min(lim, float(c[vel != 0].min()))
    lim = min(lim, float((0.01 * f["rho"] / f["rhodot"]).abs()[f["rhodot"] != 0].min()))
    big = float(f["rhodot"].abs().max())
    out["dt"] = 0.01 / big if big * lim > 0.01 else lim
    return {k: out[k] for k in ("S", "heat", "dt") + NODAL_OUT}


def _block_solve(d, e, w, s, n, b):
    """Direct solve of a 5-point system given by its bands (NY, NX): block
    elimination over the shorter axis' lines."""
    if d.shape[1] > d.shape[0]:
        return _block_solve(*(a.t().contiguous() for a in (d, s, n, e, w, b))).t().contiguous()
    rows, cols = d.shape
    eye = torch.arange(cols, device=DEV)
    inv, z = [], []
    for j in range(rows):
        A = torch.zeros((cols, cols), dtype=F64, device=DEV)
        A[eye, eye] = d[j]
        A[eye[:-1], eye[1:]] = e[j, :-1]
        A[eye[1:], eye[:-1]] = w[j, 1:]
        r = b[j]
        if j:
            A = A - n[j].view(-1, 1) * inv[-1] * s[j - 1].view(1, -1)
            r = r - n[j] * z[-1]
        inv.append(torch.linalg.inv(A))
        z.append(inv[-1] @ r)
    out = [z[-1]]
    for j in range(rows - 2, -1, -1):
        out.append(z[j] - inv[j] @ (s[j] * out[-1]))
    return torch.stack(out[::-1])


def _exact_energy(case, seed):
    w = workloads.thermal_box(case["nx"], case["ny"], seed=seed, graded=case["graded"])
    f, o = _fields(w, ["kThermal", "rho", "Cp", "lastT", "vx"]), w.options
    x, y = (torch.as_tensor(np.ascontiguousarray(a), dtype=F64).to(DEV) for a in (w.x, w.y))
    X, Y = x.view(1, -1), y.view(-1, 1)
    b = torch.as_tensor(w.nodal["heating"], dtype=F64).to(DEV).clone()
    d, e, ww, s, n = (torch.zeros_like(b) for _ in range(5))
    k, T = f["kThermal"], f["lastT"]
    ka, kb = (k[1:-1, 1:-1] + k[1:-1, :-2]) / 2, (k[1:-1, 1:-1] + k[1:-1, 2:]) / 2
    kc, kd = (k[1:-1, 1:-1] + k[:-2, 1:-1]) / 2, (k[1:-1, 1:-1] + k[2:, 1:-1]) / 2
    dx, dy = X[:, 1:] - X[:, :-1], Y[1:] - Y[:-1]
    dx1, dx2, dy1, dy2 = dx[:, :-1], dx[:, 1:], dy[:-1], dy[1:]
    mid = (slice(1, -1), slice(1, -1))
    heat = ((w.materials.materialRho[0] + f["rho"]) * f["Cp"] / w.dt)[mid]
    e[mid], ww[mid] = -2.0 / (dx1 + dx2) * kb / dx2, -2.0 / (dx1 + dx2) * ka / dx1
    n[mid], s[mid] = -2.0 / (dy1 + dy2) * kc / dy1, -2.0 / (dy1 + dy2) * kd / dy2
    d[mid] = heat - e[mid] - ww[mid] - n[mid] - s[mid]
    b[mid] += heat * T[mid]
    d[-1, 1:-1], b[-1, 1:-1] = 1.0, T[-1, 1:-1]
    if o.thermalBCTop.type[0] == 0:
        d[0, 1:-1], b[0, 1:-1] = 1.0, o.thermalBCTop.value[0]
    else:
        d[0, 1:-1], s[0, 1:-1], b[0, 1:-1] = -1.0 / dy[0], 1.0 / dy[0], 0.0
    d[:, 0] = d[:, -1] = 1.0
    age = o.slabAge * 1.0e6 * 3.15576e7
    b[:, 0] = 273.0 + (1623.0 - 273.0) * torch.erf((y - x[0] * math.tan(o.slabAngle)) / (2.0 * math.sqrt(0.7272e-6 * age)))
    root = math.cos(math.pi * (w.LX - o.rootCenter) / o.rootWidth / 2.0) ** 2 if abs(w.LX - o.rootCenter) < o.rootWidth else 0.0
    depth = o.overridingPlateThickness + o.rootThickness * root
    vx = f["vx"][:, -1]
    inflow = torch.zeros_like(y, dtype=torch.bool)
    inflow[1:] = (vx[1:] + vx[:-1]) / 2.0 < 0.0
    b[:, -1] = torch.where(y <= depth, y / depth * 1300.0 + 273.0, torch.where(inflow, torch.full_like(y, 1573.0), T[:, -1]))
    sol = _block_solve(*(a / d for a in (d, e, ww, s, n, b)))
    return {"coef": torch.cat([a.reshape(-1) for a in (d, e, ww, s, n)]), "rhs": b.reshape(-1), "T": sol.reshape(-1)}


def _exact_pressure(case, seed):
    g = _box(case)
    NX, NY = g.NX, g.NY
    rho = _blob_density(g, seed)
    x, y, xc, yc = (torch.as_tensor(a[2:2 + m], dtype=F64).to(DEV) for a, m in
                    ((g.xp, NX), (g.yp, NY), (g.xcp, NX + 1), (g.ycp, NY + 1)))
    hx, hy = (x[1:] - x[:-1]).view(1, -1), (y[1:] - y[:-1]).view(-1, 1)
    gx, gy = (xc[1:] - xc[:-1]), (yc[1:] - yc[:-1])
    d, e, w, s, n, b = (torch.zeros_like(rho) for _ in range(6))
    inn = (slice(1, None), slice(1, None))
    e[inn], w[inn] = 1.0 / hx / gx[1:].view(1, -1), 1.0 / hx / gx[:-1].view(1, -1)
    s[inn], n[inn] = 1.0 / hy / gy[1:].view(-1, 1), 1.0 / hy / gy[:-1].view(-1, 1)
    e[:, -1] = w[:, 1] = 0.0
    s[-1, :] = n[1, :] = 0.0
    top, bottom = 1.0 / hy[0, 0] / gy[0], 1.0 / hy[-1, 0] / gy[-1]
    d[inn] = -(e + w + s + n)[inn]
    pin = 4.0 / (hx[0, 0] ** 2 + hy[0, 0] ** 2)
    d[0, :] = d[:, 0] = pin
    d[1, 0] += top
    d[-1, 0] += bottom
    r2 = (rho[1:, 1:] + rho[1:, :-1]) / 2.0 - (rho[:-1, 1:] + rho[:-1, :-1]) / 2.0
    b[inn] = G * r2 / hy
    for a in (e, w, s, n, b):
        a[3, 3] = 0.0
    d[3, 3] = 4.0 / ((x[3] - x[2]) ** 2 + (y[3] - y[2]) ** 2)
    lag = torch.cat([torch.zeros_like(rho[:, :1]), rho[:, :-1]], 1)
    mean = (rho[1:] + rho[:-1] + lag[1:] + lag[:-1]) / 4.0
    b[1] += top * mean[0] * G * (yc[1] - yc[0])
    b[-1] -= bottom * mean[-1] * G * (yc[NY - 1] - yc[NY - 2])
    return _block_solve(*(a / d for a in (d, e, w, s, n, b)))


def _conv(x, W, b):
    """x (B, H, W, ci), W (taps, co, ci): a padded 3x3 (or 1x1) convolution."""
    K = 3 if W.shape[0] == 9 else 1
    p = torch.nn.functional.pad(x, (0, 0, K // 2, K // 2, K // 2, K // 2))
    h, w = x.shape[1:3]
    y = b
    for t in range(K * K):
        y = y + p[:, t // K:t // K + h, t % K:t % K + w].contiguous() @ W[t].t().contiguous()
    return y


def _exact_net(case, seed):
    X, T = _net_inputs(case, seed)
    _, params, moments = _network(case, seed)
    P = {k: [torch.as_tensor(a).to(DEV).to(F64).requires_grad_(case["kind"] == "unet_train") for a in v]
         for k, v in params.items()}
    x = torch.as_tensor((X.astype(np.uint32) << 16).view(np.float32)).to(DEV).to(F64)
    skips = []
    for i in range(case["levels"]):
        for j in (1, 2):
            x = torch.relu(_conv(x, *P["e%d_%d" % (i, j)]))
        skips.append(x)
        if i < case["levels"] - 1:
            B, H, W, C = x.shape
            x = x.reshape(B, H // 2, 2, W // 2, 2, C).mean((2, 4))
    for i in range(case["levels"] - 2, -1, -1):
        x = torch.cat([x.repeat_interleave(2, 1).repeat_interleave(2, 2), skips[i]], -1)
        for j in (1, 2):
            x = torch.relu(_conv(x, *P["d%d_%d" % (i, j)]))
    out = _conv(x, *P["out"])
    if case["kind"] == "unet_predict":
        return out
    loss = ((out[..., :3] - torch.as_tensor(T).to(DEV).to(F64)) ** 2).mean()
    loss.backward()
    grads, weights, o, t = {}, {}, ADAM, ADAM_STEPS + 1
    for k, v in P.items():
        grads[k], weights[k] = [a.grad for a in v], []
        for q, a in zip("wb", v):
            m, s = (torch.as_tensor(z).to(DEV).to(F64) for z in moments[k, q])
            m, s = o["b1"] * m + (1 - o["b1"]) * a.grad, o["b2"] * s + (1 - o["b2"]) * a.grad ** 2
            weights[k].append(a.detach() - o["lr"] * (m / (1 - o["b1"] ** t)) / ((s / (1 - o["b2"] ** t)).sqrt() + o["eps"]))
    return {"loss": float(loss.detach()), "grads": grads, "weights": weights}


def exact(case, seed):
    make = {"thermal": _exact_thermal, "ensemble": _exact_ensemble, "vep": _exact_vep, "nodal": _exact_nodal,
            "energy": _exact_energy, "pressure": _exact_pressure, "unet_train": _exact_net,
            "unet_predict": _exact_net}.get(case["kind"])
    return make(case, seed) if make else None     # tracers: which markers come and go is a matter of bits
