"""Measured cases of the BioFVM-B hot path on one MI355X: what a program that uses this
library has it do, from one small microenvironment stepped call by call to a field of two
billion voxel-substrates.

Kinds of case (``kind``):

* ``step``: one microenvironment resident on the GPU.  ``mode`` "slots" is one step through
  the two calls that replace the reference's function slots
  (``simulate_cell_sources_and_sinks`` then ``simulate_diffusion_decay``); "run" is ``steps``
  steps in one call; "graph" is the same as a replayed graph.  Options: per-voxel Dirichlet
  values, bulk source/sink rates, density gradients after the steps.
* ``moves``: a step of moving agents: new positions (already on the GPU), one step, and the
  densities at the agents' voxels, as a cell model senses them.
* ``adjoint``: a field from a CUDA tensor, a recorded run, the final field into a CUDA tensor
  and the gradients of a squared distance with respect to the initial field and the agent
  tables.
* ``batch``: uneven microenvironments advanced together as one replayed graph, then every
  field fetched to the host.

Sizes and coefficients follow the repository's benchmark (400^3 x 4 with 1M agents, 640^3 x 8,
128^3 x 2 adjoint, uneven batch), its plain 50^3 x 1 test case and the sizes of its autotuning
table (128 to 320 per axis); odd sizes are generic.
"""
from __future__ import annotations

import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "biofvm-b_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DX, DT = 20.0, 0.01
VOLUME = 4.0 / 3.0 * math.pi * 125.0  # a cell of radius 5 um
DEV = "cuda:0"


def _step(name, grid, nsub, prec, agents, mode="run", steps=1, nodes=0, bulk=False, gradients=False):
    return dict(name=name, kind="step", nx=grid[0], ny=grid[1], nz=grid[2], nsub=nsub, prec=prec, agents=agents,
                mode=mode, steps=steps, nodes=nodes, bulk=bulk, gradients=gradients)


def listed():
    return [
        # the plain small case of the tests, one step per call as the reference's drivers call it:
        # launches and host work count
        _step("slots_50cube_f64", (50, 50, 50), 1, "fp64", 1000, mode="slots"),
        # a small odd grid with per-voxel Dirichlet values, a few steps per call
        _step("run_97x61x83_nodes_f64", (97, 61, 83), 3, "fp64", 3000, steps=5, nodes=2000),
        # the usual sizes of a single simulation, between the small and the full-size workloads
        _step("run_200cube_x2_f32", (200, 200, 200), 2, "fp32", 50_000, steps=2),
        _step("slots_256cube_x4_f64", (256, 256, 256), 4, "fp64", 250_000, mode="slots"),
        # the benchmark's drop-in workload in both storage precisions
        _step("dropin_400cube_x4_f64", (400, 400, 400), 4, "fp64", 1_000_000),
        _step("dropin_400cube_x4_f32", (400, 400, 400), 4, "fp32", 1_000_000),
        # the largest workload, FP32 storage
        _step("large_640cube_x8_f32", (640, 640, 640), 8, "fp32", 1_000_000),
        # bulk sources and sinks in the step, and the gradients that chemotaxis reads, ragged grid
        _step("bulk_gradients_190x161x177_f32", (190, 161, 177), 3, "fp32", 20_000, bulk=True, gradients=True),
        # moving agents on a ragged grid
        dict(name="moves_250x230x210_x2_f64", kind="moves", nx=250, ny=230, nz=210, nsub=2, prec="fp64",
             agents=300_000),
        # the benchmark's adjoint workload, fewer steps; launch shapes by the autotuner as it does
        dict(name="adjoint_128cube_x2_f64", kind="adjoint", nx=128, ny=128, nz=128, nsub=2, prec="fp64", agents=10_000,
             steps=20, every=10, tuned=True),
        # uneven microenvironments together, autotuned and graph-replayed as in the benchmark
        # (smaller members: their fields are made on the host and fetched back to it)
        dict(name="batch_12_f64", kind="batch", members=12, lo=24, hi=128, max_sub=8, shape_seed=3, prec="fp64",
             steps=80, tuned=True),
        dict(name="batch_12_f32", kind="batch", members=12, lo=24, hi=128, max_sub=8, shape_seed=3, prec="fp32",
             steps=80, tuned=True),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi, most):
    """Three sizes, log-uniform, equal in one draw of four, at most `most` voxels."""
    while True:
        g = [_size(rng, lo, hi) for _ in range(3)]
        if rng.random() < 0.25:
            g = [g[0]] * 3
        if g[0] * g[1] * g[2] <= most:
            return g


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["moves", "adjoint", "batch"])
    prec = rng.choice(["fp64", "fp32"])
    if kind == "batch":
        return dict(kind="batch", members=rng.randint(2, 12), lo=16, hi=_size(rng, 48, 128), max_sub=rng.randint(1, 8),
                    shape_seed=rng.randrange(1 << 20), prec=prec, steps=rng.choice([5, 10, 20, 40]),
                    tuned=rng.random() < 0.5)
    if kind == "adjoint":
        nx, ny, nz = _grid(rng, 20, 160, 1 << 21)
        every = rng.choice([3, 5, 10])
        return dict(kind="adjoint", nx=nx, ny=ny, nz=nz, nsub=rng.randint(1, 3), prec=prec,
                    agents=_size(rng, 100, 20_000), steps=rng.randint(1, 20), every=every, tuned=rng.random() < 0.5)
    if kind == "moves":
        nx, ny, nz = _grid(rng, 40, 400, 1 << 25)
        return dict(kind="moves", nx=nx, ny=ny, nz=nz, nsub=rng.randint(1, 4), prec=prec,
                    agents=_size(rng, 1000, 500_000))
    nx, ny, nz = _grid(rng, 16, 512, 1 << 26)
    nsub = rng.randint(1, 8)
    while nx * ny * nz * nsub > 1 << 28:
        nsub -= 1
    big = nx * ny * nz * nsub > 1 << 25
    mode = rng.choice(["slots", "run", "run", "graph"])
    return dict(kind="step", nx=nx, ny=ny, nz=nz, nsub=nsub, prec=prec,
                agents=min(_size(rng, 100, 1_000_000), nx * ny * nz // 4), mode=mode,
                steps=1 if mode == "slots" or big else rng.choice([1, 2, 5, 10]),
                nodes=0 if big or rng.random() < 0.7 else _size(rng, 10, 5000),
                bulk=not big and rng.random() < 0.25, gradients=not big and rng.random() < 0.25)


# ------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed & 0x7FFFFFFF)


def _lognormal(shape, seed):
    t = torch.randn(shape, dtype=torch.float64, device=DEV, generator=_gen(seed))
    return t.mul_(0.5).exp_()


def _positions(rng, n, grid):
    """Cells in a ball around the centre, 3/8 of the domain per axis, as a tumour sits in it."""
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    half = np.array(grid) * DX / 2.0
    return half + d * (0.75 * half) * (rng.uniform(0, 1, n) ** (1.0 / 3.0))[:, None]


def _voxels(pos, grid):
    """Voxel of each position in the reference's numbering (x*ny + y)*nz + z."""
    i = np.clip(np.floor(pos / DX).astype(np.int64), 0, np.array(grid) - 1)
    return ((i[:, 0] * grid[1] + i[:, 1]) * grid[2] + i[:, 2]).astype(np.int32)


def _coefficients(rng, ns):
    """Diffusion and decay per substrate, Dirichlet on every other one."""
    return (10.0 ** rng.uniform(2, 5, ns), 10.0 ** rng.uniform(-3, 0, ns), rng.uniform(1.0, 40.0, ns),
            (np.arange(ns) % 2 == 0).astype(np.uint8))


def _tables(S, U):
    """temp1, temp2 of set_internal_uptake_constants with saturation 1."""
    k = (DT * VOLUME) / (DX * DX * DX)
    return S * k, (U + S) * k + 1.0


def _inputs(case, seed):
    """Host inputs of one microenvironment: coefficients, agents, options."""
    rng = np.random.default_rng(seed)
    grid, ns, n = (case["nx"], case["ny"], case["nz"]), case["nsub"], case["agents"]
    D, decay, dval, dact = _coefficients(rng, ns)
    pos = _positions(rng, n, grid)
    inp = dict(grid=grid, ns=ns, D=D, decay=decay, dval=dval, dact=dact, pos=pos, voxel=_voxels(pos, grid),
               S=rng.uniform(0, 5, (n, ns)), U=rng.uniform(0, 20, (n, ns)))
    if case.get("nodes"):
        m, nv = case["nodes"], grid[0] * grid[1] * grid[2]
        v = rng.permutation(nv)[:m]
        face = np.stack([v // (grid[1] * grid[2]), v // grid[2] % grid[1], v % grid[2]], 1)
        axis, end = rng.integers(0, 3, len(v)), rng.integers(0, 2, len(v))  # vessels on the faces
        face[np.arange(len(v)), axis] = np.where(end == 0, 0, np.array(grid)[axis] - 1)
        inp["node_voxel"] = ((face[:, 0] * grid[1] + face[:, 1]) * grid[2] + face[:, 2]).astype(np.int32)
        inp["node_value"] = rng.uniform(0.0, 50.0, (len(v), ns))
    if case.get("bulk"):
        inp["bulk"] = [rng.uniform(0.0, hi, grid + (ns,)) for hi in (1.0, 10.0, 2.0)]  # supply, target, uptake
    return inp


def _solver(case, inp):
    from biofvmb import LODSolver
    s = LODSolver(*inp["grid"], inp["ns"], DX, case["prec"])
    s.set_stream(torch.cuda.current_stream().cuda_stream)
    s.set_coefficients(inp["D"], inp["decay"], DT)
    s.set_dirichlet(inp["dval"], inp["dact"])
    if "node_voxel" in inp:
        s.set_dirichlet_nodes(inp["node_voxel"], inp["node_value"])
    if "bulk" in inp:
        s.set_bulk_rates(*inp["bulk"])
    return s


class _View:
    """A device buffer of `owner` (a solver, kept alive by the tensor that views it)."""

    def __init__(self, owner, ptr, shape, prec):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f8" if prec == "fp64" else "<f4", data=(ptr, False),
                                             version=3, strides=None)


def _device_view(owner, ptr, shape, prec):
    """A device buffer of the library as a torch tensor, without a copy."""
    return torch.as_tensor(_View(owner, ptr, shape, prec), device=DEV)


def _field(s, case):
    return _device_view(s, s.device_ptr(), (case["nsub"], case["nz"], case["ny"], case["nx"]), case["prec"])


def _moved(case, inp, seed):
    """Positions after one random move of about a voxel per axis, kept inside the domain."""
    rng = np.random.default_rng(seed)
    p = inp["pos"] + rng.normal(0.0, DX, inp["pos"].shape)
    return np.clip(p, 1.0, np.array(inp["grid"]) * DX - 1.0)


def _members(case, seed):
    r = random.Random(case["shape_seed"])
    shapes = [tuple(r.randint(case["lo"], case["hi"]) for _ in range(3)) + (r.randint(1, case["max_sub"]),)
              for _ in range(case["members"])]
    out = []
    for i, (nx, ny, nz, ns) in enumerate(shapes):
        rng = np.random.default_rng([seed, i])
        D, decay, dval, dact = _coefficients(rng, ns)
        n = int(rng.integers(0, nx * ny * nz // 64 + 1))
        pos = rng.uniform(0, 1, (n, 3)) * (np.array([nx, ny, nz]) * DX)
        t1, t2 = _tables(rng.uniform(0, 5, (n, ns)), rng.uniform(0, 20, (n, ns)))
        init = rng.uniform(0.5, 2.0, (nx, ny, nz, ns))
        out.append(dict(grid=(nx, ny, nz), ns=ns, D=D, decay=decay, dval=dval, dact=dact, init=init,
                        voxel=_voxels(pos, (nx, ny, nz)), t1=t1, t2=t2))
    return out


def prepare(case, seed):
    if case["kind"] == "batch":
        from biofvmb import Batch
        members = _members(case, seed)
        b = Batch([m["grid"] + (m["ns"],) for m in members], DX, case["prec"])
        b.set_stream(torch.cuda.current_stream().cuda_stream)
        for i, m in enumerate(members):
            b.set_coefficients(i, m["D"], m["decay"], DT)
            b.set_dirichlet(i, m["dval"], m["dact"])
            b.upload(i, m["init"])
            b.set_agents(i, m["voxel"], m["t1"], m["t2"])
        if case["tuned"]:
            b.autotune(reps=2)
        return dict(case=case, batch=b, n=len(members))
    inp = _inputs(case, seed)
    s = _solver(case, inp)
    shape = inp["grid"] + (inp["ns"],)
    init = _lognormal(shape, seed)
    s.upload(init)
    st = dict(case=case, s=s)
    n = case["agents"]
    if case["kind"] == "adjoint":
        t1, t2 = _tables(inp["S"], inp["U"])
        s.set_agents(inp["voxel"], t1, t2)
        if case["tuned"]:
            s.autotune()
        st.update(init=init, target=_lognormal(shape, seed + 1), out=torch.empty_like(init))
        return st
    s.set_agent_rates(inp["voxel"], np.full(n, VOLUME), inp["S"], inp["U"], np.ones((n, inp["ns"])), DT)
    if case["kind"] == "moves":
        moved = [_moved(case, inp, [seed, k]) for k in range(2)]
        st.update(pos=[torch.tensor(p, device=DEV) for p in moved],
                  voxel=[torch.tensor(_voxels(p, inp["grid"]), device=DEV) for p in moved],
                  sensed=torch.empty((n, inp["ns"]), dtype=torch.float64, device=DEV), turn=0)
    return st


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        b = state["batch"]
        b.run(case["steps"], graph=True)
        return [b.download(i) for i in range(state["n"])]
    s = state["s"]
    if case["kind"] == "adjoint":
        s.upload(state["init"])
        s.adjoint_forward(case["steps"], case["every"])
        rT = s.download(state["out"])
        g0, g1, g2 = s.adjoint_backward(2.0 * (rT - state["target"]))
        return dict(field=rT, grad_init=g0, grad_temp1=g1, grad_temp2=g2)
    if case["kind"] == "moves":
        k = state["turn"]
        state["turn"] = 1 - k
        s.update_agent_positions(state["pos"][k])
        s.run(1)
        sensed = s.densities_at(state["voxel"][k], state["sensed"])
        return dict(field=_field(s, case), sensed=sensed)
    if case["mode"] == "slots":
        s.simulate_cell_sources_and_sinks()
        s.simulate_diffusion_decay()
    else:
        s.run(case["steps"], graph=case["mode"] == "graph")
    out = dict(field=_field(s, case))
    if case["gradients"]:
        from biofvmb import _lib
        s.compute_gradients()
        p = ctypes.c_void_p()
        if _lib.load().bfvmb_gradient_device_ptr(ctypes.c_void_p(s.handle), ctypes.byref(p)) != _lib.OK:
            raise RuntimeError("bfvmb_gradient_device_ptr")
        out["gradients"] = _device_view(s, p.value, (3 * case["nsub"], case["nz"], case["ny"], case["nx"]),
                                        case["prec"])
    return out


# -------------------------------------------------------------------------------------- work
def work(case):
    """One pass: per step the field is read once and written once (a step needs every voxel of
    the one before) with the agents' coefficients (temp1, temp2 in FP64, an index) and densities;
    flops per voxel-substrate and sweep: forward 3 (a division counts 1), backward 2."""
    if case["kind"] == "batch":
        r = random.Random(case["shape_seed"])
        shapes = [[r.randint(case["lo"], case["hi"]) for _ in range(3)] + [r.randint(1, case["max_sub"])]
                  for _ in range(case["members"])]
        vs = sum(a * b * c * d for a, b, c, d in shapes)
        agents = sum(a * b * c * d for a, b, c, d in shapes) // 128
    else:
        vs = case["nx"] * case["ny"] * case["nz"] * case["nsub"]
        agents = case["agents"] * case["nsub"]
    e = 8 if case["prec"] == "fp64" else 4
    step = vs * 2 * e + agents * (16 + 2 * e) + agents * 4
    fl = vs * 15 + agents * 2
    if case["kind"] == "batch":
        return {"bytes": step * case["steps"] + vs * 8, "flops": fl * case["steps"]}
    if case["kind"] == "moves":
        n = case["agents"]
        return {"bytes": step + n * 24 + n * 4 + 2 * n * case["nsub"] * 8, "flops": fl + n * 6}
    if case["kind"] == "adjoint":
        # forward, and in the reverse pass the states again and the transposed step; field in
        # and out, target, seed and gradient in FP64
        return {"bytes": 3 * step * case["steps"] + 5 * vs * 8 + 2 * agents * 8, "flops": 3 * fl * case["steps"]}
    b, f = step * case["steps"], fl * case["steps"]
    if case["bulk"]:
        b, f = b + vs * 16 * case["steps"], f + vs * 5 * case["steps"]
    if case["gradients"]:
        b, f = b + vs * 4 * e, f + vs * 6
    return {"bytes": b, "flops": f}


# --------------------------------------------------------------------- the same in 64 bits
# Fields are [substrate][z][y][x] here.
class _Exact:
    def __init__(self, inp, t1, t2):
        self.nx, self.ny, self.nz = inp["grid"]
        self.ns = inp["ns"]
        c1 = inp["D"] * DT / (DX * DX)
        c2 = inp["decay"] * DT / 3.0
        self.c1 = torch.tensor(c1, device=DEV).view(-1, 1, 1)
        self.tab = []  # per axis (x, y, z): denominators and back-substitution factors
        for n in (self.nx, self.ny, self.nz):
            diag = np.repeat((1.0 + 2.0 * c1 + c2)[:, None], n, 1)
            diag[:, 0] = diag[:, -1] = 1.0 + c1 + c2
            if n == 1:
                diag[:, 0] = 1.0 + c2
            den = diag.copy()
            for k in range(1, n):
                den[:, k] = diag[:, k] - c1 * c1 / den[:, k - 1]
            self.tab.append((torch.tensor(den, device=DEV), torch.tensor(c1[:, None] / den, device=DEV)))
        self.dval, self.dact = inp["dval"], inp["dact"]
        self.nodes = None
        if "node_voxel" in inp:
            v, val = inp["node_voxel"], inp["node_value"]
            last = {int(u): k for k, u in enumerate(v)}  # a voxel listed twice keeps its last value
            k = torch.tensor(list(last.values()), device=DEV)
            self.nodes = (torch.tensor(self._offset(np.array(list(last.keys()))), device=DEV),
                          torch.tensor(val, device=DEV)[k].T.contiguous())
        # agents by rank inside their voxel: agents of one rank touch different voxels
        off = self._offset(inp["voxel"])
        order = np.argsort(off, kind="stable")
        first = np.r_[True, off[order][1:] != off[order][:-1]] if len(order) else np.zeros(0, bool)
        pos = np.arange(len(order))
        rank = pos - np.maximum.accumulate(np.where(first, pos, 0)) if len(order) else pos
        self.rounds = []
        a1, a2 = torch.tensor(t1, device=DEV), torch.tensor(t2, device=DEV)
        for r in range(int(rank.max()) + 1 if len(rank) else 0):
            ids = order[rank == r]
            i = torch.tensor(ids, device=DEV)
            self.rounds.append((torch.tensor(off[ids], device=DEV), i, a1[i].T.contiguous(), a2[i].T.contiguous()))

    def _offset(self, voxel):
        v = np.asarray(voxel, dtype=np.int64)
        x, y, z = v // (self.ny * self.nz), v // self.nz % self.ny, v % self.nz
        return (z * self.ny + y) * self.nx + x

    def dirichlet(self, f, zero=False):
        keep = None
        if self.nodes is not None and not zero:
            keep = self.nodes
        for s in range(self.ns):
            if not self.dact[s]:
                continue
            v = 0.0 if zero else float(self.dval[s])
            for face in (f[s, 0], f[s, -1], f[s, :, 0], f[s, :, -1], f[s, :, :, 0], f[s, :, :, -1]):
                face.fill_(v)
            if keep is not None:
                f[s].view(-1)[keep[0]] = keep[1][s]

    def agents(self, f, record=None):
        g = f.view(self.ns, -1)
        for off, ids, t1, t2 in self.rounds:
            r = (g[:, off] + t1) / t2
            g[:, off] = r
            if record is not None:
                record[:, ids] = r

    def agents_adjoint(self, lam, record, g1, g2):
        g = lam.view(self.ns, -1)
        for off, ids, t1, t2 in reversed(self.rounds):
            q = g[:, off] / t2
            g1[:, ids] += q
            g2[:, ids] -= q * record[:, ids]
            g[:, off] = q

    def sweep(self, f, axis):
        dim = 3 - axis  # x, y, z -> dims 3, 2, 1
        den, up = self.tab[axis]
        n = f.shape[dim]
        u = [f.select(dim, k) for k in range(n)]
        d = [den[:, k].view(-1, 1, 1) for k in range(n)]
        u[0].div_(d[0])
        for k in range(1, n):
            u[k].addcmul_(u[k - 1], self.c1).div_(d[k])
        for k in range(n - 2, -1, -1):
            u[k].addcmul_(u[k + 1], up[:, k].view(-1, 1, 1))

    def step(self, f, record=None):
        self.agents(f, record)
        self.dirichlet(f)
        for axis in range(3):
            self.sweep(f, axis)
            self.dirichlet(f)

    def step_adjoint(self, lam, record, g1, g2):
        self.dirichlet(lam, zero=True)
        for axis in (2, 1, 0):
            self.sweep(lam, axis)
            self.dirichlet(lam, zero=True)
        self.agents_adjoint(lam, record, g1, g2)


def _soa(a):
    """[x][y][z][substrate] -> [substrate][z][y][x]."""
    return a.permute(3, 2, 1, 0).contiguous()


def _gradients(f):
    out = torch.zeros((f.shape[0], 3) + tuple(f.shape[1:]), dtype=f.dtype, device=f.device)
    for a, dim in enumerate((3, 2, 1)):
        n = f.shape[dim]
        if n == 1:
            continue
        g = out[:, a]
        g.narrow(dim, 1, n - 2).copy_((f.narrow(dim, 2, n - 2) - f.narrow(dim, 0, n - 2)) / (2.0 * DX))
        g.select(dim, 0).copy_((f.select(dim, 1) - f.select(dim, 0)) / DX)
        g.select(dim, n - 1).copy_((f.select(dim, n - 1) - f.select(dim, n - 2)) / DX)
    return out.view((-1,) + tuple(f.shape[1:]))


def exact(case, seed):
    if case["kind"] == "batch":
        out = []
        for m in _members(case, seed):
            e = _Exact(m, m["t1"], m["t2"])
            f = _soa(torch.tensor(m["init"], device=DEV))
            for _ in range(case["steps"]):
                e.step(f)
            out.append(f.permute(3, 2, 1, 0).contiguous().cpu().numpy())
        return out
    inp = _inputs(case, seed)
    t1, t2 = _tables(inp["S"], inp["U"])
    f = _soa(_lognormal(inp["grid"] + (inp["ns"],), seed))
    if case["kind"] == "moves":
        inp["voxel"] = _voxels(_moved(case, inp, [seed, 0]), inp["grid"])
        e = _Exact(inp, t1, t2)
        e.step(f)
        off = torch.tensor(e._offset(inp["voxel"]), device=DEV)
        return dict(field=f, sensed=f.view(inp["ns"], -1)[:, off].T.contiguous())
    e = _Exact(inp, t1, t2)
    if case["kind"] == "adjoint":
        na = case["agents"]
        recs = [torch.zeros((e.ns, na), dtype=torch.float64, device=DEV) for _ in range(case["steps"])]
        for r in recs:
            e.step(f, r)
        rT = f.permute(3, 2, 1, 0).contiguous()
        lam = _soa(2.0 * (rT - _lognormal(inp["grid"] + (inp["ns"],), seed + 1)))
        g1 = torch.zeros((e.ns, na), dtype=torch.float64, device=DEV)
        g2 = torch.zeros_like(g1)
        for r in reversed(recs):
            e.step_adjoint(lam, r, g1, g2)
        return dict(field=rT, grad_init=lam.permute(3, 2, 1, 0).contiguous(), grad_temp1=g1.T.contiguous(),
                    grad_temp2=g2.T.contiguous())
    bulk = [_soa(torch.tensor(b, device=DEV)) for b in inp["bulk"]] if "bulk" in inp else None
    for _ in range(case["steps"]):
        if bulk is not None and case["mode"] != "slots":  # the bulk update belongs to run(), not to the slots
            supply, target, uptake = bulk
            f = (f + DT * target * supply) / (1.0 + DT * (uptake + supply))
        e.step(f)
    out = dict(field=f)
    if case["gradients"]:
        out["gradients"] = _gradients(f)
    return out
