"""Workloads of the solver and of the warm-start network, as a user's program runs them.

Every case is a dict of plain values; ``prepare`` makes what a program holds before the call (mesh, solver or
network handle, host state), ``run`` is one pass through the public entry points, ``work`` the bytes and operations
the pass cannot do without, and ``exact`` the same outputs from plain torch in float64.

Kinds:

* ``march``: the drop-in's time_integration call between two saves: hand the conservative state over, advance a number
  of Runge-Kutta steps with their residual norms (and, with ``errors``, the vortex error record of every step), take
  the state back.  On ``square`` meshes (the isentropic vortex, periodic or with the outline as Dirichlet boundary) or
  ``ogrid`` meshes (steady Euler around an airfoil with local time steps).
* ``batch``: the same for many O-grids of different sizes and conditions in one batched solver, with every instance's
  residual norms, and the wall forces at the end.
* ``residual``: one residual evaluation of a state in host memory, as a driver with its own time stepping asks for it.
* ``train``, ``step``, ``predict``: the network's training on its resident data set, one optimiser step on rows given
  by the caller, and the evaluation on all cells of a grid.
"""
import math
import zlib

import numpy as np
import torch

from fvs2d_amd import _lib
from fvs2d_amd.meshgen import Mesh
from fvs2d_amd.mlp import WarmStartNet
from fvs2d_amd.solver import BatchSolver, Scheme, Solver

GAMMA = 1.4
NET = {"depth": 5, "lr": 1e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8}
GRIDS = ((128, 64), (256, 128), (384, 192))  # per-instance resolutions of a batch
RK = {"ssp3": _lib.RK_SSP3, "ssp42": _lib.RK_SSP42, "rk4": _lib.RK_CLASSIC}
STAGES = {"ssp3": 3, "ssp42": 4, "rk4": 4}


def _march(n, grad="lsq", limiter=0, steps=100, mesh="square", periodic=True, rk="ssp3", errors=False, stencil="nn"):
    return {"kind": "march", "mesh": mesh, "n": n, "grad": grad, "limiter": limiter, "steps": steps,
            "periodic": periodic, "rk": rk, "errors": errors, "stencil": stencil}


def _ogrid(n, layers, steps, limiter=1):
    return {"kind": "march", "mesh": "ogrid", "n": n, "layers": layers, "limiter": limiter, "steps": steps,
            "grad": "lsq", "rk": "ssp42", "errors": False, "stencil": "nn"}


def listed():
    return [
        # the small vortex run of the parity workloads: 8,192 triangles, 100 steps; launches and latency count
        dict(_march(64, steps=100), name="vortex 64"),
        # the headline benchmark: 2,097,152 triangles, 200 steps, unlimited LSQ gradients
        dict(_march(1024, steps=200), name="vortex 1024"),
        # the same scheme with the Venkatakrishnan limiter, on an ordinary mesh of odd size
        dict(_march(511, limiter=1, steps=100), name="vortex 511 limited"),
        # the cell-based Green-Gauss variant, unlimited
        dict(_march(400, grad="ggcb", steps=100), name="vortex 400 ggcb"),
        # the node-based Green-Gauss variant with the limiter
        dict(_march(301, grad="ggnb", limiter=1, steps=100), name="vortex 301 ggnb limited"),
        # the scheme of the vortex example deck (face-neighbour LSQ, RK4, Dirichlet outline) on a mesh of the
        # example's size, with the error record of every step that its driver logs, between two of its saves
        dict(_march(60, steps=80, periodic=False, rk="rk4", errors=True, stencil="fn"), name="vortex 60 error log"),
        # one airfoil at the smallest batch resolution, a convergence-check interval of pseudo-time steps
        dict(_ogrid(128, 64, 250), name="airfoil 128x64"),
        # the transonic airfoil workload at its stated size
        dict(_ogrid(512, 256, 250), name="airfoil 512x256"),
        # a ragged batch of airfoils, an interval of steps and the forces
        {"kind": "batch", "instances": 12, "steps": 100, "name": "batch of 12"},
        # one residual for a driver that steps by itself: host state in, residual and wave speeds out
        {"kind": "residual", "n": 333, "grad": "lsq", "limiter": 1, "name": "residual 333"},
        # network training at its stated batch size
        {"kind": "train", "rows": 65536, "records": 262144, "steps": 10, "name": "train 65536"},
        # the warm start of one grid: the network on every cell of a 256x128 O-grid
        {"kind": "predict", "rows": 65536, "batch": 65536, "name": "predict 65536"},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["vortex"] * 5 + ["airfoil"] * 2 + ["batch", "residual", "train", "step", "predict"])
    if kind == "vortex":
        n = log(40, 640)
        periodic = rng.random() < 0.7
        return _march(n, grad=rng.choice(["lsq", "lsq", "ggcb", "ggnb"]), limiter=rng.choice([0, 0, 1]),
                      steps=log(40, 160), periodic=periodic, rk=rng.choice(["ssp3", "ssp3", "rk4"]),
                      errors=(not periodic) and rng.random() < 0.5)
    if kind == "airfoil":
        n = 2 * log(32, 192)
        return _ogrid(n, max(16, n // 2 + rng.randint(-3, 3)), log(100, 250), limiter=rng.choice([0, 1, 1]))
    if kind == "batch":
        return {"kind": "batch", "instances": rng.randint(3, 14), "steps": log(40, 120)}
    if kind == "residual":
        return {"kind": "residual", "n": log(50, 500), "grad": rng.choice(["lsq", "ggcb", "ggnb"]),
                "limiter": rng.choice([0, 1])}
    if kind == "train":
        return {"kind": "train", "rows": 64 * log(32, 1024), "records": log(20000, 400000), "steps": rng.randint(5, 12)}
    if kind == "step":
        return {"kind": "step", "rows": log(100, 30000), "batch": 32768}
    return {"kind": "predict", "rows": log(2000, 300000), "batch": 65536}


# ------------------------------------------------------------------------------------------------------- inputs
def _rng(case, seed, what=""):
    return np.random.Generator(np.random.PCG64([int(seed), zlib.crc32((case["kind"] + what).encode())]))


def _square(n, periodic, rng):
    """[-5, 5]^2 in n x n quads, each split into two triangles, interior nodes displaced by up to 10% of the spacing.
    A Dirichlet outline: two corner quads are split the other way, so that no cell has two boundary edges."""
    h = 10.0 / n
    i, j = (a.ravel() for a in np.meshgrid(np.arange(n + 1), np.arange(n + 1)))
    xy = np.stack([-5.0 + i * h, -5.0 + j * h], 1)
    inside = np.nonzero((i > 0) & (i < n) & (j > 0) & (j < n))[0]
    u = rng.random((inside.size, 2))
    r = 0.1 * h * np.sqrt(u[:, 0])
    xy[inside] += np.stack([r * np.cos(2 * np.pi * u[:, 1]), r * np.sin(2 * np.pi * u[:, 1])], 1)
    qi, qj = (a.ravel() for a in np.meshgrid(np.arange(n), np.arange(n)))
    bl = qj * (n + 1) + qi
    br, tl, tr = bl + 1, bl + n + 1, bl + n + 2
    tri = np.empty((2 * n * n, 3), np.int32)
    tri[0::2], tri[1::2] = np.stack([bl, br, tr], 1), np.stack([bl, tr, tl], 1)
    if periodic:
        return xy, tri, ((j % n) * (n + 1) + i % n).astype(np.int32), []
    flip = np.nonzero(((qi == n - 1) & (qj == 0)) | ((qi == 0) & (qj == n - 1)))[0]
    tri[2 * flip], tri[2 * flip + 1] = np.stack([bl, br, tl], 1)[flip], np.stack([br, tr, tl], 1)[flip]
    side = np.stack([i == 0, i == n, j == 0, j == n], 1)[tri]
    edge = (side & np.roll(side, -1, axis=1)).any(axis=(1, 2))
    return xy, tri, None, [("dirichlet", np.nonzero(edge)[0].astype(np.int32))]


def _airfoil(m, layers, thickness):
    """O-grid of m x layers quads, split into triangles, around a symmetric 4-digit section with a closed trailing
    edge: cosine-clustered surface nodes, first spacing 2e-3, geometric growth to 50 chords, rays that turn from the
    surface normal to the ray from mid-chord."""
    s = 2 * np.pi * np.arange(m) / m
    x = 0.5 * (1 + np.cos(s))
    y = 5 * thickness * (0.2969 * np.sqrt(x) - 0.1260 * x - 0.3516 * x ** 2 + 0.2843 * x ** 3 - 0.1036 * x ** 4)
    y = np.where(s <= np.pi, y, -y)
    y[0] = y[m // 2] = 0.0
    ang = np.arctan2(y, x - 0.5)
    t = np.stack([np.roll(x, -1) - np.roll(x, 1), np.roll(y, -1) - np.roll(y, 1)], 1)
    nrm = np.stack([t[:, 1], -t[:, 0]], 1) / np.hypot(t[:, 0], t[:, 1])[:, None]
    nrm[(nrm[:, 0] * (x - 0.5) + nrm[:, 1] * y) < 0] *= -1
    ray = np.stack([np.cos(ang), np.sin(ang)], 1)
    far = np.array([0.5, 0.0]) + 50.0 * ray
    surf = np.stack([x, y], 1)
    span = np.linalg.norm(far - surf, axis=1)
    lo, hi = 1 + 1e-12, 2.0
    for _ in range(200):
        r = 0.5 * (lo + hi)
        lo, hi = (lo, r) if 2e-3 * (r ** layers - 1) / (r - 1) > 50.0 else (r, hi)
    d = 2e-3 * (r ** np.arange(layers + 1) - 1) / (r - 1)
    xy = np.empty((layers + 1, m, 2))
    for k in range(layers):
        b = math.sqrt(d[k] / 50.0)
        way = (1 - b) * nrm + b * ray
        xy[k] = surf + (d[k] * span / 50.0 / np.linalg.norm(way, axis=1))[:, None] * way
    xy[layers] = far
    k, i = (a.ravel() for a in np.meshgrid(np.arange(layers), np.arange(m), indexing="ij"))
    a, b = k * m + i, k * m + (i + 1) % m
    tri = np.empty((2 * a.size, 3), np.int32)
    tri[0::2], tri[1::2] = np.stack([b + m, b, a], 1), np.stack([a + m, b + m, a], 1)
    wall = np.arange(0, 2 * m, 2, dtype=np.int32)
    return xy.reshape(-1, 2), tri, None, [("slip_wall", wall), ("freestream", wall + 2 * (layers - 1) * m + 1)]


def _conservative(p):
    rho, u, v, pr = p
    return np.stack([rho, rho * u, rho * v, pr / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)], -1)


def _vortex(x, y):
    """The isentropic vortex of strength 5 about the origin on the free stream (1, 1, 1, 1)."""
    c, e = 5.0 / (2 * np.pi), np.exp(0.5 * (1 - x * x - y * y))
    rho = (1.0 - c * c * (GAMMA - 1) / (2 * GAMMA) * e * e) ** (1 / (GAMMA - 1))
    return rho, 1.0 - c * y * e, 1.0 + c * x * e, rho ** GAMMA


def _freestream(mach, aoa):
    a = math.radians(aoa)
    return 1.0, mach * math.cos(a), mach * math.sin(a), 1 / GAMMA


def _conditions(rng, count):
    """Mach number, angle of attack and thickness of `count` airfoil cases."""
    return [(float(rng.uniform(0.5, 0.85)), float(rng.uniform(-2, 4)), float(rng.uniform(0.10, 0.15)))
            for _ in range(count)]


def _flow(case, seed):
    """Meshes, conditions and the start state of a solver case."""
    rng = _rng(case, seed)
    if case["kind"] == "batch":
        sizes = [GRIDS[k % 3] for k in range(case["instances"])]
        cond = _conditions(rng, len(sizes))
        meshes = [_airfoil(m, layers, c[2]) for (m, layers), c in zip(sizes, cond)]
    elif case.get("mesh") == "ogrid":
        cond = [_conditions(rng, 1)[0][:2] + (0.12,)]
        meshes = [_airfoil(case["n"], case["layers"], 0.12)]
    else:
        xy, tri, canon, bnd = _square(case["n"], case.get("periodic", True), rng)
        c = xy[tri].mean(axis=1)
        return [(xy, tri, canon, bnd)], None, _conservative(_vortex(c[:, 0], c[:, 1]))
    start = np.concatenate([np.tile(_conservative(_freestream(*c[:2])), (len(m[1]), 1)) for m, c in zip(meshes, cond)])
    return meshes, cond, start


def _scheme(case):
    steady = case["kind"] == "batch" or case.get("mesh") == "ogrid"
    grad = {"ggcb": 1, "ggnb": 2, "lsq": 3}[case.get("grad", "lsq")]
    common = dict(grad_method=grad, lsq_nn=int(case.get("stencil", "nn") == "nn"), limiter=case.get("limiter", 1),
                  recon=2, gamma=GAMMA, rk_scheme=RK[case.get("rk", "ssp42" if steady else "ssp3")], rk_order=4)
    if steady:
        return Scheme(**dict(common, rk_order=2, steady=1, cfl=1.25, dt=1.0, reorder=2))
    return Scheme(**dict(common, lvortex=1, vortex_K=5.0, vortex_inf=(1.0, 1.0, 1.0, 1.0), dt=_dt(case), reorder=1))


def _dt(case):
    return 1.1 / case["n"]  # a CFL number of about 0.5


def _records(rng, n):
    """Cell records (x, y, wall distance, Mach, angle of attack, thickness) around an airfoil, and smooth targets."""
    r, th = np.exp(rng.uniform(math.log(0.01), math.log(50.0), n)), rng.uniform(-np.pi, np.pi, n)
    raw = np.stack([0.5 + r * np.cos(th), r * np.sin(th), r * rng.uniform(0.8, 1.0, n), rng.uniform(0.5, 0.85, n),
                    rng.uniform(-2, 4, n), rng.uniform(0.10, 0.15, n)], 1).astype(np.float32)
    target = np.stack([np.sin(2 * th) * np.exp(-r), np.cos(th) / (1 + r), raw[:, 3] - 0.675, raw[:, 4] / 4], 1)
    return raw, target.astype(np.float32)


def _sizes():
    return [(68, 256)] + [(256, 256)] * (NET["depth"] - 1) + [(256, 4)]


def _weights(rng):
    """Glorot-uniform weights and small biases in the network's flat layout."""
    parts = []
    for i, o in _sizes():
        a = math.sqrt(6.0 / (i + o))
        parts += [rng.uniform(-a, a, i * o), rng.uniform(-0.05, 0.05, o)]
    return np.concatenate(parts).astype(np.float32)


def prepare(case, seed):
    if case["kind"] in ("train", "step", "predict"):
        rng = _rng(case, seed)
        net = WarmStartNet(batch=case["rows"] if case["kind"] == "train" else case["batch"], seed=0, **NET)
        net.set_params(_weights(rng))
        raw, target = _records(rng, case["records"] if case["kind"] == "train" else case["rows"])
        if case["kind"] == "train":
            net.set_data(raw, target)
        return {"case": case, "net": net, "raw": raw, "target": target}
    meshes, cond, start = _flow(case, seed)
    meshes = [Mesh(xy, len(tri), 0, tri.ravel(), bnd, canon=canon) for xy, tri, canon, bnd in meshes]
    scheme = _scheme(case)
    if case["kind"] == "batch":
        solver = BatchSolver(meshes, [c[:2] for c in cond], scheme)
    elif cond:
        solver = Solver(meshes[0], scheme, mach=cond[0][0], aoa_deg=cond[0][1])
    else:
        solver = Solver(meshes[0], scheme)
    if cond:
        solver.set_graph(True)  # as the steady drivers run
    return {"case": case, "solver": solver, "start": start}


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        loss = state["net"].train(case["steps"])
        return {"loss": loss.astype(np.float32), "weights": state["net"].get_params()}  # the loss is a float32 sum
    if case["kind"] == "step":
        loss = state["net"].step(state["raw"], state["target"])
        return {"loss": np.float32(loss), "weights": state["net"].get_params()}
    if case["kind"] == "predict":
        return state["net"].predict(state["raw"])
    solver = state["solver"]
    solver.cvar = state["start"]
    if case["kind"] == "residual":
        resid, ws = solver.compute_residual(0.0)
        return {"resid": resid, "ws": ws}
    if case["kind"] == "batch":
        norms = solver.batch_time_integration(0.0, case["steps"])
        return {"norms": norms, "forces": solver.wall_forces_batch(), "cvar": solver.cvar}
    if case["errors"]:
        norms, errors = solver.time_integration(0.0, case["steps"], vortex_error=True)
        return {"norms": norms, "errors": errors, "cvar": solver.cvar}
    return {"norms": solver.time_integration(0.0, case["steps"]), "cvar": solver.cvar}


# --------------------------------------------------------------------------------------------------------- work
def _cells(case):
    if case["kind"] == "batch":
        return sum(2 * GRIDS[k % 3][0] * GRIDS[k % 3][1] for k in range(case["instances"]))
    return 2 * case["n"] * case.get("layers", case["n"])


def work(case):
    """Solver: every stage reads and writes the state (64 B per cell) and reads the mesh (three node ids and half a
    node's coordinates per cell); per cell and stage 1.5 Roe fluxes of about 170 operations, a gradient over 12
    neighbours of 24 (LSQ) and the stage update.  Network: rows in and out, the weights once per pass, and the matrix
    products (a training step three times the forward's)."""
    if case["kind"] in ("train", "step", "predict"):
        rows, steps = case["rows"], case.get("steps", 1)
        size = sum(i * o + o for i, o in _sizes())
        flops = 2.0 * rows * sum(i * o for i, o in _sizes())
        if case["kind"] == "predict":
            return {"bytes": rows * 40.0 + 4.0 * size, "flops": flops}
        return {"bytes": steps * (rows * 40.0 + 24.0 * size), "flops": 3 * steps * flops}
    cells = float(_cells(case))
    stages = 1 if case["kind"] == "residual" else case["steps"] * STAGES[case.get("rk", "ssp42")]
    return {"bytes": cells * 84.0 * stages, "flops": cells * 600.0 * stages}


# -------------------------------------------------------------------------------- the same in float64, plain torch
class _Euler:
    """The finite-volume scheme on triangle meshes in plain torch: node-neighbour LSQ or Green-Gauss gradients,
    Venkatakrishnan's limiter, Roe's flux, all in float64."""

    def __init__(self, case, meshes, cond, dev):
        self.case, self.dev = case, dev
        nodes = np.cumsum([0] + [len(m[0]) for m in meshes])
        cells = np.cumsum([0] + [len(m[1]) for m in meshes])
        self.off = cells
        put = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        xy = put(np.concatenate([m[0] for m in meshes]))
        tri = put(np.concatenate([m[1].astype(np.int64) + o for m, o in zip(meshes, nodes)]))
        own = put(meshes[0][2].astype(np.int64))[tri] if meshes[0][2] is not None else tri
        n, nv = len(tri), len(xy)
        p = xy[tri]
        q = torch.roll(p, -1, 1)
        self.xc = p.mean(1)
        d = q - p
        self.area = torch.linalg.norm(d, dim=2)  # [n, 3]
        self.nrm = torch.stack([d[..., 1], -d[..., 0]], 2) / self.area[..., None]
        self.mid = 0.5 * (p + q) - self.xc[:, None]  # edge centres from the cell's centre, in the cell's own frame
        e1, e2 = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
        self.vol = 0.5 * (e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0])
        a, b = own, torch.roll(own, -1, 1)
        key = (torch.minimum(a, b) * nv + torch.maximum(a, b)).reshape(-1)
        order = torch.argsort(key, stable=True)
        key = key[order]
        pair = torch.nonzero(key[1:] == key[:-1])[:, 0]
        other = torch.full((3 * n,), -1, dtype=torch.int64, device=dev)  # the same edge as the neighbour's side
        other[order[pair]], other[order[pair + 1]] = order[pair + 1], order[pair]
        self.left = order[pair]  # interior edges once, as sides 3 c + e of their two cells
        self.right = order[pair + 1]
        self.bnd = torch.nonzero(other < 0)[:, 0]
        kind = torch.full((n,), -1, dtype=torch.int64, device=dev)
        for m, o in zip(meshes, cells):
            for name, c in m[3]:
                kind[put(c.astype(np.int64)) + int(o)] = {"freestream": 0, "slip_wall": 1, "dirichlet": 2}[name]
        self.kind = kind[self.bnd // 3]
        inst = torch.repeat_interleave(torch.arange(len(meshes), device=dev), put(np.diff(cells)))
        self.inst = inst
        if cond:
            self.far = put(np.array([_freestream(*c[:2]) for c in cond]))[inst[self.bnd // 3]]
        self.bxy = (self.mid + self.xc[:, None]).reshape(-1, 2)[self.bnd]
        # cells around every node: sides 3 c + l, padded
        flat = own.reshape(-1)
        by = torch.argsort(flat, stable=True)
        count = torch.bincount(flat, minlength=nv)
        first = torch.cumsum(count, 0) - count
        place = torch.arange(3 * n, device=dev) - first[flat[by]]
        around = torch.full((nv, int(count.max())), -1, dtype=torch.int64, device=dev)
        around[flat[by], place] = by
        if case.get("grad") == "ggnb":
            w = 1.0 / torch.linalg.norm(p - self.xc[:, None], dim=2)
            total = torch.zeros(nv, dtype=torch.float64, device=dev).index_add_(0, flat, w.reshape(-1))
            self.node_w, self.own, self.nv = w / total[own], own, nv
        if case.get("grad") == "ggcb":
            far = torch.where(other < 0, torch.arange(3 * n, device=dev), other).reshape(n, 3)
            d0 = torch.linalg.norm(self.mid, dim=2)
            d1 = d0.reshape(-1)[far]
            self.face_nb, self.face_w = far // 3, d0 / (d0 + d1)
        if case.get("limiter", 1) or case.get("grad", "lsq") == "lsq":
            ids, dxy = [], []
            for l in range(3):
                s = around[own[:, l]]  # [n, most]
                c = torch.clamp(s, min=0) // 3
                use = (s >= 0) & (c != torch.arange(n, device=dev)[:, None])
                for k in range(l):  # already met at an earlier node
                    use &= (own[c] != own[:, k][:, None, None]).all(2)
                here, there = p[:, l][:, None], xy[tri.reshape(-1)[torch.clamp(s, min=0)]]
                dxy.append(torch.where(use[..., None], self.xc[c] - there + here - self.xc[:, None], 0.0))
                ids.append(torch.where(use, c, -1))
                del s, c, use, here, there
            ids, dxy = torch.cat(ids, 1), torch.cat(dxy, 1)
            most = int((ids >= 0).sum(1).max())
            first = torch.argsort((ids < 0).to(torch.int8), dim=1, stable=True)[:, :most]
            self.nb, self.nb_d = torch.gather(ids, 1, first), torch.gather(dxy, 1, first[..., None].expand(-1, -1, 2))
            self.nb = torch.where(self.nb < 0, torch.arange(n, device=dev)[:, None], self.nb).T.contiguous()
            self.nb_d = self.nb_d.permute(1, 2, 0).contiguous()
            g = torch.einsum("kan,kbn->abn", self.nb_d, self.nb_d)
            det = g[0, 0] * g[1, 1] - g[0, 1] ** 2
            self.ginv = g[1, 1] / det, -g[0, 1] / det, g[0, 0] / det

    def gradient(self, w):
        grad = self.case.get("grad", "lsq")
        if grad == "lsq":
            sx, sy = torch.zeros_like(w), torch.zeros_like(w)
            for j, d in zip(self.nb, self.nb_d):
                t = w[j] - w
                sx.addcmul_(t, d[0][:, None])
                sy.addcmul_(t, d[1][:, None])
            a, b, c = (v[:, None] for v in self.ginv)
            return torch.stack([a * sx + b * sy, b * sx + c * sy], 1)  # [n, 2, 4]
        if grad == "ggcb":
            face = w[:, None] + self.face_w[..., None] * (w[self.face_nb] - w[:, None])
        else:
            node = torch.zeros(self.nv, 4, dtype=torch.float64, device=self.dev)
            node.index_add_(0, self.own.reshape(-1), (self.node_w[..., None] * w[:, None]).reshape(-1, 4))
            face = node[self.own]
            face = 0.5 * (face + torch.roll(face, -1, 1))
        out = (self.nrm * self.area[..., None])[..., None] * face[:, :, None]  # [n, 3, 2, 4]
        return out.sum(1) / self.vol[:, None, None]

    def limiter(self, w, grad):
        lo, hi = w.clone(), w.clone()
        for j in self.nb:
            q = w[j]
            torch.minimum(lo, q, out=lo)
            torch.maximum(hi, q, out=hi)
        eps2 = (5.0 * 2.0 * torch.sqrt(self.vol / math.pi))[:, None] ** 3
        phi = torch.ones_like(w)
        for e in range(3):
            b = self.mid[:, e, 0:1] * grad[:, 0] + self.mid[:, e, 1:2] * grad[:, 1]
            a = torch.where(b > 0, hi - w, lo - w)
            f = ((a * a + eps2) + 2 * b * a) / (a * a + 2 * b * b + a * b + eps2)
            phi = torch.minimum(phi, torch.where(b == 0, 1.0, f))
        return phi.amin(1)

    @staticmethod
    def roe(wl, wr, nrm):
        nx, ny = nrm[:, 0], nrm[:, 1]
        rl, ul, vl, pl = wl.unbind(1)
        rr, ur, vr, pr = wr.unbind(1)
        hl = GAMMA * pl / rl / (GAMMA - 1) + 0.5 * (ul * ul + vl * vl)
        hr = GAMMA * pr / rr / (GAMMA - 1) + 0.5 * (ur * ur + vr * vr)
        t = torch.sqrt(rr / rl)
        rho, u, v, h = t * rl, (ul + t * ur) / (1 + t), (vl + t * vr) / (1 + t), (hl + t * hr) / (1 + t)
        k = 0.5 * (u * u + v * v)
        a = torch.sqrt((GAMMA - 1) * (h - k))
        un, ut = u * nx + v * ny, v * nx - u * ny
        unl, unr = ul * nx + vl * ny, ur * nx + vr * ny
        dp, dun, dut = pr - pl, unr - unl, (vr - vl) * nx - (ur - ul) * ny

        def speed(s):
            s = s.abs()
            return torch.where(s < 0.2, 0.5 * (s * s / 0.2 + 0.2), s)

        s0 = speed(un - a) * (dp - rho * a * dun) / (2 * a * a)
        s1 = un.abs() * rho * dut
        s2 = un.abs() * (rr - rl - dp / (a * a))
        s3 = speed(un + a) * (dp + rho * a * dun) / (2 * a * a)
        diss = torch.stack([s0 + s2 + s3, s0 * (u - a * nx) - s1 * ny + s2 * u + s3 * (u + a * nx),
                            s0 * (v - a * ny) + s1 * nx + s2 * v + s3 * (v + a * ny),
                            s0 * (h - un * a) + s1 * ut + s2 * k + s3 * (h + un * a)], 1)
        fl = torch.stack([rl * unl, rl * unl * ul + pl * nx, rl * unl * vl + pl * ny, rl * unl * hl], 1)
        fr = torch.stack([rr * unr, rr * unr * ur + pr * nx, rr * unr * vr + pr * ny, rr * unr * hr], 1)
        return 0.5 * (fl + fr - diss), 0.5 * (un.abs() + a)

    def primitive(self, u):
        v = u[:, 1:3] / u[:, :1]
        return torch.cat([u[:, :1], v, (GAMMA - 1) * (u[:, 3:] - 0.5 * u[:, :1] * (v * v).sum(1, keepdim=True))], 1)

    def residual(self, u, t):
        w = self.primitive(u)
        grad = self.gradient(w)
        step = torch.einsum("ned,ndv->nev", self.mid, grad)
        if self.case.get("limiter", 1):
            step = step * self.limiter(w, grad)[:, None, None]
        sides = (w[:, None] + step).reshape(-1, 4)
        nrm, area = self.nrm.reshape(-1, 2), self.area.reshape(-1, 1)
        flux = torch.zeros_like(sides)
        ws = torch.zeros(len(sides), dtype=torch.float64, device=self.dev)
        f, s = self.roe(sides[self.left], sides[self.right], nrm[self.left])
        flux[self.left], flux[self.right] = f * area[self.left], -f * area[self.left]
        ws[self.left] = ws[self.right] = s * area[self.left, 0]
        if len(self.bnd):
            inner, nb = sides[self.bnd], nrm[self.bnd]
            ghost = inner.clone()
            ghost[:, 1:3] -= 2 * (inner[:, 1:3] * nb).sum(1, keepdim=True) * nb  # slip wall
            if bool((self.kind == 0).any()):
                ghost = torch.where((self.kind == 0)[:, None], self.far, ghost)
            if bool((self.kind == 2).any()):
                x = self.bxy.cpu().numpy() - t  # the vortex travels with the stream (1, 1)
                ghost = torch.as_tensor(np.stack(_vortex(x[:, 0], x[:, 1]), 1), device=self.dev)
            f, s = self.roe(inner, ghost, nb)
            flux[self.bnd], ws[self.bnd] = f * area[self.bnd], s * area[self.bnd, 0]
        return -flux.reshape(-1, 3, 4).sum(1) / self.vol[:, None], ws.reshape(-1, 3).sum(1)

    def march(self, u, steps, rk, dt, cfl=None):
        norms = []
        for i in range(steps):
            t, u0, acc = i * dt, u, torch.zeros_like(u)
            for k in range(STAGES[rk]):
                at = {"ssp3": (0, dt, 0.5 * dt), "rk4": (0, 0.5 * dt, 0.5 * dt, dt),
                      "ssp42": (0, dt / 3, 2 * dt / 3, dt)}[rk][k]
                r, ws = self.residual(u, t + at)
                if cfl is not None and k == 0:
                    local = (cfl * self.vol / (0.5 * ws))[:, None]
                h = dt if cfl is None else local
                if rk == "ssp3":
                    a, b = ((0, 1), (0.75, 0.25), (1 / 3, 2 / 3))[k]
                    u = a * u0 + b * (u + h * r)
                elif rk == "ssp42":
                    acc = acc + r
                    u = u0 + h * (0.25 if k == 3 else 1 / 3) * acc
                else:
                    acc = acc + (1, 2, 2, 1)[k] * r
                    u = u0 + h * acc / 6 if k == 3 else u0 + h * (0.5, 0.5, 1)[k] * r
            sq = (u - u0) ** 2
            if len(self.off) == 2:
                norms.append(torch.sqrt(sq.mean(0)))
            else:
                norms.append(torch.sqrt(torch.stack([sq[a:b].mean(0) for a, b in zip(self.off[:-1], self.off[1:])])))
        return u, torch.stack(norms)

    def forces(self, u, cond):
        """C_L, C_D of every instance from the face-extrapolated and from the cell pressure."""
        w = self.primitive(u)
        grad = self.gradient(w)
        wall = self.bnd[self.kind == 1]
        c = wall // 3
        mid, out = self.mid.reshape(-1, 2)[wall], (self.nrm * self.area[..., None]).reshape(-1, 2)[wall]
        mach = torch.tensor([x[0] for x in cond], dtype=torch.float64, device=self.dev)
        al = torch.deg2rad(torch.tensor([x[1] for x in cond], dtype=torch.float64, device=self.dev))
        res = []
        for p in (w[c, 3] + (mid * grad[c, :, 3]).sum(1), w[c, 3]):
            push = 2 / mach[self.inst[c]][:, None] ** 2 * (p - 1 / GAMMA)[:, None] * out
            f = torch.zeros(len(cond), 2, dtype=torch.float64, device=self.dev).index_add_(0, self.inst[c], push)
            res += [f[:, 1] * torch.cos(al) - f[:, 0] * torch.sin(al), f[:, 1] * torch.sin(al) + f[:, 0] * torch.cos(al)]
        return torch.stack(res, 1)


def _features(raw):
    x, y, d, m, a, t = raw.double().unbind(1)
    r, th = torch.hypot(x - 0.5, y), torch.atan2(y, x - 0.5)
    s = math.pi * torch.log1p(4 * r) / math.log1p(200.0)
    k = torch.arange(1, 17, device=raw.device, dtype=torch.float64)
    waves = [torch.stack([torch.sin(k * v[:, None]), torch.cos(k * v[:, None])], 2).reshape(len(raw), 32) for v in (s, th)]
    rest = torch.stack([torch.log1p(100 * d) / math.log1p(5000.0), (m - 0.675) / 0.175, (a - 1) / 3,
                        (t - 0.125) / 0.025], 1)
    return torch.cat(waves + [rest], 1)


def _forward(weights, x):
    at = 0
    for layer, (i, o) in enumerate(_sizes()):
        x = x @ weights[at:at + i * o].reshape(i, o) + weights[at + i * o:at + i * o + o]
        at += i * o + o
        if layer < NET["depth"]:
            x = torch.nn.functional.gelu(x)
    return x


def _mix64(z):
    """splitmix64's finaliser, by which the network draws its training rows."""
    z = (z + np.uint64(0x9E3779B97F4A7C15)).astype(np.uint64)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _network(case, seed, dev):
    rng = _rng(case, seed)
    w = torch.as_tensor(_weights(rng), device=dev).double()
    raw, target = _records(rng, case.get("records", case["rows"]))
    x, target = _features(torch.as_tensor(raw, device=dev)), torch.as_tensor(target, device=dev).double()
    if case["kind"] == "predict":
        return torch.cat([_forward(w, v) for v in x.split(65536)])
    m, v, losses = torch.zeros_like(w), torch.zeros_like(w), []
    for t in range(1, case.get("steps", 1) + 1):
        rows = slice(None)
        if case["kind"] == "train":
            with np.errstate(over="ignore"):
                slot = np.uint64(t) * np.uint64(0x100000001) + np.arange(case["rows"], dtype=np.uint64)
                rows = torch.as_tensor((_mix64(_mix64(slot)) % np.uint64(len(raw))).astype(np.int64), device=dev)
        w = w.detach().requires_grad_(True)
        loss = ((_forward(w, x[rows]) - target[rows]) ** 2).mean()
        g, = torch.autograd.grad(loss, w)
        losses.append(float(loss))
        m = NET["beta1"] * m + (1 - NET["beta1"]) * g
        v = NET["beta2"] * v + (1 - NET["beta2"]) * g * g
        w = w.detach() - NET["lr"] * (m / (1 - NET["beta1"] ** t)) / (torch.sqrt(v / (1 - NET["beta2"] ** t)) + NET["eps"])
    return {"loss": np.array(losses) if case["kind"] == "train" else losses[0], "weights": w}


def exact(case, seed):
    if case.get("stencil") == "fn" or case.get("errors"):
        return None  # the augmented face-neighbour stencil and the error record's cell lists are not restated here
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if case["kind"] in ("train", "step", "predict"):
        return _network(case, seed, dev)
    meshes, cond, start = _flow(case, seed)
    flow = _Euler(case, meshes, cond, dev)
    u = torch.as_tensor(start, device=dev)
    if case["kind"] == "residual":
        r, ws = flow.residual(u, 0.0)
        return {"resid": r, "ws": ws}
    if cond:
        u, norms = flow.march(u, case["steps"], "ssp42", 1.0, cfl=1.25)
    else:
        u, norms = flow.march(u, case["steps"], case["rk"], _dt(case))
    if case["kind"] == "batch":
        return {"norms": norms, "forces": flow.forces(u, cond), "cvar": u}
    return {"norms": norms, "cvar": u}
