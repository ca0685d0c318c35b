"""Workloads of the solver as programs run it, with their inputs, their results
and a plain 64-bit statement of what they compute.

Kinds of case:
  call   two le_step calls on a live task (the reference driver's loop body)
  job    state written from the host, N steps, state read back on the host
  steps  N steps of a live task (le_step_n), fields resident on the device
  soa    le_step_soa calls on a planar task (single steps, ring y-edge)
  sweep  le_step_x and le_step_y called one by one
  media  N steps with a per-node material plane, then the elastic energy
  batch  N steps of many independent grids of uneven sizes
  serve  simulation requests submitted to a server, drained and read back

Fields: "disk" is a disk of normal stress in a medium at rest, "waves" a
superposition of plane P and S waves that fills the grid.
"""
import math
import random

import numpy as np
import torch

import le2d_amd

DEV = "cuda" if torch.cuda.is_available() else "cpu"
H = (1.0, 1.0)
MAT = (2.0, 1.0, 1.0)  # c1, c2, rho of the reference's driver
DTYPE = {"f8": (np.float64, torch.float64), "f4": (np.float32, torch.float32)}
# arithmetic of one node and step: per sweep 6 for the invariants, 11 for each
# of 4 faces, 32 for the update
FLOPS = 2 * (6 + 44 + 32)


def listed():
    return [
        # the smallest use: a driver's le_step loop on a small grid (latency)
        {"name": "call_96x80_f8", "kind": "call", "dtype": "f8", "nx": 96, "ny": 80, "field": "disk"},
        # the reference's own case: 512^2, 100 steps, state in and out
        {"name": "job_512_f8", "kind": "job", "dtype": "f8", "nx": 512, "ny": 512, "steps": 100,
         "field": "disk"},
        # an ordinary ragged grid in single precision
        {"name": "steps_1031x517_f4", "kind": "steps", "dtype": "f4", "nx": 1031, "ny": 517,
         "steps": 20, "field": "waves"},
        # an ordinary grid in double precision
        {"name": "steps_2048_f8", "kind": "steps", "dtype": "f8", "nx": 2048, "ny": 2048,
         "steps": 20, "field": "waves"},
        # one eighth of the large grid, the slab of a sharded run
        {"name": "slab_8192x1024_f8", "kind": "steps", "dtype": "f8", "nx": 8192, "ny": 1024,
         "steps": 20, "field": "waves"},
        # the headline grid: a wave starting from a disk, double precision
        {"name": "disk_8192_f8", "kind": "steps", "dtype": "f8", "nx": 8192, "ny": 8192,
         "steps": 20, "field": "disk"},
        # the headline grid with the wave everywhere, single precision
        {"name": "waves_8192_f4", "kind": "steps", "dtype": "f4", "nx": 8192, "ny": 8192,
         "steps": 20, "field": "waves"},
        # planar storage: every call one step with the ring edge
        {"name": "soa_1500x1001_f8", "kind": "soa", "dtype": "f8", "nx": 1500, "ny": 1001,
         "steps": 4, "field": "waves"},
        # the single sweeps, as a program with its own splitting calls them
        {"name": "sweep_4096x2049_f4", "kind": "sweep", "dtype": "f4", "nx": 4096, "ny": 2049,
         "steps": 2, "field": "waves"},
        # layered medium with an inclusion, energy monitored
        {"name": "media_4100x3000_f8", "kind": "media", "dtype": "f8", "nx": 4100, "ny": 3000,
         "steps": 20, "field": "waves"},
        # a parameter study: 48 grids of uneven sizes in one launch
        {"name": "batch_48_f4", "kind": "batch", "dtype": "f4", "count": 48, "low": 128,
         "high": 1024, "steps": 20},
        # a service: requests of both precisions admitted together
        {"name": "serve_24", "kind": "serve", "count": 24, "low": 128, "high": 768, "steps": 96},
    ]


def _size(rng, low, high):
    """Log-uniform over [low, high]: multiples of 32, odd and arbitrary sizes alike."""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    how = rng.randrange(3)
    n = (n + 16) // 32 * 32 if how == 0 else n | 1 if how == 1 else n
    return min(max(n, low), high)


def draw(rng):
    kind = rng.choice(["call", "job", "steps", "steps", "steps", "soa", "sweep", "media", "batch",
                       "serve"])
    dtype = rng.choice(["f8", "f4"])
    if kind == "batch":
        low = rng.choice([48, 96, 128])
        return {"kind": kind, "dtype": dtype, "count": rng.randint(6, 48), "low": low,
                "high": _size(rng, 2 * low, 1024), "steps": rng.randint(4, 40)}
    if kind == "serve":
        return {"kind": kind, "count": rng.randint(6, 32), "low": rng.choice([64, 128]),
                "high": _size(rng, 256, 768), "steps": rng.randint(16, 128)}
    low, high, steps = {"call": (64, 512, 2), "job": (96, 1500, rng.randint(9, 120)),
                        "steps": (64, 4096, rng.randint(2, 40)), "soa": (96, 3000, rng.randint(1, 6)),
                        "sweep": (96, 4096, rng.randint(1, 4)),
                        "media": (200, 3000, rng.randint(2, 24))}[kind]
    case = {"kind": kind, "dtype": dtype, "nx": _size(rng, low, high), "ny": _size(rng, low, high),
            "field": "waves" if kind == "media" else rng.choice(["disk", "waves"])}
    if kind != "call":
        case["steps"] = steps
    return case


def work(case):
    elem = 8 if case.get("dtype", "f8") == "f8" else 4
    if case["kind"] == "serve":
        reqs = _requests(case, 0)  # sizes and steps are the same for every seed
        return {"bytes": float(sum(10 * r["nx"] * r["ny"] * np.dtype(r["dtype"]).itemsize for r in reqs)),
                "flops": float(sum(r["nx"] * r["ny"] * r["steps"] * FLOPS for r in reqs))}
    if case["kind"] == "batch":
        nodes = sum(i["nx"] * i["ny"] for i in _instances(case, 0))
    else:
        nodes = case["nx"] * case["ny"]
    steps = case.get("steps", 2)
    moved = 10 * elem * nodes + (nodes if case["kind"] == "media" else 0)
    return {"bytes": float(moved), "flops": float(nodes * steps * FLOPS)}


# ---------------------------------------------------------------------------
# Inputs.

def _waves(nx, ny, mat, seed, count=6):
    """Five fields (5, ny, nx), float64: `count` plane P and S waves of random
    directions, phases and wavelengths of 8 to 64 nodes."""
    rng = random.Random(seed)
    c1, c2, rho = mat
    mu = rho * c2 * c2
    la = rho * c1 * c1 - 2 * mu
    x = torch.arange(nx, device=DEV, dtype=torch.float64)[None, :]
    y = torch.arange(ny, device=DEV, dtype=torch.float64)[:, None]
    out = torch.zeros(5, ny, nx, device=DEV, dtype=torch.float64)
    for k in range(count):
        a = rng.uniform(0, 2 * math.pi)
        n = (math.cos(a), math.sin(a))
        kap = 2 * math.pi / math.exp(rng.uniform(math.log(8), math.log(64)))
        f = (kap * n[0] * x + (kap * n[1] * y + rng.uniform(0, 2 * math.pi))).sin_().mul_(
            rng.uniform(0.2, 1.0))
        if k % 2 == 0:  # P
            g = [n[0], n[1], -(la + 2 * mu * n[0] * n[0]) / c1, -2 * mu * n[0] * n[1] / c1,
                 -(la + 2 * mu * n[1] * n[1]) / c1]
        else:  # S
            t = (-n[1], n[0])
            g = [t[0], t[1], -2 * mu * n[0] * t[0] / c2, -mu * (n[0] * t[1] + n[1] * t[0]) / c2,
                 -2 * mu * n[1] * t[1] / c2]
        for q in range(5):
            out[q].add_(f, alpha=g[q])
    return out


def _disk_of(nx, ny, seed):
    """Centre (on half nodes, so that a node's distance is exact) and radius."""
    rng = random.Random(seed)
    r = max(2.5, min(nx, ny) / 8.0 if min(nx, ny) < 512 else 64.0)
    return ((math.floor(rng.uniform(0.3, 0.7) * nx) + 0.5, math.floor(rng.uniform(0.3, 0.7) * ny) + 0.5),
            math.floor(r) + 0.25)


def _disk(nx, ny, c, r, s=1.0):
    x = torch.arange(nx, device=DEV, dtype=torch.float64)[None, :] - c[0]
    y = torch.arange(ny, device=DEV, dtype=torch.float64)[:, None] - c[1]
    out = torch.zeros(5, ny, nx, device=DEV, dtype=torch.float64)
    inside = (x * x + y * y).sqrt() < r
    out[2][inside] = s
    out[4][inside] = s
    return out


def _problem(case, seed):
    """(dt, material, initial fields (5, ny, nx) in the case's type)."""
    nx, ny, mat = case["nx"], case["ny"], MAT
    if case["field"] == "disk":
        u = _disk(nx, ny, *_disk_of(nx, ny, seed))
    else:
        u = _waves(nx, ny, mat, seed)
    return 0.25, mat, u.to(DTYPE[case["dtype"]][1])


def _planes(case, seed):
    """Material table and ids: two layers and an inclusion."""
    rng = random.Random(seed)
    nx, ny = case["nx"], case["ny"]
    tab = [(2.0, 1.0, 1.0), (2.6, 1.4, 2.2), (1.7, 0.8, 0.7)]
    x = torch.arange(nx, device=DEV)[None, :]
    y = torch.arange(ny, device=DEV)[:, None]
    ids = torch.zeros(ny, nx, device=DEV, dtype=torch.uint8)
    ids[int(ny * rng.uniform(0.35, 0.65)):] = 1
    cx, cy, r = nx * rng.uniform(0.3, 0.7), ny * rng.uniform(0.2, 0.8), min(nx, ny) / 6.0
    ids[((x - cx) ** 2 + (y - cy) ** 2) < r * r] = 2
    return tab, ids


def _instances(case, seed):
    rng = random.Random(seed)
    sizes = random.Random(1000 * case["count"] + case["high"])  # the same sizes for every seed
    got = []
    for _ in range(case["count"]):
        nx, ny = (int(math.exp(sizes.uniform(math.log(case["low"]), math.log(case["high"] + 1))))
                  for _ in range(2))
        c1 = sizes.uniform(1.5, 4.0)
        mat = (c1, c1 * sizes.uniform(0.4, 0.7), sizes.uniform(0.5, 3.0))
        got.append({"nx": nx, "ny": ny, "mat": mat, "dt": sizes.uniform(0.3, 0.8) / c1,
                    "seed": rng.randrange(1 << 30)})
    return got


def _requests(case, seed):
    rng = random.Random(seed)
    sizes = random.Random(1000 * case["count"] + case["high"])
    got = []
    for _ in range(case["count"]):
        nx, ny = (int(math.exp(sizes.uniform(math.log(case["low"]), math.log(case["high"] + 1))))
                  for _ in range(2))
        dtype = "f4" if sizes.random() < 0.6 else "f8"
        steps = sizes.randint(case["steps"] // 2, case["steps"])
        c, r = _disk_of(nx, ny, rng.randrange(1 << 30))
        got.append({"nx": nx, "ny": ny, "steps": steps, "dtype": dtype, "c": c, "r": r})
    return got


# ---------------------------------------------------------------------------
# A program's side: tasks, batches, servers and views of their memory.

class _Memory:
    """Memory of a task or batch as an array; keeps its owner alive."""

    def __init__(self, owner, address, shape, strides, dtype, device):
        self.owner = owner
        desc = {"data": (address, False), "shape": shape, "strides": strides,
                "typestr": np.dtype(dtype).str, "version": 3}
        if device:
            desc["version"] = 2
            self.__cuda_array_interface__ = desc
        else:
            self.__array_interface__ = desc


def _device_state(state, owner, view):
    """The current device state as a tensor (5, ny, nx); one tensor per buffer is kept."""
    kept = state.setdefault("views", {})
    if view.base not in kept:
        e = view.elem
        kept[view.base] = torch.as_tensor(
            _Memory(owner, view.base, (5, view.ny, view.nx), (view.plane * e, view.pitch * e, e),
                    np.float64 if e == 8 else np.float32, True), device="cuda")
    return kept[view.base]


def _host_state(task):
    g = task.grid()
    return np.asarray(_Memory(task, g.ctypes.data, g.shape, g.strides, g.dtype, False))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        reqs = _requests(case, seed)
        budget = sum(2 * 5 * 8 * (r["nx"] + 64) * (r["ny"] + 2) for r in reqs) + (64 << 20)
        return {"kind": kind, "server": le2d_amd.Server(budget, max_live=case["count"]), "reqs": reqs}
    if kind == "batch":
        b = le2d_amd.Batch(DTYPE[case["dtype"]][0])
        insts = _instances(case, seed)
        for i in insts:
            b.add(i["nx"], i["ny"], i["dt"], H, i["mat"])
        b.commit()
        for k, i in enumerate(insts):
            u = _waves(i["nx"], i["ny"], i["mat"], i["seed"]).to(DTYPE[case["dtype"]][1])
            b.load(k, u.permute(1, 2, 0).contiguous().cpu().numpy())
        return {"kind": kind, "batch": b, "steps": case["steps"], "count": len(insts)}
    dt, mat, u = _problem(case, seed)
    soa = kind == "soa"
    task = le2d_amd.Task(case["nx"], case["ny"], dt, H, mat, le2d_amd.ST_SOA if soa else le2d_amd.ST_AOS,
                         DTYPE[case["dtype"]][0])
    state = {"kind": kind, "task": task, "steps": case.get("steps", 2)}
    if kind == "job":
        state["input"] = u.permute(1, 2, 0).contiguous().cpu().numpy()
        return state
    # straight into the host mirror, then to the device
    torch.from_numpy(task.view()).copy_(u if soa else u.permute(1, 2, 0))
    task.lib.le_mark_host_dirty(task.ref)
    if kind == "media":
        tab, ids = _planes(case, seed)
        task.set_materials(tab, ids.cpu().numpy())
    _device_state(state, task, task.device_view())
    return state


def run(state):
    kind = state["kind"]
    if kind == "serve":
        srv = state["server"]
        ids = [srv.submit(r["nx"], r["ny"], r["steps"], DTYPE[r["dtype"]][0], 0.25, H, MAT,
                          (r["c"][0], r["c"][1], r["r"], 1.0), keep=True) for r in state["reqs"]]
        srv.drain()
        return [srv.result(i) for i in ids]
    if kind == "batch":
        b = state["batch"]
        b.step(state["steps"])
        b.wait()
        return [_device_state(state, b, b.device_view(k)) for k in range(state["count"])]
    task = state["task"]
    if kind == "job":
        task.load(state["input"])
        task.step_n(state["steps"])
        return _host_state(task)
    if kind == "call":
        task.step()
        task.step()
    elif kind == "soa":
        for _ in range(state["steps"]):
            task.step()
    elif kind == "sweep":
        for _ in range(state["steps"]):
            task.step_x()
            task.step_y()
    else:
        task.step_n(state["steps"])
    if kind == "media":
        return {"energy": task.energy(), "fields": _device_state(state, task, task.device_view())}
    return _device_state(state, task, task.device_view())


# ---------------------------------------------------------------------------
# The same in plain 64-bit torch: the split-step scheme node by node.

def _consts(c1, c2, rho, dt, h):
    mu = rho * c2 * c2
    la = rho * c1 * c1 - 2 * mu
    return {"k1": dt * c1 / h, "k2": dt * c2 / h, "i1": 1 / (c1 * rho), "i2": 1 / (c2 * rho),
            "r1": c1 * rho, "r2": c2 * rho, "r3": rho * c1 * la / (la + 2 * mu)}


def _flux(um, u0, u1, k):
    du = u1 - u0
    r = ((u0 - um) + 1e-6) / (du + 1e-6)
    # max(0, max(min(1, 2r), min(2, r))) with the scheme's treatment of NaN
    a = torch.where(2 * r < 1, 2 * r, 1.0)
    b = torch.where(r < 2, r, 2.0)
    phi = torch.where(a > b, a, b).clamp_(min=0)
    return u0 + phi.mul_(0.5).mul_(1 - k).mul_(du)


def _sweep(u, axis, c, rows):
    """One sweep along `axis` (1: y, 2: x) of u (5, ny, nx); `rows`: the index of
    each window position -2 .. n+1; constants are numbers or (ny, nx) tensors."""
    vn, vt, sn, so = ((0, 1, 2, 4) if axis == 2 else (1, 0, 4, 2))
    n = u.shape[axis]
    pad = u.index_select(axis, rows)
    d = axis - 1

    def at(x, s):  # the value at distance s along the sweep
        return x.narrow(d, 2 + s, n)

    inc = []
    for f, g, ir, k in ((vn, sn, c["i1"], c["k1"]), (vt, 3, c["i2"], c["k2"])):
        for sign in (-1, 1):  # speeds +c, -c
            if isinstance(ir, float):
                w = pad[f] + pad[g] * (sign * ir)
                if sign < 0:
                    fl = _flux(w.narrow(d, 0, n + 1), w.narrow(d, 1, n + 1), w.narrow(d, 2, n + 1), k)
                else:
                    fl = _flux(w.narrow(d, 3, n + 1), w.narrow(d, 2, n + 1), w.narrow(d, 1, n + 1), k)
                left, right, w0 = fl.narrow(d, 0, n), fl.narrow(d, 1, n), at(w, 0)
            else:
                v = [at(pad[f], s) + at(pad[g], s) * (sign * ir) for s in range(-2, 3)]
                if sign < 0:
                    left, right = _flux(v[0], v[1], v[2], k), _flux(v[1], v[2], v[3], k)
                else:
                    left, right = _flux(v[3], v[2], v[1], k), _flux(v[4], v[3], v[2], k)
                w0 = v[2]
            out, into = (right, left) if sign < 0 else (left, right)
            inc.append(((w0 - k * (out - into)) - w0).mul_(0.5))
    e1, e2, e3, e4 = inc
    new = torch.empty_like(u)
    new[vn] = u[vn] + (e1 + e2)
    new[vt] = u[vt] + (e3 + e4)
    new[sn] = u[sn] + (e2 - e1) * c["r1"]
    new[so] = u[so] + (e2 - e1) * c["r3"]
    new[3] = u[3] + (e4 - e3) * c["r2"]
    return new


def _advance(u, steps, dt, mat, ring=False, ids=None, tab=None):
    ny, nx = u.shape[1:]
    if ids is None:
        cx, cy = (_consts(*mat, dt, h) for h in H)
    else:
        t = torch.tensor(tab, device=u.device, dtype=torch.float64)[ids.long()]
        cx, cy = (_consts(t[..., 0], t[..., 1], t[..., 2], dt, h) for h in H)
    xs = torch.arange(-2, nx + 2, device=u.device).clamp_(0, nx - 1)
    p = torch.arange(-2, ny + 2, device=u.device)
    ys = torch.where(p >= ny, (p - 5).clamp(min=0), p.clamp(min=0)) if ring else p.clamp(0, ny - 1)
    for _ in range(steps):
        u = _sweep(u, 2, cx, xs)
        u = _sweep(u, 1, cy, ys)
    return u


def _energy(u, tab, ids):
    t = torch.tensor(tab, device=u.device, dtype=torch.float64)[ids.long()]
    c1, c2, rho = t[..., 0], t[..., 1], t[..., 2]
    mu = rho * c2 * c2
    la = rho * c1 * c1 - 2 * mu
    e = 0.5 * rho * (u[0] ** 2 + u[1] ** 2) + (u[2] + u[4]) ** 2 / (8 * (la + mu))
    e += ((u[2] - u[4]) ** 2 / 2 + 2 * u[3] ** 2) / (4 * mu)
    return float(e.sum()) * H[0] * H[1]


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return [_advance(_disk(r["nx"], r["ny"], r["c"], r["r"]), r["steps"], 0.25, MAT)
                .permute(1, 2, 0).contiguous().cpu().numpy() for r in _requests(case, seed)]
    if kind == "batch":
        kind_t = DTYPE[case["dtype"]][1]
        return [_advance(_waves(i["nx"], i["ny"], i["mat"], i["seed"]).to(kind_t).double(),
                         case["steps"], i["dt"], i["mat"]) for i in _instances(case, seed)]
    dt, mat, u = _problem(case, seed)
    u = u.double()
    if kind == "media":
        tab, ids = _planes(case, seed)
        u = _advance(u, case["steps"], dt, mat, ids=ids, tab=tab)
        return {"energy": _energy(u, tab, ids), "fields": u}
    u = _advance(u, case.get("steps", 2), dt, mat, ring=kind == "soa")
    return u.permute(1, 2, 0).contiguous().cpu().numpy() if kind == "job" else u
